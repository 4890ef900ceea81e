// Prints, for each line "epi cin cout skip N H W" on stdin (epi: fold, pool,
// head or P; skip: the channels of a concat's first segment, 0 without), 1 if
// the binary conv would run on the matrix cores by default, 0 if on the
// popcount kernel (mfma_conv_pays, 256 compute units),
// and 1 if the matrix-core kernel takes the layer at all (mfma_conv_fits).
#include <cstdio>
#include <cstring>

#include "bnn_kernels.h"

using namespace bnn;

int main() {
  char name[8];
  int cin, cout, cs, N, H, W;
  while (scanf("%7s %d %d %d %d %d %d", name, &cin, &cout, &cs, &N, &H, &W) == 7) {
    const int epi = !strcmp(name, "fold") ? EPI_FOLD : !strcmp(name, "pool") ? EPI_POOL : !strcmp(name, "head") ? EPI_HEAD : EPI_P;
    const int cw0 = ((cs ? cs : cin) + 31) / 32, cw1 = cs ? (cin - cs + 31) / 32 : 0;
    const bool pair = (cs ? cs : cin) <= 16;
    static const uint32_t w[1] = {};
    static const float r[1] = {};
    MfmaConv mc{};
    mc.w = w;
    mc.r1 = mc.r2 = r;
    mc.coutp = mfma_coutp(cout);
    mc.mt = mfma_mt(cout);
    mc.slots = mfma_nslots(cw0, cw1, pair);
    mc.steps = (mc.slots + 3) / 4;
    printf("%d %d\n", mfma_conv_pays(mc, cin, cout, cw0, cw1, pair, epi, N, H, W, 256) ? 1 : 0,
           mfma_conv_fits(mc, cw0 + cw1, N, H, W, epi) ? 1 : 0);
  }
  return 0;
}
