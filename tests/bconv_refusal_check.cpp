// launch_bconv_mfma takes v1 concats only, whose uncovered positions read 0
// bits: one with a pad pixel (a v3 tensor's, just past its last one) is refused
// before anything is launched.  Prints the status.
#include <cstdio>

#include "bnn_kernels.h"

using namespace bnn;

int main() {
  static uint32_t words[256];
  static float rule[64];
  MfmaConv mc{};
  mc.w = mc.slot = mc.inv1 = words;
  mc.s = mc.c1 = mc.r1 = rule;
  mc.coutp = mfma_coutp(32);
  mc.mt = mfma_mt(32);
  mc.slots = mfma_nslots(1, 1, 0);
  mc.steps = (mc.slots + 3) / 4;
  BconvArgs a{};
  a.in0 = a.in1 = words;
  a.out = words;
  a.cw0 = a.cw1 = a.cwo = 1;
  a.N = 1;
  a.H = a.W = 8;
  a.h1 = a.w1 = 3;
  a.oh = a.ow = 1;
  a.uh = a.uw = 6;
  a.cin = 64;
  a.cout = 32;
  a.padoff = 3 * 3 * 4;
  printf("%d\n", (int)launch_bconv_mfma(a, mc, EPI_FOLD, nullptr));
  return 0;
}
