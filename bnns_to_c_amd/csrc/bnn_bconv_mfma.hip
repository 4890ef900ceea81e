// bnn_bconv_mfma.hip - the binary 3x3 conv on the matrix cores of gfx950, as
// an FP4 product with FP32 sums, with the rule (fold), the fused 2x2
// max-pool, the 1x1 head or the integer P as its epilogue.  Same P, bits,
// logits and dumps as the popcount kernel (csrc/bnn_conv.c:23-36,
// csrc/bnn_maxpool.c:28-48, csrc/bnn_head.c:21-34).
//
// Built with the matrix instructions' accumulators in ordinary VGPRs
// (-mllvm -amdgpu-mfma-vgpr-form): the epilogue reads all of them.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "bnn_device.h"
#include "bnn_kernels.h"
#include "bnn_mfma_f4.h"

namespace bnn {
namespace {

// The product.  v_mfma_f32_16x16x128_f8f6f4 with both operands in FP4 (E2M1:
// 0, 0.5, 1, 2, 4 and their negatives are exact) runs 128 terms at twice the
// rate of the int8 instruction's 64, and an operand element takes half a
// byte.  An activation bit needs no conversion beyond a mask: bit 4k + j of
// a packed word is nibble k of `word & (0x11111111 << j)`, which FP4 reads as
// 0 or 0.5, 1, 2 for j = 0, 1, 2 (j = 3 is shifted down to 0.5: bit 3 is the
// sign).  The weights' magnitudes make up for it (4, 2, 1, 4), so every
// product is 2*w*alpha, alpha in {0, 1}.  The accumulator starts at
// -S - c (S: the weight sum over the taps inside the image, one of 16 border
// classes, c: the centre of the channel's rule) and ends at P - c, since
// P = 2*sum(w*alpha) - S.  Every term and sum is an integer or a half below
// 2^24, so the FP32 sums are exact in any order (a layer whose tile and slot
// table fit a CU's LDS has fewer than 70,000 input channels, 18 to a sum).
//
// Work split.  A wave makes MT*16 channels x G*16 pixels, a block of four
// waves the same channels of 64*G pixels: a tile of TR rows x TW columns of a
// patch, or of TI whole patches.  The tile's words with a one-pixel zero halo
// sit in LDS, staged once for all its channels' taps, [plane of 4 words]
// [pixel][word], so one 4-byte read per lane is a whole B operand: lane
// 16q + j takes pixel j of the group and K slot 4*step + q.  A K slot is one
// (word, tap), or, for a first segment of at most 16 channels, one (row, pair
// of taps): that word holds the pixel's 16 bits and its right neighbour's.
// The weights come as ready FP4 operands ([channel group][step][m][lane][16
// bytes]); they stay in LDS for the block's life when they fit (kResident),
// else they pass through it in phases of kPhase steps, two buffers, the next
// phase's loads in flight while this one is used.
//
// Blocks are persistent and XCD-aware: block b runs on XCD b % 8, whose
// blocks walk the tiles x, x + 8, ... with a tile's channel groups side by
// side, so the words of a pixel merge in one L2.
typedef int i32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kPhase = 4;                   // K steps a streamed phase
constexpr size_t kResident = 40u * 1024;    // weight bytes of a channel group kept in LDS
constexpr uint32_t kFar = 0x80000000u;

// n / d for 0 <= n < 2^31 as mulhi(2n, mul) >> sh, for any d >= 1 without a
// branch: sh = ceil(log2 d), mul = ceil(2^(31 + sh) / d)
struct KDiv {
  uint32_t d, mul, sh;
};
inline KDiv make_kdiv(uint32_t d) {
  KDiv f{d, 0u, d > 1 ? 32u - (uint32_t)__builtin_clz(d - 1) : 0u};
  f.mul = (uint32_t)(((1ull << (31 + f.sh)) + d - 1) / d);
  return f;
}

// The tile geometry of one launch, and where its LDS regions lie.
struct MfmaTile {
  int TW, TR, TI;         // columns, rows, patches of a tile (TI > 1: whole patches)
  KDiv dpat, dcol;        // pixels (pool: 2x2 blocks) per patch of a tile, per row
  KDiv dsp, dsr;          // staged pixels per patch, per row
  KDiv dhp, dtc;          // tiles per patch, per row of tiles
  int npat;               // dpat.d * TI: pixels (blocks) of a tile
  int sub;                // tiles staged together: the next one's is subn patches or suby rows on,
  int subn, suby;         // subl bytes of a staged plane on
  uint32_t subl;
  int ns;                 // staged pixels
  int ps, planes;         // words per staged pixel and plane, planes
  uint32_t plane_b;       // bytes of a plane
  uint32_t off_tab, off_s, off_a;  // LDS bytes: slot offsets, -S - c, weights
  uint32_t ntiles;
  int ncg;                // channel groups
  int steps, slots;
  int resident;
};

// The kernel's arguments, read where they are used straight from the kernarg
// segment: held across the tile loop they took twice the scalar registers
// there are.  fresh() makes a new pointer the compiler cannot trace, so loads
// through it stay in their section.
struct MfmaParams {
  BconvArgs a;
  MfmaConv mc;
  MfmaTile T;
  uint32_t bytes0, bytes1;
};
typedef const __attribute__((address_space(4))) MfmaParams* MfmaKarg;
typedef const __attribute__((address_space(4))) KDiv* DivKarg;
__device__ __forceinline__ MfmaKarg fresh(MfmaKarg k) {
  asm volatile("" : "+s"(k));
  return k;
}
__device__ __forceinline__ uint32_t kdiv(uint32_t n, DivKarg f) { return __umulhi(2u * n, f->mul) >> f->sh; }

// waves a SIMD (blocks a CU) the registers are held to
constexpr int mfma_waves(int mt, int epi) { return (mt < 4 ? 4 : 3) - (mt > 1 && epi == EPI_P ? 1 : 0); }

template <int MT, int G, int EPI, bool RES>
__global__ __launch_bounds__(256, mfma_waves(MT, EPI)) void k_bconv_mfma(const MfmaParams) {
  const MfmaKarg kp = (MfmaKarg)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, j = lane & 15, wave = tid >> 6;
  const int H = kp->a.H, W = kp->a.W;
  const uint32_t ntiles = kp->T.ntiles, ncg = (uint32_t)kp->T.ncg;
  // block -> XCD, channel group, first tile; tiles advance by nslot * 8
  const uint32_t xcd = blockIdx.x & 7u, bi = blockIdx.x >> 3, tstep = (gridDim.x >> 3) / ncg * 8u;
  const int cg = (int)(bi % ncg);
  uint32_t tile = (bi / ncg) * 8u + xcd;
  if (tile >= ntiles) return;
  const int co0 = cg * MT * 16;

  // this lane's pixel of each group, within a tile (the same for every
  // tile): patch, row, column.  Pixels are numbered along the tile's rows,
  // group g = 16 consecutive ones; EPI_P takes 4j + g instead, so a lane's
  // four pixels are neighbours and its P leaves in 16-byte stores; a pooled
  // tile numbers its 2x2 blocks, groups 2p and 2p + 1 hold the upper and
  // lower rows of eight of them.
  uint32_t lb[G];
  int pc[G];  // patch << 20 | row << 10 | column, -1 past the tile
#pragma unroll
  for (int g = 0; g < G; ++g) {
    int ip, r, c;
    bool in;
    if (EPI == EPI_POOL) {
      const int blk = wave * (G * 4) + 8 * (g >> 1) + (j >> 1);
      in = blk < kp->T.npat;
      const uint32_t b = in ? (uint32_t)blk : 0u;
      ip = (int)kdiv(b, &kp->T.dpat);
      const uint32_t rem = b - (uint32_t)ip * kp->T.dpat.d;
      const uint32_t br = kdiv(rem, &kp->T.dcol);
      r = 2 * (int)br + (g & 1);
      c = 2 * (int)(rem - br * kp->T.dcol.d) + (j & 1);
      in = in && r < kp->T.TR && c < kp->T.TW;
    } else {
      const int l = wave * (G * 16) + (EPI == EPI_P ? G * j + g : 16 * g + j);
      in = l < kp->T.npat;
      const uint32_t b = in ? (uint32_t)l : 0u;
      ip = (int)kdiv(b, &kp->T.dpat);
      const uint32_t rem = b - (uint32_t)ip * kp->T.dpat.d;
      r = (int)kdiv(rem, &kp->T.dcol);
      c = (int)(rem - (uint32_t)r * kp->T.dcol.d);
    }
    if (!in) { ip = 0; r = 0; c = 0; }
    lb[g] = ((uint32_t)ip * kp->T.dsp.d + (uint32_t)r * kp->T.dsr.d + (uint32_t)c) * (uint32_t)(kp->T.ps * 4);
    pc[g] = in ? (ip << 20 | r << 10 | c) : -1;
  }
  // the pixel whose word this lane stores (the epilogue's lane rows)
  int po = pc[0];
#pragma unroll
  for (int g = 1; g < G; ++g)
    if ((G == 4 ? q : q >> 1) == g) po = pc[g];

  // ---- staging: piece e = words 4p .. of staged pixel i (e = p * ns + i)
  auto coords = [&](uint32_t t, int* n0, int* y0, int* x0) {
    const MfmaKarg k = fresh(kp);
    const uint32_t tp = kdiv(t, &k->T.dhp), tr = t - tp * k->T.dhp.d;  // patch (group), tile within the patch
    const uint32_t ty = kdiv(tr, &k->T.dtc);
    *n0 = (int)tp * (k->T.TI > 1 ? k->T.TI * k->T.sub : 1);
    *y0 = (int)ty * (k->T.TR * (k->T.TI > 1 ? 1 : k->T.sub));
    *x0 = (int)(tr - ty * k->T.dtc.d) * k->T.TW;
  };
  // the byte offsets of staged pixel i in the two inputs, and of its right
  // neighbour in the first (kFar: outside the image, reads 0)
  auto stage_offs = [&](MfmaKarg k, uint32_t i, int n0, int y0, int x0, uint32_t& off0, uint32_t& off1, uint32_t& offn) {
    // (recomputed for every tile: kept, it took a dozen registers a pixel)
    asm volatile("" : "+v"(i));
    const uint32_t ip = kdiv(i, &k->T.dsp), ir = i - ip * k->T.dsp.d;
    const uint32_t rr = kdiv(ir, &k->T.dsr), cc = ir - rr * k->T.dsr.d;
    const int n = n0 + (int)ip, y = y0 + (int)rr - 1, x = x0 + (int)cc - 1;
    const bool okr = n < k->a.N && (unsigned)y < (unsigned)H, ok = okr && (unsigned)x < (unsigned)W;
    const uint32_t pix = ((uint32_t)n * (uint32_t)H + (uint32_t)y) * (uint32_t)W + (uint32_t)x;
    off0 = ok ? pix * ((uint32_t)k->a.cw0 * 4u) : kFar;
    // (in the column left of the image too: column 0's bits)
    offn = okr && (unsigned)(x + 1) < (unsigned)W ? (pix + 1u) * 4u : kFar;
    off1 = kFar;
    if (k->a.cw1) {
      // nearest 2x upsample placed at (oh, ow); what it does not cover reads 0
      const int uy = y - k->a.oh, ux = x - k->a.ow;
      off1 = (unsigned)uy < (unsigned)k->a.uh && (unsigned)ux < (unsigned)k->a.uw
                 ? (((uint32_t)n * (uint32_t)k->a.h1 + (uint32_t)(uy >> 1)) * (uint32_t)k->a.w1 +
                    (uint32_t)(ux >> 1)) * ((uint32_t)k->a.cw1 * 4u)
                 : kFar;
      off1 = ok ? off1 : kFar;
    }
  };
  const uint32_t ns = (uint32_t)kp->T.ns;
  // one plane (at most four words a pixel): pixel i's words
  auto load_px = [&](MfmaKarg k, uint32_t i, int n0, int y0, int x0) -> i32x4v {
    uint32_t off0, off1, offn;
    stage_offs(k, i, n0, y0, x0, off0, off1, offn);
    const int cw0 = k->a.cw0, cw1 = k->a.cw1;
    const __amdgpu_buffer_rsrc_t r0 = make_rsrc(k->a.in0, k->bytes0);
    i32x4v v = {0, 0, 0, 0};
    if (cw0 == 4) {
      v = __builtin_bit_cast(i32x4v, __builtin_amdgcn_raw_buffer_load_b128(r0, (int)off0, 0, 0));
    } else {
      v[0] = (int)ld_u32(r0, off0, 0);
      if (cw0 > 1) v[1] = (int)ld_u32(r0, off0 + 4u, 0);
      if (cw0 > 2) v[2] = (int)ld_u32(r0, off0 + 8u, 0);
      if (k->a.pair) v[0] |= (int)(ld_u32(r0, offn, 0) << 16);
      if (cw1) {
        const __amdgpu_buffer_rsrc_t r1 = make_rsrc(k->a.in1, k->bytes1);
        const int u0 = (int)ld_u32(r1, off1, 0), u1 = cw1 > 1 ? (int)ld_u32(r1, off1 + 4u, 0) : 0,
                  u2 = cw1 > 2 ? (int)ld_u32(r1, off1 + 8u, 0) : 0;
        if (cw0 == 1) { v[1] = u0; v[2] = u1; v[3] = u2; }
        else if (cw0 == 2) { v[2] = u0; v[3] = u1; }
        else v[3] = u0;
      }
    }
    return v;
  };
  auto store_px = [&](MfmaKarg k, uint32_t i, const i32x4v& v) {
    asm volatile("" : "+v"(i));
    const int ps = k->T.ps;
    if (ps == 4) {
      *reinterpret_cast<i32x4v*>(smem + i * 16u) = v;
    } else {
      int* d = reinterpret_cast<int*>(smem) + i * (uint32_t)ps;
      d[0] = v[0];
      if (ps > 1) d[1] = v[1];
      if (ps > 2) d[2] = v[2];
    }
  };
  // several planes: pixel i, four planes' loads in flight
  auto copy_px = [&](MfmaKarg k, uint32_t i, int n0, int y0, int x0) {
    uint32_t off0, off1, offn;
    stage_offs(k, i, n0, y0, x0, off0, off1, offn);
    const int cw0 = k->a.cw0, cw = cw0 + k->a.cw1, planes = k->T.planes;
    const uint32_t pb = k->T.plane_b;
    const __amdgpu_buffer_rsrc_t r0 = make_rsrc(k->a.in0, k->bytes0);
    const __amdgpu_buffer_rsrc_t r1 = make_rsrc(k->a.in1, k->bytes1);  // (read for words past cw0 only)
#pragma unroll 1
    for (int p0 = 0; p0 < planes; p0 += 4) {
      i32x4v v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int w0 = 4 * (p0 + j);
        v[j] = i32x4v{0, 0, 0, 0};
        if (w0 + 4 <= cw0) {
          v[j] = __builtin_bit_cast(
              i32x4v, __builtin_amdgcn_raw_buffer_load_b128(r0, (int)(off0 + (uint32_t)w0 * 4u), 0, 0));
        } else if (w0 >= cw0 && w0 + 4 <= cw) {
          v[j] = __builtin_bit_cast(
              i32x4v, __builtin_amdgcn_raw_buffer_load_b128(r1, (int)(off1 + (uint32_t)(w0 - cw0) * 4u), 0, 0));
        } else if (w0 < cw) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (w0 + t < cw0) v[j][t] = (int)ld_u32(r0, off0 + (uint32_t)(w0 + t) * 4u, 0);
            else if (w0 + t < cw) v[j][t] = (int)ld_u32(r1, off1 + (uint32_t)(w0 + t - cw0) * 4u, 0);
          }
        }
      }
      if (k->a.pair && p0 == 0) v[0][0] |= (int)(ld_u32(r0, offn, 0) << 16);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (p0 + j < planes) *reinterpret_cast<i32x4v*>(smem + (uint32_t)(p0 + j) * pb + i * 16u) = v[j];
    }
  };
  const bool one = RES && kp->T.planes == 1;  // (a streamed group has more than one)
  // one plane: a thread's first kAhead pixels are loaded while the tile
  // before is multiplied
  constexpr int kAhead = 2;
  i32x4v st[kAhead];
  int n0, y0, x0;
  coords(tile, &n0, &y0, &x0);
  if (one) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      st[k] = i32x4v{0, 0, 0, 0};
      if (tid + 256u * k < ns) st[k] = load_px(kp, (uint32_t)tid + 256u * k, n0, y0, x0);
    }
  }

  // weights: step st of this channel group is MT KB at wg + st * MT KB
  const int steps = kp->T.steps;
  const i32x4v* wg = reinterpret_cast<const i32x4v*>(kp->mc.w) + (size_t)cg * steps * MT * 64;
  i32x4v* abuf = reinterpret_cast<i32x4v*>(smem + kp->T.off_a);
  const int nph = RES ? 1 : (steps + kPhase - 1) / kPhase, na = steps * MT * 64;
  constexpr int kAL = kPhase * MT / 4;  // 16-byte pieces a thread moves per phase
  i32x4v ap[kAL];
  auto a_fetch = [&](int ph) {
#pragma unroll
    for (int k = 0; k < kAL; ++k) ap[k] = wg[min(ph * (kPhase * MT * 64) + k * 256 + tid, na - 1)];
  };
  auto a_put = [&](int buf) {
#pragma unroll
    for (int k = 0; k < kAL; ++k) abuf[buf * (kPhase * MT * 64) + k * 256 + tid] = ap[k];
  };
  // slot offsets and border sums, then the weights, each batch's loads
  // issued together
  uint32_t* tab = reinterpret_cast<uint32_t*>(smem + kp->T.off_tab);
  float* stab = reinterpret_cast<float*>(smem + kp->T.off_s);
  {
    // [16 border classes][channel] -S - c1, then per channel r1, c1 - c2, r2
    constexpr int kC4 = MT * 4, kS4 = 16 * kC4, kT4 = kS4 + 3 * kC4;  // float4s
    constexpr int kTB = (kT4 + 255) / 256;
    f32x4v sv[kTB];
#pragma unroll
    for (int k = 0; k < kTB; ++k) {
      const int i = tid + 256 * k, row = i / kC4;
      const float* src = row < 16 ? kp->mc.s + (size_t)row * kp->mc.coutp : row == 16 ? kp->mc.r1 : row == 17 ? kp->mc.c12 : kp->mc.r2;
      sv[k] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
      if (i < kT4 && src) sv[k] = *reinterpret_cast<const f32x4v*>(src + co0 + i % kC4 * 4);
    }
    if constexpr (RES) {
      constexpr int kB = 5;
      for (int i = tid; i < na; i += 256 * kB) {
        i32x4v r[kB];
#pragma unroll
        for (int k = 0; k < kB; ++k) r[k] = wg[min(i + 256 * k, na - 1)];
#pragma unroll
        for (int k = 0; k < kB; ++k)
          if (i + 256 * k < na) abuf[i + 256 * k] = r[k];
      }
    } else {
      a_fetch(0);
      a_put(0);
      a_fetch(1);  // a streamed group has at least two phases
    }
    for (int s = tid; s < steps * 4; s += 256) {
      const uint32_t sl = s < kp->T.slots ? kp->mc.slot[s] : 0u;  // tap | word << 8 (past the last: any, the weights are 0)
      const uint32_t t = sl & 255u, wd = sl >> 8;
      tab[s] = (t / 3 * kp->T.dsr.d + t % 3) * (uint32_t)(kp->T.ps * 4) + (wd >> 2) * kp->T.plane_b + (wd & 3) * 4u;
    }
#pragma unroll
    for (int k = 0; k < kTB; ++k)
      if (tid + 256 * k < kT4) *reinterpret_cast<f32x4v*>(stab + (tid + 256 * k) * 4) = sv[k];
  }
  int abf = 0;

#pragma unroll 1
  for (;;) {
    const MfmaKarg ks = fresh(kp);
    if (one) {
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (tid + 256u * k < ns) store_px(ks, (uint32_t)tid + 256u * k, st[k]);
#pragma unroll 1
      for (uint32_t i = (uint32_t)tid + 256u * kAhead; i < ns; i += 512u) {
        const i32x4v v0 = load_px(ks, i, n0, y0, x0);
        i32x4v v1 = {0, 0, 0, 0};
        if (i + 256u < ns) v1 = load_px(ks, i + 256u, n0, y0, x0);
        store_px(ks, i, v0);
        if (i + 256u < ns) store_px(ks, i + 256u, v1);
      }
    } else {
#pragma unroll 1
      for (uint32_t i = (uint32_t)tid; i < ns; i += 256u) copy_px(ks, i, n0, y0, x0);
    }
    __syncthreads();
    const uint32_t next = tile + tstep;
    int n1, y1, x1;
    coords(next, &n1, &y1, &x1);
    if (one && next < ntiles) {
      const MfmaKarg kl = fresh(kp);
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (tid + 256u * k < ns) st[k] = load_px(kl, (uint32_t)tid + 256u * k, n1, y1, x1);
    }

    const int nsub = kp->T.sub;
    uint32_t sl = 0;  // LDS bytes of the sub-tile
#pragma unroll 1
    for (int sb = 0; sb < nsub; ++sb) {
    // ---- sums
    f32x4v acc[MT][G];
    {
      int cls[G];
#pragma unroll
      for (int g = 0; g < G; ++g) cls[g] = 0;
      if (x0 == 0 || x0 + kp->T.TW >= W) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int x = x0 + (pc[g] & 1023);
          cls[g] = (x == 0 ? MT * 16 : 0) + (x == W - 1 ? 2 * MT * 16 : 0);
        }
      }
      if (y0 == 0 || y0 + kp->T.TR >= H) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int y = y0 + ((pc[g] >> 10) & 1023);
          cls[g] += (y == 0 ? 4 * MT * 16 : 0) + (y == H - 1 ? 8 * MT * 16 : 0);
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][g] = *reinterpret_cast<const f32x4v*>(stab + cls[g] + m * 16 + q * 4);
    }
    {
      uint32_t w0[G], w1[G];
      i32x4v A0[MT], A1[MT];
      auto rd_w = [&](uint32_t off, uint32_t (&w)[G]) {
#pragma unroll
        for (int g = 0; g < G; ++g) w[g] = *reinterpret_cast<const uint32_t*>(smem + lb[g] + (sl + off));
      };
      auto mul = [&](const i32x4v (&A)[MT], const uint32_t (&w)[G]) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const i32x4v B = bits_f4(w[g]);
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][g] = mfma_f4(A[m], B, acc[m][g]);
        }
      };
      const uint32_t* tq = tab + q;
      const int last = steps - 1;
      rd_w(tq[0], w0);
      uint32_t on = tq[4 * min(1, last)];
      int s = 0;
#pragma unroll 1
      for (int ph = 0; ph < nph; ++ph) {
        const i32x4v* ab = abuf + abf * (kPhase * MT * 64) + lane;
        const int n = RES ? steps : min(kPhase, steps - ph * kPhase);
        auto rd_a = [&](int k, i32x4v (&A)[MT]) {
#pragma unroll
          for (int m = 0; m < MT; ++m) A[m] = ab[(k * MT + m) * 64];
        };
        rd_a(0, A0);
        int k = 0;
#pragma unroll 1
        for (; k + 2 <= n; k += 2, s += 2) {
          rd_a(k + 1, A1);
          rd_w(on, w1);
          on = tq[4 * min(s + 2, last)];
          mul(A0, w0);
          rd_a(min(k + 2, n - 1), A0);
          rd_w(on, w0);
          on = tq[4 * min(s + 3, last)];
          mul(A1, w1);
        }
        if (k < n) {
          mul(A0, w0);
          rd_w(on, w0);
          on = tq[4 * min(s + 2, last)];
          ++s;
        }
        if constexpr (!RES) {
          // the next phase (of the next tile after the last) into the other
          // buffer, which every wave left before the previous barrier
          abf ^= 1;
          a_put(abf);
          a_fetch((ph + 2) % nph);
          __syncthreads();
        }
      }
    }

    // ---- epilogue: acc = P - c1
    const MfmaKarg ke = fresh(kp);
    const int HW = H * W;
    const int cb = co0 + 4 * q;  // this lane's channels: cb + 16 m + r
    // a pixel code's patch, row and column, and whether it is in the image
    auto at = [&](int code, int* n, int* y, int* x) {
      *n = n0 + (code >> 20);
      *y = y0 + ((code >> 10) & 1023);
      *x = x0 + (code & 1023);
      return code >= 0 && *n < ke->a.N && *y < H && *x < W;
    };
    if constexpr (EPI == EPI_P) {
      bool pv[G], run = G == 4;
      size_t pp[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        int n, y, x;
        pv[g] = at(pc[g], &n, &y, &x);
        pp[g] = (size_t)n * ke->a.cout * HW + (size_t)y * W + x;
        run = run && pv[g] && pp[g] == pp[0] + (size_t)g;
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const f32x4v c1 = *reinterpret_cast<const f32x4v*>(ke->mc.c1 + cb + 16 * m);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (cb + 16 * m + r >= ke->a.cout) continue;
          int32_t* const plane = ke->a.P + (size_t)(cb + 16 * m + r) * HW;
          if (run) {
            i32x4u v;
#pragma unroll
            for (int g = 0; g < G; ++g) v[g] = (int)(acc[m][g][r] + c1[r]);
            *reinterpret_cast<i32x4u*>(plane + pp[0]) = v;
          } else {
#pragma unroll
            for (int g = 0; g < G; ++g)
              if (pv[g]) plane[pp[g]] = (int)(acc[m][g][r] + c1[r]);
          }
        }
      }
    }
    if constexpr (EPI != EPI_P) {
      constexpr int NW = (MT + 1) / 2;  // output words of the group
      const uint32_t* iv1 = ke->mc.inv1 + (co0 >> 5);
      // rule 1 per channel: |P - c1| < r1 (inverted channels flipped on the
      // packed word).  A lane has 4 channels of each 16 as a nibble at 4q
      // (m odd: 16 + 4q) of the word; the four lane rows are OR-ed together
      // by two lane swaps, which also leave lane row q with group q's pixel.
      uint32_t v[NW][G];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int h = 0; h < NW; ++h) v[h][g] = 0u;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const f32x4v r1v = *reinterpret_cast<const f32x4v*>(stab + 16 * MT * 16 + m * 16 + q * 4);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          uint32_t nib = 0;
#pragma unroll
          for (int r = 3; r >= 0; --r) nib = push_sign(nib, __builtin_fabsf(acc[m][g][r]) - r1v[r]);
          v[m >> 1][g] |= nib << (4 * q + 16 * (m & 1));
        }
      }
      if constexpr (EPI == EPI_POOL) {
        const uint32_t* iv2 = ke->mc.inv2 + (co0 >> 5);
        const int Hh = H >> 1, Wh = W >> 1;
        // the max of a block's P: the rows (groups 2p, 2p + 1), then the two
        // columns (lanes j, j ^ 1).  G = 4: the even lanes take the blocks of
        // pair 0, the odd ones those of pair 1.
        uint32_t u[NW];
#pragma unroll
        for (int h = 0; h < NW; ++h) u[h] = 0u;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const f32x4v dc = *reinterpret_cast<const f32x4v*>(stab + 17 * MT * 16 + m * 16 + q * 4);
          const f32x4v r2v = *reinterpret_cast<const f32x4v*>(stab + 18 * MT * 16 + m * 16 + q * 4);
          uint32_t nib = 0;
#pragma unroll
          for (int r = 3; r >= 0; --r) {
            const float v0 = max2(acc[m][0][r], acc[m][1][r]);
            float pm;
            if constexpr (G == 4) {
              const float v1 = max2(acc[m][2][r], acc[m][3][r]);
              pm = max2(j & 1 ? v1 : v0, swap_pair(j & 1 ? v0 : v1));
            } else {
              pm = max2(v0, swap_pair(v0));
            }
            nib = push_sign(nib, __builtin_fabsf(pm + dc[r]) - r2v[r]);
          }
          u[m >> 1] |= nib << (4 * q + 16 * (m & 1));
        }
        // lane row q -> word q / 2
        const uint32_t t = or_halves(u[0], u[NW - 1]), d = or_rows(t, t);
        const int wd = q >> 1;
        int n, y, x;
        const bool ok = at(G == 4 && (j & 1) ? pc[G - 2] : pc[0], &n, &y, &x) && y + 1 < H && x < 2 * Wh && wd < NW &&
                        (G == 4 || (j & 1) == 0) && (q & 1) == 0 && (co0 >> 5) + wd < ke->a.cwo;
        if (ok) ke->a.out2[(((size_t)n * Hh + (y >> 1)) * Wh + (x >> 1)) * ke->a.cwo + (co0 >> 5) + wd] = d ^ iv2[wd];
      }
      // lane row -> (group, word): G = 4: group q, all words; G = 2: group
      // q / 2, word q % 2
      uint32_t o[NW];
      if constexpr (G == 4) {
#pragma unroll
        for (int h = 0; h < NW; ++h) o[h] = or_rows(or_halves(v[h][0], v[h][2]), or_halves(v[h][1], v[h][3])) ^ iv1[h];
      } else {
        const uint32_t t0 = or_halves(v[0][0], v[0][1]), t1 = or_halves(v[NW - 1][0], v[NW - 1][1]);
        o[0] = or_rows(t0, t1);
      }
      int on_, oy, ox;
      const bool ov = at(po, &on_, &oy, &ox);
      if (ke->a.out != nullptr && ov) {
        uint32_t* dst = ke->a.out + (((size_t)on_ * H + oy) * W + ox) * ke->a.cwo + (co0 >> 5);
        if constexpr (G == 4) {
#pragma unroll
          for (int h = 0; h < NW; ++h)
            if ((co0 >> 5) + h < ke->a.cwo) dst[h] = o[h];
        } else {
          const int h = q & 1;
          if (h < NW && (co0 >> 5) + h < ke->a.cwo) dst[h] = o[0] ^ iv1[h];
        }
      }
      if constexpr (EPI == EPI_HEAD) {
        // one pixel per lane: bias, then the channels in order, one fused
        // step each (csrc/bnn_head.c:21-34)
        bool keep = ov;
        size_t lbase = (size_t)on_ * ke->a.ncls * HW + (size_t)oy * W + ox, lstride = HW;
        if (ke->a.pcols > 0) {
          const int prw = ke->a.prow0 + on_ / ke->a.pcols, pcl = on_ % ke->a.pcols;
          const int sy = prw * H + oy, sx = pcl * W + ox;
          keep = keep && sy < ke->a.sH && sx < ke->a.sW;
          lbase = (size_t)sy * ke->a.sW + sx;
          lstride = (size_t)ke->a.sH * ke->a.sW;
        }
        typedef const __attribute__((address_space(4))) float* const_hf;
        const const_hf hw = (const_hf)ke->a.hw, hb = (const_hf)ke->a.hb;
        float sg[MT * 16];
#pragma unroll
        for (int c = 0; c < MT * 16; ++c) sg[c] = (o[0] >> c) & 1u ? 1.0f : -1.0f;
        if (keep) {
          if (ke->a.cout == MT * 16) {
#pragma unroll 1
            for (int k = 0; k < ke->a.ncls; ++k) {
              float wv[MT * 16];
#pragma unroll
              for (int c = 0; c < MT * 16; ++c) wv[c] = hw[k * (MT * 16) + c];
              float s = hb[k];
#pragma unroll
              for (int c = 0; c < MT * 16; ++c) s = __fmaf_rn(wv[c], sg[c], s);
              ke->a.logits[lbase + (size_t)k * lstride] = s;
            }
          } else {
#pragma unroll 1
            for (int k = 0; k < ke->a.ncls; ++k) {
              float s = hb[k];
#pragma unroll
              for (int c = 0; c < MT * 16; ++c)
                if (c < ke->a.cout) s = __fmaf_rn(hw[k * ke->a.cout + c], sg[c], s);
              ke->a.logits[lbase + (size_t)k * lstride] = s;
            }
          }
        }
      }
    }
    sl += kp->T.subl;
    n0 += kp->T.subn;
    y0 += kp->T.suby;
    if (y0 >= H || n0 >= kp->a.N) break;
    }
    if (next >= ntiles) break;
    tile = next;
    n0 = n1;
    y0 = y1;
    x0 = x1;
    if (RES) __syncthreads();  // (a streamed group's last phase ended with one)
  }
}

}  // namespace

// The tile of a layer for blocks of `pb` pixels: whole patches, whole rows
// of a patch (rows up to 64 wide), or about 32 columns of wider rows; a
// pooled tile has an even number of rows and counts 2x2 blocks.  `sub` such
// tiles are staged together.
static void mfma_tile(int N, int H, int W, int cw, bool pool, int pb, int sub, MfmaTile* T) {
  const int We = pool ? (W + 1) & ~1 : W, He = pool ? (H + 1) & ~1 : H;
  int tr, tw = W, ti = 1, ntr = 1, ntc = 1;
  if ((long)We * He <= pb) {
    tr = He;
    // (at most 56 KB of staged words: two blocks a CU)
    const long per = (long)(tr + 2) * (tw + 2) * (cw < 4 ? cw : (cw + 3) / 4 * 4) * 4;
    ti = (int)std::max(1l, std::min({(long)N, (long)pb / (We * He), 56 * 1024 / per}));
  } else {
    if (We > 64) {
      ntc = (We + 31) / 32;
      tw = ((We + ntc - 1) / ntc + 3) & ~3;
      ntc = (We + tw - 1) / tw;
    }
    const int wp = pool ? (tw + 1) & ~1 : tw;
    int most = pb / wp;
    if (pool) most &= ~1;
    ntr = (He + most - 1) / most;
    tr = (He + ntr - 1) / ntr;
    if (pool) tr = (tr + 1) & ~1;
    ntr = (He + tr - 1) / tr;
  }
  if (ti == 1) sub = std::min(sub, ntr);
  const int px = pool ? (tr / 2) * ((tw + 1) / 2) : tr * tw;
  const int srows = ti > 1 ? tr + 2 : tr * sub + 2;  // staged rows of a patch
  T->TW = tw; T->TR = tr; T->TI = ti;
  T->dpat = make_kdiv((uint32_t)px);
  T->dcol = make_kdiv((uint32_t)(pool ? (tw + 1) / 2 : tw));
  T->dsp = make_kdiv((uint32_t)(srows * (tw + 2)));
  T->dsr = make_kdiv((uint32_t)(tw + 2));
  ntr = (ntr + sub - 1) / sub;
  T->dhp = make_kdiv((uint32_t)(ti > 1 ? 1 : ntr * ntc));
  T->dtc = make_kdiv((uint32_t)ntc);
  T->npat = px * ti;
  T->sub = sub;
  T->subn = ti > 1 ? ti : 0;
  T->suby = ti > 1 ? 0 : tr;
  T->ns = (ti > 1 ? ti * sub : 1) * srows * (tw + 2);
  T->ntiles = ti > 1 ? (uint32_t)((N + ti * sub - 1) / (ti * sub)) : (uint32_t)((size_t)N * ntr * ntc);
}

// LDS bytes of a layer's block; fills the regions' offsets
static size_t mfma_lds(const MfmaConv& mc, int cw, MfmaTile* T) {
  T->ps = cw < 4 ? cw : 4;
  T->planes = cw < 4 ? 1 : (cw + 3) / 4;
  T->subl = (T->subn ? T->subn * T->dsp.d : T->suby * T->dsr.d) * (uint32_t)T->ps * 4;
  T->plane_b = ((uint32_t)T->ns * T->ps * 4 + 15) & ~15u;
  T->steps = mc.steps;
  T->slots = mc.slots;
  T->ncg = mc.coutp / (16 * mc.mt);
  const size_t wb = (size_t)mc.steps * mc.mt * 1024;
  T->resident = wb <= kResident;
  T->off_tab = T->planes * T->plane_b;
  T->off_s = T->off_tab + (uint32_t)mc.steps * 16;
  T->off_a = T->off_s + (uint32_t)mc.mt * 19 * 64;
  return T->off_a + (T->resident ? wb : (size_t)2 * kPhase * mc.mt * 1024);
}

bool mfma_conv_fits(const MfmaConv& mc, int cw, int N, int H, int W, int epi) {
  if (!mc.w || H <= 0 || W <= 0) return false;
  if (epi != EPI_FOLD && epi != EPI_POOL && epi != EPI_HEAD && epi != EPI_P) return false;
  if (epi == EPI_HEAD && mc.mt > 2) return false;
  if (epi != EPI_P && !mc.r1) return false;
  if (epi == EPI_POOL && !mc.r2) return false;
  MfmaTile T{};
  mfma_tile(std::max(N, 1), H, W, cw, epi == EPI_POOL, 256, 1, &T);
  return mfma_lds(mc, cw, &T) <= 160 * 1024;
}

// A launch: its tile, the pixel groups a wave (G), LDS bytes, the blocks a CU
// holds of it, and the tile slots (blocks per channel group and XCD) and
// rounds over them.
struct MfmaPlan {
  MfmaTile T;
  int G;
  size_t lds, per_cu;
  uint32_t nts, rounds;
};
static MfmaPlan mfma_plan(const MfmaConv& mc, int cw, int N, int H, int W, int epi, int cus) {
  const bool pool = epi == EPI_POOL;
  const size_t waves = mfma_waves(mc.mt, epi);  // blocks a CU holds by registers
  MfmaPlan p{};
  mfma_tile(N, H, W, cw, pool, 256, 1, &p.T);
  p.lds = mfma_lds(mc, cw, &p.T);
  p.G = 4;
  if (epi != EPI_HEAD && (size_t)p.T.ntiles * p.T.ncg < 2 * (size_t)cus) {
    // 32 pixels a wave where 64 leave CUs without a block
    MfmaTile T2{};
    mfma_tile(N, H, W, cw, pool, 128, 1, &T2);
    const size_t l2 = mfma_lds(mc, cw, &T2);
    if (l2 <= 160 * 1024) { p.T = T2; p.lds = l2; p.G = 2; }
  } else {
    // two or four tiles staged together where that costs no round of blocks
    // (a tile's staging costs about one and a half times its sums)
    double best = 0.0;
    MfmaTile T2{};
    for (int sub = 1; sub <= 4; sub *= 2) {
      mfma_tile(N, H, W, cw, pool, 256, sub, &T2);
      const size_t l2 = mfma_lds(mc, cw, &T2);
      if (T2.sub != sub || (sub > 1 && l2 > 53 * 1024)) break;
      const size_t slots = std::max<size_t>(1, std::min<size_t>(waves, 160 * 1024 / l2)) * cus;
      const double t = (double)(((size_t)T2.ntiles * T2.ncg + slots - 1) / slots) * (sub + 1.5);
      if (sub == 1 || t < best) { best = t; p.T = T2; p.lds = l2; }
    }
  }
  // as many blocks as fit on the chip at once (LDS, registers), the tiles
  // spread evenly over them
  p.per_cu = std::max<size_t>(1, std::min<size_t>(waves, (160 * 1024) / p.lds));
  const uint32_t t8 = (p.T.ntiles + 7) / 8;
  const uint32_t most = std::max<uint32_t>(1, (uint32_t)(p.per_cu * cus / 8 / p.T.ncg));
  p.rounds = (t8 + most - 1) / most;
  p.nts = (t8 + p.rounds - 1) / p.rounds;
  return p;
}

// Folds and pools: the lesser of both kernels' estimated times in us, fitted
// to 2,238 layers timed on both (8 to 1,152 input channels, 8 to 768 output
// channels, 1 to 67,000 patches of 1 to 640 rows; eight times in ten within 9%
// here, 13% for popcount).  Summed over the layers the choice takes 20.6 ms,
// the better of the two 20.5, the popcount kernel alone 27.5, this one 22.7.
//  * popcount: a wave counts its words (9 a tap word, 5 a pair) over cog
//    channels x 1 or 4 pixels, the waves over the 1,024 SIMDs; from 60 words
//    on, and with the weights' bytes, its weight loads show (half as much
//    where fewer than half the CUs have a wave);
//  * here: K steps and rounds of tiles, by the blocks that share a CU: staging
//    by pixels and planes, sums by operands, the epilogue by outputs.
// Pairs (us, popcount : here): folds 64 -> 64, one 128x128 image, 5.0 : 7.1,
// 96 -> 192, 32x32, 5.2 : 8.1, 48 -> 16, 61 patches 113x73, 12.7 : 16.9, 256
// -> 256, 148 of 4x4, 16.4 : 10.5, 512 -> 512, 32x32, 33.8 : 12.4; pools 16 ->
// 16, 1,618 patches 70x25, 31 : 45, 32 -> 8, 6,154 of 15x19, 17 : 39, 40 ->
// 192, 192 of 35x4, 16.1 : 10.1.
// The head and P go by lines through the same pairs of times:
//  * head: 32 -> 32 at 4.8e9 bit-MACs 16.9 : 14.0; 24 -> 24 at 3.7e9 24.4 :
//    31.8;
//  * P: its stores bind, and rows of other lengths than whole groups of 16
//    leave lanes and lines partly filled, so shallow layers run here only with
//    such rows (64 -> 64, 64 x 64, 89 : 75; 16 -> 128 there 95 : 143; 64 -> 64,
//    45 x 51, 41 : 52), those from 96 channels also where many rounds of blocks
//    even the last one out (152 -> 40, 3.4e5 pixels, 62 : 43; 152 -> 64, 1.2e5
//    pixels, 28 : 36), from 224 channels at 1.5e9 bit-MACs (232 -> 24 at 1.6e9
//    15.4 : 10.2; 456 -> 168 at 1.2e9 10.3 : 16.3).
bool mfma_conv_pays(const MfmaConv& mc, int cin, int cout, int cw0, int cw1, bool pair, int epi, int N, int H, int W, int cus) {
  const int cw = cw0 + cw1;
  const double px = (double)N * H * W, macs = 9.0 * px * cin * cout;
  if (epi == EPI_HEAD || epi == EPI_P) {
    const bool pays = epi == EPI_HEAD ? macs >= 4e9 && cin >= 32
                      : cin >= 224    ? macs >= 1.5e9
                      : cin >= 176    ? macs >= 4e9
                                      : (W % 16 == 0 && cin >= 48 && macs >= 8e9) ||
                                         (cin >= 96 && macs >= 4e9 && px * ((cout + 63) / 64) >= 3e5);
    return pays && mfma_conv_fits(mc, cw, N, H, W, epi);
  }
  const bool pool = epi == EPI_POOL;
  // (deep folds on few pixels, where a popcount wave walks all words of a
  // pixel and its time outgrows the estimate: 256 -> 512, 155 patches 1x5,
  // 17.0 : 11.2, 384 -> 384, 48 of 2x3, 14.0 : 11.5)
  if (!pool && cw1 == 0 && ((cin >= 256 && macs >= 2.5e8) || cin >= 512)) return mfma_conv_fits(mc, cw, N, H, W, epi);
  int mt, cog;
  bconv_shape(epi, N, H, W, cout, &mt, &cog);
  const long waves = ((long)N * ((H + mt - 1) / mt) * ((W + mt - 1) / mt) + 63) / 64 * ((cout + cog - 1) / cog);
  const double words = 9 * cw - (pair ? 4 : 0), ws = (double)waves / (4 * cus);
  const double turns = ws < 2 ? std::ceil(ws) : ws, out = turns * cog * mt * mt;
  const double deep = turns * std::max(0.0, words - 60), kw = words * cout / 1024;
  const double pop = pool ? 4.91 + out * (0.0035 * words + 0.0188) + 0.27 * kw + 0.048 * deep
                          : 4.33 + out * (0.0036 * words + 0.0085) +
                                (0.088 * kw + 0.021 * deep) * (2 * waves < cus ? 0.5 : 1.0);
  const double planes = (cw + 3) / 4, loads = cw < 4 ? cw : 0;
  const double start = pool ? 5.87 + 0.093 * mc.steps : 5.19 + 0.071 * mc.steps;
  const double operand = pool ? 0.0077 * mc.steps + 0.0348 : 0.0100 * mc.steps + 0.0286, round = (pool ? 0.33 : 0.28) * planes;
  // (the tile is worked out only where one round of one block a CU might do:
  // 0.2 us of the host)
  if (start + round + operand * mc.mt * 2 + 0.4 >= pop || !mfma_conv_fits(mc, cw, N, H, W, epi)) return false;
  const MfmaPlan p = mfma_plan(mc, cw, N, H, W, epi, cus);
  const double blocks = 8.0 * p.T.ncg * p.nts;
  const double share = blocks <= (double)p.per_cu * cus ? std::min((double)p.per_cu, std::ceil(blocks / cus)) : blocks / cus;
  const double stage = share * p.T.ns / 256 * (pool ? 0.287 * planes + 0.0218 * loads : 0.378 * planes);
  const double here = start + p.rounds * (round + stage + operand * share * p.T.sub * mc.mt * p.G);
  return here + 0.4 < pop;  // (near ties on the popcount kernel)
}

namespace {
using MfmaFn = void (*)(const MfmaParams);
template <int MT, int G, bool RES>
MfmaFn mfma_fn(int epi) {
  switch (epi) {
    case EPI_FOLD: return k_bconv_mfma<MT, G, EPI_FOLD, RES>;
    case EPI_POOL: return k_bconv_mfma<MT, G, EPI_POOL, RES>;
    case EPI_P: return k_bconv_mfma<MT, G, EPI_P, RES>;
    case EPI_HEAD:
      if constexpr (MT <= 2 && G == 4) return k_bconv_mfma<MT, G, EPI_HEAD, RES>;
      break;
  }
  return nullptr;
}
template <bool RES>
MfmaFn mfma_fn(int mt, int G, int epi) {
  if (G == 4) return mt == 1 ? mfma_fn<1, 4, RES>(epi) : mt == 2 ? mfma_fn<2, 4, RES>(epi) : mfma_fn<4, 4, RES>(epi);
  return mt == 1 ? mfma_fn<1, 2, RES>(epi) : mt == 2 ? mfma_fn<2, 2, RES>(epi) : mfma_fn<4, 2, RES>(epi);
}
}  // namespace

hipError_t launch_bconv_mfma(const BconvArgs& a, const MfmaConv& mc, int epi, hipStream_t s) {
  if (a.N <= 0 || a.H <= 0 || a.W <= 0) return hipSuccess;
  const int cw = a.cw0 + a.cw1;
  if (!mfma_conv_fits(mc, cw, a.N, a.H, a.W, epi) || a.cout > mc.coutp) return hipErrorInvalidValue;
  if (mc.slots != mfma_nslots(a.cw0, a.cw1, a.pair)) return hipErrorInvalidValue;
  // v1 concats only: what the upsample leaves uncovered reads 0 bits (a v3
  // tensor's pad pixel lies past the range in1 is read in)
  if (a.in1 && a.padoff != kFar) return hipErrorInvalidValue;
  if (epi == EPI_P && !a.P) return hipErrorInvalidValue;
  if (epi == EPI_POOL && !a.out2) return hipErrorInvalidValue;
  if (epi == EPI_FOLD && !a.out) return hipErrorInvalidValue;
  const size_t npix = (size_t)a.N * a.H * a.W;
  if (npix * a.cw0 * 4 >= 0x80000000ull) return hipErrorInvalidValue;
  if (a.in1 && (size_t)a.N * a.h1 * a.w1 * a.cw1 * 4 >= 0x80000000ull) return hipErrorInvalidValue;
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const MfmaPlan p = mfma_plan(mc, cw, a.N, a.H, a.W, epi, device_cus());
  const MfmaTile& T = p.T;
  if ((size_t)a.N * T.dhp.d >= 0x7FFFFFFFull) return hipErrorInvalidValue;
  const MfmaFn fn = T.resident ? mfma_fn<true>(mc.mt, p.G, epi) : mfma_fn<false>(mc.mt, p.G, epi);
  if (!fn) return hipErrorInvalidValue;
  // more than 64 KB of LDS: allowed once per variant and device (bit d of
  // the variant's mask for device d)
  static std::atomic<uint64_t> attr[2][3][2][4];
  std::atomic<uint64_t>& at = attr[T.resident][mc.mt >> 1][p.G >> 2][epi];
  const uint64_t bit = 1ull << (dev & 63);
  if (!(at.load(std::memory_order_acquire) & bit)) {
    if (hipError_t e = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        e != hipSuccess)
      return e;
    at.fetch_or(bit, std::memory_order_acq_rel);
  }
  const uint32_t b0 = (uint32_t)(npix * a.cw0 * 4);
  const uint32_t b1 = a.in1 ? (uint32_t)((size_t)a.N * a.h1 * a.w1 * a.cw1 * 4) : 0u;
  hipLaunchKernelGGL(fn, dim3(8 * (unsigned)T.ncg * p.nts), dim3(256), p.lds, s, MfmaParams{a, mc, T, b0, b1});
  return hipGetLastError();
}

}  // namespace bnn
