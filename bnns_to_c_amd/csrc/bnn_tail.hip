// bnn_tail.hip - every binary layer of a 32x32 patch (enc1.c2 to dec1.c2 with
// the head; a stem model's enc1.c1 too) in one kernel on the FP4 matrix cores
// of gfx950 (csrc/bnn_model.c:168-253).  For models whose widths are at most
// 16, 32, 64, 128, 256 channels at the five levels.
#include <atomic>

#include "bnn_device.h"
#include "bnn_kernels.h"
#include "bnn_mfma_f4.h"

namespace bnn {
namespace {

// A block of 16 waves holds NP patches' activations in LDS and runs their
// layers one after another, a barrier between two.  One kernel instead of
// four to seventeen: a dependent launch costs about 4.5 us, and the deep
// levels of a patch (16 x 16 down to 2 x 2) fill no launch of their own.
//
// The product and the rules are the binary conv's (bnn_bconv_mfma.hip): FP4
// activations from masked bits, sums exact in FP32, acc = P - c1, a rule as
// |P - c| < r.  Here the weights come as sign bits too (a quarter of the
// bytes; every block reads all 250 KB of them through L2), one word a lane and
// operand: nibble k of operand register j is the FP4 code of 4, 2, 1 or 4 with
// bit 4k + j as its sign, seven instructions for an operand that meets G
// pixel groups.  A sign cannot be 0, so a K slot past the last one takes its
// activations as 0 instead, as do channels past the layer's.
//
// LDS tensors: [word][patch][d + 2][d + 2], d the level's width, a zero halo
// around every patch, word planes 16 banks apart.  A concat is its skip's
// planes and then the upsampled tensor's, which its producer writes at the
// upper level's resolution, each word to four pixels.  Tensors of at most 16
// channels hold a pixel's bits in the low half of a word and its right
// neighbour's in the high half (PAIR): three words carry the first two taps of
// each row, and the third taps are read as 16-bit halves in the second step.
//
// A level's layer is a GEMM of 16 NP d^2 / 16 pixel groups x 1 to 16 tiles of
// 16 channels; a wave keeps one set of MT tiles and walks G groups at a time.
// Pixels run in 2x2 blocks (four lanes a block), so a pool is two lane swaps.
template <int NP>
struct TailMap {
  // words of one plane (all patches): (d + 2)^2 a patch, 16 mod 64
  static constexpr int plane(int lv) {
    const int p = (32 >> lv) + 2, w = NP * p * p;
    return w + (((16 - w % 64) + 64) % 64);
  }
};

// sign bits -> FP4 codes of +-4, +-2, +-1, +-4.  (m: 0x88888888 in a vector
// register the compiler cannot see through: as a literal beside the codes it
// would take an AND and an OR instead of one v_and_or_b32.)
__device__ __forceinline__ i32x4v signs_f4(uint32_t w, uint32_t m) {
  return i32x4v{(int)(((w << 3) & m) | 0x66666666u), (int)(((w << 2) & m) | 0x44444444u),
                (int)(((w << 1) & m) | 0x22222222u), (int)((w & m) | 0x66666666u)};
}
// x of lane l ^ 2
__device__ __forceinline__ float swap_two(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, true));  // [2, 3, 0, 1]
}

typedef const __attribute__((address_space(4))) TailArgs* TailKarg;
__device__ __forceinline__ TailKarg fresh(TailKarg k) {
  asm volatile("" : "+s"(k));
  return k;
}

// The sums of G pixel groups over STEPS K steps, straight-line in batches so
// that a batch's LDS reads are under way while the one before is multiplied.
// PAIR: the first segment is a pair tensor (step 1 reads halves).  Where a
// step is one tap of four words (planes of four), its offset from the first
// step's is a constant; `off` holds the others'.  `aw` holds the weights of
// the first kTA / MT steps; a step's register takes those of the step as many
// on.
constexpr int kTA = 18;
// steps of planes of four words
constexpr int tail_full(int steps) { return steps >= 9 ? steps - steps % 9 : 0; }
template <int MT, int G, int STEPS, bool PAIR, int PLANE, int P>
__device__ __forceinline__ void tail_sums(const uint8_t* smem, const uint32_t (&lb0)[G], uint32_t (&aw)[kTA],
                                          __amdgpu_buffer_rsrc_t wu, uint32_t lane4, const int* tab, uint32_t m8,
                                          f32x4v (&acc)[MT][G]) {
  constexpr int FULL = PAIR ? 0 : tail_full(STEPS), NO = STEPS - FULL, kTC = kTA / MT;
  int o0 = 0, off[NO > 0 ? NO : 1];
  // (what two step counts share, the compiler would compute once before the
  // branch between them, for all their steps, and spill: the empty asms,
  // which differ by STEPS, keep it here)
  uint32_t lb[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    lb[g] = lb0[g];
    asm volatile("" : "+v"(lb[g]) : "i"(STEPS), "i"(P));
  }
  if constexpr (FULL > 0) o0 = tab[0];
#pragma unroll
  for (int s = 0; s < NO; ++s) off[s] = tab[4 * (FULL + s)];
  // words of a batch of kTB steps, read while the batch before is multiplied
  // (a scheduling barrier a batch: left alone the compiler reads all of a
  // layer's words first and spills)
  constexpr int kTB = MT * G >= 8 ? 2 : 3;
  auto rd = [&](int s0, uint32_t (&w)[kTB][G]) {
#pragma unroll
    for (int s = s0; s < STEPS && s < s0 + kTB; ++s) {
      // (a layer of 9, 18 or 27 steps fills its last one)
      const bool pad = PAIR ? (STEPS == 2 ? s < 2 : s == 1) : s == STEPS - 1 && STEPS % 9 != 0;
      const int of = s < FULL ? 0 : off[s < FULL ? 0 : s - FULL];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const uint8_t* at;
        if (s < FULL) at = smem + (lb[g] + (uint32_t)o0) + (4 * (s / 9) * PLANE + s % 9 / 3 * P + s % 3) * 4;
        else at = smem + lb[g] + (uint32_t)(pad ? of & 0x7FFFFFFF : of);
        if (PAIR && s == 1) w[s - s0][g] = *reinterpret_cast<const uint16_t*>(at);
        else w[s - s0][g] = *reinterpret_cast<const uint32_t*>(at);
        if (pad) w[s - s0][g] = of < 0 ? 0u : w[s - s0][g];
      }
    }
  };
  uint32_t w[2][kTB][G];
  rd(0, w[0]);
#pragma unroll
  for (int b = 0; b < STEPS; b += kTB) {
    rd(b + kTB, w[(b / kTB + 1) & 1]);
#pragma unroll
    for (int s = b; s < STEPS && s < b + kTB; ++s) {
      i32x4v A[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        uint32_t a = aw[s % kTC * MT + m];
        asm volatile("" : "+v"(a) : "i"(STEPS), "i"(P));
        A[m] = signs_f4(a, m8);
        if (s + kTC < STEPS) aw[s % kTC * MT + m] = ld_u32(wu, lane4, (uint32_t)(m * STEPS + s + kTC) * 256u);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const i32x4v B = bits_f4(w[(b / kTB) & 1][s - b][g]);
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][g] = mfma_f4(A[m], B, acc[m][g]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int NP, int NW>
struct TailWork {
  // tiles a wave and its pixel groups a turn, by level
  static constexpr int mt(int lv) { return lv == 0 ? 1 : NW == 16 ? (lv == 1 ? 2 : 1) : 2; }
  static constexpr int g(int lv) { return lv == 0 ? 4 : lv <= 2 ? NP : 1; }
};
// the weights of the first steps of a wave's tiles: entry i of aw is step i
// (one tile), or step i / 2 of tile i % 2; reads past a layer's last step
// stay inside the descriptor or give 0
__device__ __forceinline__ void tail_fetch(__amdgpu_buffer_rsrc_t wu, int steps, bool two, uint32_t lane4, uint32_t (&aw)[kTA]) {
  const uint32_t pair = two ? 256u : 512u, step = two ? (uint32_t)steps * 256u : 256u;
#pragma unroll
  for (int i = 0; i < kTA; ++i) aw[i] = ld_u32(wu, lane4, (uint32_t)(i >> 1) * pair + (uint32_t)(i & 1) * step);
}

// One layer of level LV, of 2^LV tiles of 16 channels.  A group is four 2x2
// blocks in a row of blocks (level 3: a patch, level 4: the block's patches), so
// where a lane reads and writes is a constant of the lane and the level plus
// the group's corner, which is scalar.
template <int NP, int NW, int LV>
__device__ __forceinline__ void tail_layer(TailKarg kp, int li, uint8_t* smem, int np) {
  constexpr int MT = TailWork<NP, NW>::mt(LV), G = TailWork<NP, NW>::g(LV), NCT = 1 << LV, C = NCT * 16;
  constexpr int lg = 4 - LV, QR = 1 << lg, d = 32 >> LV, p = d + 2;  // QR blocks of 2x2 a row
  constexpr int NG = NP * d * d >= 16 ? NP * d * d / 16 : 1;          // pixel groups
  constexpr int NU = NCT / MT;                                       // tile sets
  constexpr int WPU = NW / NU;                                       // waves a tile set
  constexpr bool kTurns = WPU * G < NG;                              // more than one turn a wave
  static_assert(NW % NU == 0 && NG % G == 0 && (G == 1 || LV <= 2), "work split");
  // (the lane's places at every level, hoisted out of the layer loop, would
  // fill the registers)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, q = lane >> 4, j = lane & 15;
  const int r = (j >> 1) & 1, c = j & 1, b4 = j >> 2;  // row and column in the block, block
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TailKarg k = fresh(kp);
  const __attribute__((address_space(4))) TailLayer& L = k->L[li];
  const int ct = wave % NU * MT, pg0 = wave / NU * G;  // first tile, first group
  const int steps = L.steps, kind = L.kind;
  const uint32_t lane4 = (uint32_t)lane * 4u, q16 = (uint32_t)q * 16u;
  constexpr uint32_t kTabs = (19 * C + 2 * (C / 32 > 0 ? C / 32 : 1)) * 4;  // bytes of the layer's tables
  const __amdgpu_buffer_rsrc_t tb = make_rsrc(L.tabs, kTabs);
  // row `row` of the tables (and lane-dependent bytes), this lane's four channels of tile ct + m
  auto tab4 = [&](uint32_t bytes, int row, int m) {
    return __builtin_bit_cast(f32x4v, __builtin_amdgcn_raw_buffer_load_b128(tb, (int)(bytes + q16), (row * C + (ct + m) * 16) * 4, 0));
  };
  uint32_t m8 = 0x88888888u;
  asm volatile("" : "+v"(m8));
  // a group's corner: patch, row of blocks, first block of it
  struct Corner { int n, qy, qx; };
  auto corner = [&](int pg) {
    Corner g{0, 0, 0};
    if constexpr (LV <= 2) {
      g.n = pg >> (2 * lg - 2);
      const int rem = pg & ((1 << (2 * lg - 2)) - 1);
      g.qy = rem >> (lg - 2);
      g.qx = (rem & ((1 << (lg - 2)) - 1)) * 4;
    } else if constexpr (LV == 3) {
      g.n = pg;
    }
    return g;
  };
  // the lane's pixel from its group's corner, in words: of this level's
  // window corners (lc), of the level above's pixels (lu), of the level
  // below's pixels by its block (ld)
  constexpr int p1 = d / 2 + 2, p2 = 2 * d + 2;
  int lc, lu, ld;
  if constexpr (LV <= 2) {
    lc = r * p + 2 * b4 + c;
    lu = 2 * r * p2 + 2 * (2 * b4 + c);
    ld = b4;
  } else if constexpr (LV == 3) {
    const int by = b4 >> 1, bx = b4 & 1;
    lc = (2 * by + r) * p + 2 * bx + c;
    lu = 2 * (2 * by + r) * p2 + 2 * (2 * bx + c);
    ld = by * p1 + bx;
  } else {
    const int n = b4 & (NP - 1);  // (fewer than 16 pixels: the rest repeat)
    lc = n * p * p + r * p + c;
    lu = n * p2 * p2 + 2 * r * p2 + 2 * c;
    ld = 0;
  }
  constexpr int kGs = LV <= 1 ? 8 : 2 * p;                                 // words to the turn's next group
  constexpr int kGu = LV <= 1 ? 16 : 4 * p2, kGd = LV <= 1 ? 4 : p1;
  const bool live = NP * d * d >= 16 || j < NP * d * d;  // lanes past the last pixel store nothing
  // border sums: the class bytes of the lane's pixel in a group
  auto cls_of = [&](const Corner& g) -> uint32_t {
    int v;
    if constexpr (LV <= 2) {
      v = (g.qy == 0 ? 4 - 4 * r : 0) + (g.qy == QR - 1 ? 8 * r : 0) + (g.qx == 0 ? (b4 == 0 && c == 0 ? 1 : 0) : 0) +
          (g.qx + 4 == QR ? (b4 == 3 && c == 1 ? 2 : 0) : 0);
    } else if constexpr (LV == 3) {
      const int y = 2 * (b4 >> 1) + r, x = 2 * (b4 & 1) + c;
      v = (y == 0 ? 4 : 0) + (y == 3 ? 8 : 0) + (x == 0 ? 1 : 0) + (x == 3 ? 2 : 0);
    } else {
      v = (r ? 8 : 4) + (c ? 2 : 1);
    }
    return (uint32_t)v * (C * 4u);
  };
  // what needs no other wave's work comes before the barrier: weights, the
  // rule, the first groups' border sums
  f32x4v acc[MT][G];
  auto border = [&](int pg) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const uint32_t cb = cls_of(corner(pg + g));
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m][g] = tab4(cb, 0, m);
    }
  };
  uint32_t aw[kTA];
  const __amdgpu_buffer_rsrc_t wu = make_rsrc(L.w + (uint32_t)(ct * steps * 64), (uint32_t)(MT * steps) * 256u);
  tail_fetch(wu, steps, MT == 2, lane4, aw);
  const int* tab = reinterpret_cast<const int*>(smem + k->off_tab) + L.slot * 4 + q;
  f32x4v r1v[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) r1v[m] = tab4(0u, 16, m);
  const uint32_t inv1 = __builtin_bit_cast(uint32_t, L.tabs[19 * C + (ct >> 1)]) >> (ct & 1 ? 16 : 0);
  border(pg0);
  __syncthreads();

  for (int pg = pg0; pg < NG; pg += kTurns ? WPU * G : NG) {
    if (kTurns && pg != pg0) border(pg);
    const Corner g0 = corner(pg);
    uint32_t lb[G];
#pragma unroll
    for (int g = 0; g < G; ++g) lb[g] = (uint32_t)(lc + (g0.n * p + 2 * g0.qy) * p + 2 * g0.qx + g * kGs) * 4u;
    // ---- sums: the step counts of the level's layers
    constexpr int PL = TailMap<NP>::plane(LV);
    if constexpr (LV == 0) {
      if (steps == 4) tail_sums<MT, G, 4, true, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else tail_sums<MT, G, 2, true, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
    } else if constexpr (LV == 1) {
      if (steps == 7) tail_sums<MT, G, 7, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else if (steps == 3) tail_sums<MT, G, 3, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else tail_sums<MT, G, 2, true, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
    } else if constexpr (LV == 2) {
      if (steps == 14) tail_sums<MT, G, 14, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else if (steps == 5) tail_sums<MT, G, 5, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else tail_sums<MT, G, 3, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
    } else if constexpr (LV == 3) {
      if (steps == 27) tail_sums<MT, G, 27, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else if (steps == 9) tail_sums<MT, G, 9, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else tail_sums<MT, G, 5, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
    } else {
      if (steps == 18) tail_sums<MT, G, 18, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
      else tail_sums<MT, G, 9, false, PL, p>(smem, lb, aw, wu, lane4, tab, m8, acc);
    }
    // ---- rule 1: bit = (|P - c1| < r1) ^ inv1, gathered to lane rows: G = 4
    // row q holds group q's pixels, G = 2 group q / 2, G = 1 the group in all
    uint32_t v[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      v[g] = 0;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        uint32_t nib = 0;
#pragma unroll
        for (int i = 3; i >= 0; --i) nib = push_sign(nib, __builtin_fabsf(acc[m][g][i]) - r1v[m][i]);
        v[g] |= nib << (4 * q + 16 * m);
      }
    }
    uint32_t o;
    int og;
    if constexpr (G == 4) { o = or_rows(or_halves(v[0], v[2]), or_halves(v[1], v[3])); og = q; }
    else if constexpr (G == 2) { const uint32_t t = or_halves(v[0], v[1]); o = or_rows(t, t); og = q >> 1; }
    else { const uint32_t t = or_halves(v[0], v[0]); o = or_rows(t, t); og = 0; }
    o ^= inv1;
    if constexpr (LV == 0) {
      if (kind == TAIL_HEAD) {
        // one pixel a lane: bias, then the channels in order, one fused step
        // each (csrc/bnn_head.c:21-34); the sums of the first eight come from
        // a table of their 256 sign patterns
        const TailKarg kh = fresh(kp);
        const int n = (int)blockIdx.x * NP + g0.n, y = 2 * g0.qy + r, x = 2 * (4 * q + b4) + c;
        bool keep = g0.n < np;
        size_t lbase = (size_t)n * kh->ncls * 1024 + (size_t)(y * 32 + x), lstride = 1024;
        if (kh->pcols > 0) {
          const int sy = (kh->prow0 + n / kh->pcols) * 32 + y, sx = n % kh->pcols * 32 + x;
          keep = keep && sy < kh->sH && sx < kh->sW;
          lbase = (size_t)sy * kh->sW + sx;
          lstride = (size_t)kh->sH * kh->sW;
        }
        typedef const __attribute__((address_space(4))) float* const_hf;
        const const_hf hw = (const_hf)kh->hw;
        const float* const hl = kh->hl;
        const int hc = kh->hc, ncls = kh->ncls;
        float sg[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sg[i] = (o >> (8 + i)) & 1u ? 1.0f : -1.0f;
        if (keep) {
#pragma unroll 1
          for (int t = 0; t < ncls; ++t) {
            float s = hl[t * 256 + (int)(o & 255u)];
            if (hc == 16) {
              float wv[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) wv[i] = hw[t * 16 + 8 + i];
#pragma unroll
              for (int i = 0; i < 8; ++i) s = __fmaf_rn(wv[i], sg[i], s);
            } else {
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (8 + i < hc) s = __fmaf_rn(hw[t * hc + 8 + i], sg[i], s);
            }
            kh->logits[lbase + (size_t)t * lstride] = s;
          }
        }
        continue;
      }
    }
    // where this wave's tiles sit in a tensor: word plane ct / 2, half ct % 2
    const uint32_t half = (uint32_t)(ct & 1) * 2u;
    if (kind != TAIL_UP && live && (G == 4 || (G == 2 ? (q & 1) == 0 : q == 0))) {
      uint8_t* dst = smem + (L.out + half + (uint32_t)((ct >> 1) * PL + (g0.n * p + 2 * g0.qy + 1) * p + 2 * g0.qx + 1) * 4u) +
                     (uint32_t)(lc + og * kGs) * 4u;
      if constexpr (MT == 2) {
        *reinterpret_cast<uint32_t*>(dst) = o;
      } else {
        *reinterpret_cast<uint16_t*>(dst) = (uint16_t)o;
        if (L.opair) *reinterpret_cast<uint16_t*>(dst - 2) = (uint16_t)o;  // the left neighbour's high half
      }
    }
    if constexpr (LV > 0) {
      // ---- upsampled: the word (or half) to four pixels of the level above
      if (kind == TAIL_UP && live) {
        uint8_t* dst = smem + (L.out + half + (uint32_t)((ct >> 1) * TailMap<NP>::plane(LV - 1) + (g0.n * p2 + 4 * g0.qy + 1) * p2 + 4 * g0.qx + 1) * 4u) +
                       (uint32_t)(lu + og * kGu) * 4u;
        // lane rows that hold the same pixel share the four stores
        constexpr int rep = G == 4 ? 1 : G == 2 ? 2 : 4;
        const int s0 = G == 4 ? 0 : G == 2 ? (q & 1) : q;
#pragma unroll
        for (int t = 0; t < 4 / rep; ++t) {
          const int i = t * rep + s0;
          uint8_t* const e = dst + (uint32_t)((i >> 1) * p2 + (i & 1)) * 4u;
          if constexpr (MT == 2) *reinterpret_cast<uint32_t*>(e) = o;
          else *reinterpret_cast<uint16_t*>(e) = (uint16_t)o;
        }
      }
    }
    if constexpr (LV < 4) {
      if (kind == TAIL_POOL) {
        // the max of P over a block's four lanes; G = 4: lane j ends with
        // group j % 4's, G = 2: group j % 2's
        uint32_t u = 0;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const f32x4v dc = tab4(0u, 17, m), r2 = tab4(0u, 18, m);
          uint32_t nib = 0;
#pragma unroll
          for (int i = 3; i >= 0; --i) {
            float pm;
            if constexpr (G == 4) {
              const float a = max2(c ? acc[m][1][i] : acc[m][0][i], swap_pair(c ? acc[m][0][i] : acc[m][1][i]));
              const float b = max2(c ? acc[m][3][i] : acc[m][2][i], swap_pair(c ? acc[m][2][i] : acc[m][3][i]));
              pm = max2(r ? b : a, swap_two(r ? a : b));
            } else if constexpr (G == 2) {
              const float a = max2(c ? acc[m][1][i] : acc[m][0][i], swap_pair(c ? acc[m][0][i] : acc[m][1][i]));
              pm = max2(a, swap_two(a));
            } else {
              const float a = max2(acc[m][0][i], swap_pair(acc[m][0][i]));
              pm = max2(a, swap_two(a));
            }
            nib = push_sign(nib, __builtin_fabsf(pm + dc[i]) - r2[i]);
          }
          u |= nib << (4 * q + 16 * m);
        }
        const uint32_t t0 = or_halves(u, u);
        const uint32_t dw = or_rows(t0, t0) ^ (__builtin_bit_cast(uint32_t, L.tabs[19 * C + (C < 32 ? 1 : C / 32) + (ct >> 1)]) >> (ct & 1 ? 16 : 0));
        const int gsel = G == 4 ? (j & 3) : G == 2 ? c : 0;
        if (live && q == 0 && (G == 4 || (G == 2 ? r == 0 : (j & 3) == 0))) {
          uint8_t* dst = smem + (L.down + half + (uint32_t)((ct >> 1) * TailMap<NP>::plane(LV + 1) + (g0.n * p1 + g0.qy + 1) * p1 + g0.qx + 1) * 4u) +
                         (uint32_t)(ld + gsel * kGd) * 4u;
          if constexpr (MT == 2) {
            *reinterpret_cast<uint32_t*>(dst) = dw;
          } else {
            *reinterpret_cast<uint16_t*>(dst) = (uint16_t)dw;
            if (L.dpair) *reinterpret_cast<uint16_t*>(dst - 2) = (uint16_t)dw;
          }
        }
      }
    }
  }
}

template <int NP, int NW>
__global__ __launch_bounds__(64 * NW, 4) void k_tail(const TailArgs) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const TailKarg kp = (TailKarg)__builtin_amdgcn_kernarg_segment_ptr();
  const int tid = threadIdx.x;
  // zero halos (and every unwritten bit), the slot table, then the first
  // tensor as a pair tensor
  {
    const TailKarg k = fresh(kp);
    const int nz = k->lds_words / 4;
    for (int i = tid; i < nz; i += 64 * NW) reinterpret_cast<i32x4v*>(smem)[i] = i32x4v{0, 0, 0, 0};
    int* tab = reinterpret_cast<int*>(smem + k->off_tab);
    for (int i = tid; i < k->nslot; i += 64 * NW) tab[i] = k->slots[i];
  }
  const int np = min(NP, kp->N - (int)blockIdx.x * NP);
  constexpr int PT = NP * 1024 / (64 * NW);  // input pixels a thread
  uint32_t in[PT];
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e = i * 64 * NW + tid;
    in[i] = (e >> 10) < np ? kp->in[(size_t)blockIdx.x * NP * 1024 + e] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int e = i * 64 * NW + tid, n = e >> 10, y = (e >> 5) & 31, x = e & 31;
    uint16_t* dst = reinterpret_cast<uint16_t*>(smem + kp->off_in + (uint32_t)((n * 34 * 34 + (y + 1) * 34 + x + 1) * 4));
    dst[0] = (uint16_t)in[i];
    dst[-1] = (uint16_t)in[i];
  }
  const int last = kp->nlayers;
#pragma unroll 1
  for (int li = 0; li < last; ++li) {
    const int lv = kp->L[li].lvl;
    if (lv == 0) tail_layer<NP, NW, 0>(kp, li, smem, np);
    else if (lv == 1) tail_layer<NP, NW, 1>(kp, li, smem, np);
    else if (lv == 2) tail_layer<NP, NW, 2>(kp, li, smem, np);
    else if (lv == 3) tail_layer<NP, NW, 3>(kp, li, smem, np);
    else tail_layer<NP, NW, 4>(kp, li, smem, np);
  }
}

}  // namespace

int tail_plane(int np, int lvl) { return np == 1 ? TailMap<1>::plane(lvl) : TailMap<2>::plane(lvl); }

// one patch a block of 16 waves (a block's time least) while every patch has
// a CU, else two a block of 8 waves, two blocks a CU
int tail_np(int N) { return N <= device_cus() ? 1 : 2; }

hipError_t launch_tail(const TailArgs& a, int np, hipStream_t s) {
  if (a.N <= 0) return hipSuccess;
  if (np != 1 && np != 2) return hipErrorInvalidValue;
  const size_t lds = (size_t)a.off_tab + (size_t)a.nslot * 4;
  if (lds > 80 * 1024) return hipErrorInvalidValue;
  const void* fn = np == 1 ? (const void*)k_tail<1, 16> : (const void*)k_tail<2, 8>;
  if (lds > 64 * 1024) {  // (a stem model's two patches) allowed once per variant and device
    static std::atomic<uint64_t> attr[2];
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(attr[np - 1].load(std::memory_order_acquire) & bit)) {
      if (hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024); e != hipSuccess)
        return e;
      attr[np - 1].fetch_or(bit, std::memory_order_acq_rel);
    }
  }
  const dim3 grid((unsigned)((a.N + np - 1) / np));
  if (np == 1) hipLaunchKernelGGL((k_tail<1, 16>), grid, dim3(1024), lds, s, a);
  else hipLaunchKernelGGL((k_tail<2, 8>), grid, dim3(512), lds, s, a);
  return hipGetLastError();
}

}  // namespace bnn
