// prefill_split.hip -- causal attention of few queries over the group-64
// cache on the gfx950 matrix cores (the outputs of attention_fused,
// engine.cu:236-308), for launches whose 64-query blocks are too few to fill
// the chip: a chat's next turn on a long cached history, a short prompt.
//
// prefill_mfma.hip gives one workgroup 64 queries of a whole GQA group and
// every key; 77 queries after 9000 cached tokens are 8 such workgroups, 142
// tiles each.  Here a workgroup takes 16 kQT queries of ONE query head and
// its kW waves split the keys: wave w the 64-key tiles w, w + kW, ..  Each wave
// runs on its own (a private LDS tile, no barrier) and ends with a partial
// softmax state (m, l, O) per query; the partials meet in LDS and the
// workgroup writes the rows.  No memory outside the workgroup is needed, so
// calls on several streams stay independent.
//
// One tile of a wave:
//   load     K and V rows by 16 bytes a lane, 4 neighbouring lanes to a row's
//            64 bytes (other orders fetch a fifth as fast), one tile ahead in
//            registers, then written to the wave's LDS with row r's piece p at
//            p ^ ps_sw(r);
//   S^T      = K Q^T (v_mfma_f32_16x16x32_f16): A = 16 keys x 16 dims per
//            lane group as one 16-byte LDS read, fp8 -> fp16 exactly;
//   softmax  in registers, as in prefill_tile.h (the running max moves only
//            when a numerator would overflow fp16); over H2O slots each tile
//            against its own max (slot_exp);
//   O^T     += vs (V^T P^T): V^T by ds_read_b64_tr_b8, the keys of a lane
//            group's 8 elements being those its P holds; the group's V scale
//            multiplies the tile's fp32 product, so V enters exactly.
#include "prefill_tile.h"

namespace cia {

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i32x2 lds_i32x2_t;

// 16-byte piece swizzle of LDS row r (4 pieces of 64 bytes): bits 2, 3, 4 of
// r to 01, 10, 11, pairwise independent, so that the rows sharing banks in a
// K read (16 rows of one key tile) and in a transposing V read (rows 4b .. 4b
// + 3 and 16 + 4b .. of each lane group b) take distinct pieces
__device__ __forceinline__ int ps_sw(int r) {
  return (((r >> 2) ^ (r >> 4)) & 1) | (((r >> 2) ^ (r >> 3)) & 2);
}

// What differs over the H2O slot buffer (attention_h2o's outputs,
// engine.cu:337-384): tiles of 64 slots, a scale per slot, and the mask from
// slot_pos.  The tile's slots' scales and positions pass through the wave's
// LDS; a K scale multiplies its fp32 scores, a V scale its fp16 row.
struct SlotArgs {
  const int32_t* slot_pos;
  int n_live;
};

// Numerators of one 16-query tile over 64 slots, relative to the tile's own max
// of each query: fp16 rounds the largest not at all and none of weight into
// its subnormals, wherever in the buffer the largest score lies.  (Relative to
// a running max, as over cached keys, 1024 queries over their own slots were
// 3.18e-4 off 64 bits in place of 3.14e-4, and a buffer whose output is carried
// by many slots 18 bits below the largest score 0.8 % off.)  S holds scores in
// log2 units, -inf where masked.  Returns f = 2^(tile max - m), by which the
// tile's products and sum enter O and l in fp32; m, the reference of O and l,
// moves where f would pass 2^64.
__device__ __forceinline__ float slot_exp(const f32x4 (&S)[4], float& m, float& l, f32x4 (&O)[4],
                                          f16x8 (&P)[2]) {
  float cm = -1e30f;  // (all masked: numerators 0)
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int i = 0; i < 4; i++) cm = __builtin_fmaxf(cm, S[k][i]);
  const float mt = pf_colmax(cm);
  if (__any(mt > m + 64.f)) {
    const float mn = mt > m + 64.f ? mt : m, corr = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) O[d][i] *= corr;
  }
  const float rs = pf_exp<false>(S, 1.0f, mt, 0, 0, P), f = __builtin_amdgcn_exp2f(mt - m);
  l = __builtin_fmaf(rs, f, l);
  return f;
}

constexpr int kPsORow = 68;  // floats between two queries of a wave's partial O
// bytes of a wave's LDS: the K and V tiles (and 64 slots' K scales, positions
// and V scales); then m, l and O per query
constexpr int ps_wave_bytes(bool slots, int qt) {
  const int merge = 16 * qt * (kPsORow + 2) * 4, tiles = 8192 + (slots ? 64 * 10 : 0);
  return merge > tiles ? merge : tiles;
}

// grid = 8 kv heads * 4 * nq (nq = ceil(S / (16 kQT))), block = 64 kW
template <bool kSlots, int kQT, int kW>
__global__ __launch_bounds__(64 * kW) void k_prefill_split(PrefillArgs a, SlotArgs sl) {
  constexpr int kWB = ps_wave_bytes(kSlots, kQT);
  __shared__ __attribute__((aligned(16))) uint8_t lds[kW * kWB];
  const int tid = threadIdx.x, l = tid & 63, n = l & 15, b = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (kv head g on XCD g: its L2 holds one head's cache; the queries with the
  // most keys first)
  const int g = blockIdx.x & 7, h = g * GQA + ((blockIdx.x >> 3) & 3);
  const int q0 = (a.nblk - 1 - (int)(blockIdx.x >> 5)) * 16 * kQT;
  const int qmin = a.past + q0, qlast = a.past + min(q0 + 16 * kQT - 1, a.S - 1);
  const int ntile = kSlots ? (sl.n_live + 63) >> 6 : (qlast >> 6) + 1;
  const int nfp8 = kSlots ? ntile : a.committed >> 6;
  uint8_t* kt = lds + w * kWB;
  uint8_t* vt = kt + 4096;
  float* lks = (float*)(kt + 8192);
  int* lpos = (int*)(kt + 8192 + 256);
  _Float16* lvs = (_Float16*)(kt + 8192 + 512);

  struct Tile {
    u32x4 k[4], v[4];
    uint16_t ks, vs;  // the group's; kSlots: those of slot l of the tile
    int pos;
  };
  // (uniform bases and one 32-bit lane offset)
  const uint32_t loff = (uint32_t)((l >> 2) * (NKV * D) + 16 * (l & 3));
  auto load = [&](int j, Tile& t) __attribute__((always_inline)) {
    if constexpr (kSlots) {
      // (slots past the last read it again, at a position no query sees)
      const int r0 = 64 * j, last = sl.n_live - 1;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t o = (uint32_t)(min(r0 + 16 * i + (l >> 2), last) * (NKV * D) + 16 * (l & 3));
        t.k[i] = *(const u32x4*)(a.kc8 + g * D + o);
        t.v[i] = *(const u32x4*)(a.vc8 + g * D + o);
      }
      const int r = min(r0 + l, last);
      t.ks = a.ksc[r * NKV + g];
      t.vs = a.vsc[r * NKV + g];
      t.pos = r0 + l <= last ? sl.slot_pos[r] : 0x7fffffff;
      return;
    }
    const size_t o = (size_t)j * (G * NKV * D) + g * D;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint8_t* kg = a.kc8 + o + i * (16 * NKV * D);
      const uint8_t* vg = a.vc8 + o + i * (16 * NKV * D);
      t.k[i] = *(const u32x4*)(kg + loff);
      t.v[i] = *(const u32x4*)(vg + loff);
    }
    t.ks = a.ksc[j * NKV + g];
    t.vs = a.vsc[j * NKV + g];
  };
  // lane offsets in the tiles (ps_sw of a row depends on its bits 2..4 only):
  // stores of rows 16 i + (l >> 2) by i & 1, K reads of rows 16 k + n by
  // k & 1, transposing V reads of rows 32 u + 4 b + e (e < 4) and + 12 + e
  // (e = n >> 1: lanes 2 e and 2 e + 1 of a lane group address row e's two
  // 8-byte halves of 16 dims) for dims 0..15; dims 16 d ..: ^ 16 d
  const int wo0 = 16 * l ^ 16 * ps_sw(l >> 2), wo1 = 16 * l ^ 16 * ps_sw(16 + (l >> 2));
  const int ko0 = 64 * n + 16 * (b ^ ps_sw(n)), ko1 = 64 * n + 16 * (b ^ ps_sw(16 + n));
  const int ve = n >> 1, vr = 4 * b + (ve < 4 ? ve : 12 + ve);
  const int vo = 64 * vr + 16 * ps_sw(vr) + 8 * (n & 1);
  const int nf = min(ntile, nfp8);  // FP8 tiles; tile nfp8 is the fp16 tail
  Tile cur;
  if (w < nf) load(w, cur);

  // Q^T as the B operand: lane (n, b) holds dims 16 b + 8 kb .. +7 of its query
  f16x8 qop[kQT][2];
#pragma unroll
  for (int t = 0; t < kQT; t++) {
    const int s = q0 + 16 * t + n;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
      qop[t][kb] = *(const f16x8*)(a.q + ((size_t)(s < a.S ? s : a.S - 1) * NH + h) * D + 16 * b + 8 * kb);
  }
  f32x4 O[kQT][4];
  float m[kQT], lsum[kQT];
#pragma unroll
  for (int t = 0; t < kQT; t++) {
#pragma unroll
    for (int d = 0; d < 4; d++) O[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[t] = -1e30f;
    lsum[t] = 0.f;
  }
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};

  // one tile: scores of the K operands kop(k) (16 keys each), softmax, pv(P)
  // with the factors of their products, vs over cached keys
  auto attend = [&](int j, float c, float vs, bool first, auto kop, auto pv)
      __attribute__((always_inline)) {
    f32x4 S[kQT][4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      f16x8 k0, k1;
      kop(k, k0, k1);
#pragma unroll
      for (int t = 0; t < kQT; t++) {
        S[t][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qop[t][0], zero, 0, 0, 0);
        S[t][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1, qop[t][1], S[t][k], 0, 0, 0);
      }
    }
    // (masked scores become -inf in place: c > 0 keeps them there)
    if constexpr (kSlots) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const f32x4 ks = *(const f32x4*)(lks + 16 * k + 4 * b);
        const i32x4 pos = *(const i32x4*)(lpos + 16 * k + 4 * b);
#pragma unroll
        for (int t = 0; t < kQT; t++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            S[t][k][i] = pos[i] > qmin + 16 * t + n ? -__builtin_inff() : S[t][k][i] * ks[i];
      }
    } else if (64 * j + 63 > qmin) {
#pragma unroll
      for (int t = 0; t < kQT; t++)
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            S[t][k][i] = 64 * j + 16 * k + 4 * b + i > qmin + 16 * t + n ? -__builtin_inff() : S[t][k][i];
    }
    f16x8 P[kQT][2];
    if constexpr (kSlots) {
      float f[kQT];
#pragma unroll
      for (int t = 0; t < kQT; t++) f[t] = slot_exp(S[t], m[t], lsum[t], O[t], P[t]);
      pv(P, f);
      return;
    }
#pragma unroll
    for (int t = 0; t < kQT; t++) {
      float rs = first ? __builtin_inff() : pf_exp<false>(S[t], c, m[t], 0, 0, P[t]);
      if (__any(!(rs < 3.0e38f)))
        rs = pf_remax<false>(S[t], c, first, m[t], lsum[t], O[t], 0, 0, P[t]);
      lsum[t] += rs;
    }
    float f[kQT];
#pragma unroll
    for (int t = 0; t < kQT; t++) f[t] = vs;
    pv(P, f);
  };
  int first = 1;
  asm("" : "+s"(first));  // (opaque: the loop's first pass is not peeled into code of its own)
  for (int j = w; j < nf; j += kW) {
    float c = 1.0f, vs = 1.0f;
    bool seen = true;   // by some query of the workgroup
    bool kinf = false;  // a slot's K scale is infinite
    if constexpr (kSlots) {
      seen = __any(cur.pos <= qlast);
      kinf = __any((cur.ks & 0x7FFF) == 0x7C00);
      lks[l] = h2f(cur.ks) * a.qscale;
      lpos[l] = cur.pos;
      lvs[l] = __builtin_bit_cast(_Float16, cur.vs);
    } else {
      c = __builtin_fmaxf(h2f((uint16_t)pf_late(cur.ks)) * a.qscale, 1e-30f);
      vs = h2f((uint16_t)pf_late(cur.vs));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      *(u32x4*)(kt + (i & 1 ? wo1 : wo0) + 1024 * i) = cur.k[i];
      *(u32x4*)(vt + (i & 1 ? wo1 : wo0) + 1024 * i) = cur.v[i];
    }
    if (j + kW < nf) load(j + kW, cur);
    if (!seen) continue;
    auto kop = [&](int k, f16x8& k0, f16x8& k1) __attribute__((always_inline)) {
      const u32x4 kk = *(const u32x4*)(kt + (k & 1 ? ko1 : ko0) + 1024 * k);
      k0 = pf_cvt8(kk[0], kk[1]);
      k1 = pf_cvt8(kk[2], kk[3]);
      if constexpr (kSlots)
        if (kinf) {
          // its values are infinite or 0 * inf before the product, which is
          // then NaN unless every term has one sign
          const _Float16 x = __builtin_isinf(lks[16 * k + n]) ? (_Float16)__builtin_inff() : (_Float16)1.0f;
          k0 *= x;
          k1 *= x;
        }
    };
    auto pv = [&](const f16x8 (&P)[kQT][2], const float (&f)[kQT]) __attribute__((always_inline)) {
      f16x8 sc[2];
      if constexpr (kSlots)
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const f16x4 lo = *(const f16x4*)(lvs + 32 * u + 4 * b), hi = *(const f16x4*)(lvs + 32 * u + 16 + 4 * b);
          sc[u] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
      for (int d = 0; d < 4; d++) {
        f16x8 vop[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const i32x2 raw = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
              (lds_i32x2_t*)(vt + (vo ^ 16 * d) + 2048 * u));
          vop[u] = pf_cvt8((uint32_t)raw[0], (uint32_t)raw[1]);
          if constexpr (kSlots) vop[u] *= sc[u];
        }
#pragma unroll
        for (int t = 0; t < kQT; t++) {
          f32x4 T = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[0], P[t][0], zero, 0, 0, 0);
          T = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop[1], P[t][1], T, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; i++) O[t][d][i] = __builtin_fmaf(T[i], f[t], O[t][d][i]);
        }
      }
    };
    attend(j, c, vs, first != 0, kop, pv);
    first = 0;
  }
  if (!kSlots && ntile > nfp8 && nfp8 % kW == w) {
    // the fp16 tail: K straight into operand order, V rows through the wave's
    // LDS (rows past the last token are zero), read back one value at a time
    const int nvalid = a.past + a.S - a.committed;
    auto kop = [&](int k, f16x8& k0, f16x8& k1) __attribute__((always_inline)) {
      const uint16_t* kr = a.ktail + ((size_t)(16 * k + n) * NKV + g) * D + 16 * b;
      k0 = *(const f16x8*)kr;
      k1 = *(const f16x8*)(kr + 8);
    };
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int r = 8 * i + (l >> 3);
      u32x4 v = u32x4{0u, 0u, 0u, 0u};
      if (r < nvalid) v = *(const u32x4*)(a.vtail + ((size_t)r * NKV + g) * D + 8 * (l & 7));
      *(u32x4*)(kt + r * 128 + 16 * (l & 7)) = v;
    }
    const _Float16* v16 = (const _Float16*)kt;
    auto pv = [&](const f16x8 (&P)[kQT][2], const float (&)[kQT]) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < 4; d++)
#pragma unroll
        for (int u = 0; u < 2; u++) {
          f16x8 vop;
#pragma unroll
          for (int e = 0; e < 8; e++)
            vop[e] = v16[(32 * u + 4 * b + (e < 4 ? e : 12 + e)) * D + 16 * d + n];
#pragma unroll
          for (int t = 0; t < kQT; t++)
            O[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop, P[t][u], O[t][d], 0, 0, 0);
        }
    };
    attend(nfp8, __builtin_fmaxf(a.qscale, 1e-30f), 1.0f, first != 0, kop, pv);
  }

  // ---- the wave's partial (its own LDS: the tiles are read): O[query][dim],
  // then m and l per query
  float* po = (float*)kt;
  float* pml = po + 16 * kQT * kPsORow;
#pragma unroll
  for (int t = 0; t < kQT; t++) {
    const float L = pf_colsum(lsum[t]);
#pragma unroll
    for (int d = 0; d < 4; d++) *(f32x4*)(po + (16 * t + n) * kPsORow + 16 * d + 4 * b) = O[t][d];
    if (b == 0) *(f32x2*)(pml + 2 * (16 * t + n)) = f32x2{m[t], L};
  }
  __syncthreads();
  // ---- merge: 16 neighbouring threads take a query's 64 dims
  for (int x = tid; x < 256 * kQT; x += 64 * kW) {
    const int qi = x >> 4, d = 4 * (x & 15), s = q0 + qi;
    float mw[kW], lw[kW], M = -1e30f;
#pragma unroll
    for (int p = 0; p < kW; p++) {
      const f32x2 ml = *(const f32x2*)((const float*)(lds + p * kWB) + 16 * kQT * kPsORow + 2 * qi);
      mw[p] = ml[0];
      lw[p] = ml[1];
      M = __builtin_fmaxf(M, ml[0]);
    }
    float L = 0.f;
    f32x4 o = zero;
#pragma unroll
    for (int p = 0; p < kW; p++) {
      const float wt = __builtin_amdgcn_exp2f(mw[p] - M);
      const f32x4 op = *(const f32x4*)((const float*)(lds + p * kWB) + qi * kPsORow + d);
      L = __builtin_fmaf(lw[p], wt, L);
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = __builtin_fmaf(op[i], wt, o[i]);
    }
    if (s < a.S) {
      const float inv = 1.0f / L;
      u32x2 r;
      r[0] = (uint32_t)f2h(o[0] * inv) | ((uint32_t)f2h(o[1] * inv) << 16);
      r[1] = (uint32_t)f2h(o[2] * inv) | ((uint32_t)f2h(o[3] * inv) << 16);
      *(u32x2*)(a.out + ((size_t)s * NH + h) * D + d) = r;
    }
  }
}

}  // namespace cia

using namespace cia;

namespace {

template <bool kSlots, int kQT, int kW>
int split_launch(PrefillArgs a, const SlotArgs& sl, hipStream_t s) {
  a.nblk = (a.S + 16 * kQT - 1) / (16 * kQT);
  hipLaunchKernelGGL((k_prefill_split<kSlots, kQT, kW>), dim3(8 * GQA * a.nblk), dim3(64 * kW), 0, s,
                     a, sl);
  return launch_status();
}

// Shape: one 16-query tile per wave while those units fit the chip at once
// (the more waves on the keys, the more keys there are), or while there are
// few keys; then two, so that a K / V tile's conversions serve 32 queries.
// (1 x 4, 1 x 8, 1 x 16, 2 x 4, 2 x 8 waves, us: 77 at 0 4.8 5.2 5.5 5.5 5.5;
// 77 at 1000 8.7 7.9 7.2 11.6 8.9; 77 at 9000 33 27 25 51 34; 1000 at 0 16.8
// 20.9 32 18.5 22.4; 1500 at 0 29.5 34 53 28.9 36; 200 at 4000 25 25 27 28 20;
// 1000 at 8000 175 167 180 131 125.)
template <bool kSlots>
int split_shape(const PrefillArgs& a, const SlotArgs& sl, int tiles, hipStream_t st) {
  if (NH * ((a.S + 15) / 16) <= 256) {
    if (tiles <= 8) return split_launch<kSlots, 1, 4>(a, sl, st);
    if (tiles <= 12) return split_launch<kSlots, 1, 8>(a, sl, st);
    return split_launch<kSlots, 1, 16>(a, sl, st);
  }
  if (tiles <= 20) return split_launch<kSlots, 1, 4>(a, sl, st);
  if (tiles <= 40) return split_launch<kSlots, 2, 4>(a, sl, st);
  return split_launch<kSlots, 2, 8>(a, sl, st);
}

}  // namespace

// Whether the split kernel is the faster one for S queries after `past` keys:
// both times as measured, in us.  The split kernel's grows with the (32 query
// x 64 key) tiles of all query heads, spread over every compute unit; the
// block kernel's with the tiles of one workgroup (a heavy and a light block),
// whether or not its 8 per pair of blocks fill the chip.  (Block / split: 77
// queries at 0 11.0 / 4.0, 500 at 0 20.6 / 7.5, 2048 at 0 52 / 46, 77 at 9000
// 313 / 25, 1000 at 9000 361 / 151; 3000 at 0 70 / 96, 4096 at 0 91 / 154.)
extern "C" __attribute__((visibility("hidden"))) int cia_prefill_split_wins(int S, int past) {
  const double tiles = (past + 0.5 * S) / 64.0 + 0.5;
  const double split = 4.0 + 1.15e-3 * NH * ((S + 31) / 32) * tiles;
  const int nblk = (S + kPfQ - 1) / kPfQ, wgs = 8 * ((nblk + 1) / 2);
  const double block = 10.0 + 1.3 * ((wgs + 255) / 256) * (nblk > 1 ? 2.0 : 1.0) * tiles;
  return split < block;
}

extern "C" __attribute__((visibility("hidden"))) int cia_prefill_split(
    const uint16_t* q, const uint8_t* kc8, const uint8_t* vc8, const uint16_t* ksc,
    const uint16_t* vsc, const uint16_t* ktail, const uint16_t* vtail, int committed,
    uint16_t* out, int S, int past, float scale, void* stream) {
  const PrefillArgs a{q, kc8, vc8, ksc, vsc, ktail, vtail, committed, out, S, past,
                      scale * kPfLog2e, 0};
  return split_shape<false>(a, SlotArgs{}, (past + S + 63) / 64, (hipStream_t)stream);
}

// attention_h2o's outputs for S queries over n_live slots (arguments checked
// by cia_attention_h2o)
extern "C" __attribute__((visibility("hidden"))) int cia_h2o_out(
    const uint16_t* q, const uint8_t* kf, const uint8_t* vf, const uint16_t* ks,
    const uint16_t* vs, const int32_t* slot_pos, int n_live, uint16_t* out, int S, int past,
    float scale, void* stream) {
  const PrefillArgs a{q, kf, vf, ks, vs, nullptr, nullptr, 0, out, S, past, scale * kPfLog2e, 0};
  return split_shape<true>(a, SlotArgs{slot_pos, n_live}, (n_live + 63) / 64, (hipStream_t)stream);
}
