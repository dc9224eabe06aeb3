// gemv_int4.hip -- the attention layer's INT4 group-128 projections
// (gemv_int4, engine.cu:83-109, launched by run_gemv_int4 at 626-630 for
// q/k/v_proj at 792-797 and out_proj at 858) on gfx950.
//
// Weight format (tools/export_weights.py:64-79): packed u8 [N][K/2], k even
// in the low nibble, w = (nibble - 8) * scale[n][k/128], scales fp16.
//
// Few rows of x (decode): the launch is bound by the packed weights in HBM
// (N*K/2 bytes plus N*K/64 bytes of scales) and, at the attention layer's
// sizes (3 and 2 MiB), by latency.  One wave per weight row, 8 per
// workgroup; lane l reads 16-byte chunk l of the row (32 nibbles, k = 32l ..
// 32l+31, all inside group l/4) with one 128-bit load, so one instruction
// covers a 2048-wide row.  The workgroup stages its rows of x in LDS once
// (the weight loads are already in flight) and every lane reads its 64-byte
// slice from there; the four 16-byte pieces of a slice are rotated by
// (chunk >> 2) & 3 so that each read of a 16-lane pass hits 16 distinct
// bank groups.  A nibble pair becomes two exact fp16 values nibble - 8 by
// or-ing it under the exponent of 1024 (0x6400) and subtracting 1032;
// v_dot2_f32_f16 accumulates nibble * x in fp32, and the group scale
// multiplies each lane's 32-term sum once.  One DPP / permlane reduction per
// output.  (Measured at 3072 and 2048 rows: one row per wave beats 2, 4 or
// 8; the staged x beats per-wave x loads.)
#include "common.h"
#include "int4_shape.h"

namespace cia {

struct Int4Mat {
  const uint8_t* packed;  // [N][K/2]
  const uint16_t* scales; // [N][K/128]
  int N;
  float* y32;     // fp32 output [M][N], or null
  uint16_t* y16;  // fp16 output [M][N], or null
};

struct GemvArgs {
  const uint16_t* x;  // [M][K]
  int K, M;
  int add;   // y32 += sum instead of y32 = sum
  int rows;  // total weight rows over the matrices
  Int4Mat mat[3];  // rows of mat[1] follow those of mat[0], then mat[2]
};

constexpr int kGemvWaves = 8;
// nibbles sh..sh+3 and sh+16..sh+19 of w as fp16 (nibble - 8), exact
__device__ __forceinline__ f16x2 nib_pair(uint32_t w, int sh) {
  const uint32_t v = ((w >> sh) & 0x000F000Fu) | 0x64006400u;  // 1024 + nibble
  return __builtin_bit_cast(f16x2, v) - f16x2{(_Float16)1032.0f, (_Float16)1032.0f};
}

// The x pairs matching nib_pair(w_j, 0/4/8/12) of weight word j (k = 8j ..
// 8j+7): {x0, x4}, {x1, x5}, {x2, x6}, {x3, x7} out of the x words
// 4j..4j+3 (word i holds x[2i] low, x[2i+1] high).
__device__ __forceinline__ void x_pairs(const u32x4 (&xv)[4], f16x2 (&p)[16]) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const u32x4 X = xv[j];
    p[4 * j + 0] = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(X[2], X[0], 0x05040100u));
    p[4 * j + 1] = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(X[2], X[0], 0x07060302u));
    p[4 * j + 2] = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(X[3], X[1], 0x05040100u));
    p[4 * j + 3] = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(X[3], X[1], 0x07060302u));
  }
}

// sum over one 16-byte weight chunk of (nibble - 8) * x
__device__ __forceinline__ float chunk_dot(const u32x4& w, const f16x2 (&p)[16]) {
  float d0 = 0.0f, d1 = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    d0 = __builtin_amdgcn_fdot2(nib_pair(w[j], 0), p[4 * j + 0], d0, false);
    d1 = __builtin_amdgcn_fdot2(nib_pair(w[j], 4), p[4 * j + 1], d1, false);
    d0 = __builtin_amdgcn_fdot2(nib_pair(w[j], 8), p[4 * j + 2], d0, false);
    d1 = __builtin_amdgcn_fdot2(nib_pair(w[j], 12), p[4 * j + 3], d1, false);
  }
  return d0 + d1;
}

// LDS element offset of piece p (8 fp16) of chunk c of a staged x row
__device__ __forceinline__ int xs_off(int c, int p) { return c * 32 + 8 * ((p + (c >> 2)) & 3); }

// row of the staged block holding element e (no division: kM <= 4)
template <int kM>
__device__ __forceinline__ int stage_row(int e, int K) {
  int mm = 0;
#pragma unroll
  for (int j = 1; j < kM; j++) mm += e >= j * K ? 1 : 0;
  return mm;
}

// grid = (ceil(rows / kGemvWaves), ceil(M / kM)), block = 64 * kGemvWaves.
// kStage > 0: x rows m0..m0+kM-1 (kM * K <= kStage * 4096 elements) are
// staged in LDS; 0: every lane loads its x slices itself.
template <int kM, int kStage>
__global__ __launch_bounds__(64 * kGemvWaves) void k_gemv_int4(GemvArgs a) {
  constexpr int kPer = 8 * 64 * kGemvWaves;  // elements staged per pass
  // (+8: the drop slot of the stores past the block)
  __shared__ __attribute__((aligned(16))) uint16_t xs[kStage > 0 ? kStage * kPer + 8 : 8];
  const int l = threadIdx.x & 63;
  const int row = blockIdx.x * kGemvWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.y * kM;
  const int K = a.K, nch = K >> 5, ng = K >> 7;
  // this wave's row (uniform): matrix and local row; waves past the last
  // row read it again and write nothing
  int n = row < a.rows ? row : a.rows - 1, mi = 0;
  if (n >= a.mat[0].N) {
    n -= a.mat[0].N;
    mi = 1;
    if (n >= a.mat[1].N) {
      n -= a.mat[1].N;
      mi = 2;
    }
  }
  const uint8_t* packed = mi == 0 ? a.mat[0].packed : (mi == 1 ? a.mat[1].packed : a.mat[2].packed);
  const uint16_t* scales = mi == 0 ? a.mat[0].scales : (mi == 1 ? a.mat[1].scales : a.mat[2].scales);
  const uint8_t* wp = packed + (size_t)n * (K >> 1);
  const uint16_t* sp = scales + (size_t)n * ng;
  // Loads, all branch-free so that each wait counts exactly: x first
  // (elements past the block load element 0 and are dropped), then this
  // lane's first weight chunk and its scale (lanes past the row's last
  // chunk load that chunk and discard it).  The LDS stores wait only for
  // the x loads, and the barrier only for the LDS stores.
  u32x4 st[kStage > 0 ? kStage : 1];
  if constexpr (kStage > 0) {
#pragma unroll
    for (int i = 0; i < kStage; i++) {
      int e = i * kPer + (int)threadIdx.x * 8;
      e = e < kM * K ? e : 0;
      const int mm = stage_row<kM>(e, K);
      const int src = m0 + mm < a.M ? m0 + mm : a.M - 1;
      st[i] = *(const u32x4*)(a.x + (size_t)src * K + (e - mm * K));
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  const int c0 = l < nch ? l : nch - 1;
  u32x4 wv = *(const u32x4*)(wp + 16 * c0);
  uint32_t sv = sp[c0 >> 2];  // (32-bit holder: no early wait)
  float* y32 = mi == 0 ? a.mat[0].y32 : (mi == 1 ? a.mat[1].y32 : a.mat[2].y32);
  uint16_t* y16 = mi == 0 ? a.mat[0].y16 : (mi == 1 ? a.mat[1].y16 : a.mat[2].y16);
  const int N = mi == 0 ? a.mat[0].N : (mi == 1 ? a.mat[1].N : a.mat[2].N);
  // the residual (add): fetched with the weights, so the epilogue does not
  // wait a round trip for it (the wave's lanes share the address; without
  // add, a harmless read of x[0])
  float yold[kM];
#pragma unroll
  for (int m = 0; m < kM; m++) {
    const int mm = m0 + m < a.M ? m0 + m : a.M - 1;
    const float* ysrc = a.add && y32 ? y32 + (size_t)mm * N + n : (const float*)a.x;
    yold[m] = *ysrc;
  }
  if constexpr (kStage > 0) {
#pragma unroll
    for (int i = 0; i < kStage; i++) {
      const int e = i * kPer + (int)threadIdx.x * 8;
      const int mm = stage_row<kM>(e, K), k = e - mm * K;
      *(u32x4*)(xs + (e < kM * K ? mm * K + xs_off(k >> 5, (k >> 3) & 3) : kStage * kPer)) = st[i];
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS stores
    __builtin_amdgcn_s_barrier();
  }
  float acc[kM];
#pragma unroll
  for (int m = 0; m < kM; m++) acc[m] = 0.0f;
  for (int c = l; c < nch; c += 64) {
    if (c != l) {
      wv = *(const u32x4*)(wp + 16 * c);
      sv = sp[c >> 2];
    }
#pragma unroll
    for (int m = 0; m < kM; m++) {
      u32x4 xv[4];
      if constexpr (kStage > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) xv[i] = *(const u32x4*)(xs + m * K + xs_off(c, i));
      } else {
        const uint16_t* xr = a.x + (size_t)(m0 + m < a.M ? m0 + m : a.M - 1) * K + 32 * c;
#pragma unroll
        for (int i = 0; i < 4; i++) xv[i] = *(const u32x4*)(xr + 8 * i);
      }
      f16x2 p[16];
      x_pairs(xv, p);
      acc[m] = __builtin_fmaf(chunk_dot(wv, p), h2f((uint16_t)sv), acc[m]);
    }
  }
#pragma unroll
  for (int m = 0; m < kM; m++) {
    const float v = wave_sum_fast(acc[m]);
    if (l == 0 && row < a.rows && m0 + m < a.M) {
      const size_t o = (size_t)(m0 + m) * N + n;
      if (y32) y32[o] = a.add ? yold[m] + v : v;
      if (y16) y16[o] = f2h(v);
    }
  }
}

// ---------------------------------------------------------------- GEMM
// Many rows of x (prefill): Y = X W^T on the fp16 matrix cores
// (v_mfma_f32_16x16x32_f16).  A workgroup computes a 128 (x rows) x 128
// (weight rows) tile with 8 waves (two per SIMD, so one wave's matrix
// products overlap another's dequantisation) in a 2 x 4 grid of 64 x 32
// wave tiles (4 x 2 MFMA tiles).  The K loop runs over the 128-wide scale groups: the
// products of one group accumulate from zero on the matrix cores and are
// then added with the group scale of their column in fp32, so the weights
// enter the MFMA as exact fp16 (nibble - 8) values.
//   Inside a group the k order of the four 32-k MFMA steps is permuted the
//   same way for both operands: lane group q = l >> 4 holds k = 32q + 8s ..
//   32q + 8s + 7 at step s, so one 16-byte read per lane and column tile
//   brings the nibbles of all four steps (word s is step s).
//   Operands reach LDS by DMA (global_load_lds_dwordx4: lane i's 16 bytes
//   land at the instruction's LDS base + 16 i, so the swizzles are made by
//   choosing which global chunk each lane fetches), in a ring of 3 slots
//   filled two groups ahead: per group one wait for the group's own DMA,
//   one barrier, and no staging registers.
//     X slot: 128 rows x 16 chunks; row r's chunk c at c ^ xsw(r).  A
//       16-byte read is served 32 lanes (512 bytes of banks) at a time:
//       lanes 16q + n (q = 0, 1 or 2, 3) read row n's chunks 4q + s, and
//       two rows of one parity share a 512-byte bank window, so xsw maps
//       the 8 rows of a parity to distinct offsets whose bit 2 is the
//       parity: chunk 4q + s of one q and of the other never land on one
//       bank (and the 16 rows of a read take 16 distinct offsets).
//     W slot: 128 columns x 4 chunks of nibbles; column c's chunk q at
//       q ^ ((c >> 2) & 3) (16 consecutive columns hit distinct banks).
//     scale slot: the 128 columns' fp16 scales of the group, one per dword
//       (a 2-byte LDS DMA writes each lane's value zero-extended to a dword).
constexpr int kTile = 128;
constexpr int kRing = 3;
constexpr int kGemmWaves = 8;
constexpr int kXSlot = kTile * 256;            // bytes: 128 rows x 128 fp16
constexpr int kWSlot = kTile * 64;             // bytes: 128 columns x 128 nibbles
constexpr int kSSlot = 2 * kTile * 4;          // bytes: 128 scale dwords + a drop area
constexpr int kSlot = kXSlot + kWSlot + kSSlot;

typedef __attribute__((address_space(3))) void lds_void_t;

// X slot chunk swizzle of row r: bits 1-2 of r to bits 0-1, bit 0 to bit 2,
// bit 3 stays
__device__ __forceinline__ int xsw(int r) { return ((r >> 1) & 3) | ((r & 1) << 2) | (r & 8); }
typedef __attribute__((address_space(1))) void gbl_void_t;

// 8 nibbles (one u32, k even in the low nibble) -> 8 fp16 (nibble - 8), in k order
__device__ __forceinline__ f16x8 nib8(uint32_t u) {
  const uint32_t x = u & 0x0F0F0F0Fu, y = (u >> 4) & 0x0F0F0F0Fu;
  const f16x2 off = f16x2{(_Float16)1032.0f, (_Float16)1032.0f};
  f16x8 r;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    // {lo_b, hi_b} as 16-bit values, then under the exponent of 1024
    const uint32_t sel = 0x0C000C00u | (uint32_t)(4 + b) << 16 | (uint32_t)b;
    const f16x2 h =
        __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(y, x, sel) | 0x64006400u) - off;
    r[2 * b] = h[0];
    r[2 * b + 1] = h[1];
  }
  return r;
}

// A pointer of the kernel arguments as a scalar value.  (Left visible, the
// per-column choice between the three matrices' pointers below becomes a
// choice of address and one vector load from the argument segment: a memory
// round trip before the first operand load and another before the outputs.)
template <class T>
__device__ __forceinline__ T* arg_ptr(T* p) {
  uint64_t v = (uint64_t)p;
  asm("" : "+s"(v));
  return (T*)v;
}
template <class T>
__device__ __forceinline__ T* pick(int mi, T* p0, T* p1, T* p2) {
  T *a = arg_ptr(p0), *b = arg_ptr(p1), *c = arg_ptr(p2);
  return mi == 0 ? a : (mi == 1 ? b : c);
}

// global column col (clamped) across the up to 3 matrices: matrix, row of it
struct ColRef {
  int mi, n;
};
__device__ __forceinline__ ColRef col_ref(const GemvArgs& a, int col) {
  const int c = col < a.rows ? col : a.rows - 1, n0 = a.mat[0].N, n1 = n0 + a.mat[1].N;
  const int mi = c >= n1 ? 2 : (c >= n0 ? 1 : 0);
  return ColRef{mi, c - (mi == 2 ? n1 : (mi == 1 ? n0 : 0))};
}
__device__ __forceinline__ const uint8_t* col_packed(const GemvArgs& a, ColRef c, int K) {
  return pick(c.mi, a.mat[0].packed, a.mat[1].packed, a.mat[2].packed) + (size_t)c.n * (K >> 1);
}
__device__ __forceinline__ const uint16_t* col_scales(const GemvArgs& a, ColRef c, int K) {
  return pick(c.mi, a.mat[0].scales, a.mat[1].scales, a.mat[2].scales) + (size_t)c.n * (K >> 7);
}

// What a launch does with its sums: store them (fp32), add them to y (fp32:
// out_proj into the residual), or store them as fp16 (q/k/v).
enum GemmOut { kOutF32, kOutAdd, kOutF16 };

// The output column of a lane: rows m of it at p + m * N
template <int kOut>
struct OutCol {
  float* y32;
  uint16_t* y16;
  int N;
  __device__ __forceinline__ OutCol(const GemvArgs& a, int col) {
    const ColRef c = col_ref(a, col);
    N = c.mi == 0 ? a.mat[0].N : (c.mi == 1 ? a.mat[1].N : a.mat[2].N);
    if constexpr (kOut == kOutF16)
      y16 = pick(c.mi, a.mat[0].y16, a.mat[1].y16, a.mat[2].y16) + c.n;
    else
      y32 = pick(c.mi, a.mat[0].y32, a.mat[1].y32, a.mat[2].y32) + c.n;
  }
  // the residual at row m (read ahead of the sums, so the reads of a lane's
  // rows are in flight together)
  __device__ __forceinline__ float old(int m) const {
    if constexpr (kOut == kOutAdd) return y32[(size_t)m * N];
    return 0.f;
  }
  __device__ __forceinline__ void put(int m, float v, float yold) const {
    if constexpr (kOut == kOutF16)
      y16[(size_t)m * N] = f2h(v);
    else
      y32[(size_t)m * N] = kOut == kOutAdd ? yold + v : v;
  }
};

// grid = (ceil(rows / 128), ceil(M / 128)), block = 64 * kGemmWaves.
// (Giving each XCD a contiguous run of tiles, so its L2 sees a few row
// blocks of X rather than all, measured no faster.)
template <int kOut>
__global__ __launch_bounds__(64 * kGemmWaves) void k_gemm_int4(GemvArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[kRing * kSlot];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int wm = w >> 2, wn = w & 3, n16 = l & 15, q = l >> 4;
  const int m0 = blockIdx.y * kTile, r0 = blockIdx.x * kTile;
  const int K = a.K, ng = K >> 7;
  // DMA sources of this lane (fixed across groups; + 256 g bytes for X,
  // + 64 g for W, + 2 g for the scales)
  //   X: instruction t of wave w fills rows 4 (4w + t) .. +3; lane l takes
  //      row 4 (4w + t) + (l >> 4), physical chunk l & 15
  const uint8_t* xsrc[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int r = 4 * (4 * w + t) + (l >> 4), m = m0 + r;
    const int lc = (l & 15) ^ xsw(r);
    xsrc[t] = (const uint8_t*)(a.x + (size_t)(m < a.M ? m : a.M - 1) * K) + 16 * lc;
  }
  //   W: wave w fills columns 16 w .. +15; lane l takes column 16 w + (l >> 2),
  //      physical chunk l & 3
  const int wcol = 16 * w + (l >> 2);
  const uint8_t* wsrc = col_packed(a, col_ref(a, r0 + wcol), K) + 16 * ((l & 3) ^ ((wcol >> 2) & 3));
  //   scales: waves 0, 1 fill columns 64 w + l; the others the drop area
  const uint16_t* ssrc = col_scales(a, col_ref(a, r0 + 64 * (w & 1) + l), K);
  const int sdst = kXSlot + kWSlot + (w < 2 ? 256 * w : 512);
  auto issue = [&](int g) {
    uint8_t* slot = ring + (g % kRing) * kSlot;
    const int gg = g < ng ? g : ng - 1;  // past the end: a harmless refetch
#pragma unroll
    for (int t = 0; t < 4; t++)
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(xsrc[t] + 256 * gg),
                                       (lds_void_t*)(slot + (4 * w + t) * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((gbl_void_t*)(wsrc + 64 * gg),
                                     (lds_void_t*)(slot + kXSlot + w * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((gbl_void_t*)(ssrc + gg), (lds_void_t*)(slot + sdst), 2, 0,
                                     0);
  };
  f32x4 C[4][2];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) C[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  issue(0);
  issue(1);
  for (int g = 0; g < ng; g++) {
    // this group's 6 DMAs are done once at most the next group's 6 remain
    __builtin_amdgcn_s_waitcnt(0x0F76);  // vmcnt(6)
    __builtin_amdgcn_s_barrier();        // every wave's DMA landed; slot g-1 is free
    issue(g + 2);
    const uint8_t* slot = ring + (g % kRing) * kSlot;
    const uint16_t* xs = (const uint16_t*)slot;
    const uint8_t* ws = slot + kXSlot;
    const uint32_t* ss = (const uint32_t*)(slot + kXSlot + kWSlot);
    u32x4 wq[2];
    float scl[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int c = 32 * wn + 16 * j + n16;
      wq[j] = *(const u32x4*)(ws + c * 64 + 16 * (q ^ ((c >> 2) & 3)));
      scl[j] = h2f((uint16_t)ss[c]);
    }
    f32x4 P[4][2];
#pragma unroll
    for (int s2 = 0; s2 < 4; s2++) {
      f16x8 A[4], B[2];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = 64 * wm + 16 * i + n16;
        A[i] = *(const f16x8*)(xs + r * 128 + 8 * ((4 * q + s2) ^ xsw(n16)));
      }
#pragma unroll
      for (int j = 0; j < 2; j++) B[j] = nib8(wq[j][s2]);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          P[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              A[i], B[j], s2 == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : P[i][j], 0, 0, 0);
    }
    // C += P * scale of the column (the lane's column is n16 of tile j)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) C[i][j][e] = __builtin_fmaf(P[i][j][e], scl[j], C[i][j][e]);
  }
  // outputs: lane holds rows 4q + e of tile i, column n16 of tile j; the
  // residual of a column's 16 rows is read before the first is stored
  // (rows past M read the last one)
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int col = r0 + 32 * wn + 16 * j + n16;
    const OutCol<kOut> o(a, col);
    float yo[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int m = m0 + 64 * wm + 16 * i + 4 * q + e;
        yo[i][e] = o.old(m < a.M ? m : a.M - 1);
      }
    if (col < a.rows) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int m = m0 + 64 * wm + 16 * i + 4 * q + e;
          if (m < a.M) o.put(m, C[i][j][e], yo[i][e]);
        }
    }
  }
  // (the last two DMAs refetch the final group into free slots; let them
  // land before the workgroup's LDS is released)
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
}

// ---------------------------------------------------------------- large tiles
// The tile kernel's group step is bound by vector work and LDS reads as much as
// by its products: a wave dequantises 32 columns for 64 rows.  Here a wave has
// 128 rows x (16 kNT) columns of a 256 x (64 kNT) workgroup tile, so a
// dequantised operand serves twice the rows, and the columns' scales come from
// an LDS table filled once (fetched per group, 8 waves x 64 two-byte loads in
// different rows cost the step 500 cycles of address work).  Two slots: the
// next group's DMA goes out after the barrier that ends the last group and has
// the whole step to land.  Layouts, the order of k and the sums are the tile
// kernel's: the same bits.  K up to 2048 (the LDS).
// (q/k/v of 4096 rows, kNT = 3, one round of 256 workgroups: 77 us in 128 x 128
// tiles, 55 so, 930 TFLOP/s; out_proj into the residual, kNT = 2: 69, 51.)
constexpr int kBigRows = 256;

// grid = the tiles, ceil(rows / (64 kNT)) * ceil(M / 256), up to a multiple of 8;
// block = 512
template <int kOut, int kNT>
__global__ __launch_bounds__(64 * kGemmWaves) void k_gemm_int4_big(GemvArgs a) {
  constexpr int kCols = 64 * kNT, kXB = kBigRows * 256, kWB = kCols * 64, kSlotB = kXB + kWB;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kSlotB + (kBigMaxK / 128) * kCols * 2];
  const int tid = threadIdx.x, l = tid & 63, n16 = l & 15, q = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w >> 2, wn = w & 3;
  // Workgroups go to the 8 XCDs in turn: XCD x takes the tiles x gridDim.x / 8
  // on, row tiles slowest, so that its L2 sees a few row blocks of x and not
  // all of it.
  const int nct = (a.rows + kCols - 1) / kCols;
  const int tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int m0 = tile / nct * kBigRows, r0 = tile % nct * kCols;
  if (m0 >= a.M) return;
  const int K = a.K, ng = K >> 7;
  uint16_t* ssc = (uint16_t*)(lds + 2 * kSlotB);  // [group][column]
  // DMA sources: X instruction t of wave w fills rows 4 (8w + t) .. + 3, as the
  // tile kernel's; W instruction u columns 16 u .. + 15, u = w and w + 8
  const uint8_t* xsrc[8];
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const int r = 4 * (8 * w + t) + (l >> 4), m = m0 + r;
    xsrc[t] = (const uint8_t*)(a.x + (size_t)(m < a.M ? m : a.M - 1) * K) + 16 * ((l & 15) ^ xsw(r));
  }
  const uint8_t* wsrc[2];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int c = 16 * (w + 8 * t) + (l >> 2);
    wsrc[t] = col_packed(a, col_ref(a, r0 + (c < kCols ? c : 0)), K) + 16 * ((l & 3) ^ ((c >> 2) & 3));
  }
  auto issue = [&](int g) __attribute__((always_inline)) {
    uint8_t* slot = lds + (g & 1) * kSlotB;
#pragma unroll
    for (int t = 0; t < 8; t++)
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(xsrc[t] + 256 * g),
                                       (lds_void_t*)(slot + (8 * w + t) * 1024), 16, 0, 0);
#pragma unroll
    for (int t = 0; t < 2; t++)
      if (w + 8 * t < 4 * kNT)
        __builtin_amdgcn_global_load_lds((gbl_void_t*)(wsrc[t] + 64 * g),
                                         (lds_void_t*)(slot + kXB + (w + 8 * t) * 1024), 16, 0, 0);
  };
  issue(0);
  // 16 neighbouring threads read a column's scales
#pragma unroll
  for (int e0 = 0; e0 < 16 * kCols; e0 += 64 * kGemmWaves) {
    const int c = (e0 + tid) >> 4, g = tid & 15;
    if (g < ng) ssc[g * kCols + c] = col_scales(a, col_ref(a, r0 + c), K)[g];
  }
  f32x4 C[8][kNT];
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < kNT; j++) C[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int g = 0; g < ng; g++) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): this wave's DMA (and scales) landed
    __builtin_amdgcn_s_barrier();        // every wave's did; the other slot is read
    asm volatile("" ::: "memory");
    if (g + 1 < ng) issue(g + 1);
    const uint8_t* slot = lds + (g & 1) * kSlotB;
    const uint16_t* xs = (const uint16_t*)slot + (128 * wm + n16) * 128;
    // Units of two row tiles x two k steps, in order: a unit's x operands are
    // requested before the products of the unit before it, and the columns of
    // its k steps are dequantised where the row tiles first need them.
    f16x8 A[2][4];
    auto load_a = [&](int u, f16x8 (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int s = 0; s < 2; s++)
          o[2 * i + s] = *(const f16x8*)(xs + 16 * (2 * (u >> 1) + i) * 128 +
                                         8 * ((4 * q + 2 * (u & 1) + s) ^ xsw(n16)));
    };
    u32x4 wq[kNT];
    float scl[kNT];
#pragma unroll
    for (int j = 0; j < kNT; j++) {
      const int c = 16 * (kNT * wn + j) + n16;
      wq[j] = *(const u32x4*)(slot + kXB + c * 64 + 16 * (q ^ ((c >> 2) & 3)));
      scl[j] = h2f(ssc[g * kCols + c]);
    }
    load_a(0, A[0]);
    f16x8 B[kNT][4];
    f32x4 P[2][2][kNT];  // of a pair of row tiles, and of the pair before
    auto scale_add = [&](int pr) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < kNT; j++)
#pragma unroll
          for (int e = 0; e < 4; e++)
            C[2 * pr + i][j][e] = __builtin_fmaf(P[pr & 1][i][j][e], scl[j], C[2 * pr + i][j][e]);
    };
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (u + 1 < 8) load_a(u + 1, A[(u + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const int s0 = 2 * (u & 1), pr = u >> 1;
      if (u < 2)
#pragma unroll
        for (int j = 0; j < kNT; j++) {
          B[j][s0] = nib8(wq[j][s0]);
          B[j][s0 + 1] = nib8(wq[j][s0 + 1]);
        }
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < kNT; j++)
            P[pr & 1][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                A[u & 1][2 * i + s], B[j][s0 + s], s0 + s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : P[pr & 1][i][j], 0, 0, 0);
      // the pair before is scaled between this pair's first products
      if (pr > 0 && (u & 1) == 0) {
        scale_add(pr - 1);
#pragma unroll
        for (int k = 0; k < 4 * kNT; k++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two vector instructions
        }
      }
    }
    scale_add(3);
  }
  // outputs, as the tile kernel's, a column's 32 rows at a time
#pragma unroll
  for (int j = 0; j < kNT; j++) {
    const int col = r0 + 16 * (kNT * wn + j) + n16;
    const OutCol<kOut> o(a, col);
    float yo[8][4];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int m = m0 + 128 * wm + 16 * i + 4 * q + e;
        yo[i][e] = o.old(m < a.M ? m : a.M - 1);
      }
    if (col < a.rows) {
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int m = m0 + 128 * wm + 16 * i + 4 * q + e;
          if (m < a.M) o.put(m, C[i][j][e], yo[i][e]);
        }
    }
  }
}

// ---------------------------------------------------------------- K-split GEMM
// A few to some hundred rows of x (short prompts, chat turns): too few
// 128 x 128 tiles to fill the chip, and each tile's 16 scale groups a serial
// chain.  Here a workgroup computes a (16 kMT) x (16 kNT) tile with 8 waves
// that split K: wave w takes the scale groups w, w + 8, .. (two of them at
// K = 2048), alone, with no barrier before a pass ends.
//   A lane's 16-byte loads reach 64 bytes a clock only when 4 neighbouring
//   lanes read 64 contiguous bytes (measured: 256 KB into one compute unit in
//   1.2 us; in the MFMA operand's own order, neighbouring lanes in different
//   rows, 6.2 us), so both operands are fetched 4 lanes to a row's 64 bytes
//   and change lanes afterwards:
//     x     by DMA into the wave's own LDS: instruction (i, q) brings the k =
//           32q .. 32q + 31 of row tile i's 16 rows, row r's 16-byte piece s
//           at s ^ (r >> 2) ^ (q & 1), so that the 16 rows of an operand read
//           take distinct banks.  Read back as whole operands, after which
//           the next group's DMA goes out, ahead of this group's products;
//     W     into registers, then to operand order by ds_bpermute.
//   The scales of the tile's columns are fetched once, group-fastest as they
//   lie in memory, into an LDS table.
// As in the tile kernel, a group's products accumulate from zero and are added
// in fp32 with the column's scale: the 8 waves' products of a pass of 8 groups
// meet in LDS unscaled.  From kChainsM rows on they are added in the order of
// the groups, so that an output has the tile kernel's bits, whatever the shape
// -- a q/k/v sum in another order may round to another fp16 value and that one
// to another E4M3 code in the cache.  Fewer rows, which the GEMV would take,
// are added in four chains a pass: the GEMV's sums are trees, and 16 roundings
// in a row are further off (out_proj into the residual, 2-norm from 64 bits:
// GEMV 7.2e-8, in order 7.65e-8, so 6.3e-8).
// (Two passes at K = 2048.  out_proj of 300 rows: 28.0 us in 128 x 128 tiles,
// 10.8 so; 23 rows of q/k/v: 13.2 by the GEMV, 5.1 so.)
constexpr int kKsWaves = 8;

// grid = (ceil(rows / (16 kNT)), ceil(M / (16 kMT))), block = 512; K <= kKsMaxK
template <int kOut, int kMT, int kNT, bool kChains>
__global__ __launch_bounds__(64 * kKsWaves) void k_gemm_int4_ks(GemvArgs a) {
  static_assert(kNT <= 4, "a wave's partial tile takes its x slot's place");
  __shared__ __attribute__((aligned(16))) uint8_t xs[kKsWaves * kMT * 4096];
  __shared__ float ssc[kKsMaxK / 128][16 * kNT];
  const int tid = threadIdx.x, l = tid & 63, n16 = l & 15, q = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.y * 16 * kMT, r0 = blockIdx.x * 16 * kNT;
  const int K = a.K, ng = K >> 7;
  uint8_t* xw = xs + w * kMT * 4096;
  const uint8_t* wp[kNT];
#pragma unroll
  for (int j = 0; j < kNT; j++)
    wp[j] = col_packed(a, col_ref(a, r0 + 16 * j + (l >> 2)), K) + 16 * (l & 3);
  const uint8_t* xp[kMT][2];  // the row's 64-byte pieces of even and odd q
#pragma unroll
  for (int i = 0; i < kMT; i++) {
    const int r = l >> 2, m = m0 + 16 * i + r;
    const uint8_t* row = (const uint8_t*)(a.x + (size_t)(m < a.M ? m : a.M - 1) * K);
    xp[i][0] = row + 16 * ((l & 3) ^ (r >> 2));
    xp[i][1] = row + 16 * ((l & 3) ^ (r >> 2) ^ 1);
  }
  u32x4 wq[kNT], wn[kNT];
  auto load_w = [&](int g, u32x4 (&o)[kNT]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kNT; j++) o[j] = *(const u32x4*)(wp[j] + 64 * (size_t)g);
  };
  auto load_x = [&](int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMT; i++)
#pragma unroll
      for (int c = 0; c < 4; c++)
        __builtin_amdgcn_global_load_lds((gbl_void_t*)(xp[i][c & 1] + 256 * (size_t)g + 64 * c),
                                         (lds_void_t*)(xw + (4 * i + c) * 1024), 16, 0, 0);
  };
  const int gf = w < ng ? w : 0;
  load_w(gf, wq);
  // the output tiles this wave adds up at the end (w, w + 8, ..): their
  // residual goes out with the operands
  constexpr int kTiles = kMT * kNT, kPer = (kTiles + kKsWaves - 1) / kKsWaves;
  float yo[kPer][4] = {};
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int t = w + kKsWaves * u;
    if (kOut != kOutAdd || t >= kTiles) break;
    const OutCol<kOut> o(a, r0 + 16 * (t % kNT) + n16);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int m = m0 + 16 * (t / kNT) + 4 * q + e;
      yo[u][e] = o.old(m < a.M ? m : a.M - 1);
    }
  }
  load_x(gf);
  // the scale table: 16 neighbouring threads read a column's 16 groups
  for (int g0 = 0; g0 < ng; g0 += 16)
#pragma unroll
    for (int e = tid; e < 256 * kNT; e += 64 * kKsWaves) {
      const int c = e >> 4, g = g0 + (e & 15);
      if (g < ng) ssc[g][c] = h2f(col_scales(a, col_ref(a, r0 + c), K)[g]);
    }
  // The products of this wave's groups, not scaled: of two passes, so that the
  // second's x can take the slot while the first's are in work, where they fit
  // beside the operands (2 x 3 in 128 registers, two workgroups to a compute
  // unit, and 4 x 4 in 256 do not: there x is fetched once a pass has met)
  constexpr bool kEarly = kMT * kNT <= 4 || (kMT == 4 && kNT == 3);
  f32x4 P[kEarly ? 2 : 1][kMT][kNT];
  __syncthreads();  // the scale table is in
  auto step = [&](int g, bool more, const u32x4 (&cur)[kNT], u32x4 (&nxt)[kNT], f32x4 (&Pg)[kMT][kNT]) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this group's x and W
    // lane (n16, q)'s chunk q of column n16 was loaded by lane 4 n16 + q
    u32x4 wt[kNT];
#pragma unroll
    for (int j = 0; j < kNT; j++)
#pragma unroll
      for (int s = 0; s < 4; s++)
        wt[j][s] = (uint32_t)__builtin_amdgcn_ds_bpermute(16 * n16 + 4 * q, (int)cur[j][s]);
    // two k steps at a time: the registers hold two passes' products
#pragma unroll
    for (int s0 = 0; s0 < 4; s0 += 2) {
      f16x8 A[kMT][2];
#pragma unroll
      for (int i = 0; i < kMT; i++)
#pragma unroll
        for (int s = 0; s < 2; s++)
          A[i][s] = *(const f16x8*)(xw + (4 * i + q) * 1024 + 64 * n16 + 16 * ((s0 + s) ^ (n16 >> 2) ^ (q & 1)));
      if (s0 == 2 && more) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot is read
        __builtin_amdgcn_sched_barrier(0);
        load_w(g + kKsWaves, nxt);
        load_x(g + kKsWaves);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < kNT; j++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const f16x8 B = nib8(wt[j][s0 + s]);
#pragma unroll
          for (int i = 0; i < kMT; i++)
            Pg[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                A[i][s], B, s0 + s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : Pg[i][j], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  f32x4 v[kPer];
#pragma unroll
  for (int u = 0; u < kPer; u++) v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4* part = (f32x4*)xs;  // [wave, 256 kMT apart][tile][lane] of 4 rows x 1 column
  // a pass's products meet: the tiles this wave adds up take its groups, from
  // g0, in order (kChains: in four chains); lane holds rows 4q .. 4q + 3 of
  // column n16
  auto meet = [&](int g0, const f32x4 (&Pg)[kMT][kNT]) __attribute__((always_inline)) {
    if (g0 + w < ng)
#pragma unroll
      for (int i = 0; i < kMT; i++)
#pragma unroll
        for (int j = 0; j < kNT; j++) part[w * kMT * 256 + (i * kNT + j) * 64 + l] = Pg[i][j];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; u++) {
      const int t = w + kKsWaves * u < kTiles ? w + kKsWaves * u : 0;
      if constexpr (kChains) {
        f32x4 c[4] = {};
#pragma unroll
        for (int k = 0; k < kKsWaves; k++) {
          if (g0 + k >= ng) break;
          const f32x4 pv = part[k * kMT * 256 + t * 64 + l];
          const float sc = ssc[g0 + k][16 * (t % kNT) + n16];
#pragma unroll
          for (int e = 0; e < 4; e++) c[k & 3][e] = __builtin_fmaf(pv[e], sc, c[k & 3][e]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) v[u][e] += (c[0][e] + c[1][e]) + (c[2][e] + c[3][e]);
        continue;
      }
#pragma unroll
      for (int k = 0; k < kKsWaves; k++) {
        if (g0 + k >= ng) break;
        const f32x4 pv = part[k * kMT * 256 + t * 64 + l];
        const float sc = ssc[g0 + k][16 * (t % kNT) + n16];
#pragma unroll
        for (int e = 0; e < 4; e++) v[u][e] = __builtin_fmaf(pv[e], sc, v[u][e]);
      }
    }
  };
  if constexpr (kEarly) {
    for (int g0 = 0; g0 < ng; g0 += 2 * kKsWaves) {
      const int g = g0 + w;
      if (g0 > 0) {
        __syncthreads();  // the last pass is read
        if (g < ng) {
          load_w(g, wq);
          load_x(g);
        }
      }
      if (g < ng) step(g, g + kKsWaves < ng, wq, wn, P[0]);
      if (g + kKsWaves < ng) step(g + kKsWaves, false, wn, wq, P[1]);
      meet(g0, P[0]);
      if (g0 + kKsWaves < ng) {
        __syncthreads();
        meet(g0 + kKsWaves, P[1]);
      }
    }
  } else {
    for (int g0 = 0; g0 < ng; g0 += kKsWaves) {
      const int g = g0 + w;
      if (g0 > 0) {
        __syncthreads();  // the last pass is read
        if (g < ng) load_x(g);
      }
      if (g < ng) step(g, false, wq, wn, P[0]);
      if (g + kKsWaves < ng) load_w(g + kKsWaves, wq);
      meet(g0, P[0]);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // (a wave without groups: its fetch done)
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int t = w + kKsWaves * u;
    if (t >= kTiles) break;
    const int col = r0 + 16 * (t % kNT) + n16;
    const OutCol<kOut> o(a, col);
    if (col < a.rows) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int m = m0 + 16 * (t / kNT) + 4 * q + e;
        if (m < a.M) o.put(m, v[u][e], yo[u][e]);
      }
    }
  }
}

template <int kOut, int kMT, int kNT>
static void ks_launch(const GemvArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.rows + 16 * kNT - 1) / (16 * kNT)),
                  (unsigned)((a.M + 16 * kMT - 1) / (16 * kMT)));
  if (a.M < kChainsM)
    hipLaunchKernelGGL((k_gemm_int4_ks<kOut, kMT, kNT, true>), grid, dim3(64 * kKsWaves), 0, s, a);
  else
    hipLaunchKernelGGL((k_gemm_int4_ks<kOut, kMT, kNT, false>), grid, dim3(64 * kKsWaves), 0, s, a);
}

template <int kOut, int kNT>
static void big_launch(const GemvArgs& a, long tiles, hipStream_t s) {
  hipLaunchKernelGGL((k_gemm_int4_big<kOut, kNT>), dim3((unsigned)((tiles + 7) / 8 * 8)),
                     dim3(64 * kGemmWaves), 0, s, a);
}

// the matrix-core kernels, by the launch's output form
template <int kOut>
static void gemm_launch(const GemvArgs& a, hipStream_t s) {
  const Int4Shape& sh = kInt4Shapes[int4_shape(a.M, a.rows, a.K)];
  switch (1000 * sh.xrows + sh.cols) {
    case 16016: return ks_launch<kOut, 1, 1>(a, s);
    case 16032: return ks_launch<kOut, 1, 2>(a, s);
    case 32032: return ks_launch<kOut, 2, 2>(a, s);
    case 32048: return ks_launch<kOut, 2, 3>(a, s);
    case 64048: return ks_launch<kOut, 4, 3>(a, s);
    case 64064: return ks_launch<kOut, 4, 4>(a, s);
    case 256128: return big_launch<kOut, 2>(a, int4_tiles(sh, a.M, a.rows), s);
    case 256192: return big_launch<kOut, 3>(a, int4_tiles(sh, a.M, a.rows), s);
  }
  hipLaunchKernelGGL(k_gemm_int4<kOut>, dim3((unsigned)((a.rows + kTile - 1) / kTile),
                     (unsigned)((a.M + kTile - 1) / kTile)), dim3(64 * kGemmWaves), 0, s, a);
}

template <int kM>
static void gemv_launch(const GemvArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.rows + kGemvWaves - 1) / kGemvWaves),
                  (unsigned)((a.M + kM - 1) / kM));
  const dim3 block(64 * kGemvWaves);
  const int per = 8 * 64 * kGemvWaves, need = (kM * a.K + per - 1) / per;
  if (need <= 1)
    hipLaunchKernelGGL((k_gemv_int4<kM, 1>), grid, block, 0, s, a);
  else if (need <= 2)
    hipLaunchKernelGGL((k_gemv_int4<kM, 2>), grid, block, 0, s, a);
  else if (need <= 4)
    hipLaunchKernelGGL((k_gemv_int4<kM, 4>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_gemv_int4<kM, 0>), grid, block, 0, s, a);
}

static int gemv_run(GemvArgs& a, void* stream) {
  a.rows = a.mat[0].N + a.mat[1].N + a.mat[2].N;
  hipStream_t s = (hipStream_t)stream;
  if (!int4_gemv(a.M, a.rows, a.K, a.add)) {
    if (a.mat[0].y16)
      gemm_launch<kOutF16>(a, s);
    else if (a.add)
      gemm_launch<kOutAdd>(a, s);
    else
      gemm_launch<kOutF32>(a, s);
  } else if (a.M == 1)
    gemv_launch<1>(a, s);
  else if (a.M == 2)
    gemv_launch<2>(a, s);
  else
    gemv_launch<4>(a, s);
  return launch_status();
}

static bool mat_ok(const uint8_t* packed, const uint16_t* scales) {
  return aligned(packed, 16) && aligned(scales, 2);
}

}  // namespace cia

using namespace cia;

static int gemv_common(const uint16_t* x, const uint8_t* packed, const uint16_t* scales, float* y,
                       int N, int K, int M, int add, void* stream) {
  CIA_REQUIRE(N > 0 && K > 0 && K % 128 == 0 && M >= 0, CIA_ERR_ARG);
  if (M == 0) return CIA_OK;
  CIA_REQUIRE(x && packed && scales && y, CIA_ERR_NULL);
  CIA_REQUIRE(aligned(x, 16) && mat_ok(packed, scales) && aligned(y, 4), CIA_ERR_ALIGN);
  GemvArgs a{};
  a.x = x;
  a.K = K;
  a.M = M;
  a.add = add;
  a.mat[0] = Int4Mat{packed, scales, N, y, nullptr};
  return gemv_run(a, stream);
}

extern "C" int cia_gemv_int4(const uint16_t* x, const uint8_t* packed, const uint16_t* scales,
                             float* y, int N, int K, int M, void* stream) {
  return gemv_common(x, packed, scales, y, N, K, M, 0, stream);
}

extern "C" int cia_gemv_int4_add(const uint16_t* x, const uint8_t* packed,
                                 const uint16_t* scales, float* y, int N, int K, int M,
                                 void* stream) {
  return gemv_common(x, packed, scales, y, N, K, M, 1, stream);
}

extern "C" int cia_qkv_proj_int4(const uint16_t* x, const uint8_t* wq_packed,
                                 const uint16_t* wq_scales, int Nq, const uint8_t* wk_packed,
                                 const uint16_t* wk_scales, const uint8_t* wv_packed,
                                 const uint16_t* wv_scales, int Nkv, int K, int M, uint16_t* q,
                                 uint16_t* k, uint16_t* v, void* stream) {
  CIA_REQUIRE(Nq > 0 && Nkv > 0 && K > 0 && K % 128 == 0 && M >= 0, CIA_ERR_ARG);
  if (M == 0) return CIA_OK;
  CIA_REQUIRE(x && wq_packed && wq_scales && wk_packed && wk_scales && wv_packed && wv_scales &&
                  q && k && v,
              CIA_ERR_NULL);
  CIA_REQUIRE(aligned(x, 16) && mat_ok(wq_packed, wq_scales) && mat_ok(wk_packed, wk_scales) &&
                  mat_ok(wv_packed, wv_scales) && aligned(q, 2) && aligned(k, 2) && aligned(v, 2),
              CIA_ERR_ALIGN);
  GemvArgs a{};
  a.x = x;
  a.K = K;
  a.M = M;
  a.mat[0] = Int4Mat{wq_packed, wq_scales, Nq, nullptr, q};
  a.mat[1] = Int4Mat{wk_packed, wk_scales, Nkv, nullptr, k};
  a.mat[2] = Int4Mat{wv_packed, wv_scales, Nkv, nullptr, v};
  return gemv_run(a, stream);
}
