// int4_shape.h -- which matrix-core kernel and tile an INT4 projection launch
// takes (gemv_int4.hip).  All of them give a row the same bits from kChainsM rows
// of x on, and the K-split kernel's shapes do below, so the choice is by time
// alone and may depend on the rows of W.  Plain C++, so that the rule is checked
// against measured times on the CPU.
#pragma once

namespace cia {

constexpr int kKsMaxK = 4096;   // K-split kernel: its LDS scale table's groups
constexpr int kBigMaxK = 2048;  // 256-row tiles: the LDS
// Rows of x below which the K-split kernel's sums take four chains a pass, an
// order of its own: no other matrix-core kernel runs there
constexpr int kChainsM = 56;
// The largest number of rows whose x the K-split shapes were measured with
constexpr int kKsMaxM = 2048;

enum Int4Kernel { kInt4Ks, kInt4Tile, kInt4Big };

// Time of a launch in us, with u = K / 1024 (the K-split kernel: at least 1, a
// pass of its 8 waves): a + b u for the first round of 256 workgroups (one a
// compute unit), c + d u for each further one.  Least squares of the relative
// error over 690 sizes -- 64 to 32768 rows of W, K 128 to 4096, 3 to 4096 rows
// of x -- median error 4 %.  At K = 2048, one round / two, model and measured:
// 1x1 4.6 / 6.1 (4.4 / 5.7), 1x2 5.0 / 7.4 (5.0 / 7.2), 2x2 5.9 / 9.2 (5.8 /
// 9.0), 2x3 7.6 / 12.0 (7.6 / 11.3), 4x3 9.7 / 19.2 (9.5 / 19.0), 4x4 11.8 /
// 23.4 (12.0 / 23.2), 128 x 128 26.7 / 56.8 (25 / 49), 256 x 128 36 / 86 (34 /
// 71), 256 x 192 51 / 123 (46 / 58 with the second round nearly empty).
struct Int4Shape {
  Int4Kernel kernel;
  int xrows, cols;  // of a workgroup's tile
  float a, b, c, d;
};
constexpr Int4Shape kInt4Shapes[] = {
    {kInt4Ks, 16, 16, 2.2f, 1.2f, 0.0f, 0.75f},   {kInt4Ks, 16, 32, 2.0f, 1.5f, 0.0f, 1.2f},
    {kInt4Ks, 32, 32, 2.0f, 1.95f, 0.0f, 1.65f},  {kInt4Ks, 32, 48, 1.7f, 2.95f, 0.0f, 2.2f},
    {kInt4Ks, 64, 48, 1.95f, 3.85f, 0.0f, 4.75f}, {kInt4Ks, 64, 64, 0.75f, 5.5f, 0.0f, 5.8f},
    {kInt4Tile, 128, 128, 7.2f, 9.75f, 9.5f, 10.3f},
    {kInt4Big, 256, 128, 12.1f, 12.1f, 19.3f, 15.5f},
    {kInt4Big, 256, 192, 17.0f, 16.9f, 28.3f, 21.8f}};
constexpr int kInt4NShapes = sizeof(kInt4Shapes) / sizeof(kInt4Shapes[0]);

constexpr long int4_tiles(const Int4Shape& s, int M, int rows) {
  return ((long)rows + s.cols - 1) / s.cols * (((long)M + s.xrows - 1) / s.xrows);
}

constexpr float int4_time(const Int4Shape& s, int M, int rows, int K) {
  float u = (float)K / 1024.0f;
  if (s.kernel == kInt4Ks && u < 1.0f) u = 1.0f;
  const long rounds = (int4_tiles(s, M, rows) + 255) / 256;
  return s.a + s.b * u + (float)(rounds - 1) * (s.c + s.d * u);
}

// index of the shape of least time among those that take the size
constexpr int int4_shape(int M, int rows, int K) {
  int best = -1;
  float t = 0.0f;
  for (int i = 0; i < kInt4NShapes; i++) {
    const Int4Shape& s = kInt4Shapes[i];
    if (s.kernel == kInt4Ks && (K > kKsMaxK || M > kKsMaxM)) continue;
    if (s.kernel == kInt4Big && K > kBigMaxK) continue;
    if (s.kernel != kInt4Ks && K <= kKsMaxK && M < kChainsM) continue;
    const float ti = int4_time(s, M, rows, K);
    if (best < 0 || ti < t) {
      best = i;
      t = ti;
    }
  }
  return best;
}

// Whether the GEMV runs rather than the matrix cores: for 1 and 2 rows of x, and
// for fewer than 56 where K is beyond the K-split kernel's.  Between, GEMV / K-split
// in us, K = 2048: q/k/v 2 rows 3.7 / 3.8, 3 5.0 / 4.3, 16 10.2 / 4.4; added into
// the residual (add), 2048 rows of W: 3 4.1 / 4.5, 5 5.1 / 4.4; 512: 16 4.3 / 4.5, 32
// 5.3 / 4.4; 8192: 3 7.2 / 4.8.  K = 4096, 2048 rows of W: 4 5.7 / 6.7, 5 7.7 / 6.7;
// 8192: 3 11.6 / 8.8.  K = 512, 2048: 3 3.7 / 3.2; 1152: 4 4.2 / 4.0.  So added sums take the GEMV while
// its workgroups, 8 rows of W by 4 of x, fit the chip at once.  For sums that are
// stored the line depends on K alone: a matrix must give the same bits alone and
// in a q/k/v launch, and the two kernels add in different orders.
constexpr bool int4_gemv(int M, int rows, int K, bool add) {
  if (M <= 2) return true;
  if (M >= kChainsM) return false;
  if (K > kKsMaxK) return true;
  if (add) return K > 1536 && ((long)rows + 7) / 8 * ((M + 3) / 4) <= 256;
  return K > 2048 && M < 5;
}

}  // namespace cia
