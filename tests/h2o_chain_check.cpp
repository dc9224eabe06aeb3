// Checks the buffer loads of k_h2o_chain (cuda_inf_amd/csrc/h2o_chain.h) for
// every chunk size up to a bound, all three step sizes, every lane: a load is
// either refused or inside the chunk, under each way in which the range check
// may take the scalar offset (added to the offset, taken off the size with
// 32-bit wrap-around, or left out); a row of the chunk is never refused and is
// read at its address.  Exit status 0 when all hold.
// With an argument, the loads as they would be with the step's row in the
// scalar offset: the check must refuse that (exit status 1).
#include <cstdint>
#include <cstdio>

#include "h2o_chain.h"

using namespace cia;

static long bad = 0;

static void load(ChainOff o, int bytes, int64_t size, bool row_in, int64_t want) {
  const uint32_t lane = (uint32_t)o.lane, sc = (uint32_t)o.scalar, n = (uint32_t)size;
  const bool refused[3] = {(uint64_t)lane + sc >= n, lane >= n - sc, lane >= n};
  const int64_t at = (int64_t)lane + sc;
  for (int k = 0; k < 3; k++) {
    if (!refused[k] && (at < 0 || at + bytes > size)) bad++;  // read past the chunk
    if (row_in && (refused[k] || at != want)) bad++;          // a row lost or misplaced
  }
}

int main(int argc, char**) {
  const bool scalar_rows = argc > 1;
  for (int kr = 1; kr <= 4; kr *= 2)
    for (int nq = 1; nq <= 67; nq++)
      for (int n = 0; n < (nq + kr - 1) / kr; n++)
        for (int g = 0; g < 8; g++)
          for (int lane = 0; lane < 64; lane++) {
            const int pieces = kr * 32;
            for (int c = 0; 64 * c < pieces; c++) {
              if (lane + 64 * c >= pieces) continue;
              ChainOff o = chain_q_off(kr, n, c, lane, g);
              const int rowi = (lane + 64 * c) / 8, query = n * kr + rowi / 4, head = 4 * g + rowi % 4;
              const int64_t want = (int64_t)query * kChainQRow + head * 128 + 16 * ((lane & 7) ^ (rowi & 7));
              if (scalar_rows) {
                o.scalar = (n * kr + 2 * c) * kChainQRow;
                o.lane -= o.scalar;
              }
              load(o, 16, (int64_t)nq * kChainQRow, query < nq, want);
            }
            const int r = (lane / (16 / kr)) >> 2, h = (lane / (16 / kr)) & 3, query = n * kr + r;
            load(chain_m_off(kr, n, r, g, h), 8, (int64_t)nq * kChainMRow, query < nq,
                 (int64_t)query * kChainMRow + (4 * g + h) * 8);
          }
  std::printf("%ld bad loads\n", bad);
  return bad ? 1 : 0;
}
