// h2o_chain.h -- where the attention mass chain (k_h2o_chain, h2o_attn.hip)
// reads a chunk's q rows and (m_b, w_b) pairs.  The last step's rows past the
// chunk must be refused by the buffer resource, so the whole offset is the
// lane's and the scalar offset is 0: a range check that takes the scalar
// offset off the size (offset >= size - scalar) would wrap once the scalar
// offset passed the size, as a step's second fetch does when the chunk has
// 4n + 1 queries.  Plain C++, so that the offsets are checked on the CPU.
#pragma once

namespace cia {

constexpr int kChainQRow = 32 * 64 * 2;  // bytes of a query's q rows
constexpr int kChainMRow = 32 * 8;       // bytes of a query's (m_b, w_b) in a block

// a buffer load's two offsets
struct ChainOff {
  int lane, scalar;
};

// 16-byte piece `lane` + 64 c of kv head g's q rows in step n of kr queries:
// row (query, head) lane / 8 + 8 c, its piece (lane & 7) ^ (lane / 8)
constexpr ChainOff chain_q_off(int kr, int n, int c, int lane, int g) {
  const int row = lane >> 3;
  return ChainOff{(n * kr + 2 * c + (row >> 2)) * kChainQRow + (4 * g + (row & 3)) * 128 +
                      16 * ((lane & 7) ^ row),
                  0};
}

// (m_b, w_b) of query r of step n, head h of kv head g
constexpr ChainOff chain_m_off(int kr, int n, int r, int g, int h) {
  return ChainOff{(n * kr + r) * kChainMRow + (4 * g + h) * 8, 0};
}

}  // namespace cia
