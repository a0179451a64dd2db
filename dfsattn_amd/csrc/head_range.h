// Which instance of the split attention kernel computes a head: the common
// one, or the scaled one where an operand carries an exponent (Q or K beyond
// the f16 range) or the scale lets an f16 q * c reach 2^15. Host code as well
// as device code, so that the rule can be run without a GPU.
//
// P: scale_all, H, Qb, exps ([3][H] or NULL, the exponents of Q, K and V),
// q_marks and q_block_marks. q_marks = exps where nobody has looked at Q's
// range before the attention: the words exps[0 .. H) and q_block_marks [H][Qb]
// then start at 0 and the common instance sets the words of a head and query
// block in which a row of Q leaves the range.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define DFS_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define DFS_HOST_DEVICE inline
#endif

namespace dfs {

// For the launches behind the common instance, when the marks are final.
template <typename P>
DFS_HOST_DEVICE bool head_scaled(const P& p, int h) {
  return p.scale_all || (p.exps && (p.exps[h] | p.exps[p.H + h]) != 0);
}

// For the common instance itself, whose waves ask one by one while other
// workgroups of the launch may set marks: only words that are final before the
// launch are read, or part of a workgroup could leave and the rest go on
// without its share of the column list and the tiles. A head that is marked on
// the way is gone on with, but for the marked blocks; what the scaled instance
// does says scaled_block.
template <typename P>
DFS_HOST_DEVICE bool common_skips(const P& p, int h) {
  return p.scale_all || (p.exps && ((p.q_marks ? 0 : p.exps[h]) | p.exps[p.H + h]) != 0);
}

// For the scaled instance, of a head it has: whether it does query block qb.
// Where only rows of Q left the range (marks, final by now), the common
// instance's other blocks are right: their rows' q c has the same bits and
// their scores the factor 1 in either instance. Blocks cut into parts are
// marked by the combining launch, which leaves such a head alone. 20,280
// tokens x 40 heads, one row of each beyond the range: 3.97 ms with all blocks
// of such heads done again, 1.80 so, 2.71 with Q's range known beforehand; with
// every row beyond it 2.50 and 2.93.
template <typename P>
DFS_HOST_DEVICE bool scaled_block(const P& p, int h, int qb) {
  return !p.q_marks || p.scale_all || p.exps[p.H + h] != 0 || p.q_block_marks[static_cast<int64_t>(h) * p.Qb + qb] != 0;
}

}  // namespace dfs
