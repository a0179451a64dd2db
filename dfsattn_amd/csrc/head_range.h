// Which instance of the split attention kernel computes a head: the common
// one, or the scaled one where an operand carries an exponent (Q or K beyond
// the f16 range) or the scale lets an f16 q * c reach 2^15. Host code as well
// as device code, so that the rule can be run without a GPU.
//
// P: scale_all, H, exps ([3][H] or NULL, the exponents of Q, K and V) and
// q_marks. q_marks = exps where nobody has looked at Q's range before the
// attention: the words exps[0 .. H) then start at 0 and the common instance
// sets the word of a head in which a row of Q leaves the range.
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
// the way is finished here and done again, whole, by the scaled instance.
template <typename P>
DFS_HOST_DEVICE bool common_skips(const P& p, int h) {
  return p.scale_all || (p.exps && ((p.q_marks ? 0 : p.exps[h]) | p.exps[p.H + h]) != 0);
}

}  // namespace dfs
