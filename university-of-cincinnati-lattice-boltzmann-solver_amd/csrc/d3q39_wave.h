// What the D3Q39 step kernels of both files share.
#pragma once
#include "kernels.h"

namespace uclbs {

// index s of an axis of n nodes, at most n beyond it, wrapped
__device__ __forceinline__ int wrapm(int s, int n) {
  s += (s < 0) ? n : 0;
  return s - ((s >= n) ? n : 0);
}

// a wavefront's counters, added to one of the level's slots
__device__ __forceinline__ void wave_stats39(unsigned long long* __restrict__ stats, bool active,
                                             int iters, bool noconv, int ast, bool kerr) {
  const unsigned long long act = __ballot(active);
  if (act == 0ull) return;
  unsigned long long it = 0;
#pragma unroll
  for (int bt = 0; bt < 8; ++bt)
    it += (unsigned long long)__popcll(__ballot(active && ((iters >> bt) & 1))) << bt;
  const unsigned long long nc = __popcll(__ballot(active && noconv));
  const unsigned long long nt = __popcll(__ballot(active && ast == 1));
  const unsigned long long nb = __popcll(__ballot(active && (ast == 2 || ast == 3)));
  const unsigned long long nn = __popcll(__ballot(active && ast < 0));
  const unsigned long long nk = __popcll(__ballot(active && kerr));
  if (__lane_id() == 0) {
    unsigned long long* s = stats + (size_t)(blockIdx.x & (kStatSlots - 1)) * kStatFields;
    atomicAdd(s + ST_NODES, (unsigned long long)__popcll(act));
    if (it) atomicAdd(s + ST_ITERS, it);
    if (nc) atomicAdd(s + ST_NOCONV, nc);
    if (nt) atomicAdd(s + ST_TRIVIAL, nt);
    if (nb) atomicAdd(s + ST_BOUND, nb);
    if (nn) atomicAdd(s + ST_NONPOS, nn);
    if (nk) atomicAdd(s + ST_FALLBACK, nk);
  }
}

}  // namespace uclbs
