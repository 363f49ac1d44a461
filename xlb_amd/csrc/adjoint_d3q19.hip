// Reverse-step instantiations for one lattice (kept in its own translation unit so the
// lattices compile in parallel).
#include "adjoint.hpp"

namespace xlbh {
int adjoint_dispatch_d3q19(int store, int compute, const AdjParams& p, hipStream_t s, const AdjCall& call) {
  return adjoint_dispatch_lat<XLBH_D3Q19>(store, compute, p, s, call);
}
}  // namespace xlbh
