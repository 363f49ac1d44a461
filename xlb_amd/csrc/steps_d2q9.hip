// The several-step launches of D2Q9 (steps2d.hpp).
#include "steps2d.hpp"

namespace xlbh {

static int64_t steps_2d_blocks(const StepCall& c, int steps) {
  const int side = kTile2d - 2 * steps;
  return (int64_t)((c.nx + side - 1) / side) * ((c.ny + side - 1) / side);
}

bool steps_2d_apply(int lattice, const StepCall& c, uint32_t known) {
  // What k_steps_2d implements.  Solid cells are not among them (they keep what the output buffer
  // held), nor outflow sources two cells away (they may lie outside the block).
  constexpr uint32_t kinds = 1u << XLBH_BC_NONE | 1u << XLBH_BC_EQUILIBRIUM | 1u << XLBH_BC_HALFWAY_BB |
                             1u << XLBH_BC_FULLWAY_BB | 1u << XLBH_BC_DO_NOTHING | 1u << XLBH_BC_ZOUHE_VELOCITY |
                             1u << XLBH_BC_ZOUHE_PRESSURE | 1u << XLBH_BC_REGULARIZED_VELOCITY |
                             1u << XLBH_BC_REGULARIZED_PRESSURE | 1u << XLBH_BC_EXTRAPOLATION_OUTFLOW;
  if (lattice != XLBH_D2Q9 || (c.bc_mask && (known & ~kinds) != 0)) return false;
  const bool f32 = c.store == XLBH_F32 && c.compute == XLBH_COMPUTE_F32;
  const bool f64 = c.store == XLBH_F64 && c.compute == XLBH_COMPUTE_F64;
  return (f32 || f64) && steps_2d_blocks(c, kMaxSteps2d) < (int64_t)1 << 31;
}

// A launch takes about 6 us and 1.5 us per step (the channel's; a periodic box less of both) for
// every block a CU gets: more steps share the start, but repeat more cells.  512x256: 4 steps (242
// blocks, 3.3 us per step; 5 steps, 288 blocks: 3.9); 64x64: 12 steps (1.9; 4 steps: 2.7).
int steps_2d_best(const StepCall& c, int n) {
  int best = 1;
  double cost = 0.0;
  for (int k = 1; k <= kMaxSteps2d && k <= n; ++k) {
    const double t = (double)((steps_2d_blocks(c, k) + 255) / 256) * (6.0 + 1.5 * k) / k;
    if (k == 1 || t < cost) {
      cost = t;
      best = k;
    }
  }
  return best;
}

template <int COLL, int FMT, class C>
static int launch_t(const StepCall& c, const Steps2d& g, unsigned blocks) {
  const StepParams p = step_params<XLBH_D2Q9, FMT>(c);
  if (c.bc_mask)
    hipLaunchKernelGGL((k_steps_2d<COLL, FMT, C, true>), dim3(blocks), dim3(kTile2d * kTile2d), 0, c.stream, p, g);
  else
    hipLaunchKernelGGL((k_steps_2d<COLL, FMT, C, false>), dim3(blocks), dim3(kTile2d * kTile2d), 0, c.stream, p, g);
  XLBH_LAUNCH_CHECK();
  return 0;
}

int launch_steps_2d(const StepCall& c, int steps, size_t state_bytes) {
  const int side = kTile2d - 2 * steps;
  const Steps2d g{steps, (c.ny + side - 1) / side, state_bytes};
  const unsigned blocks = (unsigned)steps_2d_blocks(c, steps);
  const bool f64 = c.compute == XLBH_COMPUTE_F64;
  switch (c.collision) {
    case XLBH_KBC:
      return f64 ? launch_t<XLBH_KBC, XLBH_F64, double>(c, g, blocks) : launch_t<XLBH_KBC, XLBH_F32, float>(c, g, blocks);
    case XLBH_SMAGORINSKY_BGK:
      return f64 ? launch_t<XLBH_SMAGORINSKY_BGK, XLBH_F64, double>(c, g, blocks)
                 : launch_t<XLBH_SMAGORINSKY_BGK, XLBH_F32, float>(c, g, blocks);
  }
  return f64 ? launch_t<XLBH_BGK, XLBH_F64, double>(c, g, blocks) : launch_t<XLBH_BGK, XLBH_F32, float>(c, g, blocks);
}

}  // namespace xlbh
