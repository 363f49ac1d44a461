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

// Times in us, from launches on 23 grids of 4 k to 2.3 M cells, wide and thin (1 x 13000 to 60000 x 2),
// with 2 to 8 steps each.
struct Times2d {
  // n steps in one launch: start + step n for the first 256 blocks (one per CU), and for every 256
  // more blocks more_start + more_step n
  double start, step, more_start, more_step;
  // one step by k_step: a launch, 256 of its blocks, and 1 MB read or written
  double single, round, mb;
};
// Every state kept: 0.2 us per step for each MB of a state beyond 4 MB (the block's segments of rows are
// not whole cache lines).
constexpr double kKeepMb2d = 0.2, kKeepFree2d = 4.0;
// [double precision][KBC][boundary cells or a force field]; Smagorinsky as BGK
constexpr Times2d kTimes2d[2][2][2] = {
    {{{4.6, 0.70, 1.7, 0.38, 2.8, 0.34, 0.087}, {6.3, 1.08, 4.1, 0.38, 3.4, 0.48, 0.102}},
     {{5.0, 1.75, 2.1, 1.29, 3.2, 0.55, 0.056}, {7.2, 2.04, 7.1, 1.59, 3.8, 0.71, 0.069}}},
    {{{5.9, 0.99, 3.8, 0.92, 3.0, 0.52, 0.096}, {7.6, 1.50, 9.6, 0.93, 3.6, 0.91, 0.077}},
     {{6.1, 2.11, 5.0, 1.86, 3.2, 0.74, 0.076}, {9.7, 2.62, 12.0, 2.06, 4.0, 1.14, 0.060}}}};

// More steps share the start of a launch, but repeat more cells (512x256 channel, us per step: 4.8 by
// k_step, 3.1 by 4 steps in 242 blocks, 3.8 by 5 in 288).  Where the arithmetic is what takes the time,
// or a block covers little of a thin grid, k_step is the faster one: KBC 1728x1331 29 us per step, 4
// steps a launch 32; 1x60000 4.4 and 7.1 (KBC FP64 4.3 and 29).  Recording 1728x1331 38 and 53, 700x350
// 5.9 and 3.8.  The fit's spread is 5 %, with KBC or Smagorinsky in more than 256 blocks 18 %.
int steps_2d_best(const StepCall& c, int n, bool keep) {
  const bool f64 = c.compute == XLBH_COMPUTE_F64;
  const Times2d& t = kTimes2d[f64][c.collision == XLBH_KBC][c.bc_mask || c.force_mode == XLBH_FORCE_FIELD];
  const dim3 g = sweep_grid(make_sweep(c.nx, c.ny, 1));
  int best = 1;
  const double mb = (double)c.nx * c.ny * 9e-6 * (f64 ? 8 : 4);
  const double kept = keep ? kKeepMb2d * std::max(0.0, mb - kKeepFree2d) : 0.0;
  double cost = t.single + t.round * ((double)g.x * g.y / 256) + t.mb * 2.0 * mb;
  for (int k = 2; k <= kMaxSteps2d && k <= n; ++k) {
    const double more = (double)((steps_2d_blocks(c, k) + 255) / 256 - 1);
    const double us = (t.start + t.step * k + more * (t.more_start + t.more_step * k)) / k + kept;
    const double spread = more == 0 || c.collision == XLBH_BGK ? 1.05 : 1.18;
    if (us * spread < cost) {
      cost = us * spread;
      best = k;
    }
  }
  return best;
}

template <int COLL, int FMT, class C>
static int launch_t(const StepCall& c, const Steps2d& g, unsigned blocks) {
  const StepParams p = step_params<XLBH_D2Q9, FMT>(c);
  // A last state goes out past the caches (512x256 channel 3.7 -> 3.3 us per step).  Kept states do if
  // they are small (235x355 channel, 3 MB: 3.7 -> 3.3); of a few MB, where rows are whole 32-byte sectors
  // and a block's segments of them are too (512x256 channel, 4 steps: 3.7 -> 3.3) or boundary cells take
  // the time (3 steps: 4.6 -> 4.1); larger, where the segments are a cache line long (FP64 1024x1000, 4
  // steps: 25.8 -> 22.6).  Else the parts of a line would go out one by one (FP32 341x365 periodic, 4.5
  // MB: 2.6 -> 3.5, 1024x1000 18.4 -> 26.2).
  const size_t segment = (kTile2d - 2 * g.steps) * sizeof(C), state = (size_t)c.nx * c.ny * 9 * sizeof(C);
  const bool rows = c.ny * sizeof(C) % 32 == 0, sectors = rows && segment % 32 == 0;
  const bool nt = g.state_bytes == 0 || state <= 4000000 || (state <= 8000000 ? sectors || (rows && c.bc_mask) : sectors && segment >= 128);
  auto go = [&](auto bcs, auto nts) {
    hipLaunchKernelGGL((k_steps_2d<COLL, FMT, C, decltype(bcs)::value, decltype(nts)::value>), dim3(blocks),
                       dim3(kTile2d * kTile2d), 0, c.stream, p, g);
  };
  using Y = std::true_type;
  using N = std::false_type;
  if (c.bc_mask && nt) go(Y{}, Y{});
  else if (c.bc_mask) go(Y{}, N{});
  else if (nt) go(N{}, Y{});
  else go(N{}, N{});
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
