// The two-step launches of D3Q19 (pair.hpp).
#include "pair.hpp"

namespace xlbh {

bool plan_pair(int lattice, const StepCall& c, uint32_t known, PairTiles& g) {
  g.blocks = 0;
  constexpr uint32_t walls = 1u << XLBH_BC_NONE | 1u << XLBH_BC_EQUILIBRIUM | 1u << XLBH_BC_HALFWAY_BB |
                             1u << XLBH_BC_FULLWAY_BB | 1u << XLBH_BC_DO_NOTHING;
  if (lattice != XLBH_D3Q19 || c.force_mode != XLBH_FORCE_NONE || (c.bc_mask && (known & ~walls) != 0)) return false;
  const bool f32 = c.store == XLBH_F32 && (c.compute == XLBH_COMPUTE_F32 || c.compute == XLBH_COMPUTE_F32_DEVIATION);
  const bool f64 = c.store == XLBH_F64 && c.compute == XLBH_COMPUTE_F64;
  if (!f32 && !f64) return false;
  const bool dev = c.compute == XLBH_COMPUTE_F32_DEVIATION;
  if (c.collision != XLBH_BGK && (c.collision != XLBH_SMAGORINSKY_BGK || dev)) return false;
  if ((uint64_t)c.ny * c.nz * (f32 ? 4 : 8) > 0xffffffffull) return false;  // 32-bit offsets inside an x-plane
  g = f32 ? pair_tiles<kPairRowsF32>(c.nx, c.ny, c.nz, 19, 4) : pair_tiles<kPairRowsF64>(c.nx, c.ny, c.nz, 19, 8);
  return g.blocks > 0;
}

int launch_pair(const StepCall& c, const PairTiles& g) {
  constexpr int L = XLBH_D3Q19, S = XLBH_SMAGORINSKY_BGK;
  if (c.compute == XLBH_COMPUTE_F64)
    return c.collision == S ? launch_pair_t<L, S, XLBH_F64, double, kPairRowsF64>(c, g)
                            : launch_pair_t<L, XLBH_BGK, XLBH_F64, double, kPairRowsF64>(c, g);
  if (c.compute == XLBH_COMPUTE_F32_DEVIATION) return launch_pair_t<L, kBgkDeviation, XLBH_F32, float, kPairRowsF32>(c, g);
  return c.collision == S ? launch_pair_t<L, S, XLBH_F32, float, kPairRowsF32>(c, g)
                          : launch_pair_t<L, XLBH_BGK, XLBH_F32, float, kPairRowsF32>(c, g);
}

}  // namespace xlbh
