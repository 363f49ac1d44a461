// Several D2Q9 steps in one launch: the same update as that many launches of k_step, with the
// states in between held in LDS.
//
// A 2-D step of the usual sizes is bound by its launch and by the latency of its loads (64x64:
// 2.9 us, 512x256: 4.5 us per step, periodic FP32), and every step pays both.  Here a block loads
// 32 x 32 cells, advances them n steps in LDS and writes the inner (32 - 2n) x (32 - 2n), which
// are the ones whose neighbours it held all along.  A thread keeps its cell for all the steps, so
// the boundary id, descriptor, missing bits, prescribed value and body force are read once, and
// where each population is pulled from (a neighbour, or the cell itself at bounce-back and
// do-nothing cells) is worked out once.  Cells go through the arithmetic of k_step, those near a
// block's edge in more than one block, so the fields are k_step's bit for bit.
//
// What is left is the arithmetic: 1024 threads take 0.7 us per step periodic and 1.2 to 1.8 us with a
// force and boundary conditions, after 3 to 6 us to start, load and store.  Square tiles keep the
// share of repeated cells small (rows of 64: 448 of 1024 cells advanced by 4 steps, here 576); with
// 64 registers two FP32 blocks share a CU (FP64: one, its states fill the LDS).  Measured, us per
// step, FP32 (FP64), before and after: channel with a force field 64x64 4.1 -> 1.9 (4.5 -> 2.4),
// 512x256 5.2 -> 3.3 (6.3 -> 4.4), 1024x512 12.3 -> 8.3 (20.2 -> 15.3), 2048x2048 73 -> 46 (136 -> 97);
// periodic 64x64 2.9 -> 0.9, 512x256 4.5 -> 2.7, 1024x512 10.3 -> 5.0, 2048x2048 62 -> 34.
#pragma once

#include "step.hpp"

namespace xlbh {

constexpr int kTile2d = 32;      // a block holds 32 x 32 cells, one per thread
constexpr int kMaxSteps2d = 12;  // at 12 steps it advances 8 x 8 of them

struct Steps2d {
  int steps;           // steps of this launch
  int tiles_y;
  size_t state_bytes;  // when every state is kept: bytes from one to the next, else 0
};

// BCS: there is a mask; NT: non-temporal stores.
template <int COLL, int FMT, class C, bool BCS, bool NT>
__global__ __launch_bounds__(kTile2d * kTile2d, sizeof(C) == 4 && COLL != XLBH_KBC ? 8 : 4) void k_steps_2d(StepParams p, Steps2d g) {
  constexpr int LAT = XLBH_D2Q9;
  constexpr LatTables T = make_tables(LAT);
  constexpr int Q = T.q;
  using R = typename Fmt<FMT>::raw;
  static_assert(__is_same(R, C), "the intermediate states are kept in the arithmetic type");
  constexpr int CELLS = kTile2d * kTile2d;
  __shared__ C lds[2 * Q * CELLS];

  const int nx = p.sw.nx, ny = p.sw.ny, n = g.steps, side = kTile2d - 2 * n;
  const int t = threadIdx.x, tx = t / kTile2d, ty = t % kTile2d;
  const int x0 = (int)blockIdx.x / g.tiles_y * side - n, y0 = (int)blockIdx.x % g.tiles_y * side - n;
  const uint32_t cell = (uint32_t)wrap(x0 + tx, nx) * ny + wrap(y0 + ty, ny);
  // steps after which the cell is still exact: its distance from the edge of the block
  const int depth = min(min(tx, kTile2d - 1 - tx), min(ty, kTile2d - 1 - ty));
  const bool inner = depth >= n && x0 + tx < nx && y0 + ty < ny;
  const R* fin = static_cast<const R*>(p.f_in);
  int id = 0;
  if constexpr (BCS) id = p.bc_mask[cell];
  C f[Q];
#pragma unroll
  for (int l = 0; l < Q; ++l) f[l] = ld_pop<FMT, C>(fin + l * p.plane + cell, T.w[l]);
  C F[3] = {C(0), C(0), C(0)};
  const bool has_force = p.force_mode != XLBH_FORCE_NONE;
  if (p.force_mode == XLBH_FORCE_UNIFORM) {
    F[0] = (C)p.fu[0];
    F[1] = (C)p.fu[1];
  } else if (p.force_mode == XLBH_FORCE_FIELD) {
#pragma unroll
    for (int d = 0; d < 2; ++d) F[d] = static_cast<const C*>(p.force_field)[(size_t)d * p.N + cell];
  }
  int kind = XLBH_BC_NONE;
  uint32_t mm = 0;
  C rb = C(1), ub[3] = {C(0), C(0), C(0)}, pv = C(0);
  int nrm[3] = {0, 0, 0};
  if (BCS && id != 0) {
    const xlbh_bc_desc* d = p.table + id;
    kind = d->kind;
    rb = (C)d->rho;
    ub[0] = (C)d->u[0];
    ub[1] = (C)d->u[1];
    mm = p.missing[cell];
    if (p.aux != nullptr) pv = static_cast<const C*>(p.aux)[cell];
    if (kind == XLBH_BC_EXTRAPOLATION_OUTFLOW) bc_normal<LAT>(mm, nrm);
  }
  int src[Q];  // where population l of the post-stream state is read in the LDS state
#pragma unroll
  for (int l = 0; l < Q; ++l) {
    src[l] = l * CELLS + t - T.c[0][l] * kTile2d - T.c[1][l];
    if constexpr (BCS) {
      if ((kind == XLBH_BC_HALFWAY_BB || kind == XLBH_BC_EXTRAPOLATION_OUTFLOW) && bit(mm, l)) src[l] = T.opp[l] * CELLS + t;
      if (kind == XLBH_BC_DO_NOTHING) src[l] = l * CELLS + t;
    }
  }
#pragma unroll
  for (int l = 0; l < Q; ++l) lds[l * CELLS + t] = f[l];
  __syncthreads();
  for (int s = 1; s <= n; ++s) {
    const C* prev = lds + ((s - 1) & 1) * (Q * CELLS);
    if (depth >= s) {
#pragma unroll
      for (int l = 0; l < Q; ++l) f[l] = prev[src[l]];
      if constexpr (BCS) {
        if (kind == XLBH_BC_EQUILIBRIUM) {
          const C us = usqr15<LAT>(ub);
#pragma unroll
          for (int l = 0; l < Q; ++l) f[l] = feq_l<LAT>(l, rb, ub, us);
        } else if (kind >= XLBH_BC_ZOUHE_VELOCITY && kind <= XLBH_BC_REGULARIZED_PRESSURE) {
          zouhe_cell<LAT>(f, mm, pv, kind == XLBH_BC_ZOUHE_VELOCITY || kind == XLBH_BC_REGULARIZED_VELOCITY,
                          kind >= XLBH_BC_REGULARIZED_VELOCITY);
        }
      }
      if (BCS && kind == XLBH_BC_FULLWAY_BB) {
#pragma unroll
        for (int l = 0; l < Q; ++l) {
          if (T.opp[l] > l) {
            const C v = f[l];
            f[l] = f[T.opp[l]];
            f[T.opp[l]] = v;
          }
        }
      } else {
        collide<LAT, COLL, C, false>(f, (C)p.omega, has_force, F, (C)p.cparam);
      }
      if (BCS && kind == XLBH_BC_EXTRAPOLATION_OUTFLOW) {
        // the source x - c_l - n is at most one cell away (the caller says so), so it is in the state
        const C cs = C(0.57735026918962584);
#pragma unroll
        for (int l = 0; l < Q; ++l) {
          if (bit(mm, l)) {
            const C faux = prev[l * CELLS + t - (T.c[0][l] + nrm[0]) * kTile2d - (T.c[1][l] + nrm[1])];
            const C fps = prev[T.opp[l] * CELLS + t];
            f[T.opp[l]] = (C(1) - cs) * fps + cs * faux;
          }
        }
      }
      if (s < n) {
        C* next = lds + (s & 1) * (Q * CELLS) + t;
#pragma unroll
        for (int l = 0; l < Q; ++l) next[l * CELLS] = f[l];
      }
      if (inner && (s == n || g.state_bytes != 0)) {
        R* out = reinterpret_cast<R*>(static_cast<char*>(p.f_out) + (g.state_bytes != 0 ? (s - 1) * g.state_bytes : 0));
#pragma unroll
        for (int l = 0; l < Q; ++l) st_pop<FMT, C, NT>(out + l * p.plane + cell, f[l], T.w[l]);
      }
    }
    __syncthreads();
  }
}

// Whether several steps of a call can run as one launch.  `known`: what may occur in the mask
// (XLBH_MASK_*, kind bits).
bool steps_2d_apply(int lattice, const StepCall& c, uint32_t known);
// Steps per launch that take the least time for a run of `n` steps (1: k_step); keep: every state is kept.
int steps_2d_best(const StepCall& c, int n, bool keep);
// `steps` steps from c.f_in to c.f_out; with state_bytes != 0 the state after step s goes to
// c.f_out + (s - 1) * state_bytes.
int launch_steps_2d(const StepCall& c, int steps, size_t state_bytes);

}  // namespace xlbh
