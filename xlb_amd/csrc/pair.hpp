// Two fused steps in one launch: the same update as two launches of k_step, with the state in
// between held on chip.
//
// One step moves 2 Q S bytes per cell and runs at the rate of that access pattern, so the only
// way past it is to move the populations less often.  A block owns a (ty x 64)-cell tile of (y, z)
// and marches along x.  At plane X it
//   1. updates the tile and one halo cell around it from f_in (first step), and leaves the result
//      in LDS;
//   2. after the barrier, updates its own cells of plane X - 1 a second time: their pulls come
//      from the first-step planes X - 2, X - 1 and X, of which LDS holds two and registers the
//      pulls of c_x = 0 (one plane back) and c_x = 1 (two planes back) read when they were there.
// Per pair of steps a cell is read 15/13 * 66/64 times (the halo, most of it from L2) and written
// once, instead of twice each.  Every cell goes through the same arithmetic as in k_step, halo
// cells more than once, so the fields are those of two k_step launches bit for bit.
//
// Tile: 15 rows of 64 cells, one wave per row, and a 16th wave for the two halo columns: rows are
// loaded and stored in whole aligned 256-byte segments, and 2 * 19 floats of 990 cells fill the
// 160 KB of LDS, so one block of 16 waves runs per CU.  FP64 takes 7 rows (140 KB; a ninth wave
// would cap the registers at 168 and spill).
// Measured on the D3Q19 BGK step, 256^3 FP32: periodic 430 -> 282 us per step, cavity 434 -> 288
// us, halfway walls 302 us; 512x256x256 860 -> 592 us; FP64 150x90x110 96 -> 65 us.  Bound by memory: a
// pair on the 256^3 cavity reads and writes 2.84 GB (1.11 times its algorithmic bytes) in 564 us, 5.0
// TB/s, the rate of a device copy; its VALU instructions take about half of that time.
// What else was tried at 256^3 periodic (us per step): loads of the next plane before the first
// update instead of after it 287 (and 320 on the cavity, whose boundary lookups then wait for
// them); 14, 12 and 7 rows 302, 295 and 315 (the last with two blocks per CU); non-temporal loads
// 404; consecutive blocks on different XCDs 313 against neighbouring tiles on one XCD 301.
#pragma once

#include "step.hpp"

namespace xlbh {

struct PairTiles {
  int nzt, nyt;  // tiles along z and y
  int ty, cx;    // rows of a tile, planes of a chunk
  int blocks;
};

constexpr int kPairPitch = 66;  // 64 cells of a row and one halo cell on each side
constexpr int kPairEq = 96;     // EquilibriumBC constants of ids below this are kept in LDS

// The collision, or the full-way bounce-back that replaces it, in place.
template <int LAT, int COLL, class C>
__device__ __forceinline__ void pair_collide(C* f, int kind, const StepParams& p) {
  constexpr LatTables T = make_tables(LAT);
  if (kind == XLBH_BC_FULLWAY_BB) {
#pragma unroll
    for (int l = 0; l < T.q; ++l) {
      if (T.opp[l] > l) {
        const C t = f[l];
        f[l] = f[T.opp[l]];
        f[T.opp[l]] = t;
      }
    }
  } else {
    const C F[3] = {C(0), C(0), C(0)};
    if constexpr (COLL == kBgkDeviation)
      bgk_deviation<LAT>(f, p.omega, false, F);
    else
      collide<LAT, COLL, C, false>(f, (C)p.omega, false, F, (C)p.cparam);
  }
}

// BCS: the mask may hold equilibrium, halfway and full-way bounce-back and do-nothing cells (no
// others); without it there is no mask.  NT: non-temporal stores, for rows of whole 128-byte lines
// (300x200x230 FP32, whose rows are not: 315 us per step without, 372 with; 256^3: 311 and 301).
template <int LAT, int COLL, int FMT, class C, int ROWS, bool BCS, bool NT>
__global__ __launch_bounds__((ROWS + 1) * 64) void k_step_pair(StepParams p, PairTiles g) {
  constexpr LatTables T = make_tables(LAT);
  constexpr int Q = T.q;
  using R = typename Fmt<FMT>::raw;
  static_assert(__is_same(R, C), "the intermediate state is kept in the arithmetic type");
  constexpr int SLOT = ROWS * kPairPitch;  // one population of one plane of the extended tile
  __shared__ C lds[2 * Q * SLOT];
  __shared__ C eqc[BCS ? kPairEq * 4 : 1];
  __shared__ uint8_t kinds[BCS ? 256 : 1];

  const int nx = p.sw.nx, ny = p.sw.ny, nz = p.sw.nz;
  // Blocks are dispatched to the 8 XCDs in turn; tile numbers that are neighbours (z fastest, then
  // y, then the chunk along x) go to one XCD, whose L2 then holds the halo lines they share.
  const uint32_t nb = gridDim.x, xcd = blockIdx.x % 8;
  const int tile = (int)(xcd * (nb / 8) + min(xcd, nb % 8) + blockIdx.x / 8);
  const int z0 = tile % g.nzt * 64, y0 = tile / g.nzt % g.nyt * g.ty, x0 = tile / (g.nzt * g.nyt) * g.cx;
  const int zl = min(64, nz - z0), yl = min(g.ty, ny - y0), xl = min(g.cx, nx - x0);

  // Row and z of the thread's cell in the extended tile: waves 0 .. ROWS - 1 hold one row each, the
  // last wave the halo columns (left and right of row lane / 2).
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const bool halo = wave == ROWS;
  const int row = halo ? lane >> 1 : wave;
  const int zi = halo ? ((lane & 1) ? zl : -1) : lane;
  const bool act = row < yl + 2 && (halo || lane < zl);
  const bool inner = act && !halo && row >= 1 && row <= yl;
  const int y = wrap1(act ? y0 + row - 1 : y0, ny), z = wrap1(act ? z0 + zi : z0, nz);
  uint32_t off[3][3];  // byte offsets of the pull sources inside an x-plane, [c_y + 1][c_z + 1]
  {
    const uint32_t yo[3] = {(uint32_t)(y == ny - 1 ? 0 : y + 1) * nz, (uint32_t)y * nz,
                            (uint32_t)(y == 0 ? ny - 1 : y - 1) * nz};
    const uint32_t zo[3] = {(uint32_t)(z == nz - 1 ? 0 : z + 1), (uint32_t)z, (uint32_t)(z == 0 ? nz - 1 : z - 1)};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int c = 0; c < 3; ++c) off[a][c] = (yo[a] + zo[c]) * (uint32_t)sizeof(R);
  }
  const uint32_t cip = (uint32_t)y * nz + z;  // the cell in its x-plane
  const uint32_t nyz = (uint32_t)ny * nz;
  const size_t xs = (size_t)nyz * sizeof(R);
  const size_t plane_bytes = (size_t)p.plane * sizeof(R);
  const char* fin = static_cast<const char*>(p.f_in);
  char* fout = static_cast<char*>(p.f_out);
  C* slot = lds + row * kPairPitch + 1 + zi;
  if constexpr (BCS) {
    for (int k = threadIdx.x; k < 256; k += (ROWS + 1) * 64) {
      kinds[k] = (uint8_t)p.table[k].kind;
      if (k < kPairEq) {
        eqc[4 * k] = (C)p.table[k].rho;
        for (int d = 0; d < 3; ++d) eqc[4 * k + 1 + d] = (C)p.table[k].u[d];
      }
    }
    __syncthreads();
  }

  using gchar = const __attribute__((address_space(1))) char;
  // The empty asm statements keep the scalar base and the 32-bit lane offset apart (the
  // scalar-base form of loads and stores) and keep both from being hoisted out of the march as
  // one 64-bit vector address per population.
  auto at = [&](size_t base, uint32_t o, double w) -> C {
    gchar* s = (gchar*)(fin + base);
    asm("" : "+s"(s), "+v"(o));
    return ld_pop<FMT, C>(reinterpret_cast<const R*>((const char*)(s + o)), w);
  };
  auto next = [&](int X) { return X == nx - 1 ? 0 : X + 1; };
  auto ld_id = [&](int X) -> int { return BCS ? p.bc_mask[(size_t)X * nyz + cip] : 0; };
  auto pull = [&](int X, C* v) {
    const size_t xo[3] = {(size_t)next(X) * xs, (size_t)X * xs, (size_t)(X == 0 ? nx - 1 : X - 1) * xs};
    size_t lp = 0, pb = plane_bytes;
    asm volatile("" : "+s"(pb));
#pragma unroll
    for (int l = 0; l < Q; ++l, lp += pb)
      v[l] = at(lp + xo[T.c[0][l] + 1], off[T.c[1][l] + 1][T.c[2][l] + 1], T.w[l]);
  };
  // The streaming-step boundary conditions of a cell with id `id` and kind `kind` on v; own(l): its
  // own pre-stream population l.
  auto walls = [&](C* v, int id, int kind, uint32_t mm, auto&& own) {
    if (kind == XLBH_BC_HALFWAY_BB) {
#pragma unroll
      for (int l = 0; l < Q; ++l)
        if (bit(mm, l)) v[l] = own(T.opp[l]);
    } else if (kind == XLBH_BC_DO_NOTHING) {
#pragma unroll
      for (int l = 0; l < Q; ++l) v[l] = own(l);
    } else if (kind == XLBH_BC_EQUILIBRIUM) {
      C rb, ub[3];
      // two separate loads, not one through a selected pointer (a flat load, which would also
      // wait for every global load in flight)
      if (id < kPairEq) {
        rb = eqc[4 * id];
        for (int d = 0; d < 3; ++d) ub[d] = eqc[4 * id + 1 + d];
        asm volatile("" : "+v"(rb));
      } else {
        rb = (C)p.table[id].rho;
        for (int d = 0; d < 3; ++d) ub[d] = (C)p.table[id].u[d];
        asm volatile("" : "+v"(rb));
      }
      const C us = usqr15<LAT>(ub);
#pragma unroll
      for (int l = 0; l < Q; ++l) v[l] = feq_l<LAT>(l, rb, ub, us);
    }
  };

  C pf[Q];             // the next plane's pulls
  int idn, idm = 0;    // ids of the next and of the previous plane
  uint32_t mmm = 0;    // missing bits of the previous plane
  {
    const int X = x0 == 0 ? nx - 1 : x0 - 1;
    idn = ld_id(X);
    pull(X, pf);
  }
  C c0[Q], cp1[Q], cp2[Q];  // first-step pulls waiting: c_x = 0 of the last plane, c_x = 1 of the last two
#pragma unroll
  for (int l = 0; l < Q; ++l) c0[l] = cp1[l] = cp2[l] = C(0);
  // Plane X = x0 - 1 + i.  LDS buffer i & 1 holds its first-step state.  One barrier per plane is
  // enough: the buffer written at plane X + 1 was last read by other threads at plane X - 1, before
  // the barrier of plane X.
  for (int i = 0; i < xl + 2; ++i) {
    const int X = wrap1(x0 - 1 + i, nx);
    C* buf = slot + (i & 1) * (Q * SLOT);
    const int id = idn;
    uint32_t mm = 0;
    if (act) {
      const int kind = BCS ? kinds[id] : 0;
      if (BCS && kind != 0) {
        const size_t base = (size_t)X * xs;
        size_t pb = plane_bytes;
        asm volatile("" : "+s"(pb));
        if (kind == XLBH_BC_HALFWAY_BB) mm = p.missing[(size_t)X * nyz + cip];
        walls(pf, id, kind, mm, [&](int l) { return at(base + l * pb, off[1][1], T.w[l]); });
      }
      pair_collide<LAT, COLL, C>(pf, kind, p);
#pragma unroll
      for (int l = 0; l < Q; ++l) buf[l * SLOT] = pf[l];
    }
    asm volatile("" ::: "memory");
    idn = ld_id(next(X));
    if (i < xl + 1) pull(next(X), pf);
    asm volatile("" ::: "memory");
    __syncthreads();
    C h[Q];
    const int Xo = X == 0 ? nx - 1 : X - 1;
    if (inner && i >= 2) {
#pragma unroll
      for (int l = 0; l < Q; ++l)
        h[l] = T.c[0][l] == 0 ? c0[l] : (T.c[0][l] > 0 ? cp2[l] : buf[l * SLOT - T.c[1][l] * kPairPitch - T.c[2][l]]);
      const int kind = BCS ? kinds[idm] : 0;
      if (BCS && kind != 0) {
        const C* own = slot + ((i - 1) & 1) * (Q * SLOT);
        walls(h, idm, kind, mmm, [&](int l) { return own[l * SLOT]; });
      }
      pair_collide<LAT, COLL, C>(h, kind, p);
    }
    // The next plane's loads are waited for here, ahead of the stores: a wait at the top of the
    // loop would include the stores.
#pragma unroll
    for (int l = 0; l < Q; ++l) asm volatile("" : "+v"(pf[l]));
    if constexpr (BCS) asm volatile("" : "+v"(idn));
    if (inner) {
      if (i >= 2) {
        gchar* s = (gchar*)(fout + (size_t)Xo * xs);
        size_t pb = plane_bytes;
        asm volatile("" : "+s"(pb));
#pragma unroll
        for (int l = 0; l < Q; ++l) {
          uint32_t o = off[1][1];
          asm("" : "+s"(s), "+v"(o));
          R* d = reinterpret_cast<R*>(const_cast<char*>((const char*)s) + o);
          if constexpr (NT)
            st_pop<FMT, C>(d, h[l], T.w[l]);
          else
            *d = h[l];
          s += pb;
        }
      }
      asm volatile("" ::: "memory");  // the reads below stay behind the second update: fewer live values in it
#pragma unroll
      for (int l = 0; l < Q; ++l) {
        const C* m = buf + (l * SLOT - T.c[1][l] * kPairPitch - T.c[2][l]);
        if (T.c[0][l] == 0) c0[l] = *m;
        if (T.c[0][l] > 0) {
          cp2[l] = cp1[l];
          cp1[l] = *m;
        }
      }
    }
    idm = id;
    mmm = mm;
  }
}

// Tiles for a grid, or blocks = 0 where two launches of k_step take less time.  Both sides are
// estimates from measured times: a block takes 6.5 us per plane (FP32; FP64 5.3 us) whether or not
// the other CUs are busy, plus three planes to start and end a chunk; k_step streams 5.8 TB/s and
// takes 2 us to start.  (64^3 FP32: pair 25 us, two steps 18 us; 128^3: 91 and 110 us.)
template <int ROWS>
PairTiles pair_tiles(int nx, int ny, int nz, int q, int bytes) {
  constexpr int kCus = 256;
  PairTiles g;
  g.nzt = (nz + 63) / 64;
  g.nyt = (ny + ROWS - 3) / (ROWS - 2);
  g.ty = (ny + g.nyt - 1) / g.nyt;
  const int64_t tiles = (int64_t)g.nzt * g.nyt;
  g.cx = nx;
  double best = 0.0;
  for (int n = 1; n <= nx && (n == 1 || tiles * (n - 1) < 4 * kCus); ++n) {
    const int cx = (nx + n - 1) / n;
    const double t = (double)((tiles * ((nx + cx - 1) / cx) + kCus - 1) / kCus) * (cx + 3);
    if (best == 0.0 || t < best) {
      best = t;
      g.cx = cx;
    }
  }
  const int64_t blocks = tiles * ((nx + g.cx - 1) / g.cx);
  const double pair_us = best * (bytes == 8 ? 5.3 : 6.5);
  const double single_us = (double)nx * ny * nz * 2.0 * q * bytes / 5.8e6 + 2.0;
  g.blocks = pair_us < 2.0 * single_us && blocks < (int64_t)1 << 31 ? (int)blocks : 0;
  return g;
}

template <int LAT, int COLL, int FMT, class C, int ROWS>
int launch_pair_t(const StepCall& c, const PairTiles& g) {
  const StepParams p = step_params<LAT, FMT>(c);
  const bool nt = (size_t)c.nz * sizeof(C) % 128 == 0;
  auto go = [&](auto bcs, auto nts) {
    hipLaunchKernelGGL((k_step_pair<LAT, COLL, FMT, C, ROWS, decltype(bcs)::value, decltype(nts)::value>),
                       dim3(g.blocks), dim3((ROWS + 1) * 64), 0, c.stream, p, g);
  };
  auto with_nt = [&](auto bcs) {
    if (nt)
      go(bcs, std::true_type{});
    else
      go(bcs, std::false_type{});
  };
  if (c.bc_mask)
    with_nt(std::true_type{});
  else
    with_nt(std::false_type{});
  XLBH_LAUNCH_CHECK();
  return 0;
}

// Rows of a tile by precision.
constexpr int kPairRowsF32 = 15, kPairRowsF64 = 7;

// Whether two steps of a call can run as one launch, and its tiles (g.blocks > 0).  `known`: what
// may occur in the mask (XLBH_MASK_*, XLBH_KIND bits).
bool plan_pair(int lattice, const StepCall& c, uint32_t known, PairTiles& g);
int launch_pair(const StepCall& c, const PairTiles& g);

}  // namespace xlbh
