// Several D2Q9 steps per launch (temporal blocking), the path of sim.LBM runs.
//
// A run of n reference steps is the operations
//   C   collide the caller's post-streaming field in place
//   F   pull, walls, collide (n - 1 times)
//   S   pull, walls: the caller's post-streaming result
// Done one per launch, each reads and writes the whole field: bound by HBM where
// the field exceeds the last-level cache, and by the launches (5-9 us each) where it
// is small.  Here a workgroup takes a tile through k operations: the first reads
// the tile and k - 1 cells around it from memory, the following work on the
// populations in LDS, each on one ring of cells less, and the last writes the
// tile.  Memory is read and written once per k operations; the rings are computed
// by several workgroups.
//
// The grid is a torus to the tiles (streaming is periodic, walls rewrite their
// cells afterwards), and the tiles are shifted so that the seam x = 0 and y = 0
// lies SX and SY cells inside a tile: every wall cell that a tile computes then
// has its inward neighbours in the tile's region, and the cells across the seam that the
// wall schemes read at the corners are computed like any others.  Tiles away
// from the seam hold no wall cell and wrap no index.
//
// Every cell is computed by the expressions of the one-operation passes
// (step.hpp), and 16-bit storages keep their codes in LDS too, so a run gives the
// populations that the passes one by one give.
#pragma once
#include "step_impl.hpp"

namespace vsx {

struct MultiArgs {
  int32_t k;                  // operations of this launch (2 .. kRunOps)
  int32_t first, last;        // operation 1 is C / operation k is S
  int32_t nty, tiles;         // tiles along y, all tiles
  int32_t store;              // field stores: 0 plain, 1 non-temporal, 2 written through
  uint32_t magic[kRunOps];    // magic[e] = ceil(2^20 / (TY + 2 e)): division by the row length of a region
};

// TX x TY tile, NT threads; a region of RX x RW cells in LDS
template <int TX_, int TY_, int NT_>
struct MultiCfg {
  static constexpr int TX = TX_, TY = TY_, KL = kRunOps, NT = NT_;
  static constexpr int RX = TX + 2 * (KL - 1), RW = TY + 2 * (KL - 1), RC = RX * RW;
  // waves per SIMD: two workgroups of 768 threads per CU, one of 1024 (whose wall
  // units then keep their three sets of populations in registers)
  static constexpr int WAVES = NT > 768 ? 4 : 6;
  // distance of the seam from its tile's edge: the wall cells on both sides of it,
  // their inward neighbours and those neighbours' own lie KL cells and more inside
  static constexpr int SX = KL + 2 > 8 ? 16 : 8, SY = TY >= 64 ? 16 : SX;
  static_assert(KL + 2 <= SX && SX + 3 <= TX && SY + 3 <= TY, "wall cells lie inside their tile");
  static_assert(NT % 64 == 0 && NT / 64 >= (RX > 64 || RW > 64 ? 12 : 8), "a wave for every wall and corner unit");
};

// The region in LDS is updated in place (the AA pattern: Bailey, Myre, Walsh, Lilja, Saar,
// "Accelerating lattice Boltzmann fluid flow simulations using graphics processors",
// ICPP 2009).  After an odd operation s population i
// of cell x lies at b[i][x]; the next one pulls b[i][x - c_i] and writes its
// result to b[opp i][x + c_i], the places it read; the one after that finds
// its pulled populations at b[opp i][x] and writes b[i][x].  So the cells of an
// operation read and write disjoint places and need no second buffer (which,
// at four operations, left one workgroup per CU instead of two).
// Pulled populations of region cell l in operation s > 1 ...
template <class ST, class CF>
__device__ __forceinline__ void lds_pull(const StepCtx &c, const typename ST::T *b, int s, int l, float (&f)[9]) {
  if (s & 1) {
#pragma unroll
    for (int i = 0; i < 9; ++i) f[i] = ST::cvt(b[D2Q9::opp[i] * CF::RC + l], c.shift[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) f[i] = ST::cvt(b[i * CF::RC + l - D2Q9::cx[i] * CF::RW - D2Q9::cy[i]], c.shift[i]);
  }
}
// ... its populations before that streaming ...
template <class ST, class CF>
__device__ __forceinline__ void lds_local(const StepCtx &c, const typename ST::T *b, int s, int l, float (&f)[9]) {
  if (s & 1) {
#pragma unroll
    for (int i = 0; i < 9; ++i)
      f[i] = ST::cvt(b[D2Q9::opp[i] * CF::RC + l + D2Q9::cx[i] * CF::RW + D2Q9::cy[i]], c.shift[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) f[i] = ST::cvt(b[i * CF::RC + l], c.shift[i]);
  }
}
// ... and its result.
template <class ST, class CF>
__device__ __forceinline__ void lds_put(const StepCtx &c, typename ST::T *b, int s, int l, const float (&f)[9]) {
  if (s & 1) {
#pragma unroll
    for (int i = 0; i < 9; ++i) b[i * CF::RC + l] = ST::enc(f[i], c.shift[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i)
      b[D2Q9::opp[i] * CF::RC + l + D2Q9::cx[i] * CF::RW + D2Q9::cy[i]] = ST::enc(f[i], c.shift[i]);
  }
}

// One workgroup's operations, in units of a wavefront: 64 consecutive cells of
// the region, or (SEAM) up to 64 cells of one wall, or one corner cell.  SEAM: the
// region may hold wall cells and wrap around the grid; otherwise it lies inside the
// grid away from the walls.  Each wall and corner unit has a wave of its own: as
// lanes of the cells' waves the walls' chains followed one another in a few
// waves, which the whole tile then waited for (256^2 cavity: 7.3 against 4.4 us per
// step).  A wall cell also reads places of its neighbour and, before streaming,
// its own, which other cells write: all wall reads come before a barrier.
template <int COLL, class ST, class CF, bool SEAM>
__device__ __forceinline__ void multi_tile(const StepCtx &c, const void *__restrict__ src, void *__restrict__ dst,
                                           const MultiArgs &a, int x0, int y0, typename ST::T *lds) {
  using T = typename ST::T;
  using F32 = Store<VSX_STORE_F32>;
  const float *sf = static_cast<const float *>(src);
  const T *ss = static_cast<const T *>(src);
  constexpr int M = CF::KL - 1;   // region cell (M, M) is the tile's first cell
  constexpr int NW = CF::NT / 64;
  const int nx = c.dims[0], ny = c.dims[1];
  const int org[3] = {0, 0, 0};
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // the last tile of an axis ends where the first begins
  const int vx = min(CF::TX, nx - CF::SX - x0), vy = min(CF::TY, ny - CF::SY - y0);
  // region coordinate of each wall (left, right, bottom, top), far off the
  // region where there is none; this wave's unit of walls and corners (-1: none):
  // 2 f + h = half h of wall f, 8 + q = corner q (bit 0: right, bit 1: top)
  int wl[4], unit = -1, n_list = 0;
  if constexpr (SEAM) {
    const int at[4] = {0, nx - 1, 0, ny - 1};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int n = f < 2 ? nx : ny;
      int p = at[f] - (f < 2 ? x0 : y0) + M;
      p = p < 0 ? p + n : (p >= n ? p - n : p);
      wl[f] = c.order[f] >= 0 && p < (f < 2 ? vx : vy) + 2 * M ? p : -4 * CF::RC;
    }
    auto add = [&](int v) { unit = n_list++ == wave ? v : unit; };
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (wl[q & 1] >= 0 && wl[2 + (q >> 1)] >= 0) add(8 + q);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (wl[f] >= 0) add(2 * f);
      if (wl[f] >= 0 && (f < 2 ? CF::RW : CF::RX) > 64) add(2 * f + 1);
    }
  }
  for (int s = 1; s <= a.k; ++s) {
    const int e = a.k - s, w = CF::TY + 2 * e, cells = w * (CF::TX + 2 * e);
    const bool in_place = a.first && s == 1, collide = !(a.last && s == a.k);
    auto coords = [&](int lx, int ly, int (&co)[3]) {
      co[0] = x0 - M + lx;
      co[1] = y0 - M + ly;
      co[2] = 0;
      if constexpr (SEAM) {
        co[0] = wrap(co[0], nx);
        co[1] = wrap(co[1], ny);
      }
    };
    auto pull_at = [&](const int (&co)[3], int l, int dx, int dy, float (&v)[9]) {
      if (s > 1) {
        lds_pull<ST, CF>(c, lds, s, l + dx * CF::RW + dy, v);
      } else if constexpr (SEAM) {
        pull<D2Q9, ST>(c, ss, co[0] + dx, co[1] + dy, 0, v);
      } else {
        const uint32_t cell = (uint32_t)co[0] * ny + co[1];
#pragma unroll
        for (int i = 0; i < 9; ++i)
          v[i] = ST::ld(ss + (size_t)i * c.n, cell - (uint32_t)(D2Q9::cx[i] * ny + D2Q9::cy[i]), c.shift[i]);
      }
    };
    auto emit = [&](const int (&co)[3], int l, float (&f)[9]) {
      const uint32_t cell = (uint32_t)co[0] * ny + co[1];
      if (COLL == VSX_COLL_BGK && in_place) finish<D2Q9, COLL, true>(c, cell, co, org, false, f);
      else if (collide) finish<D2Q9, COLL>(c, cell, co, org, false, f);
      if (s < a.k) lds_put<ST, CF>(c, lds, s, l, f);
      else if (a.last) store_cell<D2Q9, F32>(c, static_cast<float *>(dst), cell, f);
      else if (a.store == 1) store_cell<D2Q9, Streamed<ST>>(c, static_cast<T *>(dst), cell, f);
      else if (a.store == 2) store_cell<D2Q9, Through<ST>>(c, static_cast<T *>(dst), cell, f);
      else store_cell<D2Q9, ST>(c, static_cast<T *>(dst), cell, f);
    };
    const bool walls = SEAM && n_list > 0 && !in_place;
    if constexpr (SEAM) {
      if (walls) {
        bool on = false;   // this lane has a wall cell
        int lx = M, ly = M, co[3];
        float f[9], nb[9], pre[9];
        const int fa = unit < 8 ? unit >> 1 : unit & 1, fb = unit < 8 ? -1 : 2 + ((unit >> 1) & 1);
        if (unit >= 0) {
          if (unit < 8) {
            const int p = 64 * (unit & 1) + lane, at = fa & 2 ? (fa & 1 ? wl[3] : wl[2]) : (fa & 1 ? wl[1] : wl[0]);
            const int x = fa < 2 ? at : p, y = fa < 2 ? p : at;
            on = x >= M - e && x < M + vx + e && y >= M - e && y < M + vy + e &&
                 (fa < 2 ? y != wl[2] && y != wl[3] : x != wl[0] && x != wl[1]);
            lx = on ? x : M;
            ly = on ? y : M;
          } else {
            // a corner cell: four lanes as in edge_cells, lane bit 0 / 1: moved inward along x / y
            const int x = unit & 1 ? wl[1] : wl[0], y = unit & 2 ? wl[3] : wl[2];
            on = lane < 4 && x >= M - e && x < M + vx + e && y >= M - e && y < M + vy + e;
            lx = on ? x + (lane & 1 ? (unit & 1 ? -1 : 1) : 0) : M;
            ly = on ? y + (lane & 2 ? (unit & 2 ? -1 : 1) : 0) : M;
          }
          coords(lx, ly, co);
          pull_at(co, lx * CF::RW + ly, 0, 0, f);
          const VsxWall &wall = c.p.walls[c.order[fa]];
#pragma unroll
          for (int i = 0; i < 9; ++i) nb[i] = pre[i] = 0.f;
          if (fb < 0 && wall_needs_neighbor(wall) && on)
            pull_at(co, lx * CF::RW + ly, fa < 2 ? (fa & 1 ? -1 : 1) : 0, fa < 2 ? 0 : (fa & 1 ? -1 : 1), nb);
          if (wall_needs_pre(wall) || (fb >= 0 && wall_needs_pre(c.p.walls[c.order[fb]]))) {
            if (s == 1) local<D2Q9, ST>(c, ss, (uint32_t)co[0] * ny + co[1], pre);
            else lds_local<ST, CF>(c, lds, s, lx * CF::RW + ly, pre);
          }
        }
        if (s > 1 && s < a.k) __syncthreads();
        if (unit >= 0) {
          const bool swap = fb >= 0 && c.order[fb] < c.order[fa];   // the corner's walls in list order
          for (int j = 0; j < (fb < 0 ? 1 : 2); ++j) {
            const int face = (j == 0) != swap ? fa : fb, ax = face >> 1;
            const VsxWall &wall = c.p.walls[c.order[face]];
            if (fb >= 0) {
#pragma unroll
              for (int i = 0; i < 9; ++i) nb[i] = __shfl_xor(f[i], 1 << ax, 64);
            }
            if (on && (fb < 0 || !((lane >> ax) & 1)))
              apply_wall<D2Q9>(wall, ax == 0 ? co[1] : co[0], f, Held<9>{nb}, Held<9>{pre});
          }
          if (on && (fb < 0 || lane == 0)) emit(co, lx * CF::RW + ly, f);
        }
      }
    }
    // the other cells, first by the waves without a wall unit
    const int n_wall = walls ? n_list : 0;
#pragma unroll 1
    for (int u = wave < n_wall ? wave + NW - n_wall : wave - n_wall; u * 64 < cells; u += NW) {
      const int t = u * 64 + lane;
      const int ix = (int)((uint32_t)t * a.magic[e] >> 20), iy = t - ix * w;
      const int lx = M - e + ix, ly = M - e + iy, l = lx * CF::RW + ly;
      if (t >= cells || ix >= vx + 2 * e || iy >= vy + 2 * e) continue;
      if (SEAM && walls && (lx == wl[0] || lx == wl[1] || ly == wl[2] || ly == wl[3])) continue;
      int co[3];
      coords(lx, ly, co);
      float f[9];
      if (in_place) local<D2Q9, F32>(c, sf, (uint32_t)co[0] * ny + co[1], f);
      else pull_at(co, l, 0, 0, f);
      emit(co, l, f);
    }
    if (s < a.k) __syncthreads();
  }
}

template <int COLL, class ST, class CF>
__global__ __attribute__((amdgpu_flat_work_group_size(CF::NT, CF::NT), amdgpu_waves_per_eu(CF::WAVES))) void
k_multi2d(StepCtx c_arg, const void *__restrict__ src,
                                                    void *__restrict__ dst, MultiArgs a) {
  const StepCtx &c = kernel_ctx();
  __shared__ typename ST::T lds[9 * CF::RC];
  // neighbouring tiles on the same XCD (workgroups go to the 8 XCDs in turn), so
  // that the rings they share are read from its L2
  const int q = a.tiles / 8, r = a.tiles % 8, xcd = blockIdx.x % 8;
  const int tile = xcd * q + min(xcd, r) + (int)(blockIdx.x / 8);
  const int x0 = (tile / a.nty) * CF::TX - CF::SX, y0 = (tile % a.nty) * CF::TY - CF::SY;
  // the region and the cells it pulls from lie inside the grid, without wall cells
  const bool inside = x0 - CF::KL > 0 && y0 - CF::KL > 0 && x0 + CF::TX + CF::KL < c.dims[0] &&
                      y0 + CF::TY + CF::KL < c.dims[1];
  if (inside) multi_tile<COLL, ST, CF, false>(c, src, dst, a, x0, y0, lds);
  else multi_tile<COLL, ST, CF, true>(c, src, dst, a, x0, y0, lds);
}

// ------------------------------------------------------------------ host side

template <int COLL, class ST, class CF>
int run_multi(const StepCtx &c, const float *f_in, float *f_out, void *wa, void *wb, int n, hipStream_t s) {
  MultiArgs a;
  a.nty = (c.dims[1] + CF::TY - 1) / CF::TY;
  a.tiles = a.nty * ((c.dims[0] + CF::TX - 1) / CF::TX);
  const size_t bytes = sizeof(typename ST::T);
  a.store = (size_t)c.n * 9 * bytes > kLastLevelCacheBytes ? 1 : write_through(c.n, 9, c.dims[1], bytes) ? 2 : 0;
  for (int e = 0; e < kRunOps; ++e) a.magic[e] = ((1u << 20) + CF::TY + 2 * e - 1) / (CF::TY + 2 * e);
  // n + 1 operations in launches of equal size (2 and more each)
  const int64_t ops = (int64_t)n + 1, launches = run_launches(n);
  const void *cur = f_in;
  void *bufs[2] = {wa, wb};
  for (int64_t j = 0, done = 0; j < launches; ++j) {
    a.k = (int)((ops - done + launches - j - 1) / (launches - j));
    a.first = j == 0;
    a.last = j == launches - 1;
    void *dst = a.last ? f_out : bufs[j & 1];
    const int full = a.k - a.first - a.last;   // without the opening collision and the closing streaming
    if (full > 0) timer_begin(s);
    hipLaunchKernelGGL((k_multi2d<COLL, ST, CF>), dim3(a.tiles), dim3(CF::NT), 0, s, c, cur, dst, a);
    if (full > 0) timer_end(s, a.k, full);
    VSX_CHECK_LAUNCH();
    cur = dst;
    done += a.k;
  }
  return VSX_OK;
}

// The tile: large ones repeat less work on their rings and leave two workgroups per CU; small
// ones give each of the 256 CUs one where the grid has few cells (a step takes 4 us
// then, as long as a CU needs for one operation of a small region).  us per
// step, tiles of 16 x 16 | 16 x 32 | 20 x 64 | 40 x 64 (16-bit storage, whose region
// takes half the LDS), and one launch per operation: 256^2 cavity 3.8 | 4.3 | 5.9 and
// 8.2; 362^2 4.9 | 4.3 | 5.9 and 9.1; 512^2 6.9 | 5.5 | 5.9 and 11.2; 1031 x 777
// 18.0 | 12.3 | 8.0 and 15.0; 4000 x 2050 158 | 100 | 51 and 145; FP16S 1031 x 777
// 8.7 | 9.7 (20 x 64 | 40 x 64) and 11.2; 2048^2 29.3 | 26.4 and 32.9; 4000 x 2050 54.8 | 48.3 and 78.
// What bounds the large tiles is VALU issue: at 4000 x 2050 FP32 BGK it is busy throughout, LDS 23 %
// of the time, HBM at 31 % of peak; 237 instructions per cell and operation, rings included.
// Six operations per launch: with four the large tiles took 60 us at 4000 x 2050.
template <int COLL, class ST>
int run_multi_tiles(const StepCtx &c, const float *f_in, float *f_out, void *wa, void *wb, int n, hipStream_t s) {
  auto tiles = [&](int tx, int ty) {
    return (int64_t)((c.dims[0] + tx - 1) / tx) * ((c.dims[1] + ty - 1) / ty);
  };
  if (tiles(16, 16) <= 256) return run_multi<COLL, ST, MultiCfg<16, 16, 1024>>(c, f_in, f_out, wa, wb, n, s);
  if (tiles(16, 32) <= 512) return run_multi<COLL, ST, MultiCfg<16, 32, 1024>>(c, f_in, f_out, wa, wb, n, s);
  if constexpr (sizeof(typename ST::T) == 2) {
    if (tiles(40, 64) >= 512) return run_multi<COLL, ST, MultiCfg<40, 64, 768>>(c, f_in, f_out, wa, wb, n, s);
  }
  return run_multi<COLL, ST, MultiCfg<20, 64, 768>>(c, f_in, f_out, wa, wb, n, s);
}

// One instantiation per storage, each in a translation unit of its own.
template <class ST>
int multi2d_run_any(const StepCtx &c, const float *f_in, float *f_out, void *wa, void *wb, int n, hipStream_t s) {
  switch (c.p.collision) {
    case VSX_COLL_BGK: return run_multi_tiles<VSX_COLL_BGK, ST>(c, f_in, f_out, wa, wb, n, s);
    case VSX_COLL_MRT: return run_multi_tiles<VSX_COLL_MRT, ST>(c, f_in, f_out, wa, wb, n, s);
    case VSX_COLL_KBC: return run_multi_tiles<VSX_COLL_KBC, ST>(c, f_in, f_out, wa, wb, n, s);
    default: return run_multi_tiles<VSX_COLL_REG, ST>(c, f_in, f_out, wa, wb, n, s);
  }
}

}  // namespace vsx
