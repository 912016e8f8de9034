// Fused pull-scheme LBM step, generic over the lattice.
//
// The reference composes a time step from pure functions
//   macroscopic -> equilibrium -> collision -> forcing -> streaming -> walls
// (README.md:105-121, examples/2d/lid_driven_cavity.py:55-64,
// examples/2d/poiseuille_channel.py:80-128).  Here the stored state is the
// POST-COLLISION population field; one pass per cell
//   1. pulls f_i(x) = f_post_i(x - c_i) (periodic),
//   2. applies the ordered wall list to wall cells,
//   3. computes rho, u, adds the body force, collides and forces in registers,
//   4. writes the new post-collision populations of the cell.
// So every population is read once and written once per step (Q loads + Q
// stores = 72 B/cell D2Q9, 152 B/cell D3Q19 in FP32).  A run of N reference
// steps is one COLLIDE pass (the input is a post-streaming state), N-1 FULL
// passes and one STREAM pass that recovers the reference's post-streaming state.
//
// Wall cells: the reference applies each wall to the whole streamed array, in
// order, so a later wall can read cells an earlier wall rewrote (NEE reads the
// neighbour line) and the last writer wins at corners.  A cell on exactly one
// wall whose update reads no cell rewritten by an earlier wall is finished in
// the bulk kernel (one extra pull for the neighbour line).  The remaining cells
// (on walls of several axes) go to the first blocks of the same launch, a group
// of 2^D lanes per cell (edge_cells); they exist only when such cells do.
#pragma once
#include <cstddef>
#include <type_traits>
#include <utility>

#include "cell.hpp"
#include "common.hpp"
#include "lattice.hpp"
#include "wall.hpp"

namespace vsx {

// Body-force window written by the immersed-boundary kernels (device pointers).
struct Window {
  const int32_t *origin;   // [3] clamped window origin, or null (no window)
  const float *g;          // [D][S0][S1(][S2)]
  int32_t size[3];
};

// Sum over the stencil slots that land on window cell k of mf[m][a] * W[slot]
// (ib/stencil.py:81-110 as a gather), in slot order.
constexpr int kS3 = 64;   // stencil points per marker (4 x 4 x 4)
__device__ __forceinline__ void gather_cell3(const float *__restrict__ mf, const float *__restrict__ W,
                                             const int32_t *__restrict__ cell_ptr,
                                             const int32_t *__restrict__ cell_slot, int64_t k, float (&s)[3]) {
  s[0] = s[1] = s[2] = 0.f;
  const int e1 = cell_ptr[k + 1];
  int e = cell_ptr[k];
  for (; e + 4 <= e1; e += 4) {   // four slots' loads in flight, summed in slot order
    int slot[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) slot[u] = cell_slot[e + u];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = slot[u] / kS3;
      const float w = W[slot[u]];
#pragma unroll
      for (int a = 0; a < 3; ++a) s[a] += mf[3 * m + a] * w;
    }
  }
  for (; e < e1; ++e) {
    const int slot = cell_slot[e];
    const int m = slot / kS3;
    const float w = W[slot];
#pragma unroll
    for (int a = 0; a < 3; ++a) s[a] += mf[3 * m + a] * w;
  }
}

// Every wave waits for the lines of the argument segment that it reads before its
// first load, so what all kernels read there shares one line: the grid, the walls'
// order and the window's pointers.  The whole fills lines too.
struct alignas(64) StepCtx {
  VsxLbm p;
  alignas(64) int32_t dims[3];   // nx, ny, nz (nz = 1 in 2D)
  // Walls by location, so device code indexes walls only by compile-time
  // location: order[LOC] = position of the wall at LOC in p.walls (-1: none,
  // -2: several walls at LOC), at[LOC] = that wall.
  int32_t order[6];
  int64_t n;               // cells
  Window win;
  VsxWall at[6];
  float shift[19];         // 16-bit storage: stored value = f_i - shift[i] = f_i - feq_i(1, p.store_u)
};
static_assert(offsetof(StepCtx, win) % 64 + 2 * sizeof(void *) <= 64, "win.origin and win.g on the line of dims");

// 3D steps: the forces `F` [M][3] of the markers, gathered by the window's cells
// themselves (null: read from win.g); stencil weights and cell -> slot lists of
// vsx_ib3d_transpose_stencil; also stored in win.g.  Behind the rest, and in 3D only:
// within Window these 32 bytes moved fields across lines (us per step, within Window ->
// here and dims .. win.g on one line: periodic 32^3 KBC 4.64 -> 4.44, 64^3 9.00 -> 8.85,
// 65 x 64 x 63 11.56 -> 11.37, 96^3 24.5 -> 24.2, batch of 64 244.0 -> 239.8; with dims and order on
// two lines a 96 x 65 channel x 20 took 68.9 us instead of 67.9).
struct StepCtx3 : StepCtx {
  const float *F = nullptr, *W = nullptr;
  const int32_t *cell_ptr = nullptr, *cell_slot = nullptr;
};
template <class L>
using CtxOf = std::conditional_t<L::D == 3, StepCtx3, StepCtx>;

// The kernel's StepCtx argument, addressed in the kernarg segment (it is always
// the first kernel parameter, at offset 0).  Taking the context by reference
// from here, instead of from the by-value parameter, keeps the compiler from
// making a private per-lane copy of the ~1.4 KB block whenever a reference to
// it reaches a function that is not inlined.
template <class CTX = StepCtx>
__device__ __forceinline__ const CTX &kernel_ctx() {
  return *reinterpret_cast<const CTX *>((const char *)__builtin_amdgcn_kernarg_segment_ptr());
}

// Cell index (< 2^31 cells, checked on the host).  Populations are addressed as
// (uniform base of population i) + (32-bit cell offset), so every load is a
// scalar-base + 32-bit vector-offset access.
template <class L>
__device__ __forceinline__ uint32_t cell_of(const StepCtx &c, int x, int y, int z) {
  return ((uint32_t)x * (uint32_t)c.dims[1] + (uint32_t)y) * (uint32_t)c.dims[2] + (uint32_t)z;
}

__device__ __forceinline__ int wrap(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

template <class L, class SRC>
__device__ __forceinline__ void pull(const StepCtx &c, const typename SRC::T *__restrict__ src, int x, int y, int z,
                                     float (&f)[L::Q]) {
#pragma unroll
  for (int i = 0; i < L::Q; ++i) {
    const int xs = wrap(x - L::cx[i], c.dims[0]);
    const int ys = wrap(y - L::cy[i], c.dims[1]);
    const int zs = L::D == 3 ? wrap(z - L::cz[i], c.dims[2]) : 0;
    f[i] = SRC::ld(src + (size_t)i * c.n, cell_of<L>(c, xs, ys, zs), c.shift[i]);
  }
}

template <class L, class SRC>
__device__ __forceinline__ void local(const StepCtx &c, const typename SRC::T *__restrict__ src, uint32_t cell,
                                      float (&f)[L::Q]) {
#pragma unroll
  for (int i = 0; i < L::Q; ++i) f[i] = SRC::ld(src + (size_t)i * c.n, cell, c.shift[i]);
}

// component a of a coordinate triple, by selects (no dynamic register indexing)
__device__ __forceinline__ int comp3(const int (&v)[3], int a) { return a == 0 ? v[0] : (a == 1 ? v[1] : v[2]); }

// coordinates of the inward neighbour across wall `loc`
template <class L>
__device__ __forceinline__ void inward(int loc, const int (&co)[3], int (&cn)[3]) {
  const int a = L::w_axis[loc], sg = L::w_sign[loc];
  cn[0] = co[0] + (a == 0 ? sg : 0);
  cn[1] = co[1] + (a == 1 ? sg : 0);
  cn[2] = co[2] + (a == 2 ? sg : 0);
}

template <class L>
__device__ __forceinline__ bool on_wall(const StepCtx &c, int loc, const int (&co)[3]) {
  const int a = L::w_axis[loc];
  return comp3(co, a) == (L::w_sign[loc] > 0 ? 0 : comp3(c.dims, a) - 1);
}

// index of a cell along the wall (matches the per-node wall arrays)
template <class L>
__device__ __forceinline__ int64_t wall_node(const StepCtx &c, int loc, const int (&co)[3]) {
  const int a = L::w_axis[loc];
  if (a == 0) return (int64_t)co[1] * c.dims[2] + co[2];
  if (a == 1) return (int64_t)co[0] * c.dims[2] + co[2];
  return (int64_t)co[0] * c.dims[1] + co[1];
}

// Post-streaming, post-walls populations of cell co after walls [0, J).
// TAG only separates instantiations: an out-of-line function takes its register
// budget from the kernels that call it, so a kernel with a tight budget calls
// its own copy.
template <class L, class SRC, int J, int TAG = 0>
__device__ __noinline__ void wall_state(const StepCtx &c, const typename SRC::T *__restrict__ src, const int (&co)[3],
                                        float (&f)[L::Q]) {
  if constexpr (J == 0) {
    pull<L, SRC>(c, src, co[0], co[1], co[2], f);
  } else {
    wall_state<L, SRC, J - 1, TAG>(c, src, co, f);
    if (J - 1 < c.p.n_walls) {
      const VsxWall &w = c.p.walls[J - 1];
      if (on_wall<L>(c, w.loc, co)) {
        float fn[L::Q];
#pragma unroll
        for (int i = 0; i < L::Q; ++i) fn[i] = 0.f;
        if (wall_needs_neighbor(w)) {
          int cn[3];
          inward<L>(w.loc, co, cn);
          wall_state<L, SRC, J - 1, TAG>(c, src, cn, fn);
        }
        apply_wall<L>(w, wall_node<L>(c, w.loc, co), f, Held<L::Q>{fn},
                      [&](float (&fp)[L::Q]) { local<L, SRC>(c, src, cell_of<L>(c, co[0], co[1], co[2]), fp); });
      }
    }
  }
}

// Calls f(std::integral_constant<int, I>) for I = 0 .. N-1 (compile-time loop).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <class L, int LOC>
__device__ __forceinline__ bool on_wall_at(const StepCtx &c, const int (&co)[3]) {
  constexpr int a = L::w_axis[LOC];
  return co[a] == (L::w_sign[LOC] > 0 ? 0 : c.dims[a] - 1);
}

// Wall class of a cell: -1 on no wall; LOC when the cell is on exactly one wall
// (at location LOC) and that wall reads no neighbour rewritten by an earlier
// wall, so one pull and one wall update reproduce the ordered sequence; -2
// otherwise (cells on walls of several axes, left to edge_cells).
template <class L>
__device__ __forceinline__ int wall_class(const StepCtx &c, const int (&co)[3]) {
  int loc_on = -1, count = 0;
  static_for<L::n_walls>([&](auto LC) {
    constexpr int LOC = decltype(LC)::value;
    if (c.order[LOC] != -1 && on_wall_at<L, LOC>(c, co)) {
      loc_on = LOC;
      count += c.order[LOC] == -2 ? 2 : 1;
    }
  });
  if (count == 0) return -1;
  if (count > 1) return -2;
  int result = loc_on;
  static_for<L::n_walls>([&](auto LC) {
    constexpr int LOC = decltype(LC)::value;
    if (LOC == loc_on && wall_needs_neighbor(c.at[LOC])) {
      int cn[3];
      inward<L>(LOC, co, cn);
      static_for<L::n_walls>([&](auto L2C) {
        constexpr int L2 = decltype(L2C)::value;
        if (c.order[L2] >= 0 && c.order[L2] < c.order[LOC] && on_wall_at<L, L2>(c, cn)) result = -2;
      });
    }
  });
  return result;
}

// The wall of a cell of wall class cls >= 0 (the wall location) on its pulled
// populations.  In 2D the neighbour's loads are issued before anything waits for
// the cell's own: a second round trip in the wall tiles, the last to start,
// lengthens a launch (1024^2 VIV step 21.2 -> 22.4 us).  In 3D the registers that
// this holds cost more.
template <class L, class SRC>
__device__ __forceinline__ void single_wall(const StepCtx &c, const typename SRC::T *__restrict__ src,
                                            const int (&co)[3], int cls, float (&f)[L::Q]) {
  static_for<L::n_walls>([&](auto LC) {
    constexpr int LOC = decltype(LC)::value;
    if (LOC != cls) return;
    const VsxWall &w = c.at[LOC];
    auto nb = [&](float (&fn)[L::Q]) {
      int cn[3];
      inward<L>(LOC, co, cn);
      pull<L, SRC>(c, src, cn[0], cn[1], cn[2], fn);
    };
    auto pre = [&](float (&fp)[L::Q]) { local<L, SRC>(c, src, cell_of<L>(c, co[0], co[1], co[2]), fp); };
    if constexpr (L::D == 2) {
      float fn[L::Q];
#pragma unroll
      for (int i = 0; i < L::Q; ++i) fn[i] = 0.f;
      if (wall_needs_neighbor(w)) nb(fn);
      apply_wall_at<L, LOC>(w, wall_node<L>(c, LOC, co), f, Held<L::Q>{fn}, pre);
    } else {
      apply_wall_at<L, LOC>(w, wall_node<L>(c, LOC, co), f, nb, pre);
    }
  });
}

// Populations of a cell of wall class cls >= 0.
template <class L, class SRC>
__device__ __forceinline__ void single_wall_state(const StepCtx &c, const typename SRC::T *__restrict__ src,
                                                  const int (&co)[3], int cls, float (&f)[L::Q]) {
  pull<L, SRC>(c, src, co[0], co[1], co[2], f);
  single_wall<L, SRC>(c, src, co, cls, f);
}

// Post-streaming, post-walls populations of any cell.
template <class L, class SRC, int TAG = 0>
__device__ __forceinline__ void cell_state(const StepCtx &c, const typename SRC::T *__restrict__ src, const int (&co)[3],
                                           float (&f)[L::Q]) {
  const int cls = c.p.n_walls > 0 ? wall_class<L>(c, co) : -1;
  if (cls == -1) pull<L, SRC>(c, src, co[0], co[1], co[2], f);
  else if (cls >= 0) single_wall_state<L, SRC>(c, src, co, cls, f);
  else wall_state<L, SRC, L::n_walls, TAG>(c, src, co, f);
}

// Whether any cell can be of class -2: two walls on different axes (shared
// corners) or two walls at the same location.
template <class L>
inline bool walls_need_edge(const VsxLbm &p) {
  for (int i = 0; i < p.n_walls; ++i)
    for (int j = i + 1; j < p.n_walls; ++j)
      if (L::w_axis[p.walls[i].loc] != L::w_axis[p.walls[j].loc] || p.walls[i].loc == p.walls[j].loc) return true;
  return false;
}

// body force at a cell: uniform + optional full field + immersed-boundary window
// (window origin `org`, used when `win`)
template <class L>
__device__ __forceinline__ void body_force(const CtxOf<L> &c, uint32_t cell, const int (&co)[3], const int (&org)[3],
                                           bool win, float (&g)[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) g[a] = a < L::D ? c.p.g_uniform[a] : 0.f;
  if (c.p.g) {
#pragma unroll
    for (int a = 0; a < L::D; ++a) g[a] += c.p.g[(size_t)a * c.n + cell];
  }
  if (win) {
    int r[3];
    bool in = true;
#pragma unroll
    for (int a = 0; a < L::D; ++a) {
      r[a] = co[a] - org[a];
      in = in && r[a] >= 0 && r[a] < c.win.size[a];
    }
    if (in) {
      int k = r[0];
#pragma unroll
      for (int a = 1; a < L::D; ++a) k = k * c.win.size[a] + r[a];
      const int wn = c.win.size[0] * c.win.size[1] * (L::D == 3 ? c.win.size[2] : 1);
      if constexpr (L::D == 3) {
        if (c.F) {
          float s[3];
          gather_cell3(c.F, c.W, c.cell_ptr, c.cell_slot, k, s);
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const_cast<float *>(c.win.g)[a * wn + k] = s[a];
            g[a] += s[a];
          }
          return;
        }
      }
#pragma unroll
      for (int a = 0; a < L::D; ++a) {
        // 2D: the force window may come from the IB workgroup of this launch;
        // 3D: it was written by an earlier launch
        if constexpr (L::D == 2) g[a] += ld_agent(&c.win.g[a * wn + k]);
        else g[a] += c.win.g[a * wn + k];
      }
    }
  }
}

// window origin of the bulk kernels: read from the window buffer (device)
template <class L>
__device__ __forceinline__ bool window_origin_of(const StepCtx &c, int (&org)[3]) {
  org[0] = org[1] = org[2] = 0;
  if (!c.win.origin) return false;
#pragma unroll
  for (int a = 0; a < L::D; ++a) org[a] = c.win.origin[a];
  return true;
}

// collision + forcing of one cell, composed as in the reference examples:
//   Guo: u* = u + g / (2 rho) in the equilibrium and the forcing term (poiseuille_channel.py:99-128)
//   EDM: uncorrected u, f += F(g, u)                               (poiseuille_channel.py:84-97)
// Which of BGK's two products is rounded is written out (IN_PLACE: the unforced
// collision that opens a run): left to the compiler it depends on the code around,
// and kernels that run the same operation then differ in the last bit.
template <class L, int COLL, bool IN_PLACE = false>
__device__ __forceinline__ void collide_force(float (&f)[L::Q], float rho, const float (&u)[3], const float (&g)[3],
                                              int forcing, float omega, const float *rates) {
  const bool has_g = forcing != VSX_FORCE_NONE && (g[0] != 0.f || g[1] != 0.f || g[2] != 0.f);
  float ue[3] = {u[0], u[1], u[2]};
  if (has_g && forcing == VSX_FORCE_GUO) {
#pragma unroll
    for (int a = 0; a < L::D; ++a) ue[a] = u[a] + g[a] * 0.5f / rho;
  }
  float feq[L::Q];
  equilibrium<L>(rho, ue, feq);
  float F[L::Q];
  if (has_g) {
    const float (&uf)[3] = forcing == VSX_FORCE_GUO ? ue : u;
    const float ug = dot3<L>(g, uf);
#pragma unroll
    for (int i = 0; i < L::Q; ++i) F[i] = guo_i<L>(i, uf, g, ug);
  }
  bool forced = false;
  if constexpr (COLL == VSX_COLL_BGK) {
    const float a = 1.f - omega;
#pragma unroll
    for (int i = 0; i < L::Q; ++i)
      f[i] = IN_PLACE ? __builtin_fmaf(omega, feq[i], a * f[i]) : __builtin_fmaf(a, f[i], omega * feq[i]);
  } else if constexpr (COLL == VSX_COLL_KBC) {
    if constexpr (L::Q == 9) kbc_d2q9(f, feq, omega);
    else kbc_d3q19<L>(f, feq, omega);
  } else if constexpr (COLL == VSX_COLL_REG) {
    if constexpr (L::Q == 9) reg_d2q9(f, feq, omega);
    else reg_d3q19<L>(f, feq, omega);
  } else {  // MRT
    if constexpr (L::Q == 9) {
      float r[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) r[k] = rates[k];
      if (has_g && forcing == VSX_FORCE_GUO) {
        mrt_d2q9<true>(f, feq, F, r);
        forced = true;
      } else {
        mrt_d2q9<false>(f, feq, F, r);
      }
    } else {
      forced = has_g && forcing == VSX_FORCE_GUO;
      if (forced) mrt_d3q19<true>(f, feq, F, rates);
      else mrt_d3q19<false>(f, feq, F, rates);
    }
  }
  if (has_g && !forced) {
    const float s = forcing == VSX_FORCE_GUO ? (1.f - 0.5f * omega) : 1.f;
#pragma unroll
    for (int i = 0; i < L::Q; ++i) f[i] += F[i] * s;
  }
}

template <class L, class DST>
__device__ __forceinline__ void store_cell(const StepCtx &c, typename DST::T *__restrict__ dst, uint32_t cell,
                                           const float (&f)[L::Q]) {
#pragma unroll
  for (int i = 0; i < L::Q; ++i) DST::st(dst + (size_t)i * c.n, cell, f[i], c.shift[i]);
}

// finish() of a cell that carries no body force (no g field, no uniform g, not
// in the IB window): the forced branches are compiled out.
template <class L, int COLL, bool IN_PLACE = false>
__device__ __forceinline__ void finish_unforced(const StepCtx &c, float (&f)[L::Q]) {
  float rho, u[3];
  macroscopic<L>(f, rho, u);
  if constexpr (COLL == VSX_COLL_MRT && L::Q == 9) {
    float r[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) r[k] = c.p.mrt_rates[k];
    mrt_d2q9_unforced(f, rho, u, r);
  } else {
    const float g[3] = {0.f, 0.f, 0.f};
    collide_force<L, COLL, IN_PLACE>(f, rho, u, g, VSX_FORCE_NONE, c.p.omega, c.p.mrt_rates);
  }
}

template <class L, int COLL, bool IN_PLACE = false>
__device__ __forceinline__ void finish(const CtxOf<L> &c, uint32_t cell, const int (&co)[3], const int (&org)[3],
                                       bool win, float (&f)[L::Q]) {
  bool unforced = !win && !c.p.g;
#pragma unroll
  for (int a = 0; a < L::D; ++a) unforced = unforced && c.p.g_uniform[a] == 0.f;
  if (unforced) {
    finish_unforced<L, COLL, IN_PLACE>(c, f);
    return;
  }
  float rho, u[3], g[3];
  macroscopic<L>(f, rho, u);
  body_force<L>(c, cell, co, org, win, g);
  collide_force<L, COLL>(f, rho, u, g, c.p.forcing, c.p.omega, c.p.mrt_rates);
}

// ------------------------------------------------------------------ cells on several walls
// Lines of cells on the walls of two axes, and whole faces that carry two
// walls (host list, make_edges).
constexpr int kMaxEdges = 16;
struct EdgeList {
  int32_t n = 0;                   // entries
  int32_t loc[kMaxEdges][2];       // an edge: the two faces; a face: {loc, -1}
  int64_t begin[kMaxEdges + 1];    // first cell of each entry
};

// The cells of wall class -2.  The state of such a cell after wall w needs the
// state of its inward neighbour across w after the walls before w, and so on:
// for a cell on the walls of m axes, the 2^m cells reached by moving inward
// along any of these axes.  A group of 2^D lanes holds them, lane bit a set =
// moved inward along axis a; every lane pulls its own cell, then the walls are
// taken in list order, each lane on the wall reading its neighbour's populations
// from the lane of that bit.  Replayed by one thread as a recursion over the walls
// (scratch arrays, one chain of loads per level) these cells took 17 us of a
// 256^2 cavity step and 120 us of a 121 x 113 x 127 one, as a kernel of their own.
template <class L, int COLL, int PHASE, class SRC, class DST>
__device__ __forceinline__ void edge_cells(const CtxOf<L> &c, const EdgeList &E, int64_t t,
                                           const typename SRC::T *__restrict__ src,
                                           typename DST::T *__restrict__ dst) {
  constexpr int G = 1 << L::D;
  const int member = (int)(t % G);
  int64_t j = t / G;
  bool active = j < E.begin[E.n];
  int e = 0;
  for (int k = 1; k < E.n; ++k) e = j >= E.begin[k] ? k : e;
  j = active ? j - E.begin[e] : 0;
  int co[3] = {0, 0, 0};
  const int la = E.loc[e][0], lb = E.loc[e][1];
  const int a = L::w_axis[la], b = lb >= 0 ? L::w_axis[lb] : -1;
  // the free axes, fastest last (2D: axis 2 has one cell)
#pragma unroll
  for (int ax = 2; ax >= 0; --ax) {
    if (ax == a) {
      co[ax] = L::w_sign[la] > 0 ? 0 : c.dims[ax] - 1;
    } else if (ax == b) {
      co[ax] = L::w_sign[lb] > 0 ? 0 : c.dims[ax] - 1;
    } else {
      co[ax] = (int)(j % c.dims[ax]);
      j /= c.dims[ax];
    }
  }
  // inward direction per axis (0: on no wall of that axis)
  int s[3] = {0, 0, 0}, cn[3];
  static_for<L::n_walls>([&](auto LC) {
    constexpr int LOC = decltype(LC)::value;
    if (c.order[LOC] != -1 && on_wall_at<L, LOC>(c, co)) s[L::w_axis[LOC]] = L::w_sign[LOC];
  });
  // a cell on the walls of three axes is taken with the edge of axes 0 and 1,
  // a face's border with the edges
  if (b < 0) active = active && (s[0] != 0) + (s[1] != 0) + (s[2] != 0) == 1;
  else if (a + b != 1) active = active && !(s[0] && s[1] && s[2]);
#pragma unroll
  for (int ax = 0; ax < 3; ++ax) cn[ax] = co[ax] + ((member >> ax) & 1 ? s[ax] : 0);
  const uint32_t cell = cell_of<L>(c, cn[0], cn[1], cn[2]);
  float f[L::Q];
  pull<L, SRC>(c, src, cn[0], cn[1], cn[2], f);
  for (int k = 0; k < c.p.n_walls; ++k) {
    const VsxWall &w = c.p.walls[k];
    const int ax = L::w_axis[w.loc], sg = L::w_sign[w.loc];
    const bool on = comp3(s, ax) == sg && !((member >> ax) & 1);
    float fn[L::Q];
#pragma unroll
    for (int i = 0; i < L::Q; ++i) fn[i] = 0.f;
    if (wall_needs_neighbor(w)) {
#pragma unroll
      for (int i = 0; i < L::Q; ++i) fn[i] = __shfl_xor(f[i], 1 << ax, 64);
    }
    if (on)
      apply_wall<L>(w, wall_node<L>(c, w.loc, cn), f, Held<L::Q>{fn},
                    [&](float (&fp)[L::Q]) { local<L, SRC>(c, src, cell, fp); });
  }
  if (!active || member != 0) return;
  if constexpr (PHASE == VSX_PHASE_FULL) {
    int org[3];
    const bool win = window_origin_of<L>(c, org);
    finish<L, COLL>(c, cell, cn, org, win, f);
  }
  store_cell<L, DST>(c, dst, cell, f);
}

// ------------------------------------------------------------------ kernels
// Bulk: one thread per cell; blockIdx.x tiles the contiguous axis, blockIdx.y
// (and z in 3D) the others, so a wavefront touches 64 consecutive cells.
// k_bulk_walls: walls on several axes; the
// first `edge_rows` rows of the outermost grid axis hold the cells on several
// walls.  Their long chains (a few waves) run beside the bulk.  waves_per_eu sets
// the registers of both paths: in 2D those of the bulk path, what the edge path needs
// above it is spilled there; in 3D the bulk path with its walls spills too below
// 128 registers (MRT cavity, us per operation at 5, 4, 3 waves: 32^3 18.3, 13.6,
// 12.5; 96^3 36.0, 35.4, 39.4; 121 x 113 x 127 84.7, 68.6, 66.4).
template <class L>
constexpr int bulk_waves() {
  return L::D == 2 ? 8 : 4;
}

template <class L, int COLL, int PHASE, class SRC, class DST>
__device__ __forceinline__ void bulk_cells(const CtxOf<L> &c, int outer, const typename SRC::T *__restrict__ src,
                                           typename DST::T *__restrict__ dst) {
  int co[3];
  if constexpr (L::D == 2) {
    co[1] = blockIdx.x * blockDim.x + threadIdx.x;
    co[0] = outer;
    co[2] = 0;
    if (co[1] >= c.dims[1]) return;
  } else {
    co[2] = blockIdx.x * blockDim.x + threadIdx.x;
    co[1] = blockIdx.y;
    co[0] = outer;
    if (co[2] >= c.dims[2]) return;
  }
  const uint32_t cell = cell_of<L>(c, co[0], co[1], co[2]);
  int org[3];
  const bool win = window_origin_of<L>(c, org);
  float f[L::Q];
  if constexpr (PHASE == VSX_PHASE_COLLIDE) {
    local<L, SRC>(c, src, cell, f);
  } else {
    const int cls = c.p.n_walls > 0 ? wall_class<L>(c, co) : -1;
    if (cls < -1) return;   // cells on several walls: edge_cells
    pull<L, SRC>(c, src, co[0], co[1], co[2], f);
    // A wall across the contiguous axis takes one lane of a row's first or last
    // wave: the wave runs the wall update for it and goes on together. (With a path
    // of its own, finish and store included, such a wave did everything twice;
    // collected in blocks of their own, such lanes read the ends of every row a
    // second time on another XCD.  20 steps of a 121 x 113 x 127 MRT cavity, where
    // every wave has such a lane: 2.00, 1.97 and 1.75 ms.)
    if (cls >= 0) single_wall<L, SRC>(c, src, co, cls, f);
  }
  if constexpr (PHASE != VSX_PHASE_STREAM) finish<L, COLL, PHASE == VSX_PHASE_COLLIDE>(c, cell, co, org, win, f);
  store_cell<L, DST>(c, dst, cell, f);
}

template <class L, int COLL, int PHASE, class SRC, class DST>
__global__ __launch_bounds__(256) void k_bulk(CtxOf<L> c_arg, const typename SRC::T *__restrict__ src,
                                              typename DST::T *__restrict__ dst) {
  bulk_cells<L, COLL, PHASE, SRC, DST>(kernel_ctx<CtxOf<L>>(), L::D == 2 ? blockIdx.y : blockIdx.z, src, dst);
}

template <class L, int COLL, int PHASE, class SRC, class DST>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 256),
                          amdgpu_waves_per_eu(bulk_waves<L>(), bulk_waves<L>()))) void
k_bulk_walls(CtxOf<L> c_arg, const typename SRC::T *__restrict__ src, typename DST::T *__restrict__ dst, EdgeList E,
            int edge_rows) {
  const auto &c = kernel_ctx<CtxOf<L>>();
  const int outer = L::D == 2 ? blockIdx.y : blockIdx.z;
  if (outer < edge_rows) {
    const int64_t row = L::D == 2 ? (int64_t)outer : (int64_t)outer * gridDim.y + blockIdx.y;
    edge_cells<L, COLL, PHASE, SRC, DST>(c, E, (row * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x, src, dst);
    return;
  }
  bulk_cells<L, COLL, PHASE, SRC, DST>(c, outer - edge_rows, src, dst);
}

}  // namespace vsx
