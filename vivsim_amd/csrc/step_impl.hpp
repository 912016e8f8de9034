// Host-side launch logic of the fused steps (validation, template dispatch,
// the N-step driver).  Included by step2d.hip and step3d.hip.
#pragma once
#include "step.hpp"

namespace vsx {

template <class L>
int validate_lbm(const VsxLbm *p) {
  if (!p) return fail(VSX_ERR_VALUE, "null parameters");
  if (p->nx < 3 || p->ny < 3 || (L::D == 3 ? p->nz < 3 : p->nz != 1))
    return fail(VSX_ERR_VALUE, "bad grid %d x %d x %d", p->nx, p->ny, p->nz);
  if ((int64_t)p->nx * p->ny * p->nz >= ((int64_t)1 << 31)) return fail(VSX_ERR_VALUE, "grid too large (>= 2^31 cells)");
  if (p->collision < VSX_COLL_BGK || p->collision > VSX_COLL_REG) return fail(VSX_ERR_VALUE, "unknown collision %d", p->collision);
  if (p->forcing < VSX_FORCE_NONE || p->forcing > VSX_FORCE_EDM) return fail(VSX_ERR_VALUE, "unknown forcing %d", p->forcing);
  if (p->storage < VSX_STORE_F32 || p->storage > VSX_STORE_E3M12S) return fail(VSX_ERR_VALUE, "unknown storage %d", p->storage);
  if (p->n_walls < 0 || p->n_walls > L::n_walls) return fail(VSX_ERR_VALUE, "bad wall count %d", p->n_walls);
  for (int k = 0; k < p->n_walls; ++k) {
    const VsxWall &w = p->walls[k];
    if (w.loc < 0 || w.loc >= L::n_walls) return fail(VSX_ERR_KEY, "unknown wall location %d", w.loc);
    if (w.kind < VSX_WALL_NEE || w.kind > VSX_WALL_SPECULAR) return fail(VSX_ERR_VALUE, "unknown wall kind %d", w.kind);
    if (w.mode < VSX_MODE_PLAIN || w.mode > VSX_MODE_FORCE_CORRECTED) return fail(VSX_ERR_VALUE, "unknown wall mode %d", w.mode);
  }
  return VSX_OK;
}

template <class L>
CtxOf<L> make_ctx(const VsxLbm &p, Window win) {
  CtxOf<L> c;
  c.p = p;
  c.win = win;
  c.dims[0] = p.nx;
  c.dims[1] = p.ny;
  c.dims[2] = L::D == 3 ? p.nz : 1;
  c.n = (int64_t)c.dims[0] * c.dims[1] * c.dims[2];
  for (int l = 0; l < 6; ++l) {
    c.order[l] = -1;
    c.at[l] = VsxWall{};
  }
  for (int k = 0; k < p.n_walls; ++k) {
    const int l = p.walls[k].loc;
    c.order[l] = c.order[l] == -1 ? k : -2;
    c.at[l] = p.walls[k];
  }
  // shift of the 16-bit storages: feq_i(1, store_u) (lbm/basic.py:114-135 at rho = 1)
  const float u0 = p.store_u[0], u1 = p.store_u[1], u2 = L::D == 3 ? p.store_u[2] : 0.f;
  const float usq = u0 * u0 + u1 * u1 + u2 * u2;
  for (int i = 0; i < 19; ++i) c.shift[i] = 0.f;
  for (int i = 0; i < L::Q; ++i) {
    const float cu = L::cx[i] * u0 + L::cy[i] * u1 + L::cz[i] * u2;
    c.shift[i] = L::w[i] * (1.f + 3.f * cu + 4.5f * cu * cu - 1.5f * usq);
  }
  return c;
}

template <class L>
void bulk_grid(const StepCtx &c, dim3 &grid, dim3 &block) {
  const int inner = L::D == 2 ? c.dims[1] : c.dims[2];
  int b = ((inner + 63) / 64) * 64;
  if (b > 256) b = 256;
  block = dim3(b);
  if (L::D == 2) grid = dim3((inner + b - 1) / b, c.dims[0]);
  else grid = dim3((inner + b - 1) / b, c.dims[1], c.dims[0]);
}

// The lines and faces of edge_cells: every pair of walled faces of two axes, and
// every face with two walls.
template <class L>
EdgeList make_edges(const StepCtx &c) {
  EdgeList E;
  int64_t cells = 0;
  auto add = [&](int la, int lb) {
    const int a = L::w_axis[la], b = lb >= 0 ? L::w_axis[lb] : -1;
    int64_t m = 1;
    for (int k = 0; k < 3; ++k)
      if (k != a && k != b) m *= c.dims[k];
    E.loc[E.n][0] = la;
    E.loc[E.n][1] = lb;
    E.begin[E.n++] = cells;
    cells += m;
  };
  for (int la = 0; la < L::n_walls; ++la) {
    if (c.order[la] == -1) continue;
    for (int lb = la + 1; lb < L::n_walls; ++lb)
      if (c.order[lb] != -1 && L::w_axis[lb] != L::w_axis[la]) add(la, lb);
    if (c.order[la] == -2) add(la, -1);
  }
  E.begin[E.n] = cells;
  return E;
}

template <class L, int COLL, int PHASE, class SRC, class DST>
void launch_bulk(const CtxOf<L> &c, const typename SRC::T *src, typename DST::T *dst, dim3 grid, dim3 block,
                 hipStream_t s) {
  if constexpr (PHASE != VSX_PHASE_COLLIDE) {
    if (c.p.n_walls > 0 && walls_need_edge<L>(c.p)) {
      const EdgeList E = make_edges<L>(c);
      const int64_t blocks = ((E.begin[E.n] << L::D) + block.x - 1) / block.x;
      const int64_t per_row = (int64_t)grid.x * (L::D == 2 ? 1 : grid.y);
      const int rows = (int)((blocks + per_row - 1) / per_row);
      (L::D == 2 ? grid.y : grid.z) += rows;
      hipLaunchKernelGGL((k_bulk_walls<L, COLL, PHASE, SRC, DST>), grid, block, 0, s, c, src, dst, E, rows);
      return;
    }
  }
  hipLaunchKernelGGL((k_bulk<L, COLL, PHASE, SRC, DST>), grid, block, 0, s, c, src, dst);
}

template <class L, int PHASE, class SRC, class DST>
int launch_phase(const CtxOf<L> &c, const void *src, void *dst, hipStream_t s) {
  dim3 grid, block;
  bulk_grid<L>(c, grid, block);
  auto S = static_cast<const typename SRC::T *>(src);
  auto D = static_cast<typename DST::T *>(dst);
  if constexpr (PHASE == VSX_PHASE_FULL) timer_begin(s);
  if constexpr (PHASE == VSX_PHASE_STREAM) {
    launch_bulk<L, VSX_COLL_BGK, PHASE, SRC, DST>(c, S, D, grid, block, s);
  } else {
    switch (c.p.collision) {
      case VSX_COLL_BGK: launch_bulk<L, VSX_COLL_BGK, PHASE, SRC, DST>(c, S, D, grid, block, s); break;
      case VSX_COLL_MRT: launch_bulk<L, VSX_COLL_MRT, PHASE, SRC, DST>(c, S, D, grid, block, s); break;
      case VSX_COLL_KBC: launch_bulk<L, VSX_COLL_KBC, PHASE, SRC, DST>(c, S, D, grid, block, s); break;
      default: launch_bulk<L, VSX_COLL_REG, PHASE, SRC, DST>(c, S, D, grid, block, s); break;
    }
  }
  if constexpr (PHASE == VSX_PHASE_FULL) timer_end(s);
  VSX_CHECK_LAUNCH();
  return VSX_OK;
}

// runtime (phase, src storage, dst storage) -> template instantiation
template <class L, class ST>
int phase_dispatch(const CtxOf<L> &c, const void *src, bool src_f32, void *dst, bool dst_f32, int phase, hipStream_t s) {
  using F32 = Store<VSX_STORE_F32>;
  switch (phase) {
    case VSX_PHASE_COLLIDE:
      return src_f32 ? launch_phase<L, VSX_PHASE_COLLIDE, F32, ST>(c, src, dst, s)
                     : launch_phase<L, VSX_PHASE_COLLIDE, ST, ST>(c, src, dst, s);
    case VSX_PHASE_FULL:
      // an FP32 work buffer larger than the last-level cache: non-temporal
      // field stores; below it, stores written through (FP32 only, which keeps
      // the kernel count of the generic step down)
      if constexpr (std::is_same_v<ST, Store<VSX_STORE_F32>>) {
        if ((size_t)c.n * L::Q * sizeof(float) > kLastLevelCacheBytes)
          return launch_phase<L, VSX_PHASE_FULL, ST, Streamed<ST>>(c, src, dst, s);
        if (write_through(c.n, L::Q, c.dims[L::D - 1], sizeof(float)))
          return launch_phase<L, VSX_PHASE_FULL, ST, Through<ST>>(c, src, dst, s);
      }
      return launch_phase<L, VSX_PHASE_FULL, ST, ST>(c, src, dst, s);
    case VSX_PHASE_STREAM:
      return dst_f32 ? launch_phase<L, VSX_PHASE_STREAM, ST, F32>(c, src, dst, s)
                     : launch_phase<L, VSX_PHASE_STREAM, ST, ST>(c, src, dst, s);
    default:
      return fail(VSX_ERR_VALUE, "unknown phase %d", phase);
  }
}

template <class L>
int step_any(const CtxOf<L> &c, const void *src, bool src_f32, void *dst, bool dst_f32, int phase, hipStream_t s) {
  switch (c.p.storage) {
    case VSX_STORE_F32: return phase_dispatch<L, Store<VSX_STORE_F32>>(c, src, true, dst, true, phase, s);
    case VSX_STORE_F16S: return phase_dispatch<L, Store<VSX_STORE_F16S>>(c, src, src_f32, dst, dst_f32, phase, s);
    case VSX_STORE_BF16S: return phase_dispatch<L, Store<VSX_STORE_BF16S>>(c, src, src_f32, dst, dst_f32, phase, s);
    default: return phase_dispatch<L, Store<VSX_STORE_E3M12S>>(c, src, src_f32, dst, dst_f32, phase, s);
  }
}

template <class L>
int step_entry(const VsxLbm *p, const void *src, int src_f32, void *dst, int dst_f32, int phase, void *stream) {
  int rc = validate_lbm<L>(p);
  if (rc) return rc;
  VSX_REQUIRE(src && dst && src != dst, "step needs distinct source and destination buffers");
  const CtxOf<L> c = make_ctx<L>(*p, Window{nullptr, nullptr, {0, 0, 0}});
  return step_any<L>(c, src, src_f32 != 0, dst, dst_f32 != 0, phase, as_stream(stream));
}

// The multi-operation runs (multi2d.hpp), per storage; operations per launch.
constexpr int kRunOps = 6;
// launches of a run of n steps, n + 1 operations (64 bits: n may be the largest int)
inline int64_t run_launches(int n) { return ((int64_t)n + kRunOps) / kRunOps; }
int multi2d_run_f32(const StepCtx &, const float *, float *, void *, void *, int, hipStream_t);
int multi2d_run_f16(const StepCtx &, const float *, float *, void *, void *, int, hipStream_t);
int multi2d_run_bf16(const StepCtx &, const float *, float *, void *, void *, int, hipStream_t);
int multi2d_run_e3m12(const StepCtx &, const float *, float *, void *, void *, int, hipStream_t);

// Whether a run goes through them: sides that hold the seam and its rings inside
// a tile, at most one wall per face, and no launch (run_multi) that reads a buffer
// it writes.  (Sides from 22 on would hold the seam and its rings without meeting
// their own copy; below 40 that has been neither tested nor timed.)  Single passes also take an input that is work_a (collided in place) and
// an output that is the work buffer idle at the end.
inline bool multi2d_takes(const StepCtx &c, const float *f_in, const float *f_out, const void *wa, const void *wb,
                          int n) {
  for (int l = 0; l < 4; ++l)
    if (c.order[l] == -2) return false;
  if (c.dims[0] < 40 || c.dims[1] < 40) return false;
  const size_t f = 9 * (size_t)c.n * sizeof(float), w = 9 * (size_t)c.n * store_bytes(c.p.storage);
  auto apart = [](const void *a, size_t na, const void *b, size_t nb) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return x + na <= y || y + nb <= x;
  };
  const int64_t launches = run_launches(n);
  if (launches == 1) return apart(f_in, f, f_out, f);
  return apart(f_in, f, wa, w) && apart(f_out, f, launches % 2 ? wb : wa, w);
}

inline int multi2d_run(const StepCtx &c, const float *f_in, float *f_out, void *wa, void *wb, int n, hipStream_t s) {
  switch (c.p.storage) {
    case VSX_STORE_F32: return multi2d_run_f32(c, f_in, f_out, wa, wb, n, s);
    case VSX_STORE_F16S: return multi2d_run_f16(c, f_in, f_out, wa, wb, n, s);
    case VSX_STORE_BF16S: return multi2d_run_bf16(c, f_in, f_out, wa, wb, n, s);
    default: return multi2d_run_e3m12(c, f_in, f_out, wa, wb, n, s);
  }
}

// n reference steps: COLLIDE(f_in -> a), FULL x (n-1) (a <-> b), STREAM(-> f_out)
template <class L>
int run_entry(const VsxLbm *p, const float *f_in, float *f_out, void *wa, void *wb, int n, void *stream) {
  int rc = validate_lbm<L>(p);
  if (rc) return rc;
  VSX_REQUIRE(f_in && f_out && wa, "null buffer");
  VSX_REQUIRE(n >= 0, "negative step count");
  VSX_REQUIRE(n <= 1 || wb, "need two work buffers for more than one step");
  hipStream_t s = as_stream(stream);
  const CtxOf<L> c = make_ctx<L>(*p, Window{nullptr, nullptr, {0, 0, 0}});
  if (n == 0) {
    if (f_out != f_in) VSX_HIP(hipMemcpyAsync(f_out, f_in, sizeof(float) * L::Q * c.n, hipMemcpyDeviceToDevice, s));
    return VSX_OK;
  }
  if constexpr (L::D == 2) {
    if (multi2d_takes(c, f_in, f_out, wa, wb, n)) return multi2d_run(c, f_in, f_out, wa, wb, n, s);
  }
  rc = step_any<L>(c, f_in, true, wa, false, VSX_PHASE_COLLIDE, s);
  if (rc) return rc;
  void *cur = wa, *nxt = wb;
  for (int t = 1; t < n; ++t) {
    rc = step_any<L>(c, cur, false, nxt, false, VSX_PHASE_FULL, s);
    if (rc) return rc;
    void *tmp = cur;
    cur = nxt;
    nxt = tmp;
  }
  return step_any<L>(c, cur, false, f_out, true, VSX_PHASE_STREAM, s);
}

}  // namespace vsx
