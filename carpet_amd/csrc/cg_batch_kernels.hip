// cg_batch_kernels.hip -- kernels of the batched level step.
//
// The transfers of one phase that share a kernel become one launch over a
// device-resident list of work items -- (descriptor, tile) pairs, transfers
// by decreasing size, each transfer's tiles in spatial order -- arranged in
// 8 segments, one per XCD, every transfer striped over all 8 in slabs of
// equal cost.  Two launch modes:
//  * persistent mode (default for tensor tiles): resident-capacity
//    workgroups take items from per-XCD counters, their own segment first,
//    then the others' (work stealing); items are taken in order, so the
//    tiles in flight on an XCD are neighbours that march through z together
//    and share halo rows in its L2; the loop ends for every workgroup once
//    all counters pass their segment ends, so the grid always drains;
//  * grid mode (default for pointwise runs): one workgroup per item;
//    workgroup b runs on XCD b % 8 (the hardware dispatches workgroups
//    round-robin over the XCDs) and takes slot b / 8 of that XCD's segment.
// Phases are separate launches in stream order (a kernel boundary makes one
// phase's results visible to the next across all XCD L2s), and the counters
// are cleared by a small kernel at the start of the step, so the whole step
// can be captured as one hipGraph.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <queue>
#include <vector>

#include "cg_batch_dev.hpp"

namespace cg {

// 256-point items per workgroup of pointwise classes of small regions in
// grid mode (k_grid_point_n)
#ifndef CG_POINT_NI
#define CG_POINT_NI 4
#endif

// destination stores of the pointwise kernels: nontemporal (1) or plain (0)
#ifndef CG_POINT_NT
#define CG_POINT_NT 1
#endif
__device__ __forceinline__ void point_store(double v, gdst_t p) {
  if constexpr (CG_POINT_NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// regions thin in x and long in y may take the 4x16-base tiles
#ifndef CG_SLIM_TILES
#define CG_SLIM_TILES 1
#endif

// tensor transfers of at most this many tiles run whole on one XCD
#ifndef CG_WHOLE_XCD_ITEMS
#define CG_WHOLE_XCD_ITEMS 16
#endif
constexpr int WHOLE_XCD_ITEMS = CG_WHOLE_XCD_ITEMS;

// default work items: pointwise = PT_DEFAULT consecutive destination points
// (x fastest); tensor = one x/y tile over ZCHUNK_DEFAULT coarse z bases
constexpr int PT_DEFAULT = 4096;
constexpr int ZCHUNK_DEFAULT = 16;



// points per thread and round of the pointwise kernel: items of 256, 512,
// 1024 points take one round of 1, 2, 4 points per thread, larger items
// rounds of 8 (a plain copy streams fastest with one point per thread and
// many small workgroups; stencils with several loads per point prefer more
// independent points per thread)
constexpr int pu_of(int pt) { return pt >= 2048 ? 8 : pt >= 1024 ? 4 : pt >= 512 ? 2 : 1; }

// coarse cells [tile*pt, tile*pt + pt) of a TVD region (fx/fxy divide by
// the parent-cell extents), each with all its children, NTL time levels
template <int NTL>
__device__ __forceinline__ void tvd_item(const PointArgs &a, unsigned tile, int pt) {
  int qx0, qy0, qz0, nqx, nqy, nqz;
  tvd_range(a, 0, &qx0, &nqx);
  tvd_range(a, 1, &qy0, &nqy);
  tvd_range(a, 2, &qz0, &nqz);
  const unsigned nxy = (unsigned)nqx * (unsigned)nqy;
  const unsigned tot = nxy * (unsigned)nqz; // < 2^31 (checked on the host)
  const unsigned e0 = tile * (unsigned)pt;
  const unsigned e1 = min(tot, e0 + (unsigned)pt);
  // TU cells per thread per round: every cell's loads before any store
  constexpr int TU = NTL == 1 ? 4 : 2;
  for (unsigned eb = e0; eb < e1; eb += 256u * TU) {
    TvdCell v[TU][NTL];
    int q[TU][3];
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      const unsigned e = eb + u * 256u + threadIdx.x;
      q[u][0] = -1;
      if (e < e1) {
        const unsigned k = fastdiv(e, a.fxy);
        const unsigned r = e - k * nxy;
        const unsigned j = fastdiv(r, a.fx);
        const unsigned i = r - j * (unsigned)nqx;
        q[u][0] = qx0 + (int)i;
        q[u][1] = qy0 + (int)j;
        q[u][2] = qz0 + (int)k;
#pragma unroll
        for (int tl = 0; tl < NTL; ++tl)
          v[u][tl] = tvd_load(a, tl, q[u][0], q[u][1], q[u][2]);
      }
    }
#pragma unroll
    for (int u = 0; u < TU; ++u)
      if (q[u][0] >= 0)
        tvd_store<NTL>(a, q[u][0], q[u][1], q[u][2], v[u]);
  }
}

// points [tile*pt, tile*pt + pt) of a region, x fastest; for TVD the
// items count the region's coarse parent cells
template <int OP, int PU>
__device__ __forceinline__ void point_item(const PointArgs &a, unsigned tile, int pt) {
  if constexpr (OP == PO_TVD) {
    if (a.ntl == 1)
      tvd_item<1>(a, tile, pt);
    else if (a.ntl == 2)
      tvd_item<2>(a, tile, pt);
    else
      tvd_item<3>(a, tile, pt);
  } else {
    const unsigned nx = (unsigned)a.nxp;
    const unsigned nxy = nx * (unsigned)a.n[1];
    const unsigned tot = nxy * (unsigned)a.n[2]; // < 2^31 (checked on the host)
    const unsigned e0 = tile * (unsigned)pt;
    const unsigned e1 = min(tot, e0 + (unsigned)pt);
    // PU points per thread per round: all loads first, then all stores, so
    // that PU loads per thread are in flight at once
    for (unsigned eb = e0; eb < e1; eb += 256u * PU) {
      double v[PU];
      long long o[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const unsigned e = eb + u * 256u + threadIdx.x;
        const unsigned k = fastdiv(e, a.fxy);
        const unsigned r = e - k * nxy;
        const unsigned j = fastdiv(r, a.fx);
        const int i = (int)(r - j * nx) - a.sx;
        o[u] = -1;
        if (e < e1 && i >= 0 && i < a.n[0]) {
          v[u] = point_value<OP>(a, i, (int)j, (int)k);
          o[u] = i + a.dj * j + a.dk * k;
        }
      }
#pragma unroll
      for (int u = 0; u < PU; ++u)
        if (o[u] >= 0)
          point_store(v[u], (gdst_t)a.dst + o[u]);
    }
  }
}

template <int OP, int PU>
__global__ __launch_bounds__(256) void k_persist_point(
    const PointArgs *__restrict__ descs, const Item *__restrict__ items,
    const int *__restrict__ seg, int *counter, int pt) {
  __shared__ int s_item;
  for (;;) {
    const int it = dequeue(counter, seg, &s_item);
    if (it < 0)
      return;
    const Item w = items[it];
    point_item<OP, PU>(descs[w.desc], w.tile, pt);
  }
}

template <int OP, int PU>
__global__ __launch_bounds__(256) void k_grid_point(const PointArgs *__restrict__ descs,
                                                    const Item *__restrict__ items,
                                                    const int *__restrict__ seg, int pt) {
  const int it = grid_item(seg);
  if (it < 0)
    return;
  const Item w = items[it];
  point_item<OP, PU>(descs[w.desc], w.tile, pt);
}

// Grid mode for classes of 256-point items: workgroup b takes NI
// consecutive slots of its XCD's segment (slots (b/8)*NI ..), one point of
// each per thread, and issues the loads of all NI items before the first
// store.  Regions of a hierarchy's ghost shells are a few hundred points;
// with one item per workgroup each thread has a single load in flight and
// the launch is bound by workgroup latency.
template <int OP, int NI>
__global__ __launch_bounds__(256) void k_grid_point_n(const PointArgs *__restrict__ descs,
                                                      const Item *__restrict__ items,
                                                      const int *__restrict__ seg) {
  static_assert(OP != PO_TVD, "TVD items run per coarse cell");
  const int x = blockIdx.x & 7;
  const int i0 = seg[x] + (int)(blockIdx.x >> 3) * NI, i1 = seg[x + 1];
  double v[NI];
  gdst_t q[NI]; // destination of each value, null outside the item
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    q[u] = nullptr;
    const int it = i0 + u;
    if (it < i1) {
      const Item w = items[it];
      const PointArgs &a = descs[w.desc];
      const unsigned nx = (unsigned)a.nxp;
      const unsigned nxy = nx * (unsigned)a.n[1];
      const unsigned tot = nxy * (unsigned)a.n[2];
      const unsigned e = w.tile * 256u + threadIdx.x;
      const unsigned k = fastdiv(e, a.fxy);
      const unsigned r = e - k * nxy;
      const unsigned j = fastdiv(r, a.fx);
      const int i = (int)(r - j * nx) - a.sx;
      if (e < tot && i >= 0 && i < a.n[0]) {
        v[u] = point_value<OP>(a, i, (int)j, (int)k);
        q[u] = (gdst_t)a.dst + (i + a.dj * j + a.dk * k);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < NI; ++u)
    if (q[u])
      point_store(v[u], q[u]);
}

// TVD items run per coarse cell with their own unrolling: one instance
// points per thread and round instantiated for an operator: TVD always 8
// (per coarse cell), the staggered operators 1 (up to 64 taps per point and
// time level), the others as asked
template <int OP> constexpr int pu_inst(int pu) {
  return OP == PO_TVD ? 8 : (OP == PO_STAGGER || OP == PO_RESTRICT_STAGGER) ? 1 : pu;
}

__global__ void k_zero_counters(int *c, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    c[i] = 0;
}

// ---------------------------------------------------------------------------
namespace {

struct Group {
  int phase, is_tensor, kind, order, ntl, op, prec;
  int small; // tensor regions routed to the 8x8-base (2) or 4x16-base (3) tiles, else 0
  int bigsh; // other tensor regions: the wide (0) or narrow (1) shape, per region
  std::vector<int> members; // transfer indices
  bool same(const Group &g) const {
    return phase == g.phase && is_tensor == g.is_tensor && kind == g.kind &&
           order == g.order && ntl == g.ntl && op == g.op && prec == g.prec && small == g.small &&
           bigsh == g.bigsh;
  }
};

int line_span(int kind, int order) {
  int span = 0;
  with_line(kind, order, [&](auto tag) -> int {
    using L = decltype(tag);
    span = L::TMAXALL - L::TMINALL;
    return 0;
  });
  return span;
}

// Lanes a region keeps busy in tiles of shape sh: tiles x (planes + stencil
// span) x (tile width) x (tile rows + span), the work of the window loads
// and of the x- and y-passes.
double tile_busy(const TensorArgs &a, int kind, int order, int ntl, int prec, int sh) {
  const int span = line_span(kind, order);
  int cx, cy, th;
  tile_shape(ntl, prec, &cx, &cy, &th, sh);
  return (double)tiles_x(a, cx, tile_shift(a, cx, prec ? 4 : 8, tile_cost(kind, order, ntl, prec))) * tiles_y(a, cy) *
         (a.nq[2] + span) * cx * (cy + span);
}

// An FP64 region goes to the small tiles when they keep at most 1/1.3 of
// the lanes busy that the better of the two large shapes would: a small
// tile's lane costs more (more tiles per region, each with its own ramp-up
// planes and halo).  (Measured, both workloads in one process: the level
// step of a 3-level hierarchy, whose boundary prolongation regions are 3-
// and 6-point shells, 1.14 ms against 1.61 ms without small tiles; 2000
// regions of 8-96 points per axis 19.41 ms against 19.53 ms, and 19.83 ms
// when routing at the break-even point 1.0.)
// Of the two small shapes: 4x16 for regions at most 4 bases across in x
// (one tile wide) where it keeps fewer lanes busy than 8x8 -- ghost and
// buffer faces normal to x -- else 8x8.  (Routing every region by the
// lane count alone sent 2000 regions of 8-96 points per axis with
// 5-12 bases in x to the 4x16 tiles: 18.59 ms per step against 17.46.)
int small_tiles(const ProlongPlan &p, int ntl, int prec) {
  if (prec != CG_PREC_F64)
    return 0;
  auto busy = [&](int sh) { return tile_busy(p.t, p.kind, p.order, ntl, prec, sh); };
  const double big = std::min(busy(0), busy(1));
  const double b2 = busy(2), b3 = busy(3);
  const int sh = CG_SLIM_TILES && p.t.nq[0] <= 4 && b3 < b2 ? 3 : 2;
  return (sh == 3 ? b3 : b2) * 1.3 <= big ? sh : 0;
}

// Regions of one kernel whose shapes fall into three classes or more run as
// one class on the 8x8 tiles where the chip holds few rounds of those: every
// class beyond the first costs a launch, a fork and a join of streams, and a
// tail.  Up to 32 tiles a CU that is more than the better shapes give; up to
// 128 only if the small tiles keep at most a quarter more lanes busy.  (In
// several classes against one: 300 regions of 5-31 points per axis x 3, order
// 3, 2 levels 62 against 29 us, from a graph 45 against 33; a 3-level
// hierarchy of 64^3 coarse points x 4 116 against 86 us, of 128^3 x 12, which
// keeps its classes, 475 against 488 us; 432 boxes x 4 1.274 against 1.240
// ms; 1000 regions of 8-60 points 626 against 598 us.)  Fewer than 128 regions,
// and the phases of the bit mask keep, which the caller has named a mode for,
// keep their classes, so that they can run beside each other or in turn
// (cg_batch_set_phase_mode).
constexpr long long MERGE_POINTS = 1 << 18; // per region
void merge_small_classes(const std::vector<Transfer> &tr, std::vector<Group> &per, int ncu, unsigned keep) {
  std::vector<char> done(per.size(), 0);
  for (size_t i = 0; i < per.size(); ++i) {
    if (done[i] || !per[i].is_tensor || per[i].prec != CG_PREC_F64 || (keep >> per[i].phase & 1))
      continue;
    std::vector<size_t> same;
    long long items = 0;
    double busy = 0, busy8 = 0;
    bool small = true;
    int seen = 0; // shapes, a bit each
    for (size_t j = i; j < per.size(); ++j) {
      const Group &g = per[j];
      if (!g.is_tensor || g.phase != per[i].phase || g.kind != per[i].kind || g.order != per[i].order ||
          g.ntl != per[i].ntl || g.prec != per[i].prec)
        continue;
      same.push_back(j);
      done[j] = 1;
      seen |= 1 << (g.small ? g.small : g.bigsh);
      const TensorArgs &a = tr[j].pr.t;
      small = small && tr[j].dst_points() <= MERGE_POINTS;
      busy += tile_busy(a, g.kind, g.order, g.ntl, g.prec, g.small ? g.small : g.bigsh);
      busy8 += tile_busy(a, g.kind, g.order, g.ntl, g.prec, 2);
      const int sx = tile_shift(a, 8, 8, tile_cost(g.kind, g.order, g.ntl, g.prec));
      items += (long long)tiles_x(a, 8, sx) * tiles_y(a, 8) * ((a.nq[2] + 7) / 8);
    }
    if (small && __builtin_popcount((unsigned)seen) >= 3 && same.size() >= 128 &&
        items <= (busy8 <= 1.25 * busy ? 128LL : 32LL) * ncu)
      for (size_t j : same) {
        per[j].small = 2;
        per[j].bigsh = 0;
      }
  }
}

// one transfer's descriptor in launch l: a tensor transfer resolved to one
// time level (its target time matches level 0 exactly) inside a class of
// more levels keeps nlev = 1 and reads level 0 for every level slot; a
// same-level interpolation resolved to a copy stays an interpolation of one
// level
TensorArgs tensor_desc(const BatchLaunch &l, const Transfer &t, int sx = -1) {
  TensorArgs a = t.pr.t;
  for (int k = a.nlev; k < l.ntl; ++k)
    a.src[k] = a.src[0];
  a.sx = sx;
  TileCfg cfg;
  int th = 0;
  tile_shape(l.ntl, l.prec, &cfg.cx, &cfg.cy, &th, l.shape);
  cfg.zchunk = l.zchunk;
  cfg.es = l.prec ? 4 : 8;
  cfg.cost = tile_cost(l.kind, l.order, l.ntl, l.prec);
  (void)tensor_tiles(a, cfg);
  return a;
}

// work units of a pointwise transfer per axis: row slots, or TVD's coarse
// parent cells
void point_units(const BatchLaunch &l, const PointArgs &a, long long *u) {
  for (int d = 0; d < 3; ++d)
    u[d] = l.op == PO_TVD ? ((a.off[d] + a.n[d] - 1) >> 1) - (a.off[d] >> 1) + 1 : d == 0 ? a.nxp : a.n[d];
}

// nxp > 0: the row slots that the transfer's items were cut with
PointArgs point_desc(const BatchLaunch &l, const Transfer &t, int sx = 0, int nxp = 0) {
  PointArgs a = t.is_prolong ? t.pr.p : t.pt.a;
  if (l.op == PO_INTERP && !t.is_prolong && t.pt.op == PO_COPY) {
    a.ntl = 1;
    a.s[0] = 1.0;
  }
  a.sx = 0;
  a.nxp = a.n[0];
  if (l.op != PO_TVD)
    point_rows(l.op, a);
  if (nxp > 0) {
    a.sx = sx;
    a.nxp = nxp;
  }
  long long u[3];
  point_units(l, a, u);
  // (planes of 2^31 units and more are refused: no divisor, which cut to 32
  // bits may be 0)
  if (u[0] * u[1] < (1LL << 31)) {
    a.fx = make_fastdiv((unsigned)u[0]);
    a.fxy = make_fastdiv((unsigned)(u[0] * u[1]));
  }
  return a;
}

template <int SH> const void *tensor_fn_sh(const BatchLaunch &l, int *threads) {
  switch (l.kind) {
  case LK_VLAG: return batch_tensor_fn_kind<LK_VLAG, SH>(l, threads);
  case LK_CLAG: return batch_tensor_fn_kind<LK_CLAG, SH>(l, threads);
  case LK_ENO: return batch_tensor_fn_kind<LK_ENO, SH>(l, threads);
  case LK_VENO: return batch_tensor_fn_kind<LK_VENO, SH>(l, threads);
  }
  return nullptr;
}

template <int SH>
int tensor_run_sh(const BatchLaunch &l, const TensorArgs *td, const Item *items, const int *seg, int *ctr,
                  hipStream_t st) {
  switch (l.kind) {
  case LK_VLAG: return batch_tensor_kind<LK_VLAG, SH>(l, td, items, seg, ctr, st);
  case LK_CLAG: return batch_tensor_kind<LK_CLAG, SH>(l, td, items, seg, ctr, st);
  case LK_ENO: return batch_tensor_kind<LK_ENO, SH>(l, td, items, seg, ctr, st);
  case LK_VENO: return batch_tensor_kind<LK_VENO, SH>(l, td, items, seg, ctr, st);
  }
  return -1;
}

template <int OP> const void *persist_point_pu(int pu) {
  switch (pu_inst<OP>(pu)) {
  case 1: return reinterpret_cast<const void *>(&k_persist_point<OP, 1>);
  case 2: return reinterpret_cast<const void *>(&k_persist_point<OP, 2>);
  case 4: return reinterpret_cast<const void *>(&k_persist_point<OP, 4>);
  }
  return reinterpret_cast<const void *>(&k_persist_point<OP, pu_inst<OP>(8)>);
}

const void *persist_point_fn(int op, int pt) {
  const int pu = pu_of(pt);
  switch (op) {
  case PO_COPY: return persist_point_pu<PO_COPY>(pu);
  case PO_RESTRICT_VC: return persist_point_pu<PO_RESTRICT_VC>(pu);
  case PO_RESTRICT_CC: return persist_point_pu<PO_RESTRICT_CC>(pu);
  case PO_INTERP: return persist_point_pu<PO_INTERP>(pu);
  case PO_TVD: return persist_point_pu<PO_TVD>(pu);
  case PO_RESTRICT_CC_O3: return persist_point_pu<PO_RESTRICT_CC_O3>(pu);
  case PO_RESTRICT_CC_O5: return persist_point_pu<PO_RESTRICT_CC_O5>(pu);
  case PO_MONO5: return persist_point_pu<PO_MONO5>(pu);
  case PO_STAGGER: return persist_point_pu<PO_STAGGER>(pu);
  case PO_RESTRICT_STAGGER: return persist_point_pu<PO_RESTRICT_STAGGER>(pu);
  case PO_RESTRICT_VC2: return persist_point_pu<PO_RESTRICT_VC2>(pu);
  }
  return nullptr;
}

const void *launch_fn(const BatchLaunch &l, int *threads) {
  if (!l.is_tensor) {
    *threads = 256;
    return persist_point_fn(l.op, l.pt);
  }
  switch (l.shape) {
  case 0: return tensor_fn_sh<0>(l, threads);
  case 1: return tensor_fn_sh<1>(l, threads);
  case 2: return tensor_fn_sh<2>(l, threads);
  case 3: return tensor_fn_sh<3>(l, threads);
  }
  return nullptr;
}

} // namespace

void batch_device_free(BatchDevice &dev) {
  for (hipStream_t s : dev.aux)
    (void)hipStreamSynchronize(s);
  for (hipStream_t s : dev.aux)
    (void)hipStreamDestroy(s);
  for (hipEvent_t e : dev.join)
    (void)hipEventDestroy(e);
  for (hipEvent_t e : dev.fork)
    (void)hipEventDestroy(e);
  dev.aux.clear();
  dev.join.clear();
  dev.fork.clear();
  if (dev.blob)
    (void)hipFree(dev.blob);
  if (dev.counters)
    (void)hipFree(dev.counters);
  dev.blob = nullptr;
  dev.counters = nullptr;
  dev.launches.clear();
  dev.blob_bytes = 0;
  dev.ncounters = 0;
}

static int ilog2(long long v) {
  int r = 0;
  while (v > 1) {
    v >>= 1;
    ++r;
  }
  return r;
}

void batch_launch_descs(const BatchLaunch &l, const std::vector<Transfer> &tr, char *out) {
  for (size_t i = 0; i < l.members.size(); ++i) {
    const Transfer &t = tr[l.members[i]];
    if (l.is_tensor) {
      const TensorArgs a = tensor_desc(l, t, l.sx[i]);
      std::memcpy(out + i * sizeof(TensorArgs), &a, sizeof a);
    } else {
      const PointArgs a = point_desc(l, t, l.sx[i], l.nxp[i]);
      std::memcpy(out + i * sizeof(PointArgs), &a, sizeof a);
    }
  }
}

int batch_device_build(BatchDevice &dev, const std::vector<Transfer> &tr,
                       const std::vector<int> &phase, const std::vector<int> &prec,
                       const std::vector<int> &cls_ntl, std::vector<char> &shapes, int tile_cfg,
                       const TuneMap *tuned, int only, unsigned keep_phases) {
  batch_device_free(dev);
  // group transfers by (phase, kernel)
  const bool chosen = !shapes.empty();
  std::vector<Group> groups, per;
  for (size_t i = 0; i < tr.size(); ++i) {
    Group g{};
    g.phase = phase[i];
    g.prec = prec[i];
    if (tr[i].is_prolong && tr[i].pr.kind != PK_TVD && tr[i].pr.kind != PK_MONO5 &&
        tr[i].pr.kind != PK_STAGGER) {
      g.is_tensor = 1;
      g.small = chosen ? 0 : small_tiles(tr[i].pr, cls_ntl[i], prec[i]);
      // the large shape that keeps fewer lanes busy on this region -- tiles x
      // (planes + stencil span) x (tile width) x (tile rows + span), the work
      // of the window loads and of the x- and y-passes -- with a 25% margin
      // for the wide tile, which is faster per lane on large regions
      // (single 512^3 patch: narrow 0.81x the busy lanes of wide, yet 4%
      // slower).  Per region rather than per class: 0.6% faster on 2000
      // regions of 8-96 points per axis, 1.8% and 1.2% on the level steps
      // of the 3-level and the 2000-box hierarchies.
      // FP32 rows that lose their place in a 128-byte line from row to row take
      // the wide tile from a smaller margin on: a narrow tile's row is one line
      // long and goes out in two parts (6 x 256^3 in unpadded rows, order 9: 295
      // us narrow, 156 wide, at 0.73 of the busy lanes).
      g.bigsh = 0;
      if (!chosen && !g.small) {
        const ProlongPlan &p = tr[i].pr;
        const bool split = prec[i] == CG_PREC_MIXED && (p.t.dj % 32 || p.t.dk % 32);
        const double b0 = tile_busy(p.t, p.kind, p.order, cls_ntl[i], prec[i], 0);
        const double b1 = tile_busy(p.t, p.kind, p.order, cls_ntl[i], prec[i], 1);
        g.bigsh = b1 < (split ? 0.6 : 0.75) * b0 ? 1 : 0;
      }
      g.kind = tr[i].pr.kind;
      g.order = tr[i].pr.order;
      g.ntl = cls_ntl[i];
      g.op = -1;
    } else {
      g.is_tensor = 0;
      g.kind = g.order = -1;
      g.ntl = 1;
      g.op = !tr[i].is_prolong            ? tr[i].pt.op
             : tr[i].pr.kind == PK_MONO5   ? PO_MONO5
             : tr[i].pr.kind == PK_STAGGER ? PO_STAGGER
                                           : PO_TVD;
    }
    per.push_back(g);
  }
  int dev_id = 0, ncu = 0;
  hipError_t he = hipGetDevice(&dev_id);
  if (he != hipSuccess)
    return hip_error(he, "hipGetDevice");
  he = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev_id);
  if (he != hipSuccess)
    return hip_error(he, "hipDeviceGetAttribute");
  if (!chosen) {
    merge_small_classes(tr, per, ncu, keep_phases);
    shapes.resize(tr.size());
  }
  for (size_t i = 0; i < tr.size(); ++i) {
    if (chosen) {
      per[i].small = shapes[i] >= 2 ? shapes[i] : 0;
      per[i].bigsh = shapes[i] == 1;
    } else {
      shapes[i] = (char)(per[i].small ? per[i].small : per[i].bigsh);
    }
    const Group &g = per[i];
    auto it = std::find_if(groups.begin(), groups.end(), [&](const Group &x) { return x.same(g); });
    if (it == groups.end()) {
      groups.push_back(g);
      it = groups.end() - 1;
    }
    it->members.push_back((int)i);
  }
  std::stable_sort(groups.begin(), groups.end(),
                   [](const Group &a, const Group &b) { return a.phase < b.phase; });

  // host image of the blob: per launch, descriptors then items (8-byte aligned)
  std::vector<char> host;
  auto append = [&](const void *p, size_t n) {
    size_t off = (host.size() + 15) / 16 * 16;
    host.resize(off + n);
    if (n)
      std::memcpy(host.data() + off, p, n);
    return off;
  };
  for (size_t gi = 0; gi < groups.size(); ++gi) {
    const Group &g = groups[gi];
    if (only >= 0 && (int)gi != only)
      continue;
    if (g.prec != CG_PREC_F64 && (!g.is_tensor || fp64_only(g.kind)))
      return set_error(CG_ERR_OPERATOR, "mixed precision applies to Lagrange prolongation only");
    BatchLaunch l{};
    l.phase = g.phase;
    l.is_tensor = g.is_tensor;
    l.kind = g.kind;
    l.order = g.order;
    l.ntl = g.ntl;
    l.op = g.op;
    l.prec = g.prec;
    // key of the tuner cache: kernel class + box-size histogram bucket
    // (log2 of the median destination points per transfer) + count bucket
    long long median_pts = 0, class_pts = 0;
    int levels = 1; // the most time levels that a member combines
    {
      std::vector<long long> pts;
      for (int m : g.members)
        pts.push_back(tr[m].dst_points());
      for (long long n : pts)
        class_pts += n;
      for (int m : g.members)
        levels = std::max(levels, !tr[m].is_prolong ? tr[m].pt.a.ntl : g.is_tensor ? tr[m].pr.ntl : tr[m].pr.p.ntl);
      std::nth_element(pts.begin(), pts.begin() + pts.size() / 2, pts.end());
      median_pts = pts[pts.size() / 2];
      char key[128];
      snprintf(key, sizeof key, "%s k%d o%d t%d p%d op%d h%d n%d",
               !g.is_tensor ? "point" : g.small == 3 ? "tensor4" : g.small ? "tensor8" : g.bigsh == 1 ? "tensorN" : "tensor",
               g.kind, g.order, g.ntl, g.prec, g.op, ilog2(median_pts),
               ilog2((long long)g.members.size()));
      l.key = key;
    }
    l.zchunk = tile_cfg < 0 ? ZCHUNK_DEFAULT : tile_cfg;
    l.pt = PT_DEFAULT;
    // pointwise classes of small regions (median under 2048 points, such as
    // the ghost and restriction slabs of a hierarchy's components): items of
    // 256 points, one per thread, so a region spreads over several
    // workgroups (the tuner's choice on such classes)
    l.ni = 1;
    if (!g.is_tensor && median_pts < 2048) {
      l.pt = 256;
      l.ni = CG_POINT_NI;
    }
    // TVD items count coarse parent cells (8 fine points each): 1024 cells
    // (8 variables of 192^3 -> 384^3: 0.98 ms against 1.00 ms with 512, 1.01
    // with 2048 and 1.10 with 256); cell restriction of order 3 1024 points, of
    // order 5, 216 terms each, 512 (60 of 60x40x40 and of 100x40x40 points: 376
    // and 605 us, against 408 and 653 with 1024)
    else if (g.op == PO_TVD || g.op == PO_RESTRICT_CC_O3)
      l.pt = 1024;
    else if (g.op == PO_RESTRICT_CC_O5)
      l.pt = 512;
    // cell-centred restriction (8 children per point): 256 (the 384^3 ->
    // 192^3 restriction of the same set, at 256, 512, 1024 and 4096: 0.70,
    // 0.74, 0.76 and 0.79 ms)
    else if (g.op == PO_RESTRICT_CC)
      l.pt = 256;
    // copies 1024 slots, injections 512 (2000 regions of 8-96 points per
    // axis x 4, at 512, 1024, 2048 and 4096: copies 1.53, 1.29, 1.45 and
    // 1.53 ms, injections 0.279, 0.304, 0.311 and 0.317 ms)
    else if (g.op == PO_COPY)
      l.pt = 1024;
    else if (g.op == PO_RESTRICT_VC)
      l.pt = 512;
    // tensor tiles of very large regions (median 2^25 points and up):
    // persistent grid (its workgroups take the tiles in order, so
    // neighbouring tiles march through z together and share halo rows in
    // L2); other tensor classes and pointwise runs: one workgroup per item.
    // (Persistent against one per item: 4 x 512^3 order 5, 3 levels, a pass
    // among those of other arrays 1343 and 1377 us, alone 1381 and 1357; 8 x
    // 384^3 with FP32 storage 597 and 602 us, alone 664 and 637; the same
    // arrays again and again 1284 and 1243, 641 and 615; 4 x 384^3 cell
    // ENO<3>, 3 levels, equal; below the line 5 x 256^3 vertex ENO, 3 levels,
    // 378 and 323.)  Regions of 2^20 points and up whose items fit one round
    // of resident workgroups have a mode of their own (one_round, below).
    l.wpc = g.is_tensor && !g.small && median_pts >= (1LL << 25) ? 0 : -1;
    // tile shape: the class's (its regions were routed by shape)
    l.shape = !g.is_tensor ? 0 : g.small ? g.small : g.bigsh;
    if (tuned) {
      auto it = tuned->find(l.key);
      if (it != tuned->end()) {
        l.zchunk = it->second.zchunk;
        l.pt = it->second.pt;
        l.wpc = it->second.wpc;
        // items per workgroup: 1, 2, 4, 8 or 16 (the largest of these not
        // above the cached value)
        l.ni = 1;
        while (l.ni < 16 && 2 * l.ni <= it->second.ni)
          l.ni *= 2;
        if (!g.is_tensor && l.wpc == -2) // static rounds: tensor tiles only
          l.wpc = -1;
        if (g.is_tensor && !g.small && it->second.shape >= 0 && it->second.shape < 2)
          l.shape = it->second.shape;
      }
    }
    // two columns a thread in narrow tiles from order 5 on and classes of 2^20
    // points: 104 drawn classes of FP32 storage 2.5% faster, 70 of them by 1% or
    // more, 2 slower (8 x 192x50x100 order 7 24.1 us with rows, 21.6 with columns;
    // 10 x 68x34x205 order 9, 3 levels, 30.9 and 32.5); lower orders and smaller
    // classes 0.3% slower (11 x 52x51x93 cell order 2, 2 levels, 8.8 and 9.3)
    l.cols = g.is_tensor && g.prec == CG_PREC_MIXED &&
             (l.shape == 0 || (l.shape == 1 && g.order >= 5 && class_pts >= (1LL << 20))) &&
             std::all_of(g.members.begin(), g.members.end(),
                         [&](int m) { return column_pairs(tensor_desc(l, tr[m])); });
    // persistent grid: resident workgroups per CU x CUs, a multiple of the
    // 8 XCDs
    int threads = 0;
    const void *fn = launch_fn(l, &threads);
    if (!fn)
      return set_error(CG_ERR_ORDER, "no persistent kernel for this transfer class");
    const int per_cu = resident_per_cu(fn, threads, dev_id);
    const int full_grid = std::max(8, (per_cu * ncu) / 8 * 8);
    // transfers largest first; a transfer's items in spatial order (x tile
    // fastest, then y, then z chunk), so consecutive items are neighbours
    std::vector<int> members = g.members;
    std::stable_sort(members.begin(), members.end(), [&](int x, int y) {
      return tr[x].dst_points() > tr[y].dst_points();
    });
    std::vector<Item> items;
    std::vector<double> cost;
    std::vector<int> first; // first item of each transfer, plus the end
    if (g.is_tensor) {
      TileCfg cfg;
      int tthreads = 0;
      tile_shape(g.ntl, g.prec, &cfg.cx, &cfg.cy, &tthreads, l.shape);
      // z chunk: the one whose items finish soonest on the resident
      // workgroups, under greedy list scheduling in dispatch order (what the
      // work counters and the dispatcher do) with an item's cost its planes
      // plus the ramp-up of the stencil span; a chunk adds those ramp-up
      // planes, and whole-region items leave workgroups idle when regions
      // are few.  Near-ties go to the longer chunk (neighbouring tiles
      // then march through z together and share halo rows in L2).
      if (tile_cfg < 0 && !(tuned && tuned->count(l.key))) {
        const int span = line_span(g.kind, g.order), tc = tile_cost(g.kind, g.order, g.ntl, g.prec);
        std::vector<double> mk;
        const int zcs[6] = {128, 64, 32, 16, 8, 4};
        for (int zc : zcs) {
          std::priority_queue<double, std::vector<double>, std::greater<double>> q;
          for (int w = 0; w < full_grid; ++w)
            q.push(0.0);
          for (int m : members) {
            const TensorArgs &a = tr[m].pr.t;
            const long long nxy =
                (long long)tiles_x(a, cfg.cx, tile_shift(a, cfg.cx, g.prec ? 4 : 8, tc)) *
                tiles_y(a, cfg.cy);
            for (int z0 = 0; z0 < a.nq[2]; z0 += zc)
              for (long long t = 0; t < nxy; ++t) {
                const double at = q.top();
                q.pop();
                q.push(at + std::min(zc, a.nq[2] - z0) + span + 1);
              }
          }
          double end = 0;
          for (; !q.empty(); q.pop())
            end = std::max(end, q.top());
          mk.push_back(end);
        }
        // ENO kinds (data-dependent stencils, several times the arithmetic
        // per plane) march slower and drift further apart: at most 64
        // planes (8 variables of 192^3 -> 384^3 with ENO<3>: 1.64 ms at 64
        // against 1.74 ms at 128)
        const int first = fp64_only(g.kind) ? 1 : 0;
        const double best = *std::min_element(mk.begin() + first, mk.end());
        for (int i = first; i < 6; ++i)
          if (mk[i] <= 1.03 * best) {
            l.zchunk = zcs[i];
            break;
          }
      }
      std::vector<TensorArgs> descs;
      for (int m : members) {
        const TensorArgs a = tensor_desc(l, tr[m]);
        const long long nt = (long long)a.ntiles[0] * a.ntiles[1] * a.ntiles[2];
        const unsigned d = (unsigned)descs.size();
        descs.push_back(a);
        l.sx.push_back(a.sx);
        first.push_back((int)items.size());
        for (long long t = 0; t < nt; ++t) {
          items.push_back(Item{d, (unsigned)t});
          // cost ~ coarse planes (with the halo) x tile area: a tile's
          // lanes are busy whether or not the region fills it
          const int tz = (int)(t / ((long long)a.ntiles[0] * a.ntiles[1]));
          const int nz = std::min(a.zchunk, a.nq[2] - tz * a.zchunk) + 5;
          cost.push_back((double)nz * cfg.cx * cfg.cy);
        }
      }
      l.desc_off = append(descs.data(), descs.size() * sizeof(TensorArgs));
      l.desc_bytes = descs.size() * sizeof(TensorArgs);
    } else {
      std::vector<PointArgs> descs;
      for (int m : members) {
        const PointArgs a = point_desc(l, tr[m]);
        long long u[3];
        point_units(l, a, u);
        const long long tot = u[0] * u[1] * u[2];
        if (tot >= (1LL << 31) - l.pt)
          return set_error(CG_ERR_ARG, "region too large for the batch");
        const unsigned d = (unsigned)descs.size();
        descs.push_back(a);
        l.sx.push_back(a.sx);
        l.nxp.push_back(a.nxp);
        first.push_back((int)items.size());
        const long long nt = (tot + l.pt - 1) / l.pt;
        for (long long t = 0; t < nt; ++t) {
          items.push_back(Item{d, (unsigned)t});
          cost.push_back((double)std::min<long long>(l.pt, tot - t * l.pt));
        }
      }
      l.desc_off = append(descs.data(), descs.size() * sizeof(PointArgs));
      l.desc_bytes = descs.size() * sizeof(PointArgs);
    }
    l.members = members;
    first.push_back((int)items.size());
    l.nitems = (int)items.size();
    // One segment per XCD.  Every transfer is striped over the XCDs: its
    // items are cut into 8 contiguous parts of equal cost (spatial slabs,
    // e.g. ranges of y tiles) and part x goes to XCD x, so all XCDs work on
    // the same transfer at the same time, as one launch per transfer would,
    // with each slab's halos shared in one L2.  A tensor transfer of at
    // most WHOLE_XCD_ITEMS tiles goes whole to the XCD with the least work
    // so far: its tiles' stencil halos overlap, and on one XCD the rows two
    // tiles share are fetched from HBM once, where striped over XCDs every
    // tile fetches them into its own L2.  A pointwise transfer with fewer
    // than 8 items gives each item to the least-loaded XCD.
    const bool one = g.is_tensor && !g.small && median_pts >= (1LL << 20) && l.nitems <= full_grid;
    auto split = [&](const std::vector<double> &w, std::vector<int> *part) {
      double load[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      for (size_t m = 0; m + 1 < first.size(); ++m) {
        const int i0 = first[m], i1 = first[m + 1];
        if (g.is_tensor && i1 - i0 <= WHOLE_XCD_ITEMS) {
          const int x = (int)(std::min_element(load, load + 8) - load);
          for (int i = i0; i < i1; ++i) {
            part[x].push_back(i);
            load[x] += w[i];
          }
          continue;
        }
        if (i1 - i0 < 8) {
          for (int i = i0; i < i1; ++i) {
            const int x = (int)(std::min_element(load, load + 8) - load);
            part[x].push_back(i);
            load[x] += w[i];
          }
          continue;
        }
        // TVD writes eight values per cell it reads, and writes to memory best
        // when the XCDs work close together: blocks of 64 items in turn, from
        // the XCD with the least work so far, where the class writes more than
        // 1 GiB.  Below that much of it stays in the last-level cache, and slabs
        // read each coarse plane on fewer XCDs.  (Slabs, and blocks of 16, 32
        // and 64 items, us: 8 x 384^3 of 1 level 987, 890, 896, 894, of 3 levels
        // 1403, 1380, 1381, 1353; 20 x 230^3, 1 level, 514, 476, 485, 487; 8 x
        // 256^3, 1 level, 186, 219, 194, 189; 8 x 200^3, 2 levels, 101, 121, 101,
        // 99.  The cell restriction back of 8 x 384^3, which reads: 717 in slabs,
        // 757 in blocks of 16.)  One level above 2 GiB takes blocks of 16: 8 x
        // 384^3 with that restriction after it 1649 us a step, 1679 in blocks of
        // 64.
        const int block = levels == 1 && class_pts > (1LL << 28) ? 16 : 64;
        if (g.op == PO_TVD && class_pts > (1LL << 27) && i1 - i0 >= 8 * block) {
          const int x0 = (int)(std::min_element(load, load + 8) - load);
          for (int i = i0; i < i1; ++i) {
            const int x = (x0 + (i - i0) / block) % 8;
            part[x].push_back(i);
            load[x] += w[i];
          }
          continue;
        }
        double total = 0;
        for (int i = i0; i < i1; ++i)
          total += w[i];
        double acc = 0;
        int x = 0;
        for (int i = i0; i < i1; ++i) {
          // item i belongs to the part its cost midpoint falls in
          const double mid = acc + 0.5 * w[i];
          while (x < 7 && mid >= total * (x + 1) / 8.0)
            ++x;
          part[x].push_back(i);
          load[x] += w[i];
          acc += w[i];
        }
      }
    };
    std::vector<int> part[8];
    split(cost, part);
    // Classes of regions from 2^20 points whose items fit one round of resident
    // workgroups, one or two to a CU: a segment longer than its XCD holds at once
    // takes a second round, so the XCDs get equal numbers of items instead where
    // that ends sooner (4 x 250x120x120 order 11, 3 levels, 256 items: 147 us with
    // 36 on one XCD, 84 with 32 on each; where the second round is of short chunks,
    // equal cost is the better split: 6 x 180^3 cell ENO<3>, 3 levels, 562 us
    // against 600).  Three and more workgroups to a CU share its rate, and the
    // second round fills in as the first drains (equal cost and equal numbers, three
    // to a CU, us: 6 x 67x145x161 vertex ENO<3>, 2 levels, 43 and 52; 9 x 139x66x209
    // cell order 3, 2 levels, 54 and 59; 12 x 160^3 FP32 storage, order 3, 50 and 54.
    // Of 34 such classes 5 were faster with equal numbers, by 9% at most.)
    if (one && per_cu <= 2) {
      auto end = [&](const std::vector<int> *pt) {
        double e = 0;
        for (int x = 0; x < 8; ++x) {
          std::priority_queue<double, std::vector<double>, std::greater<double>> q;
          for (int k = 0; k < full_grid / 8; ++k)
            q.push(0.0);
          for (int i : pt[x]) {
            e = std::max(e, q.top() + cost[i]);
            q.push(q.top() + cost[i]);
            q.pop();
          }
        }
        return e;
      };
      std::vector<int> even[8];
      split(std::vector<double>(cost.size(), 1.0), even);
      if (end(even) < 0.8 * end(part))
        for (int x = 0; x < 8; ++x)
          part[x].swap(even[x]);
    }
    int segb[9], longest = 1;
    {
      std::vector<Item> ordered;
      ordered.reserve(items.size());
      segb[0] = 0;
      for (int x = 0; x < 8; ++x) {
        for (int i : part[x])
          ordered.push_back(items[i]);
        segb[x + 1] = (int)ordered.size();
        longest = std::max(longest, segb[x + 1] - segb[x]);
      }
      items.swap(ordered);
      l.seg_off = append(segb, sizeof segb);
    }
    l.item_off = append(items.data(), items.size() * sizeof(Item));
    l.counter = (int)dev.launches.size();
    // one workgroup per item then, all of them resident, without counters (and
    // the launch that clears them, 5-7 us); as it fills the GPU by itself it runs
    // in turn with its phase's other classes (104x104x97 points and three thin
    // faces, order 5, 3 levels: 19 us in turn, 34 side by side; 118x98x98 and 24
    // of 20^3: 22 and 34).  A tuned class runs as its parameters say.
    l.one_round = one && !(tuned && tuned->count(l.key));
    if (l.one_round)
      l.wpc = 0;
    if (l.wpc == -1 || l.one_round) {
      // grid mode: 8 x the longest segment (in groups of ni items)
      const int ni = (!g.is_tensor && l.pt == 256 && g.op != PO_TVD) ? l.ni : 1;
      const long long groups = (longest + ni - 1) / ni;
      if (8 * groups > 0x7fffffffLL)
        return set_error(CG_ERR_ARG, "too many work items for one launch");
      l.grid = (int)(8 * groups);
    } else {
      const long long all = std::max(8, (l.nitems + 7) / 8 * 8);
      // persistent (counters or static rounds): a multiple of 8 workgroups
      const long long grid =
          l.wpc > 0 ? std::max(8LL, (long long)l.wpc * ncu / 8 * 8) : full_grid;
      l.grid = (int)std::min(grid, all);
    }
    dev.launches.push_back(l);
  }
  dev.ncounters = (int)dev.launches.size();
  if (host.empty())
    return CG_OK;
  he = hipMalloc(&dev.blob, host.size());
  if (he != hipSuccess)
    return set_error(CG_ERR_NOMEM, "batch descriptors: %s", hipGetErrorString(he));
  dev.blob_bytes = host.size();
  he = hipMemcpy(dev.blob, host.data(), host.size(), hipMemcpyHostToDevice);
  if (he != hipSuccess)
    return hip_error(he, "batch descriptor upload");
  he = hipMalloc(&dev.counters, sizeof(int) * 8 * std::max(1, dev.ncounters));
  if (he != hipSuccess)
    return set_error(CG_ERR_NOMEM, "batch counters: %s", hipGetErrorString(he));
  return CG_OK;
}

static int run_launch(BatchDevice &dev, const BatchLaunch &l, hipStream_t st);

// helper streams (default priority, non-blocking) and the fork/join events
// of the launches that share a phase
static int ensure_aux(BatchDevice &dev, size_t n) {
  if (dev.fork.empty()) {
    hipEvent_t e;
    hipError_t he = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (he != hipSuccess)
      return hip_error(he, "hipEventCreate");
    dev.fork.push_back(e);
  }
  while (dev.aux.size() < n) {
    hipStream_t s;
    hipEvent_t e;
    hipError_t he = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
    if (he != hipSuccess)
      return hip_error(he, "hipStreamCreate");
    dev.aux.push_back(s);
    he = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (he != hipSuccess)
      return hip_error(he, "hipEventCreate");
    dev.join.push_back(e);
  }
  return CG_OK;
}

size_t batch_phase_end(const BatchDevice &dev, size_t i) {
  size_t j = i + 1;
  while (j < dev.launches.size() && dev.launches[j].phase == dev.launches[i].phase)
    ++j;
  return j;
}

// The launches of one phase write disjoint regions (dh's lists never send
// one point twice), so the classes of a phase may run side by side: the
// first on st, the others on helper streams forked from st by an event and
// joined back before the next phase.  Under stream capture the fork and
// join become branches of the graph.
static int run_phase(BatchDevice &dev, size_t i, size_t j, bool side, hipStream_t st) {
  const size_t extra = side ? j - i - 1 : 0;
  if (extra > 0) {
    if (int e = ensure_aux(dev, extra))
      return e;
    hipError_t he = hipEventRecord(dev.fork[0], st);
    for (size_t k = 0; k < extra && he == hipSuccess; ++k)
      he = hipStreamWaitEvent(dev.aux[k], dev.fork[0], 0);
    if (he != hipSuccess)
      return hip_error(he, "phase fork");
  }
  for (size_t k = i; k < j; ++k) {
    int e = run_launch(dev, dev.launches[k], (k == i || !side) ? st : dev.aux[k - i - 1]);
    if (e)
      return e;
  }
  for (size_t k = 0; k < extra; ++k) {
    hipError_t he = hipEventRecord(dev.join[k], dev.aux[k]);
    if (he == hipSuccess)
      he = hipStreamWaitEvent(st, dev.join[k], 0);
    if (he != hipSuccess)
      return hip_error(he, "phase join");
  }
  return CG_OK;
}

static bool phase_beside(const BatchDevice &dev, size_t i) {
  return dev.beside.size() != dev.launches.size() || dev.beside[i] != 0;
}

int batch_device_run(BatchDevice &dev, hipStream_t st) {
  if (dev.launches.empty())
    return CG_OK;
  // only persistent launches use the work counters
  bool persistent = false;
  for (const BatchLaunch &l : dev.launches)
    persistent = persistent || (l.wpc >= 0 && !l.one_round);
  if (persistent)
    hipLaunchKernelGGL(k_zero_counters, dim3((8 * dev.ncounters + 255) / 256), dim3(256), 0, st,
                       dev.counters, 8 * dev.ncounters);
  for (size_t i = 0; i < dev.launches.size();) {
    const size_t j = batch_phase_end(dev, i);
    if (int e = run_phase(dev, i, j, phase_beside(dev, i), st))
      return e;
    i = j;
  }
  return CG_OK;
}

int batch_device_run_phase(BatchDevice &dev, size_t i, size_t j, bool side, hipStream_t st) {
  if (i >= j || j > dev.launches.size())
    return set_error(CG_ERR_ARG, "no launches [%zu, %zu)", i, j);
  hipLaunchKernelGGL(k_zero_counters, dim3((8 * dev.ncounters + 255) / 256), dim3(256), 0, st,
                     dev.counters, 8 * dev.ncounters);
  return run_phase(dev, i, j, side, st);
}

int batch_device_run_one(BatchDevice &dev, int idx, hipStream_t st) {
  if (idx < 0 || idx >= (int)dev.launches.size())
    return set_error(CG_ERR_ARG, "no launch %d", idx);
  hipLaunchKernelGGL(k_zero_counters, dim3((8 * dev.ncounters + 255) / 256), dim3(256), 0, st,
                     dev.counters, 8 * dev.ncounters);
  return run_launch(dev, dev.launches[idx], st);
}

static int run_launch(BatchDevice &dev, const BatchLaunch &l, hipStream_t st) {
  const void *descs = dev.blob + l.desc_off;
  const Item *items = reinterpret_cast<const Item *>(dev.blob + l.item_off);
  const int *seg = reinterpret_cast<const int *>(dev.blob + l.seg_off);
  int *ctr = dev.counters + 8 * l.counter;
  const bool grid_mode = l.wpc == -1;
  int rc = 0;
  if (l.is_tensor) {
    const TensorArgs *td = static_cast<const TensorArgs *>(descs);
    switch (l.shape) {
    case 0: rc = tensor_run_sh<0>(l, td, items, seg, ctr, st); break;
    case 1: rc = tensor_run_sh<1>(l, td, items, seg, ctr, st); break;
    case 2: rc = tensor_run_sh<2>(l, td, items, seg, ctr, st); break;
    case 3: rc = tensor_run_sh<3>(l, td, items, seg, ctr, st); break;
    default: rc = -1;
    }
  } else {
    const PointArgs *pd = static_cast<const PointArgs *>(descs);
    auto go_pu = [&](auto opc, auto puc) {
      constexpr int OP = decltype(opc)::value;
      constexpr int PU = decltype(puc)::value;
      if constexpr (OP != PO_TVD) {
        if (grid_mode && l.pt == 256 && l.ni > 1) {
          switch (l.ni) {
          case 2: hipLaunchKernelGGL((k_grid_point_n<OP, 2>), dim3(l.grid), dim3(256), 0, st, pd, items, seg); break;
          case 4: hipLaunchKernelGGL((k_grid_point_n<OP, 4>), dim3(l.grid), dim3(256), 0, st, pd, items, seg); break;
          case 8: hipLaunchKernelGGL((k_grid_point_n<OP, 8>), dim3(l.grid), dim3(256), 0, st, pd, items, seg); break;
          default: hipLaunchKernelGGL((k_grid_point_n<OP, 16>), dim3(l.grid), dim3(256), 0, st, pd, items, seg);
          }
          return 0;
        }
      }
      if (grid_mode)
        hipLaunchKernelGGL((k_grid_point<OP, PU>), dim3(l.grid), dim3(256), 0, st, pd, items, seg, l.pt);
      else
        hipLaunchKernelGGL((k_persist_point<OP, PU>), dim3(l.grid), dim3(256), 0, st, pd, items, seg,
                           ctr, l.pt);
      return 0;
    };
    auto go = [&](auto opc) {
      constexpr int OP = decltype(opc)::value;
      switch (pu_inst<OP>(pu_of(l.pt))) {
      case 1: return go_pu(opc, std::integral_constant<int, pu_inst<OP>(1)>{});
      case 2: return go_pu(opc, std::integral_constant<int, pu_inst<OP>(2)>{});
      case 4: return go_pu(opc, std::integral_constant<int, pu_inst<OP>(4)>{});
      }
      return go_pu(opc, std::integral_constant<int, pu_inst<OP>(8)>{});
    };
    switch (l.op) {
    case PO_COPY: rc = go(std::integral_constant<int, PO_COPY>{}); break;
    case PO_RESTRICT_VC: rc = go(std::integral_constant<int, PO_RESTRICT_VC>{}); break;
    case PO_RESTRICT_CC: rc = go(std::integral_constant<int, PO_RESTRICT_CC>{}); break;
    case PO_INTERP: rc = go(std::integral_constant<int, PO_INTERP>{}); break;
    case PO_TVD: rc = go(std::integral_constant<int, PO_TVD>{}); break;
    case PO_RESTRICT_CC_O3: rc = go(std::integral_constant<int, PO_RESTRICT_CC_O3>{}); break;
    case PO_RESTRICT_CC_O5: rc = go(std::integral_constant<int, PO_RESTRICT_CC_O5>{}); break;
    case PO_MONO5: rc = go(std::integral_constant<int, PO_MONO5>{}); break;
    case PO_STAGGER: rc = go(std::integral_constant<int, PO_STAGGER>{}); break;
    case PO_RESTRICT_STAGGER: rc = go(std::integral_constant<int, PO_RESTRICT_STAGGER>{}); break;
    case PO_RESTRICT_VC2: rc = go(std::integral_constant<int, PO_RESTRICT_VC2>{}); break;
    default: rc = -1;
    }
  }
  if (rc)
    return set_error(CG_ERR_ORDER, "no batch kernel for this transfer class");
  hipError_t he = hipGetLastError();
  if (he != hipSuccess)
    return hip_error(he, "batch launch");
  return CG_OK;
}

} // namespace cg
