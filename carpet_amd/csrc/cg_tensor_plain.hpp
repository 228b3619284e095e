// cg_tensor_plain.hpp -- per-call tensor prolongation launches, one
// template per line kind; instantiated in cg_tensor_{vlag,clag,eno}.hip so
// the three kinds compile in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include "cg_tiles.hpp"

namespace cg {

// NTL: levels of the passes; NSRC: source levels (NSRC > NTL: combined at
// the window store)
// 512-thread workgroups of orders up to 5 held to 128 VGPRs, two per CU
// (the O=5, 3-level tile otherwise takes 130 and runs one per CU)
template <class L, int NTL, int CX, int CY, int IPT, int PR, int NSRC, bool COLS>
__global__ __launch_bounds__(2 * CX * CY / IPT) __attribute__((amdgpu_waves_per_eu(
    (2 * CX * CY / IPT >= 512 && L::R <= 6) ? 4 : 1))) void k_tensor(TensorArgs a) {
  __shared__ __align__(16) double smem[tile_lds<L, NTL, CX, CY>()];
  tensor_tile<L, NTL, CX, CY, IPT, PR, 1, pipe_fits<L, NTL, CX, CY>(), NSRC, COLS>(
      a, xcd_remap(blockIdx.x, gridDim.x), smem);
}

template <class L, int NSRC, int PR, bool COLS>
int launch_tensor_c(const TensorArgs &a0, const TileCfg &cfg0, hipStream_t s) {
  constexpr int NTL = pass_levels(NSRC, PR);
  using T = TileShape<NTL, 0, PR>;
  TensorArgs a = a0;
  TileCfg cfg = cfg0;
  cfg.cx = T::CX;
  cfg.cy = T::CY;
  constexpr int threads = tile_threads<NTL, 0, PR>();
  const auto kernel = &k_tensor<L, NTL, T::CX, T::CY, T::IPT, PR, NSRC, COLS>;
  // of the kernel, the same on every gfx950
  static const Resident res = resident_workgroups(reinterpret_cast<const void *>(kernel), threads);
  cfg.zchunk = call_chunk(a, cfg, threads, L::TMAXALL - L::TMINALL, res.per_cu, res.cus);
  const long long nblk = tensor_tiles(a, cfg);
  if (nblk <= 0 || nblk > 0x7fffffffLL)
    return -1;
  hipLaunchKernelGGL(kernel, dim3((unsigned)nblk), dim3(threads), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

// FP32 storage takes column pairs for regions of 2^24 points and up; below that
// a call has few tiles, and two rows a thread are the faster ones (rows against
// columns: 160^3, order 3, 1 level 127.6 and 135.7 us; 256^3 110 and 101, order 5,
// 3 levels 121 and 115)
template <class L, int NSRC, int PR>
int launch_tensor_t(const TensorArgs &a, const TileCfg &cfg, hipStream_t s) {
  if constexpr (PR == 1) {
    using T = TileShape<1, 0, PR>;
    TensorArgs b = a;
    b.sx = tile_shift(a, T::CX, cfg.es, cfg.cost);
    if ((long long)a.n[0] * a.n[1] * a.n[2] >= (1LL << 24) && column_pairs(b))
      return launch_tensor_c<L, NSRC, PR, true>(a, cfg, s);
  }
  return launch_tensor_c<L, NSRC, PR, false>(a, cfg, s);
}

// prec: precision mode (Prec in cg_tiles.hpp); the FP32-storage modes
// (1, 2) exist for the Lagrange kinds only
template <int KIND>
int launch_tensor_kind(int order, int ntl, int prec, const TensorArgs &a, const TileCfg &cfg,
                       hipStream_t s) {
  return with_order<KIND>(order, [&](auto tag) -> int {
    using L = decltype(tag);
    auto by_ntl = [&](auto prc) -> int {
      constexpr int PR = decltype(prc)::value;
      switch (ntl) {
      case 1: return launch_tensor_t<L, 1, PR>(a, cfg, s);
      case 2: return launch_tensor_t<L, 2, PR>(a, cfg, s);
      case 3: return launch_tensor_t<L, 3, PR>(a, cfg, s);
      }
      return -1;
    };
    if (prec == 0)
      return by_ntl(std::integral_constant<int, 0>{});
    if constexpr (!fp64_only(KIND)) {
      if (prec == 1)
        return by_ntl(std::integral_constant<int, 1>{});
      if (prec == 2)
        return by_ntl(std::integral_constant<int, 2>{});
    }
    return -1;
  });
}

} // namespace cg
