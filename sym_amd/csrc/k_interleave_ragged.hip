// k_interleave_ragged.hip - planar -> interleaved relayouts (a small padded
// inner axis) whose pixel count or plane stride fits no whole pixel groups:
// an image with an odd number of pixels starts every plane after the first
// inside a group.
//
// The items of k_interleave (G pixels: one load per plane, one packed run of
// G*CP output elements, two items 64 apart per lane) at whatever alignment
// they have. The last group of a plane may be cut: its planes are read from
// the plane's last G pixels and moved down in registers, its run is stored in
// at most four pieces per 16 bytes. Bound by memory.
#include "kernels.h"

namespace relx {
namespace {

template <int WIN, int WOUT, int CP, int CH>
__global__ __launch_bounds__(kBlock) void k_interleave_rag(KArgs a) {
  constexpr int G = interleave_pixels(WIN, WOUT, CP);
  constexpr int BI = G * WIN, BO = G * CP * WOUT;
  constexpr int NO = BO >= 16 ? BO / 16 : 1;
  constexpr int U = 2;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const uint32_t stride = gridDim.x * (kBlock / 64) * (64 * U);
  asm volatile("" ::"s"(a.src), "s"(a.dst), "s"(a.work), "s"(a.fill), "s"(a.sbase), "s"(a.dbase),
               "s"(a.i_ssc), "s"(a.i_loc), "s"(a.i_vc), "s"(stride), "s"(a.r_len));
  hot(a.i_ng);
  hot_levels<kBatchLevels>(a);
  for (uint32_t base = wave * (64 * U) + lane; base < a.work; base += stride) {
    vec4 in[U][CP];
    bool valid[U][CP];
    int64_t dof[U];
    uint32_t p0[U], back[U]; // first pixel, pixels the loads start before it
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = base + 64u * u < a.work ? base + 64u * u : base;
      const uint32_t rest = fdiv(i, a.i_ng);
      int64_t sbase = a.sbase;
      dof[u] = a.dbase;
      const bool pad = decompose<kBatchLevels>(a.lv, rest, sbase, dof[u]);
      p0[u] = (i - rest * a.i_ng.d) * G; // the pixel axis is unpadded
      back[u] = p0[u] + G > a.r_len ? p0[u] + G - a.r_len : 0u;
      dof[u] += static_cast<int64_t>(p0[u]) * CP;
#pragma unroll
      for (int ch = 0; ch < CP; ++ch) {
        const int32_t vc = ch - a.i_loc;
        valid[u][ch] = !pad && static_cast<uint32_t>(vc) < static_cast<uint32_t>(a.i_vc);
        in[u][ch] = ldu_n<BI>(valid[u][ch] ? a.src + (sbase + vc * a.i_ssc + (p0[u] - back[u])) * WIN
                                           : g_unused_src);
      }
    }
    auto emit = [&](auto uc) {
      constexpr int u = decltype(uc)::value;
      uint32_t flat[G * CP];
#pragma unroll
      for (int ch = 0; ch < CP; ++ch) {
        uint32_t v[G];
        if (!valid[u][ch]) {
#pragma unroll
          for (int e = 0; e < G; ++e)
            v[e] = a.fill;
        } else {
          if (back[u])
            in[u][ch] = down_bytes(in[u][ch], back[u] * WIN);
          unpack<WIN, G>(&in[u][ch], v);
          chain_vec<CH, G>(a, v, 0);
        }
#pragma unroll
        for (int e = 0; e < G; ++e)
          flat[e * CP + ch] = v[e];
      }
      vec4 out[NO];
      out[0] = vec4{0u, 0u, 0u, 0u};
      pack<WOUT, G * CP>(flat, out);
      uint8_t *dst = a.dst + dof[u] * WOUT;
      if (back[u] == 0) {
#pragma unroll
        for (int j = 0; j < NO; ++j)
          stu_n<(BO < 16 ? BO : 16)>(dst + j * 16, out[j]);
      } else {
        const int32_t n = static_cast<int32_t>((G - back[u]) * CP * WOUT);
#pragma unroll
        for (int j = 0; j < NO; ++j) {
          if (n >= (j + 1) * 16)
            stu_n<16>(dst + j * 16, out[j]);
          else if (n > j * 16)
            stu_cut(dst + j * 16, out[j], static_cast<uint32_t>(n - j * 16));
        }
      }
    };
    emit(std::integral_constant<int, 0>{});
    if (base + 64u < a.work)
      emit(std::integral_constant<int, 1>{});
  }
}

template <int WIN, int WOUT, int CH, int CP> hipError_t rag_cp(const KArgs &a, hipStream_t s) {
  constexpr int BO = interleave_pixels(WIN, WOUT, CP) * CP * WOUT;
  if constexpr (BO == 4 || BO == 8 || BO % 16 == 0) {
    const dim3 grid(grid_for((static_cast<int64_t>(a.work) + 1) / 2)), block(kBlock);
    hipLaunchKernelGGL((k_interleave_rag<WIN, WOUT, CP, CH>), grid, block, 0, s, a);
    return hipGetLastError();
  } else {
    return hipErrorInvalidValue;
  }
}

template <int WIN, int WOUT, int CH> hipError_t rag_launch(const KArgs &a, hipStream_t s) {
  switch (a.cpad) {
  case 2:
    return rag_cp<WIN, WOUT, CH, 2>(a, s);
  case 4:
    return rag_cp<WIN, WOUT, CH, 4>(a, s);
  case 8:
    return rag_cp<WIN, WOUT, CH, 8>(a, s);
  default:
    return hipErrorInvalidValue;
  }
}

} // namespace

RELX_DISPATCH_FAST(interleave_ragged_fast, rag_launch)
RELX_DISPATCH_GENERIC(interleave_ragged_generic, rag_launch)

} // namespace relx
