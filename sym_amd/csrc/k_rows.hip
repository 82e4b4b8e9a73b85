// k_rows.hip - relayouts with the innermost axis contiguous on both sides
// that the stream kernel cannot take: rows of any length and alignment, with
// pads (k_rows), and flat tensors whose channels change inside a vector or
// whose length is not a multiple of one (k_flat).
//
// Bound by memory; both keep the stream kernel's shape (16 bytes per item on
// the wider side, two items 64 apart per lane). Element-wise -> here, buffers
// of three calls in turn: f32 [8000,1003] padded to 1024 columns -> int8
// 42.3 -> 9.4 us (4.3 TB/s; a 16-byte copy of these 40 MB 4.7); f32
// [5000,4097] -> int8 102 -> 18.7 us; int8 [2816,7863] dequantized per row ->
// f16 121 -> 11.4 us (5.9 TB/s).
#include "kernels.h"

namespace relx {
namespace {

// v moved up by n < 16 bytes, zeros before it.
__device__ __forceinline__ vec4 up_bytes(vec4 v, uint32_t n) {
  if (n & 8)
    v = vec4{0u, 0u, v.x, v.y};
  if (n & 4)
    v = vec4{0u, v.x, v.y, v.z};
  const uint64_t b = (n & 3) * 8;
  return vec4{v.x << b, static_cast<uint32_t>(((uint64_t{v.y} << 32 | v.x) << b) >> 32),
              static_cast<uint32_t>(((uint64_t{v.z} << 32 | v.y) << b) >> 32),
              static_cast<uint32_t>(((uint64_t{v.w} << 32 | v.z) << b) >> 32)};
}

// Item i of a row covers destination columns [i*V, i*V + V) of it (the last
// item may be cut). Its source vector starts at its own column where all of it
// is valid; where a pad begins or ends inside it, at the nearest column that
// keeps the load inside the row's valid columns (there are at least V), and
// its elements move into place in registers.
template <int WIN, int WOUT, int L, int CH, bool NTS>
__global__ __launch_bounds__(kBlock) void k_rows(KArgs a) {
  constexpr int V = 16 / (WIN > WOUT ? WIN : WOUT);
  constexpr int BI = V * WIN, BO = V * WOUT;
  constexpr int U = 2;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const uint32_t stride = gridDim.x * (kBlock / 64) * (64 * U);
  asm volatile("" ::"s"(a.src), "s"(a.dst), "s"(a.work), "s"(a.fill), "s"(a.sbase), "s"(a.dbase),
               "s"(stride), "s"(a.r_len), "s"(a.r_off), "s"(a.r_lo), "s"(a.r_hi));
  hot_levels<L>(a);
  hot_chain<CH>(a);
  for (uint32_t base = wave * (64 * U) + lane; base < a.work; base += stride) {
    int64_t dof[U];
    bool pad[U];
    int32_t col[U], at[U]; // the item's first column, the column its load starts at
    vec4 in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i0 = base + 64u * u;
      const uint32_t i = i0 < a.work ? i0 : base;
      int64_t sof = a.sbase;
      dof[u] = a.dbase;
      // the innermost level counts items; its valid range is all of it
      pad[u] = decompose<L>(a.lv, i, sof, dof[u]);
      const uint32_t row = fdiv(i, a.lv[L - 1].div);
      const int32_t p = static_cast<int32_t>(i - row * a.lv[L - 1].div.d) * V;
      col[u] = p + a.r_off;
      at[u] = min(max(col[u], a.r_lo), a.r_hi - V);
      pad[u] |= col[u] >= a.r_hi || col[u] + V <= a.r_lo;
      // sof counts from column r_off of the row
      in[u] = ldu_n<BI>(pad[u] ? g_unused_src : a.src + (sof + (at[u] - col[u])) * WIN);
    }
    VecParams par[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      par[u] = fetch_params<CH>(a, dof[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && base + 64u * u >= a.work)
        break;
      const int32_t d = at[u] - col[u];
      if (d < 0)
        in[u] = down_bytes(in[u], static_cast<uint32_t>(-d * WIN) & 15u);
      else if (d > 0)
        in[u] = up_bytes(in[u], static_cast<uint32_t>(d * WIN) & 15u);
      uint32_t v[V];
      unpack<WIN, V>(&in[u], v);
      chain_vec_p<CH, V, true>(a, v, dof[u], par[u]);
      if (pad[u] || d != 0) {
#pragma unroll
        for (int e = 0; e < V; ++e)
          if (pad[u] || col[u] + e < a.r_lo || col[u] + e >= a.r_hi)
            v[e] = a.fill;
      }
      vec4 out = {0u, 0u, 0u, 0u};
      pack<WOUT, V>(v, &out);
      const int32_t left = static_cast<int32_t>(a.r_len) - (col[u] - a.r_off);
      uint8_t *dst = a.dst + dof[u] * WOUT;
      if (left >= V)
        stu_n<BO, NTS>(dst, out);
      else
        stu_cut(dst, out, static_cast<uint32_t>(left * WOUT));
    }
  }
}

// Parameter entries of V consecutive elements of a flat tensor from offset
// `o`: channels of rs >= V elements (DevStage::vec 2, or 0 where no vector
// holds two: c0, then c1 from element `left` on), or one channel per element
// (vec 1 or 3: c0 + e, wrapping at re >= V).
struct FlatChan {
  uint32_t c0, c1, left;
};

__device__ __forceinline__ FlatChan flat_chan(const DevStage &s, uint32_t o) {
  const uint32_t q = fdiv(o, s.ch_rs_div);
  FlatChan f;
  f.left = s.ch_rs_div.d - (o - q * s.ch_rs_div.d);
  f.c0 = q - fdiv(q, s.ch_re_div) * s.ch_re_div.d;
  f.c1 = f.c0 + 1 == s.ch_re_div.d ? 0 : f.c0 + 1;
  return f;
}

template <int V>
__device__ __forceinline__ void flat_params(const KArgs &a, const DevStage &s, uint32_t o, bool zps,
                                            float (&sc)[V], int32_t (&zp)[V]) {
  const FlatChan f = flat_chan(s, o);
  if (s.vec & 1) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const uint32_t c = f.c0 + e, w = c >= s.ch_re_div.d ? c - s.ch_re_div.d : c;
      sc[e] = a.pf[s.scale_off + w];
      zp[e] = zps ? a.pi[s.zp_off + (s.zp_per_ch ? w : 0u)] : 0;
    }
    return;
  }
  const bool one = s.vec == 0;
  const float s0 = a.pf[s.scale_off + f.c0], s1 = a.pf[s.scale_off + (one ? f.c0 : f.c1)];
  int32_t z0 = 0, z1 = 0;
  if (zps) {
    z0 = a.pi[s.zp_off + (s.zp_per_ch ? f.c0 : 0u)];
    z1 = a.pi[s.zp_off + (s.zp_per_ch && !one ? f.c1 : s.zp_per_ch ? f.c0 : 0u)];
  }
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const bool first = static_cast<uint32_t>(e) < f.left;
    sc[e] = first ? s0 : s1;
    zp[e] = first ? z0 : z1;
  }
}

template <int CH, int V>
__device__ __forceinline__ void chain_flat(const KArgs &a, uint32_t (&v)[V], int64_t o,
                                           const float (&sc)[V], const int32_t (&zp)[V]) {
  if constexpr (CH == kChainGeneric) {
    for (int k = 0; k < a.chain.n; ++k) {
      const DevStage &s = a.chain.st[k];
      if (s.op == kOpQuantize || s.op == kOpDequantize) {
        float fs[V];
        int32_t fz[V];
        flat_params<V>(a, s, static_cast<uint32_t>(o), s.op == kOpDequantize, fs, fz);
#pragma unroll
        for (int e = 0; e < V; ++e)
          v[e] = s.op == kOpQuantize ? op_quant(v[e], fs[e]) : op_dequant(v[e], fs[e], fz[e]);
      } else {
        stage_vec<V>(a, s, v, o);
      }
    }
  } else if constexpr (chain_param_stage(CH) < 0) {
    chain_vec<CH, V>(a, v, o);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      if constexpr (CH == kChainDeqF16)
        v[e] = op_f32_f16(op_dequant(v[e], sc[e], zp[e]));
      else if constexpr (CH == kChainDeq)
        v[e] = op_dequant(v[e], sc[e], zp[e]);
      else if constexpr (CH == kChainF16Quant)
        v[e] = quant_value(op_f16_f32_value(v[e]), sc[e]);
      else
        v[e] = op_quant(v[e], sc[e]);
    }
  }
}

// A flat tensor: r_len elements, `work` whole vectors; the last r_len mod V
// elements one by one on the first lanes.
template <int WIN, int WOUT, int CH>
__global__ __launch_bounds__(kBlock) void k_flat(KArgs a) {
  constexpr int V = 16 / (WIN > WOUT ? WIN : WOUT);
  constexpr int BI = V * WIN, BO = V * WOUT;
  constexpr int U = 2;
  constexpr bool NTL = RELX_NT_LOAD(kFamStream, WIN, WOUT, 1);
  constexpr bool NTS = RELX_NT_STORE(kFamStream, WIN, WOUT, 1);
  constexpr int PS = chain_param_stage(CH);
  constexpr bool kZp = CH == kChainDeqF16 || CH == kChainDeq;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const uint32_t stride = gridDim.x * (kBlock / 64) * (64 * U);
  asm volatile("" ::"s"(a.src), "s"(a.dst), "s"(a.work), "s"(a.sbase), "s"(a.dbase), "s"(stride),
               "s"(a.r_len));
  hot_chain<CH>(a);
  const uint8_t *src = a.src + a.sbase * WIN;
  uint8_t *dst = a.dst + a.dbase * WOUT;
  for (uint32_t base = wave * (64 * U) + lane; base < a.work; base += stride) {
    vec4 in[U];
    float sc[U][V];
    int32_t zp[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = base + 64u * u < a.work ? base + 64u * u : base;
      in[u] = ld_n<BI, NTL>(src + static_cast<int64_t>(i) * BI);
    }
    if constexpr (PS >= 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t i = base + 64u * u < a.work ? base + 64u * u : base;
        flat_params<V>(a, a.chain.st[PS], static_cast<uint32_t>(a.dbase) + i * V, kZp, sc[u], zp[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = base + 64u * u;
      if (u > 0 && i >= a.work)
        break;
      uint32_t v[V];
      unpack<WIN, V>(&in[u], v);
      chain_flat<CH, V>(a, v, a.dbase + static_cast<int64_t>(i) * V, sc[u], zp[u]);
      vec4 out = {0u, 0u, 0u, 0u};
      pack<WOUT, V>(v, &out);
      st_n<BO, NTS>(dst + static_cast<int64_t>(i) * BO, out);
    }
  }
  const uint32_t tail = a.r_len % V;
  if (blockIdx.x == 0 && threadIdx.x < tail) {
    const int64_t i = static_cast<int64_t>(a.work) * V + threadIdx.x;
    uint32_t v[1] = {static_cast<uint32_t>(load_el(src + i * WIN, WIN))};
    float sc[1];
    int32_t zp[1];
    if constexpr (PS >= 0)
      flat_params<1>(a, a.chain.st[PS], static_cast<uint32_t>(a.dbase + i), kZp, sc, zp);
    chain_flat<CH, 1>(a, v, a.dbase + i, sc, zp);
    store_el(dst + i * WOUT, v[0], WOUT);
  }
}

template <int WIN, int WOUT, int L, int CH> void rows_levels(const KArgs &a, hipStream_t s) {
  const dim3 grid(grid_for((static_cast<int64_t>(a.work) + 1) / 2)), block(kBlock);
  if (a.r_nts)
    hipLaunchKernelGGL((k_rows<WIN, WOUT, L, CH, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_rows<WIN, WOUT, L, CH, false>), grid, block, 0, s, a);
}

template <int WIN, int WOUT, int CH> hipError_t rows_launch(const KArgs &a, hipStream_t s) {
  if (a.family == kFamFlat) {
    const dim3 grid(grid_for((static_cast<int64_t>(a.work) + 1) / 2)), block(kBlock);
    hipLaunchKernelGGL((k_flat<WIN, WOUT, CH>), grid, block, 0, s, a);
    return hipGetLastError();
  }
  switch (a.nlev) {
  case 2:
    rows_levels<WIN, WOUT, 2, CH>(a, s);
    break;
  case 4:
    rows_levels<WIN, WOUT, 4, CH>(a, s);
    break;
  case 8:
    rows_levels<WIN, WOUT, 8, CH>(a, s);
    break;
  default:
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

} // namespace

RELX_DISPATCH_FAST(rows_fast, rows_launch)
RELX_DISPATCH_GENERIC(rows_generic, rows_launch)

} // namespace relx
