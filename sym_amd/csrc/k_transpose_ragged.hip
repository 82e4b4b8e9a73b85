// k_transpose_ragged.hip - LDS-tiled transposes of any extents and row
// alignments.
//
// The tile kernels of kernels.h move whole tiles whose rows are 16-byte
// aligned. Here the last tile along q or c may be cut and rows start at any
// element. A lane moves its vector with one 16-byte access at whatever
// alignment it has. The last vector of a cut source row is read from its
// row's last 16 bytes (q has at least a vector, so it starts inside the row)
// and the elements that the vector before it brings are not written to LDS;
// the last vector of a cut destination row is stored in at most four pieces.
//
// Bound by memory: a tile row that starts inside a 128-byte line shares that
// line with the next tile, so the line is fetched, or written in part, twice
// unless both tiles run on one XCD at about the same time. Hence the orders
// and cache policies of ragged_policy (program.cpp). Measured against the
// element-wise kernel, buffers of three calls in turn: f32 [16,1001,770] ->
// bf16 [16,770,1001] (74 MB) 74.9 -> 12.9 us, 5.7 TB/s (18.0 from HBM, buffers
// of twelve calls); int8 [1027,4099] -> f32 (21 MB) 32.7 -> 7.7 us; int8
// [3637,7047] -> f32 (128 MB) 178 -> 28.5 us; f32 [262143,64] (134 MB) 96 ->
// 27 us; int8 [4096,11007] -> f16 (135 MB) 305 -> 23.8 us. Reading the
// arguments in one batch and the parameters beside the tile loads is 1-6% of
// these.
#include "kernels.h"

namespace relx {
namespace {

// Tile position and extents of a block (block-uniform).
struct RagTile {
  int64_t sbase, dbase; // element offsets of the tile's first source and destination element
  int qn, cn;           // q and c inside the tile
};

template <int TQ, int TC> __device__ __forceinline__ RagTile rag_tile(const KArgs &a, uint32_t t) {
  uint32_t tq, tc, r2;
  tile_of(a, t, tq, tc, r2);
  RagTile p{a.sbase, a.dbase, 0, 0};
  decompose<kBatchLevels>(a.lv, r2, p.sbase, p.dbase); // transposes carry no pads
  const uint32_t q0 = tq * TQ, c0 = tc * TC;
  p.sbase += static_cast<int64_t>(c0) * a.t_ssc + q0;
  p.dbase += static_cast<int64_t>(q0) * a.t_dsq + c0;
  p.qn = static_cast<int>(min(static_cast<uint32_t>(TQ), a.t_qn - q0));
  p.cn = static_cast<int>(min(static_cast<uint32_t>(TC), a.t_cn - c0));
  return p;
}

// Every argument a block reads, in one batch of scalar loads (see hot() in
// kernels.h).
template <int CH> __device__ __forceinline__ void rag_hot(const KArgs &a) {
  asm volatile("" ::"s"(a.src), "s"(a.dst), "s"(a.work), "s"(a.sbase), "s"(a.dbase), "s"(a.t_full),
               "s"(a.t_flags), "s"(a.t_ssc), "s"(a.t_dsq), "s"(a.t_qn), "s"(a.t_cn), "s"(gridDim.x));
  hot(a.t_plane);
  hot(a.t_group);
  hot(a.t_g);
  hot(a.t_tail);
  hot(a.t_nc);
  hot_levels<kBatchLevels>(a);
  hot_chain<CH>(a);
}

// The tile's source vectors: lane vid of VPR vectors per row. `back`: how far
// a cut vector starts before its place.
template <int WIN, int VPR, int NI, bool NT>
__device__ __forceinline__ void rag_load_nt(const KArgs &a, const RagTile &p, vec4 (&in)[NI]) {
  constexpr int VI = 16 / WIN;
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int vid = threadIdx.x + j * kBlock;
    const int row = vid / VPR, col = vid % VPR * VI;
    const int at = min(col, p.qn - VI);
    in[j] = ldu_n<16, NT>(row < p.cn && col < p.qn ? a.src + (p.sbase + row * a.t_ssc + at) * WIN
                                               : g_unused_src);
  }
}

template <int WIN, int VPR, int NI>
__device__ __forceinline__ void rag_load(const KArgs &a, const RagTile &p, vec4 (&in)[NI]) {
  if (a.t_flags & kTileNtLoad) // block-uniform
    rag_load_nt<WIN, VPR, NI, true>(a, p, in);
  else
    rag_load_nt<WIN, VPR, NI, false>(a, p, in);
}

// Each lane's elements into LDS through put(row, column, value).
template <int WIN, int VPR, int NI, typename Put>
__device__ __forceinline__ void rag_to_lds(const RagTile &p, const vec4 (&in)[NI], Put put) {
  constexpr int VI = 16 / WIN;
  if (p.qn % VI == 0) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int vid = threadIdx.x + j * kBlock;
      const int row = vid / VPR, col = vid % VPR * VI;
      uint32_t v[VI];
      unpack<WIN, VI>(&in[j], v);
#pragma unroll
      for (int e = 0; e < VI; ++e)
        put(row, col + e, v[e]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int vid = threadIdx.x + j * kBlock;
      const int row = vid / VPR, col = vid % VPR * VI;
      if (row >= p.cn || col >= p.qn)
        continue;
      const int back = col + VI > p.qn ? col + VI - p.qn : 0;
      uint32_t v[VI];
      unpack<WIN, VI>(&in[j], v);
#pragma unroll
      for (int e = 0; e < VI; ++e)
        if (e >= back)
          put(row, col - back + e, v[e]);
    }
  }
}

template <int WIN, int WOUT, int CH, int TQ, int TC, bool NTS>
__global__ __launch_bounds__(kBlock) void k_transpose_rag(KArgs a) {
  constexpr int kPitch = TQ + 1;
  __shared__ uint32_t tile[TC * kPitch]; // [c][q]
  constexpr int VI = 16 / WIN, VO = 16 / WOUT;
  constexpr int VPRI = TQ / VI, VPRO = TC / VO;
  constexpr int NI = TC * VPRI / kBlock, NO = TQ * VPRO / kBlock;
  static_assert(NI * kBlock == TC * VPRI && NO * kBlock == TQ * VPRO, "whole tiles per block");
  rag_hot<CH>(a);
  const uint32_t t = (a.t_flags & kTileXcd) ? xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
  if (t >= a.work)
    return;
  const RagTile p = rag_tile<TQ, TC>(a, t);
  vec4 in[NI];
  rag_load<WIN, VPRI, NI>(a, p, in);
  VecParams par[NO];
#pragma unroll
  for (int j = 0; j < NO; ++j) {
    const int vid = threadIdx.x + j * kBlock;
    par[j] = fetch_params<CH>(a, p.dbase + vid / VPRO * a.t_dsq + vid % VPRO * VO);
  }
  rag_to_lds<WIN, VPRI, NI>(p, in, [&](int row, int col, uint32_t x) { tile[row * kPitch + col] = x; });
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NO; ++j) {
    const int vid = threadIdx.x + j * kBlock;
    const int row = vid / VPRO, col = vid % VPRO * VO;
    if (row >= p.qn || col >= p.cn)
      continue;
    uint32_t v[VO];
#pragma unroll
    for (int e = 0; e < VO; ++e)
      v[e] = tile[(col + e) * kPitch + row];
    const int64_t dof = p.dbase + row * a.t_dsq + col;
    chain_vec_p<CH, VO, true>(a, v, dof, par[j]);
    vec4 out;
    pack<WOUT, VO>(v, &out);
    if (col + VO <= p.cn)
      stu_n<16, NTS>(a.dst + dof * WOUT, out);
    else
      stu_cut(a.dst + dof * WOUT, out, static_cast<uint32_t>(p.cn - col) * WOUT);
  }
}

// One-byte sources: a tile of 128 c by 128 q kept in LDS as bytes already
// transposed ([q][c]), as transpose_b_body.
template <int WOUT, int CH, int TQ, int TC, bool NTS>
__global__ __launch_bounds__(kBlock) void k_transpose_rag_b(KArgs a) {
  constexpr int PAD = WOUT == 1 ? 16 : 8, PT = TC + PAD; // LDS reads of VO bytes stay aligned
  __shared__ __align__(16) uint8_t tile[TQ * PT];        // [q][c]
  constexpr int VPRI = TQ / 16, NI = TC * VPRI / kBlock;
  constexpr int VO = 16 / WOUT, VPRO = TC / VO;
  constexpr int NO = TQ * VPRO / kBlock;
  rag_hot<CH>(a);
  const uint32_t t = (a.t_flags & kTileXcd) ? xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
  if (t >= a.work)
    return;
  const RagTile p = rag_tile<TQ, TC>(a, t);
  vec4 in[NI];
  rag_load<1, VPRI, NI>(a, p, in);
  const int col = threadIdx.x % VPRO * VO;
  // the store phase's parameters, in flight with the tile loads where a lane
  // stores few vectors
  constexpr bool kEarly = NO <= 4;
  VecParams early[kEarly ? NO : 1];
  if constexpr (kEarly) {
#pragma unroll
    for (int j = 0; j < NO; ++j)
      early[j] = fetch_params<CH>(a, p.dbase + (threadIdx.x / VPRO + j * (kBlock / VPRO)) * a.t_dsq + col);
  }
  rag_to_lds<1, VPRI, NI>(p, in, [&](int row, int col, uint32_t x) {
    tile[col * PT + row] = static_cast<uint8_t>(x);
  });
  __syncthreads();
#pragma unroll 4
  for (int j = 0; j < NO; ++j) {
    const int row = threadIdx.x / VPRO + j * (kBlock / VPRO);
    if (row >= p.qn || col >= p.cn)
      break;
    const uint8_t *tp = tile + row * PT + col;
    const int64_t dof = p.dbase + row * a.t_dsq + col;
    VecParams par;
    if constexpr (kEarly)
      par = early[j];
    else
      par = fetch_params<CH>(a, dof);
    vec4 w = {0u, 0u, 0u, 0u};
    if constexpr (VO == 16) {
      w = *reinterpret_cast<const vec4 *>(tp);
    } else if constexpr (VO == 8) {
      const uint2 b = *reinterpret_cast<const uint2 *>(tp);
      w.x = b.x;
      w.y = b.y;
    } else {
      w.x = *reinterpret_cast<const uint32_t *>(tp);
    }
    uint32_t val[VO];
    unpack<1, VO>(&w, val);
    chain_vec_p<CH, VO, true>(a, val, dof, par);
    vec4 out;
    pack<WOUT, VO>(val, &out);
    if (col + VO <= p.cn)
      stu_n<16, NTS>(a.dst + dof * WOUT, out);
    else
      stu_cut(a.dst + dof * WOUT, out, static_cast<uint32_t>(p.cn - col) * WOUT);
  }
}

template <int WIN, int WOUT, int CH, int TQ, int TC, bool NTS>
hipError_t ragged_tile_launch(const KArgs &a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.work)), block(kBlock);
  if constexpr (WIN == 1)
    hipLaunchKernelGGL((k_transpose_rag_b<WOUT, CH, TQ, TC, NTS>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((k_transpose_rag<WIN, WOUT, CH, TQ, TC, NTS>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <int WIN, int WOUT, int CH> hipError_t ragged_launch(const KArgs &a, hipStream_t s) {
  const bool nts = (a.t_flags & kTileNtStore) != 0;
  constexpr int LQ = ragged_large_q(WIN), LC = kRaggedLargeC;
  if (a.t_wq == kRaggedTile && a.t_wc == kRaggedTile)
    return nts ? ragged_tile_launch<WIN, WOUT, CH, kRaggedTile, kRaggedTile, true>(a, s)
               : ragged_tile_launch<WIN, WOUT, CH, kRaggedTile, kRaggedTile, false>(a, s);
  if (a.t_wq == LQ && a.t_wc == LC && !nts)
    return ragged_tile_launch<WIN, WOUT, CH, LQ, LC, false>(a, s);
  return hipErrorInvalidValue;
}

} // namespace

RELX_DISPATCH_FAST(transpose_ragged_fast, ragged_launch)
RELX_DISPATCH_GENERIC(transpose_ragged_generic, ragged_launch)

} // namespace relx
