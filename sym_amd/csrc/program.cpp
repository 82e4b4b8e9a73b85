// program.cpp - turn a bound plan into device launch programs.
//
// prepareProgram's checks (libreloc/src/TypedExecute.cpp:292-403) are
// restated here: every stage must be one of the implemented policy tables,
// quantize reciprocals are formed once in binary32 from the declared scale,
// and channel maps that are a single result coordinate (possibly `dN mod K`
// with K >= the extent) are recognised so the fast kernels can index
// parameters without evaluating expressions. The fill written into pads is
// the original fill folded to the result type (fillAt,
// libreloc/src/TypedExecute.cpp:422-464).
#include "runtime.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "index.h"

// Rows of m per permute block: at most this many source bytes over all C.
#ifndef RELX_PERMUTE_SOURCE_BYTES
#define RELX_PERMUTE_SOURCE_BYTES 8192
#endif
// A permute block reads G of the C channels of each source row, at most this
// many bytes of the row (G halves from C while it is more), and the blocks run
// group by group: the resident blocks then write the result planes of one
// group, not all C. Measured on the MI355X over buffers spanning 2.4 GB, C5's
// [8,4096,32,128] f16 -> int8 launch: 74.1 us with all 32 heads per block
// (2 rows), 68.2 us with 16 (2 rows of 4 KiB), 66.3 us with 16 and one row
// per block (RELX_PERMUTE_SOURCE_BYTES), against 65.2 us for a 16-byte copy
// of the same bytes; [64,4096,..] 572 -> 498 us.
#ifndef RELX_PERMUTE_GROUP_BYTES
#define RELX_PERMUTE_GROUP_BYTES 4096
#endif


namespace relx {

FastDiv make_div(int64_t d64) {
  FastDiv f{};
  const uint32_t d = static_cast<uint32_t>(d64 < 1 ? 1 : d64);
  f.d = d;
  uint32_t s = 0;
  while (s < 32 && (uint64_t{1} << s) < d)
    ++s;
  f.s = s;
  // m = floor(2^32 * (2^s - d) / d) + 1
  const unsigned __int128 num = (static_cast<unsigned __int128>(1) << 32) *
                                ((static_cast<unsigned __int128>(1) << s) - d);
  f.m = static_cast<uint32_t>(num / d + 1);
  return f;
}

namespace {

uint8_t op_of(const BoundStage &s) {
  if (s.transform == kCast) {
    if (s.in.f32() && s.out.f16() && s.policy == kIeeeRne)
      return kOpF32toF16;
    if (s.in.f16() && s.out.f32() && s.policy == kExact)
      return kOpF16toF32;
    if (s.in.f32() && s.out.bf16() && s.policy == kIeeeRne)
      return kOpF32toBF16;
    if (s.in.bf16() && s.out.f32() && s.policy == kExact)
      return kOpBF16toF32;
    fail("unsupported_stage",
         "only cast f32->f16/bf16 ieee_rne and f16/bf16->f32 exact are implemented");
  }
  if (s.transform == kQuantize) {
    if (!(s.in.f32() && s.out.i8() && s.policy == kSymmetricRne))
      fail("unsupported_stage", "only quantize f32->s8 symmetric_rne is implemented");
    return kOpQuantize;
  }
  if (!(s.in.i8() && s.out.f32() && s.policy == kAffine))
    fail("unsupported_stage", "only dequantize s8->f32 affine is implemented");
  return kOpDequantize;
}

int64_t sext(uint64_t bits, uint32_t width) {
  if (width >= 64)
    return static_cast<int64_t>(bits);
  const uint64_t mask = (uint64_t{1} << width) - 1;
  uint64_t v = bits & mask;
  if (v >> (width - 1))
    v |= ~mask;
  return static_cast<int64_t>(v);
}

} // namespace

// --------------------------------------------------------------- stages

void prepare_stages(const Bound &b, Prepared &p) {
  const size_t rank = b.result_extents.size();
  p.res_strides.assign(rank, 1);
  for (size_t j = rank; j-- > 1;)
    p.res_strides[j - 1] = p.res_strides[j] * b.result_extents[j];
  for (size_t k = 0; k < b.stages.size(); ++k) {
    const BoundStage &s = b.stages[k];
    HostStage h;
    h.op = op_of(s);
    h.in_width = s.in.width();
    h.out_width = s.out.width();
    const std::string where = "stage " + std::to_string(k) + ": ";
    if (h.op == kOpQuantize || h.op == kOpDequantize) {
      if (!s.scale.present || !s.scale.type.f32() ||
          s.scale.bytes.size() != static_cast<size_t>(s.scale.length) * 4)
        fail("invalid_parameter", where + "scale is absent or malformed");
      h.scale.resize(static_cast<size_t>(s.scale.length));
      std::memcpy(h.scale.data(), s.scale.bytes.data(), s.scale.bytes.size());
      for (float v : h.scale)
        if (!(v > 0.0f) || v == __builtin_inff())
          fail("invalid_parameter", where + "scale is not finite and strictly positive");
      h.zero_point.assign(1, 0);
      if (s.zero_point.present) {
        const uint32_t w = s.zero_point.type.width();
        if (s.zero_point.type.kind != kInteger || !w || w > 8 ||
            s.zero_point.bytes.size() != static_cast<size_t>(s.zero_point.length) * w)
          fail("invalid_parameter", where + "zero point is malformed");
        h.zero_point.resize(static_cast<size_t>(s.zero_point.length));
        for (int64_t i = 0; i < s.zero_point.length; ++i) {
          uint64_t raw = 0;
          std::memcpy(&raw, s.zero_point.bytes.data() + i * w, w);
          const int64_t v = sext(raw, s.zero_point.type.bits);
          if (v < -128 || v > 127)
            fail("invalid_parameter", where + "zero point outside [-128, 127]");
          h.zero_point[static_cast<size_t>(i)] = static_cast<int32_t>(v);
        }
      }
      if (h.op == kOpQuantize) {
        for (int32_t zp : h.zero_point)
          if (zp != 0)
            fail("invalid_parameter", where + "symmetric_rne admits only zero point 0");
        h.inv.resize(h.scale.size());
        for (size_t i = 0; i < h.scale.size(); ++i)
          h.inv[i] = 1.0f / h.scale[i]; // fl32(1/scale), formed once
      }
    }
    if (s.has_channel) {
      if (h.scale.empty())
        fail("invalid_parameter", where + "per-channel stage without scales");
      h.len = static_cast<int64_t>(h.scale.size());
      if (h.zero_point.size() > 1 && h.zero_point.size() != h.scale.size())
        fail("invalid_parameter", where + "zero point length disagrees with the scale");
      h.mode = kChanExpr;
      const Expr &c = s.channel;
      if (!c.empty() && c[0].op == kPushDim && c[0].value >= 0 &&
          static_cast<size_t>(c[0].value) < rank) {
        const int dim = static_cast<int>(c[0].value);
        bool is_dim = c.size() == 1;
        if (c.size() == 3 && c[2].op == kMod && (c[1].op == kPushConst || c[1].op == kPushSym)) {
          const int64_t mod = c[1].op == kPushConst ? c[1].value
                                                    : b.symbols[static_cast<size_t>(c[1].value)];
          if (mod > 0 && b.result_extents[static_cast<size_t>(dim)] <= mod)
            is_dim = true;
        }
        if (is_dim) {
          h.mode = kChanDim;
          h.dim = dim;
        }
      }
      if (h.mode == kChanExpr) {
        for (const Token &t : c) {
          ChanToken ct{t.op, 0, t.value};
          if (t.op == kPushSym) {
            ct.op = kPushConst;
            ct.value = b.symbols[static_cast<size_t>(t.value)];
          }
          h.tokens.push_back(ct);
        }
      }
    } else {
      h.mode = kChanNone;
      h.len = 1;
      if (h.scale.size() > 1 || h.zero_point.size() > 1)
        fail("invalid_parameter", where + "per-tensor stage with more than one parameter");
    }
    p.stages.push_back(std::move(h));
  }
}

// Fill bits at boundary `to` (every pad settled), folded through the stages
// after each pad's entry stage; nullopt-like `has` = false without pads.
bool fill_at(const Bound &b, const Prepared &p, uint32_t to, uint64_t &bits) {
  if (b.fills.empty()) {
    if (!b.typed && !b.layout.pads.empty()) {
      bits = b.layout.pads.front().bits;
      return true;
    }
    return false;
  }
  bool have = false;
  for (const PlanFill &f : b.fills) {
    if (f.stage > to)
      fail("pads_not_settled", "a pad enters after boundary " + std::to_string(to));
    uint64_t v = f.bits;
    for (uint32_t k = f.stage; k < to; ++k) {
      const HostStage &s = p.stages[k];
      if (s.mode != kChanNone)
        fail("fill_crosses_channel_stage",
             "a pad fill would cross per-channel stage " + std::to_string(k));
      v = host_apply(s, v, 0);
    }
    if (have && v != bits)
      fail("mixed_fills_unsupported",
           "pads carry different values at boundary " + std::to_string(to));
    bits = v;
    have = true;
  }
  if (to == p.stages.size() && !b.layout.pads.empty() && b.layout.pads.front().bits != bits)
    fail("fill_mismatch", "folded fill disagrees with the layout's fused fill");
  return have;
}

uint64_t host_apply(const HostStage &s, uint64_t x, int64_t c) {
  switch (s.op) {
  case kOpF32toF16:
    return f32_to_f16_bits(static_cast<uint32_t>(x));
  case kOpF16toF32:
    return f16_to_f32_bits(static_cast<uint16_t>(x));
  case kOpF32toBF16:
    return f32_to_bf16_bits(static_cast<uint32_t>(x));
  case kOpBF16toF32:
    return bf16_to_f32_bits(static_cast<uint16_t>(x));
  case kOpQuantize: {
    float f;
    const uint32_t b = static_cast<uint32_t>(x);
    std::memcpy(&f, &b, 4);
    return static_cast<uint8_t>(quantize_one(f, s.inv[static_cast<size_t>(c)]));
  }
  default: {
    const int32_t q = static_cast<int8_t>(static_cast<uint8_t>(x));
    const int32_t zp = s.zero_point.size() == 1 ? s.zero_point[0]
                                                : s.zero_point[static_cast<size_t>(c)];
    const float y = static_cast<float>(q - zp) * s.scale[static_cast<size_t>(c)];
    uint32_t r;
    std::memcpy(&r, &y, 4);
    return r;
  }
  }
}

// ------------------------------------------------------------ programs

namespace {

bool dense_dst(const BoundLayout &L, const std::vector<int64_t> &pext) {
  int64_t running = 1;
  for (size_t k = pext.size(); k-- > 0;) {
    if (L.dst_strides[k] != running)
      return false;
    running *= pext[k];
  }
  return true;
}

// Per-vector channel behaviour for V consecutive destination elements whose
// dense offset is a multiple of V: 0 constant, 1 +1 per element, -1 neither.
int vec_mode(const HostStage &s, const Prepared &p, const Bound &b, int64_t V) {
  if (s.mode == kChanNone)
    return 0;
  if (s.mode != kChanDim)
    return -1;
  const int64_t rs = p.res_strides[static_cast<size_t>(s.dim)];
  const int64_t re = b.result_extents[static_cast<size_t>(s.dim)];
  if (re > s.len)
    return -1; // a coordinate could leave the table: keep the checked kernel
  if (rs % V == 0)
    return 0;
  if (rs == 1 && re % V == 0)
    return 1;
  return -1;
}

// Channel behaviour along a destination row of `len` elements (the innermost
// coalesced axis, whose rows start at multiples of len): 0 constant along the
// row, 1 the column itself, -1 neither.
int row_mode(const HostStage &s, const Prepared &p, const Bound &b, int64_t len) {
  if (s.mode == kChanNone)
    return 0;
  if (s.mode != kChanDim)
    return -1;
  const int64_t rs = p.res_strides[static_cast<size_t>(s.dim)];
  const int64_t re = b.result_extents[static_cast<size_t>(s.dim)];
  if (re > s.len)
    return -1;
  if (rs % len == 0)
    return 0;
  if (rs == 1 && re == len)
    return 1;
  return -1;
}

// Channel behaviour of V consecutive elements of a flat tensor from any
// offset (DevStage::vec of k_flat): 0 per tensor, 2 at most two channels, 3 +1
// per element and at most one wrap, -1 none of these.
int flat_mode(const HostStage &s, const Prepared &p, const Bound &b, int64_t V) {
  if (s.mode == kChanNone)
    return 0;
  if (s.mode != kChanDim)
    return -1;
  const int64_t rs = p.res_strides[static_cast<size_t>(s.dim)];
  const int64_t re = b.result_extents[static_cast<size_t>(s.dim)];
  if (re > s.len)
    return -1;
  if (rs == 1 && re >= V)
    return 3;
  return rs >= V ? 2 : -1;
}

bool interleave_family(int family) {
  return family == kFamInterleave || family == kFamRaggedInterleave;
}

bool transpose_family(int family) {
  return family == kFamTranspose || family == kFamRaggedTranspose;
}

// Families whose work items are vectors of the innermost axis.
bool row_family(int family) {
  return family == kFamStream || family == kFamRows || family == kFamFlat;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Bytes above which little of a launch is still in the 256 MB Infinity Cache
// when its buffers come round again.
constexpr int64_t kColdBytes = int64_t{96} << 20;

// A stage takes another parameter entry for each element of a vector.
bool channel_per_element(const KArgs &a) {
  for (int i = 0; i < a.chain.n; ++i)
    if (a.chain.st[i].vec == 1)
      return true;
  return false;
}

// Tile widths, order and cache policy of a ragged transpose launch that moves
// `bytes` and is c_ext wide along c. A row that starts inside a line shares it
// with the next tile. Figures are over buffers of three calls in turn, which
// small launches find in the Infinity Cache in part; a second one is over
// twelve, which none do.
//   Destination rows that start on 64-byte boundaries: streaming stores of
//   64 x 64 tiles (int8 [4096,11007] -> f16 24.5 us against 34.8 cached).
//   Others are written in part by two tiles, which streaming would send to
//   memory as two partial writes (f32 [16,1001,770] -> f16 16.5 against 13.0
//   us cached). Large launches (kColdBytes) of planes wider than one 64 x 64
//   tile along c take large tiles, which have fewer such lines, and streaming
//   loads (f32 [32,2047,513] -> f16, 202 MB, 38.8 and 46.5 us, small tiles
//   with cached loads 47.4 and 48.4). Narrower planes would leave half of a
//   large tile empty (f32 [32768,24,40] 89.0 us, small 51.1; f32 -> f16
//   [8192,16,128] 44.6, small 23.0), and a channel per element of a row, whose
//   entries every vector loads, leaves them behind at any width (int8 -> f16
//   [8208,8192] scaled along c 144, small 101). Smaller launches take 64 x 64 tiles, of
//   which more run at once (int8 [1027,4099] -> f32, 21 MB, 8.6 against 14.2
//   us; [3637,7047] -> f16, 77 MB, 14.9 and 23.8, large 20.9 and 22.4).
//   Streaming loads, where rows share lines: large launches only (f32
//   [16,1001,770] -> f16 13.0 against 15.6 us; f16 [8,4001,1001] 27.8 and
//   32.0 with large tiles, cached 30.6 and 30.9). Launches whose lines are all
//   their own keep cached loads at any size: f32 [64,262000] 22.9 and 26.8 us,
//   streaming 25.5 and 25.6; [16,1040,784] -> f16 12.8 and 18.3, streaming
//   15.0 and 18.8.
// Each XCD takes a contiguous run of tiles (74 MB activation above: 18.6 ->
// 13.0 us), so tiles that share a line meet in one L2, except where no line
// is shared: words whose rows are all aligned (f32 [262000,64] 22.9 -> 21.0
// us without).
void ragged_policy(KArgs &a, int64_t bytes, int64_t c_ext) {
  auto aligned = [&](int64_t base, int64_t stride, int64_t batch, int w) {
    return (base * w) % 64 == 0 && (stride * w) % 64 == 0 && (batch * w) % 64 == 0;
  };
  bool src = true, dst = true;
  for (int j = 0; j < kBatchLevels; ++j) {
    src = src && aligned(a.sbase, a.t_ssc, a.lv[j].ss, a.win);
    dst = dst && aligned(a.dbase, a.t_dsq, a.lv[j].ds, a.wout);
  }
  const bool cold = bytes >= kColdBytes, xcd = a.win == 1 || !src || !dst;
  const bool large = !dst && cold && c_ext > kRaggedTile && !channel_per_element(a);
  a.t_wq = static_cast<uint16_t>(large ? ragged_large_q(a.win) : kRaggedTile);
  a.t_wc = static_cast<uint16_t>(large ? kRaggedLargeC : kRaggedTile);
  a.t_flags = (xcd ? kTileXcd : 0u) | (cold && xcd ? kTileNtLoad : 0u) | (dst ? kTileNtStore : 0u);
}

// Aligned transpose boxes of at least this many elements whose last tiles are
// cut run as one ragged launch, and a device-resident call's whatever their
// size (f32 [128,96] -> f16 transposed 11.0 us a pass as tiles and a strip,
// 7.0 as one launch; [72,200], with two strips, 14.7 and 7.0). A smaller box
// of a transfer keeps its whole tiles and strips, and so do the boxes of
// tiles_and_strips.
constexpr int64_t kRaggedWholeElements = int64_t{1} << 14;

// The ragged transpose needs one vector of q and takes c extents from here on:
// a tile is 64 c wide whatever c is, and the element-wise kernel's stores are
// then the better ones (f32 [64,3,50177] -> f16 [64,50177,3] 32 us element-wise,
// 55 in tiles; [32,6,20001] 17.4 and 14.1, [32,12,20001] 27.3 and 14.3; along
// q, [32,20001,4] 15.0 and 12.6, [32,20001,12] 40.8 and 13.1).
constexpr int64_t kRaggedMinC = 6;
// Elements a tile must hold on average. A tile costs one block's load, barrier
// and store whatever it holds, about a nanosecond each with the chip full, so
// many planes that each fill little of theirs are the element-wise kernel's
// (f32, tiles and element-wise: [131072,12,12], 144 a tile, 133.7 and 43.4 us;
// [131072,16,16], 256, 127.3 and 78.5; [2796,6,1000], 375, 72.1 and 39.5;
// [2796,1000,6], 375, 60.4 and 65.2; [32768,64,8], 512, 37.1 and 42.9;
// [32768,24,40], 960, 51.1 and 76.6; f16 [65536,16,16] 59.1 and 42.0,
// [32768,64,8] 30.1 and 39.3). Dequantizing an element at a time costs almost
// twice as much: int8 -> f16 [174762,6,16], 96 a tile, 164 and 73.5 us;
// [65536,16,16] 63.3 and 71.0; [13981,6,200], 300, 68.1 and 72.3.
constexpr int64_t kRaggedTileElements = 384;
constexpr int64_t kRaggedTileDequantized = 256;

// A chain that a direct permute of planes of `rs` elements and C channels can
// run: a compile-time one whose parameter stage is per tensor or along c.
bool direct_chain(const Bound &b, const Prepared &p, uint32_t k, int chain_code, int64_t rs, int64_t C) {
  if (chain_code == kChainGeneric)
    return false;
  const int at = chain_param_stage(chain_code);
  if (at < 0)
    return true;
  const HostStage &s = p.stages[k + static_cast<uint32_t>(at)];
  if (s.mode == kChanNone)
    return true;
  return s.mode == kChanDim && p.res_strides[static_cast<size_t>(s.dim)] == rs &&
         b.result_extents[static_cast<size_t>(s.dim)] == C;
}

// Channels G (a divisor of C, at most RELX_PERMUTE_GROUP_BYTES of a source
// row) and rows T of a direct permute's block whose power-of-two pair (G, T)
// holds fewer than 256 vectors of 16 bytes: the pair whose blocks keep the
// most of their 256 lanes busy, the cut last m-tile counted, over at most
// three vectors per lane; among equals the longer row part. f16 -> int8 on the
// MI355X, general kernel and power-of-two rule -> here: [8,1024,40,128] 42.5 ->
// 21.7 us (10 channels of one row, 160 vectors -> 8 of two, 256),
// [16,1024,32,96] 45.5 -> 26.9 us (192 -> 768), [33,999,8,128] 35.9 -> 18.0 us
// (odd m: 128 -> 256).
// Pairs that fill three quarters of the lanes and store runs of 192 bytes or
// more only widen G: more rows make a block of several rounds, whose loads
// and stores alternate (f32 [16,1024,32,96], 8 channels: one row 65.1 us, four
// 71.9; f32 -> f16 54.0 and 54.2, 384-byte runs; runs of 96 bytes above gain).
// So do blocks of 256 vectors and more, which keep their pair (f32
// [8,1024,7,256], 7 channels of one row, 448 vectors, 20.4 us, four rows of one
// 22.5; f16 [128,196,12,64] 14.5 and 14.6, int8 -> f16 [8,1024,24,128] 14.2 and
// 15.8).
void permute_block(int64_t C, int64_t M, int64_t E, int win, int wout, int64_t &G, int64_t &T) {
  const bool rows = T * G * E * win / 16 < 192 || T * E * wout < 192;
  const int64_t t_lo = rows ? 1 : T, t_hi = rows ? std::min<int64_t>(8, M) : T;
  double best = 0.0;
  for (int64_t g = C; g >= 1; --g) {
    if (C % g || (g * E * win > RELX_PERMUTE_GROUP_BYTES && g > 1))
      continue;
    for (int64_t t = t_lo; t <= t_hi; ++t) {
      const int64_t n = t * g * E * win / 16;
      if (t * g * E * wout > 32768 || (n > 3 * 256 && t > 1))
        continue;
      const double use = static_cast<double>(n) / static_cast<double>(ceil_div(n, 256) * 256) *
                         static_cast<double>(M) / static_cast<double>(ceil_div(M, t) * t);
      if (use > best + 1e-9) {
        best = use;
        G = g;
        T = t;
      }
    }
  }
}

} // namespace

std::unique_ptr<DeviceProgram> build_program(const Bound &b, const Prepared &p, uint32_t k) {
  const BoundLayout &L = b.layout;
  const int r = static_cast<int>(L.extents.size());
  if (r > kMaxRank)
    fail("unsupported_layout", "more than " + std::to_string(kMaxRank) + " coalesced axes");
  const uint32_t nst = static_cast<uint32_t>(p.stages.size());
  if (k > nst)
    fail("invalid_boundary", "wire boundary beyond the last stage");
  if (nst - k > static_cast<uint32_t>(kMaxStages))
    fail("unsupported_stage", "too many device stages");
  auto dp = std::make_unique<DeviceProgram>();
  dp->boundary = k;
  KArgs &a = dp->base;
  std::memset(&a, 0, sizeof(a));
  a.rank = r;
  const int win = b.typed ? static_cast<int>(k == 0 ? b.source_type.width()
                                                    : p.stages[k - 1].out_width)
                          : static_cast<int>(L.element_size);
  const int wout = static_cast<int>(L.element_size);
  a.win = win;
  a.wout = wout;
  std::vector<int64_t> pext(static_cast<size_t>(r)), lo(static_cast<size_t>(r), 0);
  bool any_pad = false, inner_pad = false;
  for (int i = 0; i < r; ++i) {
    pext[static_cast<size_t>(i)] = L.extents[static_cast<size_t>(i)];
    a.vext[i] = L.extents[static_cast<size_t>(i)];
    a.ss[i] = L.src_strides[static_cast<size_t>(i)];
    a.ds[i] = L.dst_strides[static_cast<size_t>(i)];
  }
  for (const BoundPad &pd : L.pads) {
    pext[static_cast<size_t>(pd.axis)] += pd.lo + pd.hi;
    lo[static_cast<size_t>(pd.axis)] = pd.lo;
    any_pad = true;
    if (pd.axis == r - 1)
      inner_pad = true;
  }
  for (int i = 0; i < r; ++i) {
    a.pext[i] = pext[static_cast<size_t>(i)];
    a.lo[i] = lo[static_cast<size_t>(i)];
  }
  uint64_t fill = 0;
  a.has_fill = fill_at(b, p, nst, fill) ? 1 : 0;
  a.fill64 = fill;
  a.fill = static_cast<uint32_t>(fill);

  // result coordinates (channels); layout plans have none
  a.res_rank = static_cast<int32_t>(b.result_extents.size());
  for (int j = 0; j < a.res_rank && j < kMaxRank; ++j) {
    a.rs[j] = p.res_strides[static_cast<size_t>(j)];
    a.re[j] = b.result_extents[static_cast<size_t>(j)];
  }
  if (a.res_rank > kMaxRank)
    fail("unsupported_layout", "result rank above the device limit");

  // stages [k, n): parameters packed into one float and one int table
  Chain &ch = a.chain;
  ch.n = static_cast<int32_t>(nst - k);
  bool needs_expr = false;
  for (uint32_t i = k; i < nst; ++i) {
    const HostStage &h = p.stages[i];
    DevStage &d = ch.st[i - k];
    d.op = h.op;
    d.mode = h.mode;
    d.ch_rs_div = make_div(1); // per tensor: entry 0
    d.ch_re_div = make_div(1);
    if (h.mode == kChanDim) {
      d.ch_rs = p.res_strides[static_cast<size_t>(h.dim)];
      d.ch_re = b.result_extents[static_cast<size_t>(h.dim)];
      if (d.ch_rs < (int64_t{1} << 32) && d.ch_re < (int64_t{1} << 32)) {
        d.ch_rs_div = make_div(d.ch_rs);
        d.ch_re_div = make_div(d.ch_re);
      }
    }
    d.len = static_cast<uint32_t>(h.len);
    d.scale_off = static_cast<uint32_t>(dp->pf.size());
    const std::vector<float> &f = h.op == kOpQuantize ? h.inv : h.scale;
    dp->pf.insert(dp->pf.end(), f.begin(), f.end());
    d.zp_off = static_cast<uint32_t>(dp->pi.size());
    dp->pi.insert(dp->pi.end(), h.zero_point.begin(), h.zero_point.end());
    d.zp_per_ch = h.zero_point.size() > 1 ? 1 : 0;
    if (h.mode == kChanExpr) {
      needs_expr = true;
      if (ch.ntok + static_cast<int>(h.tokens.size()) > kMaxChanTokens)
        fail("unsupported_stage", "channel expression too long for the device");
      d.tok_begin = ch.ntok;
      d.tok_count = static_cast<int32_t>(h.tokens.size());
      for (const ChanToken &t : h.tokens)
        ch.tok[ch.ntok++] = t;
    }
  }
  if (dp->pf.empty())
    dp->pf.push_back(0.0f);
  if (dp->pi.empty())
    dp->pi.push_back(0);

  int64_t wire_elems = 1;
  if (b.typed) {
    for (int64_t e : b.source_extents)
      wire_elems *= e;
  } else {
    int64_t span = 0; // layout plans: the source span the strides reach
    for (int i = 0; i < r; ++i)
      span += (a.vext[i] - 1) * a.ss[i];
    wire_elems = span + 1;
  }
  dp->wire_elems = wire_elems;
  dp->wire_bytes = wire_elems * win;
  // Bounds proofs the kernels rely on: every source offset the valid box
  // reaches lies inside the wire, every destination offset inside the result.
  int64_t src_span = 0, dst_span = 0, total = 1;
  for (int i = 0; i < r; ++i) {
    if (a.ss[i] < 0 || a.ds[i] < 0)
      fail("unsupported_layout", "negative stride");
    int64_t t;
    if (__builtin_mul_overflow(a.vext[i] - 1, a.ss[i], &t) ||
        __builtin_add_overflow(src_span, t, &src_span) ||
        __builtin_mul_overflow(a.pext[i] - 1, a.ds[i], &t) ||
        __builtin_add_overflow(dst_span, t, &dst_span) ||
        __builtin_mul_overflow(total, a.pext[i], &total))
      fail("integer_overflow", "layout offsets overflow");
  }
  if (src_span >= wire_elems)
    fail("unsupported_layout", "the plan reads beyond its source (span " +
                                   std::to_string(src_span + 1) + " > " +
                                   std::to_string(wire_elems) + " elements)");
  dp->dst_elems = std::max(total, dst_span + 1);

  // ------------------------------------------------------ family choice
  const bool widths_ok = (win == 1 || win == 2 || win == 4) && (wout == 1 || wout == 2 || wout == 4);
  const bool dense = dense_dst(L, pext);
  int family = kFamGeneric;
  // stream items: 16 bytes on the wider side
  const int V = widths_ok ? 16 / std::max(win, wout) : 0;
  // per-channel stages in the fast kernels index with a 32-bit result offset
  const bool off32 = dp->dst_elems < (int64_t{1} << 32);
  auto channels_ok = [&](int64_t vlen) {
    for (uint32_t i = k; i < nst; ++i) {
      const int m = vec_mode(p.stages[i], p, b, vlen);
      if (m < 0 || (p.stages[i].mode == kChanDim && !off32))
        return false;
      ch.st[i - k].vec = static_cast<uint8_t>(m);
    }
    return true;
  };
  // the same for kernels whose vectors start at any element of a row but
  // never leave it (the channel is constant along a row, or the row's column),
  // and for flat tensors
  const int64_t row_len = r > 0 ? pext[static_cast<size_t>(r - 1)] : 1;
  auto row_channels_ok = [&](bool flat = false) {
    for (uint32_t i = k; i < nst; ++i) {
      const int m = flat ? flat_mode(p.stages[i], p, b, V) : row_mode(p.stages[i], p, b, row_len);
      if (m < 0 || (p.stages[i].mode == kChanDim && !off32))
        return false;
      ch.st[i - k].vec = static_cast<uint8_t>(m);
    }
    return true;
  };
  // stage sequences with a compile-time kernel body
  int chain_code = kChainGeneric;
  {
    std::vector<uint8_t> ops;
    for (uint32_t i = k; i < nst; ++i)
      ops.push_back(p.stages[i].op);
    using V8 = std::vector<uint8_t>;
    if (ops.empty())
      chain_code = kChainNone;
    else if (ops == V8{kOpF32toF16})
      chain_code = kChainF32F16;
    else if (ops == V8{kOpF16toF32})
      chain_code = kChainF16F32;
    else if (ops == V8{kOpDequantize, kOpF32toF16})
      chain_code = kChainDeqF16;
    else if (ops == V8{kOpDequantize})
      chain_code = kChainDeq;
    else if (ops == V8{kOpF16toF32, kOpQuantize})
      chain_code = kChainF16Quant;
    else if (ops == V8{kOpQuantize})
      chain_code = kChainQuant;
    else if (ops == V8{kOpF32toBF16})
      chain_code = kChainF32BF16;
    else if (ops == V8{kOpBF16toF32})
      chain_code = kChainBF16F32;
  }
  if (widths_ok && dense && !needs_expr && !any_pad && r >= 3 && r - 3 <= kBatchLevels) {
    // permute: destination [batch..., c, m, e] from a source holding
    // (m, c, e) contiguously -- two axes swapped above a contiguous inner
    // block (an activation's [B,S,H,D] -> [B,H,S,D])
    const int c = r - 3, m = r - 2, e = r - 1;
    const int64_t E = a.vext[e], C = a.vext[c], M = a.vext[m];
    const int VI = 16 / win;
    bool ok = a.ss[e] == 1 && a.ds[e] == 1 && a.ss[c] == E && a.ss[m] == C * E &&
              a.ds[m] == E && a.ds[c] == M * E && E % VI == 0 && (E * wout) % 16 == 0 &&
              C > 1 && M > 1;
    for (int i = 0; i < c; ++i)
      ok = ok && a.ss[i] % VI == 0;
    // G channels per block (RELX_PERMUTE_GROUP_BYTES)
    int64_t G = C;
    while (G % 2 == 0 && G * E * win > RELX_PERMUTE_GROUP_BYTES)
      G /= 2;
    // T rows of m per block: at most RELX_PERMUTE_SOURCE_BYTES of source over
    // all C (at least one row), an LDS tile of at most 32 KiB, T dividing M
    int64_t T = 0;
    if (ok) {
      T = 1;
      while (T * 2 <= M && M % (T * 2) == 0 && T * 2 * C * E * win <= RELX_PERMUTE_SOURCE_BYTES &&
             T * 2 * G * E * wout <= 32768)
        T *= 2;
      ok = T * G * E * wout <= 32768;
    }
    // blocks of fewer vectors than lanes take another G and T where the
    // launches run the direct kernel, whose last m-tile may be cut
    if (ok && T * G * E / VI < 256 && c <= 1 && direct_chain(b, p, k, chain_code, M * E, C))
      permute_block(C, M, E, win, wout, G, T);
    if (ok && channels_ok(VI)) {
      family = kFamPermute;
      a.vec = VI;
      a.p_t = static_cast<uint32_t>(T);
      a.p_g = static_cast<uint32_t>(G);
      a.p_lds = static_cast<uint32_t>(T * G * E * wout);
    }
  }
  if (family == kFamGeneric && widths_ok && dense && !needs_expr) {
    // stream: innermost axis contiguous on both sides, unpadded
    // a single contiguous axis need not be a multiple of the vector: its
    // launches then run k_flat, which takes the tail too (prefix_launches)
    if (a.ss[r - 1] == 1 && a.ds[r - 1] == 1 && !inner_pad &&
        (a.vext[r - 1] % V == 0 || (r == 1 && a.vext[0] >= V))) {
      bool ok = true;
      for (int i = 0; i < r - 1; ++i)
        ok = ok && a.ss[i] % V == 0;
      if (ok && channels_ok(V)) {
        family = kFamStream;
        a.vec = V;
        a.nlev = r <= 1 ? 1 : r <= 2 ? 2 : r <= 4 ? 4 : 8;
      }
    }
    // rows, flat: the same axes where the vectors do not fit (at least one
    // vector of valid elements; 32-bit columns)
    if (family == kFamGeneric && a.ss[r - 1] == 1 && a.ds[r - 1] == 1 && a.vext[r - 1] >= V &&
        row_len < kMaxLaunchWork - 64) {
      if (r == 1 && !any_pad && row_channels_ok(true))
        family = kFamFlat;
      else if (row_channels_ok())
        family = kFamRows;
      if (family != kFamGeneric) {
        a.vec = V;
        a.nlev = r <= 2 ? 2 : r <= 4 ? 4 : 8;
      }
    }
    // transpose: dst-inner axis has a source stride, another axis is
    // source-contiguous; tile-aligned extents, no pads
    if (family == kFamGeneric && !any_pad && r >= 2 && r - 2 <= kBatchLevels && a.ss[r - 1] != 1) {
      int qa = -1;
      for (int i = 0; i < r - 1; ++i)
        if (a.ss[i] == 1 && a.vext[i] > 1)
          qa = i;
      const int VI = 16 / win, VO = 16 / wout;
      // extents need not be multiples of 64: boxes with cut tiles run as
      // ragged launches (prefix_launches)
      if (qa >= 0 && a.vext[qa] >= 64 && a.vext[r - 1] >= 64 && a.ss[r - 1] % VI == 0 &&
          a.ds[qa] % VO == 0) {
        bool ok = true;
        for (int i = 0; i < r - 1; ++i)
          if (i != qa)
            ok = ok && a.ss[i] % VI == 0 && a.ds[i] % VO == 0;
        int64_t tiles = (a.vext[qa] / 64) * (a.vext[r - 1] / 64);
        for (int i = 0; i < r - 1; ++i)
          if (i != qa)
            tiles *= a.vext[i];
        ok = ok && tiles < (int64_t{1} << 22); // one block per tile
        if (ok && channels_ok(VO)) {
          family = kFamTranspose;
          dp->qa = qa;
          dp->ca = r - 1;
          // one-byte sources take tiles 128 q wide when q allows it (each
          // tile row then reads a whole 128-byte line); with two- and
          // four-byte results, 128 c wide too, kept in LDS as bytes, when c
          // allows it
          a.t_wq = win == 1 && a.vext[qa] % 128 == 0 ? 128 : 64;
          a.t_wc = a.t_wq == 128 && wout >= 2 && a.vext[r - 1] % 128 == 0 ? 128 : 64;
        }
      }
    }
    // ragged transpose: the same axes at any extents and alignments (checked
    // after the interleave, whose few channels would leave most of a tile
    // empty)
    auto ragged_transpose = [&] {
      if (any_pad || r < 2 || r - 2 > kBatchLevels || a.ss[r - 1] == 1)
        return false;
      int qa = -1;
      for (int i = 0; i < r - 1; ++i)
        if (a.ss[i] == 1 && a.vext[i] > 1)
          qa = i;
      if (qa < 0 || a.vext[qa] < 16 / win || a.vext[r - 1] < kRaggedMinC)
        return false;
      a.t_wq = a.t_wc = kRaggedTile; // boxes start at multiples (large tiles: any start)
      const int64_t plane_tiles = ceil_div(a.vext[qa], a.t_wq) * ceil_div(a.vext[r - 1], a.t_wc);
      int64_t tiles = plane_tiles;
      for (int i = 0; i < r - 1; ++i)
        if (i != qa)
          tiles *= a.vext[i];
      bool dequantizes = false;
      for (uint32_t i = k; i < nst; ++i)
        dequantizes = dequantizes || p.stages[i].op == kOpDequantize;
      if (tiles >= (int64_t{1} << 22) ||
          a.vext[qa] * a.vext[r - 1] < plane_tiles * (dequantizes ? kRaggedTileDequantized : kRaggedTileElements) ||
          !row_channels_ok())
        return false;
      dp->qa = qa;
      dp->ca = r - 1;
      return true;
    };
    // interleave: [batch..., P, C(pad)] planar source
    if (family == kFamGeneric && r >= 2 && r - 2 <= kBatchLevels && a.ss[r - 1] != 1 &&
        a.ss[r - 2] == 1 && a.ds[r - 2] == pext[static_cast<size_t>(r - 1)]) {
      const int64_t cp = pext[static_cast<size_t>(r - 1)];
      const int G = interleave_pixels(win, wout, static_cast<int>(cp));
      const int64_t bo = G * cp * wout;
      bool pa_pad = lo[static_cast<size_t>(r - 2)] != 0 || pext[static_cast<size_t>(r - 2)] != a.vext[r - 2];
      bool ok = (cp == 2 || cp == 4 || cp == 8) && !pa_pad && a.vext[r - 2] >= G &&
                (bo == 4 || bo == 8 || bo % 16 == 0);
      for (uint32_t i = k; i < nst; ++i)
        ok = ok && p.stages[i].mode == kChanNone;
      // whole groups at aligned planes, or any
      bool whole = a.vext[r - 2] % G == 0 && a.ss[r - 1] % G == 0;
      for (int i = 0; i < r - 2; ++i)
        whole = whole && a.ss[i] % G == 0;
      if (ok) {
        family = whole ? kFamInterleave : kFamRaggedInterleave;
        a.vec = G;
        a.cpad = static_cast<int32_t>(cp);
      }
    }
    if (family == kFamGeneric && ragged_transpose())
      family = kFamRaggedTranspose;
  }
  if (family == kFamGeneric)
    for (uint32_t i = k; i < nst; ++i)
      ch.st[i - k].vec = 0;
  dp->family = family;
  // the fast families prove every channel; so do element-wise stages per tensor
  // or along a dimension no longer than its table
  for (uint32_t i = k; i < nst && family == kFamGeneric; ++i) {
    const HostStage &h = p.stages[i];
    dp->reports = dp->reports || h.mode == kChanExpr ||
                  (h.mode == kChanDim && b.result_extents[static_cast<size_t>(h.dim)] > h.len);
  }
  a.chain_code = chain_code;
  static const char *names[] = {"generic", "stream", "transpose", "interleave", "permute",
                                "generic", "generic", "generic", "generic"};
  dp->kernel = names[family];

  // ------------------------------------------------------- chunk axis
  dp->chunk_axis = -1;
  dp->chunk_align = 1;
  {
    int ax = -1;
    for (int i = 0; i < r; ++i)
      if (a.vext[i] > 1 && (ax < 0 || a.ss[i] > a.ss[ax]))
        ax = i;
    if (ax >= 0) {
      int64_t rest = 0;
      for (int i = 0; i < r; ++i)
        if (i != ax)
          rest += (a.vext[i] - 1) * a.ss[i];
      if (a.ss[ax] * a.vext[ax] == wire_elems && rest < a.ss[ax]) {
        dp->chunk_axis = ax;
        dp->chunk_stride = a.ss[ax];
        if (row_family(family) && ax == r - 1)
          dp->chunk_align = V;
        else if (transpose_family(family) && (ax == dp->qa || ax == dp->ca))
          dp->chunk_align = ax == dp->qa ? a.t_wq : a.t_wc;
        else if (interleave_family(family) && ax == r - 2)
          dp->chunk_align = a.vec;
        // an interleave launch writes every channel of its pixels, so its
        // boxes never split the channel axis
        if (interleave_family(family) && ax == r - 1)
          dp->chunk_axis = -1;
        // a permute block takes T rows of m and all of c and e
        if (family == kFamPermute) {
          if (ax == r - 2)
            dp->chunk_align = a.p_t;
          else if (ax >= r - 3)
            dp->chunk_axis = -1;
        }
      }
    }
  }
  return dp;
}

namespace {

struct Box {
  int64_t lo[kMaxRank], ext[kMaxRank];
};

// Work items of a box for the program's family.
int64_t box_work(const DeviceProgram &dp, const Box &b) {
  const KArgs &a = dp.base;
  const int r = a.rank;
  int64_t n = 1;
  for (int i = 0; i < r; ++i) {
    int64_t e = b.ext[i];
    if (row_family(dp.family) && i == r - 1)
      e = dp.family == kFamRows ? ceil_div(e, a.vec) : e / a.vec;
    else if (transpose_family(dp.family) && (i == dp.qa || i == dp.ca))
      e = ceil_div(e, i == dp.qa ? a.t_wq : a.t_wc);
    else if (interleave_family(dp.family) && i == r - 2)
      e = ceil_div(e, a.vec);
    else if (interleave_family(dp.family) && i == r - 1)
      e = 1;
    else if (dp.family == kFamPermute && i == r - 2)
      e = ceil_div(e, a.p_t); // cut only where the direct kernel runs
    else if (dp.family == kFamPermute && i == r - 3)
      e /= a.p_g;
    else if (dp.family == kFamPermute && i > r - 3)
      e = 1;
    n *= e;
  }
  return n;
}

// Coordinates a split of axis i must keep together (0: never split).
int64_t split_align(const DeviceProgram &dp, int i) {
  const int r = dp.base.rank;
  if (row_family(dp.family) && i == r - 1)
    return dp.base.vec;
  if (transpose_family(dp.family) && (i == dp.qa || i == dp.ca))
    return i == dp.qa ? dp.base.t_wq : dp.base.t_wc;
  if (interleave_family(dp.family) && i == r - 2)
    return dp.base.vec;
  if (interleave_family(dp.family) && i == r - 1)
    return 0;
  if (dp.family == kFamPermute && i == r - 2)
    return dp.base.p_t;
  if (dp.family == kFamPermute && i > r - 4)
    return 0;
  return 1;
}

// Axes whose coordinates the decomposition levels carry (the others are the
// 2-D block of the transpose/interleave kernels).
bool level_axis(const DeviceProgram &dp, int i) {
  const int r = dp.base.rank;
  if (transpose_family(dp.family))
    return i != dp.qa && i != dp.ca;
  if (interleave_family(dp.family))
    return i < r - 2;
  if (dp.family == kFamPermute)
    return i < r - 3;
  return true;
}

// Largest element offset the levels of box b reach from its base, on the
// source and the destination side; contrib[i] the larger of axis i's two.
int64_t level_span(const DeviceProgram &dp, const Box &b, int64_t *contrib) {
  int64_t ss = 0, ds = 0;
  for (int i = 0; i < dp.base.rank; ++i) {
    contrib[i] = 0;
    if (!level_axis(dp, i) || b.ext[i] <= 1)
      continue;
    const int64_t s = (b.ext[i] - 1) * dp.base.ss[i], d = (b.ext[i] - 1) * dp.base.ds[i];
    ss += s;
    ds += d;
    contrib[i] = std::max(s, d);
  }
  return std::max(ss, ds);
}

// Split a fast-family box until it has fewer than 2^31 work items and level
// spans below 2^31 elements: halve (keeping alignment) the splittable axis
// with the largest span contribution, or the outermost one for work alone.
void split_box(const DeviceProgram &dp, const Box &b, std::vector<Box> &out) {
  if (dp.family == kFamGeneric) {
    out.push_back(b);
    return;
  }
  int64_t contrib[kMaxRank];
  const bool wide = level_span(dp, b, contrib) >= kMaxLaunchWork;
  if (!wide && box_work(dp, b) < kMaxLaunchWork) {
    out.push_back(b);
    return;
  }
  int axis = -1;
  for (int i = 0; i < dp.base.rank; ++i) {
    const int64_t al = split_align(dp, i);
    if (al == 0 || b.ext[i] <= al)
      continue;
    if (axis < 0 || (wide && contrib[i] > contrib[axis]))
      axis = i;
  }
  if (axis < 0)
    fail("unsupported_layout", "a launch box cannot be split below 2^31 elements");
  const int64_t al = split_align(dp, axis);
  const int64_t half = (b.ext[axis] / al + 1) / 2 * al; // extents are multiples of al
  Box c = b;
  c.ext[axis] = half;
  split_box(dp, c, out);
  c.lo[axis] = b.lo[axis] + half;
  c.ext[axis] = b.ext[axis] - half;
  split_box(dp, c, out);
}

Level trivial_level() {
  Level l{};
  l.div = make_div(1);
  l.vlo = 0;
  l.vcnt = 1;
  return l;
}

// Level of axis i counting units of `unit` coordinates (unit > 1 only on
// unpadded axes whose box start is a multiple of unit). The valid units of
// the box are [vlo, vlo + vcnt).
Level axis_level(const KArgs &a, const Box &b, int i, int64_t unit) {
  Level l{};
  const int64_t n = b.ext[i] / unit;
  l.div = make_div(n);
  const int64_t vmin = (a.lo[i] - b.lo[i]) / unit, vmax = vmin + a.vext[i] / unit;
  const int64_t lo = std::min(std::max<int64_t>(vmin, 0), n), hi = std::min(std::max<int64_t>(vmax, 0), n);
  l.vlo = static_cast<uint32_t>(lo);
  l.vcnt = static_cast<uint32_t>(hi - lo);
  if (n > 1) { // a single coordinate never moves the offset
    const int64_t ss = a.ss[i] * unit, ds = a.ds[i] * unit;
    if (ss >= kMaxLaunchWork || ds >= kMaxLaunchWork || n >= kMaxLaunchWork)
      fail("internal_launch_check", "a level stride exceeds 32 bits");
    l.ss = static_cast<uint32_t>(ss);
    l.ds = static_cast<uint32_t>(ds);
  }
  return l;
}

int64_t box_elements(const Box &b, int rank) {
  int64_t n = 1;
  for (int i = 0; i < rank; ++i)
    n *= b.ext[i];
  return n;
}

// The element-wise launch of box b, whose box_lo and box_ext are set: in 32
// bits where its elements, the offsets its axes reach and the result offsets
// its channels divide allow.
void element_args(const DeviceProgram &dp, const Box &b, KArgs &a) {
  const int r = a.rank;
  a.work64 = box_elements(b, r);
  a.work = 0;
  a.family = kFamGeneric;
  int64_t ss = 0, ds = 0;
  for (int i = 0; i < r; ++i) {
    ss += (b.ext[i] - 1) * a.ss[i];
    ds += (b.ext[i] - 1) * a.ds[i];
  }
  bool channels = true;
  for (int k = 0; k < a.chain.n; ++k)
    channels = channels && (a.chain.st[k].mode != kChanDim || dp.dst_elems < (int64_t{1} << 32));
  if (a.work64 >= kMaxLaunchWork || std::max(ss, ds) >= kMaxLaunchWork || !channels)
    return;
  a.family = kFamElement;
  a.work = static_cast<uint32_t>(a.work64);
  a.nlev = r <= 2 ? 2 : r <= 4 ? 4 : 8;
  a.sbase = a.dbase = 0;
  for (int i = 0; i < kMaxRank; ++i)
    a.lv[i] = trivial_level();
  for (int i = 0; i < r; ++i) {
    a.lv[a.nlev - r + i] = axis_level(a, b, i, 1);
    a.sbase += (b.lo[i] - a.lo[i]) * a.ss[i];
    a.dbase += b.lo[i] * a.ds[i];
  }
}

// Large aligned transpose boxes (kColdBytes) with cut tiles that keep their
// whole tiles on the tile kernel and run the strips past them as ragged
// launches:
// - a channel per element of rows that start off 64-byte boundaries: such rows
//   want large tiles, which such chains make slow (ragged_policy). int8 -> f16
//   [8208,8192] scaled along c 88.9 us, one ragged launch 144 (small tiles
//   101); f32 -> int8 78.9 and 91.6.
// - one-byte sources of four-byte results whose source rows lie multiples of 8
//   KiB apart: a ragged tile reads 64-byte halves of lines that fall on the
//   same sets, and the other halves are gone when the next tile wants them; the
//   tile kernel's rows are whole lines. int8 -> f32 [4112,8192] 34.7 us, one
//   ragged launch 50.6; [8208,8192] 59.7 and 65.8; rows 6 or 12 KiB apart 32.2
//   and 26.0, 52.9 and 51.2.
bool tiles_and_strips(const DeviceProgram &dp, const Box &b) {
  const KArgs &a = dp.base;
  if (box_elements(b, a.rank) * (a.win + a.wout) < kColdBytes)
    return false;
  if (a.win == 1 && a.wout == 4 && a.ss[dp.ca] % 8192 == 0)
    return true;
  bool aligned = true;
  for (int i = 0; i < a.rank; ++i)
    aligned = aligned && (i == dp.ca || b.ext[i] <= 1 || (a.ds[i] * a.wout) % 64 == 0);
  return !aligned && channel_per_element(a);
}

// Arguments of an edge box: the element-wise kernel over the box.
KArgs edge_args(const DeviceProgram &dp, const Box &b) {
  KArgs a = dp.base;
  for (int i = 0; i < a.rank; ++i) {
    a.box_lo[i] = b.lo[i];
    a.box_ext[i] = b.ext[i];
  }
  element_args(dp, b, a);
  return a;
}

bool pow2(int64_t x) { return x > 0 && (x & (x - 1)) == 0; }

// A byte-tile transpose launch indexes the parameters of its dequantize ->
// f16 chain by destination row (kTileRowChannel) when the stage has one
// channel per
// destination row of the box. For a result offset o = D + q * dsq + c of
// box row q < Q and column c < C (the box is one plane: no batch levels),
// chan_of(o) = (o / rs) mod re = D / dsq + q exactly when rs = dsq,
// (D mod dsq) + C <= dsq (the box's columns stay inside one row) and
// D / dsq + Q <= re (no wrap). t_choff = D / dsq.
bool row_channel(KArgs &a, const Box &b, int qa, int ca) {
  if (a.chain_code != kChainDeqF16 || a.wout != 2)
    return false;
  const DevStage &s = a.chain.st[0];
  const int64_t dsq = a.ds[qa];
  if (s.mode != kChanDim || s.vec != 0 || s.ch_rs != dsq || a.ds[ca] != 1 || dsq <= 0)
    return false;
  for (int j = 0; j < kBatchLevels; ++j)
    if (a.lv[j].div.d != 1)
      return false;
  if (a.dbase % dsq + b.ext[ca] > dsq || a.dbase / dsq + b.ext[qa] > s.ch_re)
    return false;
  a.t_choff = static_cast<uint32_t>(a.dbase / dsq);
  return true;
}

// The zero points of channels [c0, c0 + n) of a dequantize stage are all 0.
bool zero_points_zero(const DeviceProgram &dp, const DevStage &s, int64_t c0, int64_t n) {
  const int64_t lo = s.zp_off + (s.zp_per_ch ? c0 : 0), hi = lo + (s.zp_per_ch ? n : 1);
  if (lo < 0 || hi > static_cast<int64_t>(dp.pi.size()))
    return false;
  for (int64_t i = lo; i < hi; ++i)
    if (dp.pi[static_cast<size_t>(i)] != 0)
      return false;
  return true;
}

// A permute launch runs the direct body when its batch entries lie along one
// level (the outer levels are unit levels) and the parameter stage, if any,
// takes a vector's entry from the block's own c coordinate: with shifts when
// G*E, E and the 16-byte vectors of a run are powers of two (make_div then
// gives m = 1 and s = log2 d) and T divides the box's m, else with divisions
// and a last m-tile that may be cut. For a stage per channel along c
// (rs = M*E, re = C) at result offset o = D + c*M*E + m*E + e, with m < M,
// e < E and D the offset of the block's batch entry, (o / (M*E)) mod C = c
// exactly when D is a multiple of C*M*E: every batch level's destination
// stride is, and the launch origin is one plus an offset inside a plane
// (below M*E; a launch may start at any m). A per-tensor stage takes entry 0.
int permute_direct(KArgs &a, int64_t C, int64_t M, int64_t E) {
  a.p_cmask = 0;
  if (a.chain_code == kChainGeneric)
    return kPermuteGeneral;
  const int body = pow2(a.p_ge.d) && pow2(a.p_e.d) && pow2(a.p_run.d) && a.p_m % a.p_t == 0
                       ? kPermuteShift
                       : kPermuteDiv;
  const int k = chain_param_stage(a.chain_code);
  // Blocks of several vectors per lane without parameters, from four-byte
  // sources: the direct kernel saves no channel there, and the general one has
  // four vectors of a lane in flight for its two (f32 -> f16 [8,512,3,1024]
  // 13.6 us, direct 14.5; f32 [16,1024,5,128] 14.8 and 15.3, [8,1024,7,256]
  // 20.6 and 20.4; f16 [64,512,6,32] 6.4 and 5.5, int8 [8,1024,16,80] 6.4 and
  // 5.0).
  if (body == kPermuteDiv && a.win == 4 && k < 0 && a.p_m % a.p_t == 0 &&
      a.p_t * a.p_ge.d * 4 / 16 > 256)
    return kPermuteGeneral;
  // the direct kernel takes a batch entry's offsets from the innermost level
  for (int j = 0; j + 1 < kBatchLevels; ++j)
    if (a.lv[j].div.d != 1 || a.lv[j].vcnt != 1)
      return kPermuteGeneral;
  if (k < 0)
    return body;
  const DevStage &s = a.chain.st[k];
  if (s.vec != 0)
    return kPermuteGeneral;
  if (s.mode == kChanNone)
    return body;
  const int64_t plane = C * M * E;
  if (s.mode != kChanDim || s.ch_rs != M * E || s.ch_re != C || a.dbase % plane >= M * E)
    return kPermuteGeneral;
  for (int j = 0; j < kBatchLevels; ++j)
    if (a.lv[j].div.d > 1 && a.lv[j].ds % plane != 0)
      return kPermuteGeneral;
  a.p_cmask = ~0u;
  return body;
}

// Valid source columns [lo, hi) of a box along the innermost axis.
void valid_columns(const DeviceProgram &dp, const Box &b, int64_t &lo, int64_t &hi) {
  const KArgs &a = dp.base;
  const int i = a.rank - 1;
  lo = std::max<int64_t>(0, b.lo[i] - a.lo[i]);
  hi = std::min(a.vext[i], b.lo[i] + b.ext[i] - a.lo[i]);
}

// `family`: the program's own, or kFamRaggedTranspose for a box of a
// transpose program whose last tiles are cut.
KArgs launch_args(const DeviceProgram &dp, const Box &b, int family) {
  if (family == kFamGeneric)
    return edge_args(dp, b);
  KArgs a = dp.base;
  const int r = a.rank;
  for (int i = 0; i < r; ++i) {
    a.box_lo[i] = b.lo[i];
    a.box_ext[i] = b.ext[i];
  }
  // box origin: destination offset of its first padded coordinate, source
  // offset of the valid coordinate it corresponds to (interleave channels are
  // addressed by the kernel itself)
  a.sbase = 0;
  a.dbase = 0;
  for (int i = 0; i < r; ++i) {
    if (interleave_family(dp.family) && i == r - 1)
      continue;
    a.sbase += (b.lo[i] - a.lo[i]) * a.ss[i];
    a.dbase += b.lo[i] * a.ds[i];
  }
  for (int i = 0; i < kMaxRank; ++i)
    a.lv[i] = trivial_level();
  int64_t work = box_work(dp, b);
  a.family = family;
  // batch levels of the 2-D families: every axis but skip0/skip1, outer first
  auto batch = [&](int skip0, int skip1) {
    int idx[kMaxRank], n = 0;
    for (int i = 0; i < r; ++i)
      if (i != skip0 && i != skip1)
        idx[n++] = i;
    for (int j = 0; j < n; ++j)
      a.lv[kBatchLevels - n + j] = axis_level(a, b, idx[j], 1);
  };
  switch (family) {
  case kFamStream:
    for (int i = 0; i < r; ++i)
      a.lv[a.nlev - r + i] = axis_level(a, b, i, i == r - 1 ? a.vec : 1);
    break;
  case kFamFlat: // a.work whole vectors and the tail
    a.r_len = static_cast<uint32_t>(b.ext[0]);
    work = b.ext[0] / a.vec;
    break;
  case kFamRows: {
    for (int i = 0; i < r - 1; ++i)
      a.lv[a.nlev - r + i] = axis_level(a, b, i, 1);
    const int64_t n = ceil_div(b.ext[r - 1], a.vec);
    Level &l = a.lv[a.nlev - 1]; // items of the row
    l.div = make_div(n);
    l.ss = l.ds = static_cast<uint32_t>(a.vec);
    l.vlo = 0;
    l.vcnt = static_cast<uint32_t>(n);
    a.r_len = static_cast<uint32_t>(b.ext[r - 1]);
    a.r_off = static_cast<int32_t>(b.lo[r - 1] - a.lo[r - 1]);
    int64_t lo, hi;
    valid_columns(dp, b, lo, hi);
    a.r_lo = static_cast<int32_t>(lo);
    a.r_hi = static_cast<int32_t>(hi);
    // rows whose vectors are aligned stream their stores; others share a
    // vector's line with the next row
    bool aligned = (a.dbase * a.wout) % 16 == 0;
    for (int i = 0; i < r - 1; ++i)
      aligned = aligned && (a.ds[i] * a.wout) % 16 == 0;
    a.r_nts = aligned ? 1 : 0;
    break;
  }
  case kFamTranspose:
    batch(dp.qa, dp.ca);
    {
      // orders (measured on C3's int8 -> f16 transpose, 8 KiB result rows):
      // 128-wide tiles q fastest with each q-tile's c-tiles rotated, so the
      // blocks in flight write their rows at different column offsets
      // (30.0 -> 27.1 us); 64-wide one-byte tiles q fastest, grouped by XCD
      // so that the two halves of each source line meet in one L2; wider
      // elements in groups of kTileGroup q-tiles
      const int64_t nq = b.ext[dp.qa] / a.t_wq, nc = b.ext[dp.ca] / a.t_wc;
      const bool bytes = a.win == 1, wide = a.t_wq == 128;
      const int64_t g = bytes ? nq : std::min<int64_t>(kTileGroup, nq);
      const int64_t full = nq / g * g;
      a.t_plane = make_div(nq * nc);
      a.t_group = make_div(g * nc);
      a.t_g = make_div(g);
      a.t_tail = make_div(nq - full > 0 ? nq - full : 1);
      a.t_nc = make_div(nc);
      a.t_full = static_cast<uint32_t>(full);
      a.t_flags = (bytes && !wide ? kTileXcd : 0u) | (wide ? kTileSkew : 0u);
      if (keeps_source(a.win, a.wout) && box_elements(b, r) * a.win <= kKeepBytes)
        a.t_flags |= kTileKeep;
      a.t_choff = 0;
      if (a.t_wc == 128 && row_channel(a, b, dp.qa, dp.ca)) {
        a.t_flags |= kTileRowChannel;
        if (zero_points_zero(dp, a.chain.st[0], a.t_choff, b.ext[dp.qa]))
          a.t_flags |= kTileZeroPoint0;
      }
    }
    a.t_ssc = a.ss[dp.ca];
    a.t_dsq = a.ds[dp.qa];
    break;
  case kFamRaggedTranspose: {
    batch(dp.qa, dp.ca);
    a.t_ssc = a.ss[dp.ca];
    a.t_dsq = a.ds[dp.qa];
    ragged_policy(a, box_elements(b, r) * (a.win + a.wout), b.ext[dp.ca]);
    const int64_t nq = ceil_div(b.ext[dp.qa], a.t_wq), nc = ceil_div(b.ext[dp.ca], a.t_wc);
    work = box_elements(b, r) / (b.ext[dp.qa] * b.ext[dp.ca]) * nq * nc;
    const int64_t g = std::min<int64_t>(kTileGroup, nq), full = nq / g * g;
    a.t_plane = make_div(nq * nc);
    a.t_group = make_div(g * nc);
    a.t_g = make_div(g);
    a.t_tail = make_div(nq - full > 0 ? nq - full : 1);
    a.t_nc = make_div(nc);
    a.t_full = static_cast<uint32_t>(full);
    a.t_choff = 0;
    a.t_qn = static_cast<uint32_t>(b.ext[dp.qa]);
    a.t_cn = static_cast<uint32_t>(b.ext[dp.ca]);
    break;
  }
  case kFamPermute: {
    int idx[kMaxRank], n = 0;
    for (int i = 0; i < r - 3; ++i)
      idx[n++] = i;
    for (int j = 0; j < n; ++j)
      a.lv[kBatchLevels - n + j] = axis_level(a, b, idx[j], 1);
    const int64_t E = a.vext[r - 1], C = a.vext[r - 3], M = a.vext[r - 2], T = a.p_t;
    a.p_m = static_cast<uint32_t>(b.ext[r - 2]);
    a.p_tiles = make_div(ceil_div(b.ext[r - 2], T));
    a.p_cgt = make_div(work / (C / a.p_g));
    a.p_ce = make_div(C * E);
    a.p_ge = make_div(int64_t{a.p_g} * E);
    a.p_e = make_div(E);
    a.p_run = make_div(T * E * a.wout / 16);
    a.p_dsc = M * E;
    a.p_direct = permute_direct(a, C, M, E);
    if (a.p_direct == kPermuteGeneral && a.p_m % T)
      fail("internal_launch_check", "a cut m-tile outside the direct permute");
    break;
  }
  case kFamInterleave:
  case kFamRaggedInterleave:
    batch(r - 2, r - 1);
    a.r_len = static_cast<uint32_t>(b.ext[r - 2]);
    a.i_ng = make_div(ceil_div(b.ext[r - 2], a.vec));
    a.i_ssc = a.ss[r - 1];
    a.i_loc = static_cast<int32_t>(a.lo[r - 1]);
    a.i_vc = static_cast<int32_t>(a.vext[r - 1]);
    break;
  default:
    break;
  }
  a.work = static_cast<uint32_t>(work);
  a.work64 = family == kFamFlat ? b.ext[0] : work; // a flat box may be a tail alone
  return a;
}

} // namespace

// Launch arguments for valid coordinates [v0, v1) of the chunk axis (the
// whole box when the axis is -1). The first/last chunk also cover the axis'
// leading/trailing pad. One entry per launch.
std::vector<KArgs> box_launches(const DeviceProgram &dp, int64_t v0, int64_t v1, bool first,
                                bool last) {
  const KArgs &a = dp.base;
  if (dp.chunk_axis < 0)
    return axis_launches(dp, -1, 0, 0);
  const int ax = dp.chunk_axis;
  const int64_t plo = first ? 0 : v0 + a.lo[ax];
  const int64_t phi = last ? a.pext[ax] : v1 + a.lo[ax];
  return axis_launches(dp, ax, plo, phi);
}

int64_t axis_align(const DeviceProgram &dp, int i) { return split_align(dp, i); }

std::vector<KArgs> axis_launches(const DeviceProgram &dp, int axis, int64_t plo, int64_t phi) {
  return prefix_launches(dp, nullptr, axis, plo, phi);
}

std::vector<KArgs> prefix_launches(const DeviceProgram &dp, const int64_t *fixed, int axis,
                                   int64_t plo, int64_t phi, bool resident) {
  const KArgs &a = dp.base;
  Box b{};
  for (int i = 0; i < a.rank; ++i) {
    b.lo[i] = 0;
    b.ext[i] = a.pext[i];
  }
  if (axis >= 0) {
    for (int i = 0; fixed && i < axis; ++i) {
      b.lo[i] = fixed[i];
      b.ext[i] = 1;
    }
    b.lo[axis] = plo;
    b.ext[axis] = phi - plo;
  }
  std::vector<KArgs> out;
  std::vector<Box> edges;
  // A transpose box whose q or c extent is not a multiple of the tile runs
  // as one ragged launch; a transfer's small one, and those of
  // tiles_and_strips, keep their whole tiles on the tile kernel and run the strips past them (the q strip over the whole c
  // range, the c strip beside the whole q tiles) as ragged launches.
  int family = dp.family;
  if (family == kFamStream && a.rank == 1 && b.ext[0] % a.vec != 0)
    family = kFamFlat; // the tail past the last vector in the same launch
  if (family == kFamRows) { // a chunk of fewer valid columns than a vector
    int64_t lo, hi;
    valid_columns(dp, b, lo, hi);
    if (hi - lo < a.vec)
      return {edge_args(dp, b)};
  }
  // a chunk of fewer pixels than a group
  if (family == kFamRaggedInterleave && b.ext[a.rank - 2] < a.vec)
    return {edge_args(dp, b)};
  if (family == kFamTranspose && (b.ext[dp.qa] % a.t_wq || b.ext[dp.ca] % a.t_wc)) {
    if ((resident || box_elements(b, a.rank) >= kRaggedWholeElements) && !tiles_and_strips(dp, b)) {
      family = kFamRaggedTranspose;
    } else {
      const int q = dp.qa, c = dp.ca;
      const int64_t mq = b.ext[q] / a.t_wq * a.t_wq, mc = b.ext[c] / a.t_wc * a.t_wc;
      if (mq < b.ext[q]) {
        Box e = b;
        e.lo[q] = b.lo[q] + mq;
        e.ext[q] = b.ext[q] - mq;
        edges.push_back(e);
      }
      if (mc < b.ext[c] && mq > 0) {
        Box e = b;
        e.ext[q] = mq;
        e.lo[c] = b.lo[c] + mc;
        e.ext[c] = b.ext[c] - mc;
        edges.push_back(e);
      }
      b.ext[q] = mq;
      b.ext[c] = mc;
    }
  }
  std::vector<Box> boxes;
  if (box_elements(b, a.rank) > 0)
    split_box(dp, b, boxes);
  out.reserve(boxes.size() + edges.size());
  for (const Box &x : boxes)
    if (box_elements(x, a.rank) > 0)
      out.push_back(launch_args(dp, x, family));
  for (const Box &x : edges)
    if (box_elements(x, a.rank) > 0)
      out.push_back(launch_args(dp, x, kFamRaggedTranspose));
  return out;
}

namespace {

[[noreturn]] void bad_launch(const DeviceProgram &dp, const std::string &what) {
  fail("internal_launch_check", std::string(dp.kernel) + " launch: " + what);
}

template <int L>
bool decompose_n(const Level *lv, uint32_t i, int64_t &sof, int64_t &dof) {
  return decompose<L>(lv, i, sof, dof);
}

bool decompose_rt(int n, const Level *lv, uint32_t i, int64_t &sof, int64_t &dof) {
  switch (n) {
  case 1:
    return decompose_n<1>(lv, i, sof, dof);
  case 2:
    return decompose_n<2>(lv, i, sof, dof);
  case 3:
    return decompose_n<3>(lv, i, sof, dof);
  case 4:
    return decompose_n<4>(lv, i, sof, dof);
  default:
    return decompose_n<8>(lv, i, sof, dof);
  }
}

struct Checker {
  const DeviceProgram &dp;
  const KArgs &a;
  int64_t wire, dst; // elements
  size_t npf, npi;
  int64_t wire_lo; // first wire element the launch may read

  // n elements from `off`, accessed as one vector of n * width bytes when
  // `vec` (which must then be aligned to its size)
  void src_run(int64_t off, int64_t n, bool vec) const {
    if (off < wire_lo || off + n > wire)
      bad_launch(dp, "source run [" + std::to_string(off) + ", " + std::to_string(off + n) +
                         ") outside wire elements [" + std::to_string(wire_lo) + ", " +
                         std::to_string(wire) + ")");
    if (vec && (off * a.win) % (n * a.win) != 0)
      bad_launch(dp, "unaligned " + std::to_string(n * a.win) + "-byte source access at element " +
                         std::to_string(off));
  }
  void dst_run(int64_t off, int64_t n, bool vec) const {
    if (off < 0 || off + n > dst)
      bad_launch(dp, "destination run [" + std::to_string(off) + ", " + std::to_string(off + n) +
                         ") outside " + std::to_string(dst) + " result elements");
    if (vec && (off * a.wout) % (n * a.wout) != 0)
      bad_launch(dp, "unaligned " + std::to_string(n * a.wout) +
                         "-byte destination access at element " + std::to_string(off));
  }
  // The source element that the element-wise map gives dense result offset o
  // (-1: a pad): what a kernel of another family must read for it.
  int64_t source_of(int64_t o) const {
    int64_t s = 0;
    for (int k = 0; k < a.rank; ++k) {
      const int64_t v = (o / a.ds[k]) % a.pext[k] - a.lo[k];
      if (v < 0 || v >= a.vext[k])
        return -1;
      s += v * a.ss[k];
    }
    return s;
  }
  void same_source(int64_t o, int64_t s) const {
    if (source_of(o) != s)
      bad_launch(dp, "result element " + std::to_string(o) + " takes source element " +
                         std::to_string(s) + ", its map gives " + std::to_string(source_of(o)));
  }
  // channels of V consecutive result elements from dense offset o, as the
  // fast kernels index them (constant, or +1 per element)
  void channels(int64_t o, int V) const {
    for (int k = 0; k < a.chain.n; ++k) {
      const DevStage &s = a.chain.st[k];
      const uint32_t c = chan_of(s, o);
      const uint32_t last = chan_of(s, o + V - 1);
      const uint32_t want = s.vec ? c + static_cast<uint32_t>(V - 1) : c;
      if (last != want)
        bad_launch(dp, "channel pattern of stage " + std::to_string(k) + " breaks inside a vector");
      const bool reads_params = s.op == kOpQuantize || s.op == kOpDequantize;
      if (want >= s.len ||
          (reads_params && (s.scale_off + want >= npf ||
                            s.zp_off + (s.zp_per_ch ? want : 0u) >= npi)))
        bad_launch(dp, "parameter index outside its table at stage " + std::to_string(k));
    }
  }
};

} // namespace

void verify_launch(const DeviceProgram &dp_in, const KArgs &a, int64_t wire_lo, int64_t wire_hi) {
  DeviceProgram edge;
  if (a.family != dp_in.family) { // a launch of another family than the program's
    edge = dp_in;
    edge.family = a.family;
  }
  const DeviceProgram &dp = a.family != dp_in.family ? edge : dp_in;
  const Checker ck{dp,          a,           wire_hi < 0 ? dp.wire_elems : wire_hi,
                   dp.dst_elems, dp.pf.size(), dp.pi.size(),
                   wire_lo};
  if (dp.family != kFamGeneric) { // the levels' 32-bit offsets cannot wrap
    int64_t ss = 0, ds = 0;
    for (const Level &l : a.lv) {
      ss += (int64_t{l.div.d} - 1) * l.ss;
      ds += (int64_t{l.div.d} - 1) * l.ds;
      if (int64_t{l.vlo} + l.vcnt > l.div.d)
        bad_launch(dp, "a level's valid range leaves its extent");
    }
    if (ss >= kMaxLaunchWork || ds >= kMaxLaunchWork)
      bad_launch(dp, "level offsets exceed 31 bits");
  }
  const int win = a.win, wout = a.wout;
  switch (dp.family) {
  case kFamStream: {
    if (a.work64 >= kMaxLaunchWork || a.work != a.work64)
      bad_launch(dp, "work above 2^31");
    const int V = a.vec;
    for (uint32_t i = 0; i < a.work; ++i) {
      int64_t sof = a.sbase, dof = a.dbase;
      const bool pad = decompose_rt(a.nlev, a.lv, i, sof, dof);
      ck.dst_run(dof, V, true);
      if (!pad) {
        ck.src_run(sof, V, true);
        ck.channels(dof, V);
      }
    }
    break;
  }
  case kFamTranspose: {
    if (a.work64 > (int64_t{1} << 22) || a.work != a.work64)
      bad_launch(dp, "more tiles than one launch takes");
    const int VO = 16 / wout;
    const int64_t TQ = a.t_wq, TC = a.t_wc;
    if (!(TQ == 64 || (TQ == 128 && win == 1)) || !(TC == 64 || (TC == 128 && TQ == 128)) ||
        a.t_nc.d != a.t_group.d / a.t_g.d || (a.t_flags & ~(kTileXcd | kTileSkew | kTileRowChannel | kTileZeroPoint0 | kTileKeep)) ||
        ((a.t_flags & kTileKeep) && !keeps_source(win, wout)) ||
        ((a.t_flags & kTileSkew) && (a.t_flags & kTileXcd)) || (TC == 128 && (a.t_flags & kTileXcd)) ||
        ((a.t_flags & kTileRowChannel) && TC != 128))
      bad_launch(dp, "tile geometry disagrees with the kernel");
    std::vector<bool> seen(a.work, false); // the order must be a bijection
    for (uint32_t blk = 0; blk < a.work; ++blk) { // grid = one block per tile
      const uint32_t t = (a.t_flags & kTileXcd) ? xcd_tile(blk, a.work) : blk;
      if (t >= a.work)
        bad_launch(dp, "a block maps past the last tile");
      uint32_t tq, tc, r2;
      tile_of(a, t, tq, tc, r2);
      const uint32_t nc = a.t_group.d / a.t_g.d, nq = a.t_plane.d / nc;
      if (tq >= nq || tc >= nc)
        bad_launch(dp, "tile coordinates outside the plane");
      const size_t id = (static_cast<size_t>(r2) * nq + tq) * nc + tc;
      if (id >= seen.size() || seen[id])
        bad_launch(dp, "the tile order visits a tile twice");
      seen[id] = true;
      int64_t sbase = a.sbase, dbase = a.dbase;
      if (decompose_rt(kBatchLevels, a.lv, r2, sbase, dbase))
        bad_launch(dp, "a transpose tile reaches a pad");
      const int64_t q0 = int64_t{tq} * TQ, c0 = int64_t{tc} * TC;
      // a tile row moves as 16-byte vectors: TC source rows of TQ elements,
      // TQ destination rows of TC
      for (int64_t row = 0; row < TC; row += TC - 1) {
        const int64_t so = sbase + (c0 + row) * a.t_ssc + q0;
        ck.src_run(so, TQ, false);
        if ((so * win) % 16 != 0)
          bad_launch(dp, "a tile row is not 16-byte aligned");
      }
      for (int64_t row = 0; row < TQ; row += TQ - 1) {
        const int64_t d = dbase + (q0 + row) * a.t_dsq + c0;
        ck.dst_run(d, TC, false);
        if ((d * wout) % 16 != 0)
          bad_launch(dp, "a tile row is not 16-byte aligned");
      }
      if ((a.t_ssc * win) % 16 != 0 || (a.t_dsq * wout) % 16 != 0)
        bad_launch(dp, "row strides break 16-byte alignment");
      const bool rowch = (a.t_flags & kTileRowChannel) != 0;
      if (rowch && (r2 != 0 || a.chain_code != kChainDeqF16 || a.chain.st[0].vec != 0))
        bad_launch(dp, "row-indexed parameters with a chain or batch they do not fit");
      if ((a.t_flags & kTileZeroPoint0) &&
          (!rowch || !zero_points_zero(dp, a.chain.st[0], a.t_choff, int64_t{a.t_plane.d} /
                                                                       a.t_nc.d * TQ)))
        bad_launch(dp, "a launch that leaves zero points out reads one that is not 0");
      for (int64_t row = 0; row < TQ; ++row)
        for (int64_t cv = 0; cv < TC; cv += VO) {
          const int64_t o = dbase + (q0 + row) * a.t_dsq + c0 + cv;
          ck.channels(o, VO);
          if (rowch && chan_of(a.chain.st[0], o) != a.t_choff + static_cast<uint32_t>(q0 + row))
            bad_launch(dp, "a row-indexed launch reads another parameter entry");
        }
    }
    break;
  }
  case kFamFlat: {
    const int V = a.vec;
    if (a.work64 >= kMaxLaunchWork || a.r_len != a.work64 || a.r_len / V != a.work)
      bad_launch(dp, "work disagrees with the elements");
    for (uint32_t i = 0; i <= a.work; ++i) { // the last one: the tail, element by element
      const int n = i < a.work ? V : static_cast<int>(a.r_len % V);
      if (n == 0)
        break;
      const int64_t s0 = a.sbase + int64_t{i} * V, d0 = a.dbase + int64_t{i} * V;
      ck.src_run(s0, n, n == V);
      ck.dst_run(d0, n, n == V);
      ck.same_source(d0, s0);
      ck.same_source(d0 + n - 1, s0 + n - 1);
      for (int k = 0; k < a.chain.n; ++k) { // the entries k_flat takes
        const DevStage &s = a.chain.st[k];
        const uint32_t o = static_cast<uint32_t>(d0), c0 = chan_of(s, o), re = s.ch_re_div.d;
        const uint32_t left = s.ch_rs_div.d - o % s.ch_rs_div.d;
        for (int e = 0; e < n; ++e) {
          uint32_t c = c0;
          if (s.vec & 1)
            c = c0 + e >= re ? c0 + e - re : c0 + e;
          else if (s.vec != 0 && static_cast<uint32_t>(e) >= left)
            c = c0 + 1 == re ? 0 : c0 + 1;
          if (c != chan_of(s, d0 + e) || c >= s.len)
            bad_launch(dp, "a flat launch reads another parameter entry");
        }
      }
    }
    break;
  }
  case kFamRows: {
    if (a.work64 >= kMaxLaunchWork || a.work != a.work64)
      bad_launch(dp, "work above 2^31");
    const int V = a.vec;
    const FastDiv &row_div = a.lv[a.nlev - 1].div;
    if (a.r_hi - a.r_lo < V || ceil_div(a.r_len, V) != row_div.d)
      bad_launch(dp, "columns disagree with the row's items");
    for (uint32_t i = 0; i < a.work; ++i) { // the kernel's arithmetic
      int64_t sof = a.sbase, dof = a.dbase;
      bool pad = decompose_rt(a.nlev, a.lv, i, sof, dof);
      const int32_t p = static_cast<int32_t>(i - fdiv(i, row_div) * row_div.d) * V;
      const int32_t col = p + a.r_off, at = std::min(std::max(col, a.r_lo), a.r_hi - V);
      pad |= col >= a.r_hi || col + V <= a.r_lo;
      const int n = std::min<int>(V, static_cast<int>(a.r_len) - p);
      ck.dst_run(dof, n, a.r_nts && n == V);
      for (int e = 0; e < n; ++e)
        ck.same_source(dof + e, pad || col + e < a.r_lo || col + e >= a.r_hi ? -1 : sof + e);
      if (!pad) {
        if (std::abs(at - col) >= V)
          bad_launch(dp, "a vector moves by its whole width");
        ck.src_run(sof + (at - col), V, false);
        ck.channels(dof, n);
      }
    }
    break;
  }
  case kFamRaggedTranspose: {
    if (a.work64 > (int64_t{1} << 22) || a.work != a.work64)
      bad_launch(dp, "more tiles than one launch takes");
    const int VO = 16 / wout;
    const int64_t TQ = a.t_wq, TC = a.t_wc, Q = a.t_qn, C = a.t_cn;
    const int64_t nq = ceil_div(Q, TQ), nc = ceil_div(C, TC);
    const bool large = TC == kRaggedLargeC;
    if (TQ != (large ? ragged_large_q(win) : kRaggedTile) || !(large || TC == kRaggedTile) || Q < 1 ||
        C < 1 || (a.t_flags & ~(kTileXcd | kTileNtLoad | kTileNtStore)) ||
        (large && (a.t_flags & kTileNtStore)) || a.t_nc.d != nc || int64_t{a.t_plane.d} != nq * nc)
      bad_launch(dp, "tile geometry disagrees with the kernel");
    std::vector<bool> seen(a.work, false); // the order must be a bijection
    for (uint32_t blk = 0; blk < a.work; ++blk) {
      const uint32_t t = (a.t_flags & kTileXcd) ? xcd_tile(blk, a.work) : blk;
      if (t >= a.work)
        bad_launch(dp, "a block maps past the last tile");
      uint32_t tq, tc, r2;
      tile_of(a, t, tq, tc, r2);
      if (tq >= nq || tc >= nc)
        bad_launch(dp, "tile coordinates outside the plane");
      const size_t id = (static_cast<size_t>(r2) * nq + tq) * nc + tc;
      if (id >= seen.size() || seen[id])
        bad_launch(dp, "the tile order visits a tile twice");
      seen[id] = true;
      int64_t sbase = a.sbase, dbase = a.dbase;
      if (decompose_rt(kBatchLevels, a.lv, r2, sbase, dbase))
        bad_launch(dp, "a transpose tile reaches a pad");
      const int64_t q0 = tq * TQ, c0 = tc * TC;
      const int64_t qn = std::min(TQ, Q - q0), cn = std::min(TC, C - c0);
      // rows of qn elements; the last vector of a cut row ends with the row
      // and may start before the tile, inside the same source row (strides
      // are not negative: the first and last row reach the furthest)
      const int64_t before = std::max<int64_t>(0, 16 / win - qn);
      if (a.box_lo[dp.qa] + q0 < before)
        bad_launch(dp, "a cut vector starts before its row");
      for (int64_t row : {int64_t{0}, cn - 1})
        ck.src_run(sbase + (c0 + row) * a.t_ssc + q0 - before, qn + before, false);
      for (int64_t row = 0; row < qn; ++row) {
        const int64_t d = dbase + (q0 + row) * a.t_dsq + c0;
        ck.dst_run(d, cn, false);
        for (int64_t c : {int64_t{0}, cn - 1})
          ck.same_source(d + c, sbase + (c0 + c) * a.t_ssc + q0 + row);
        for (int64_t cv = 0; cv < cn; cv += VO)
          ck.channels(d + cv, static_cast<int>(std::min<int64_t>(VO, cn - cv)));
      }
    }
    break;
  }
  case kFamRaggedInterleave:
  case kFamInterleave: {
    if (a.work64 >= kMaxLaunchWork || a.work != a.work64)
      bad_launch(dp, "work above 2^31");
    const bool rag = dp.family == kFamRaggedInterleave;
    const int G = a.vec, CP = a.cpad;
    for (int k = 0; k < a.chain.n; ++k)
      if (a.chain.st[k].mode != kChanNone)
        bad_launch(dp, "per-channel stage in an interleave program");
    if (a.r_len < static_cast<uint32_t>(G) || a.i_ng.d != ceil_div(a.r_len, G))
      bad_launch(dp, "pixel groups disagree with the box");
    if (!rag && (a.i_ssc * win) % (G * win) != 0)
      bad_launch(dp, "plane stride breaks the alignment of plane loads");
    if (G != interleave_pixels(win, wout, CP))
      bad_launch(dp, "pixels per item disagree with the kernel");
    for (uint32_t i = 0; i < a.work; ++i) {
      const uint32_t rest = fdiv(i, a.i_ng);
      const uint32_t g = i - rest * a.i_ng.d;
      int64_t sbase = a.sbase, dbase = a.dbase;
      const bool pad = decompose_rt(kBatchLevels, a.lv, rest, sbase, dbase);
      const int64_t p0 = int64_t{g} * G, back = std::max<int64_t>(0, p0 + G - a.r_len);
      if (back && !rag)
        bad_launch(dp, "a cut pixel group");
      ck.dst_run(dbase + p0 * CP, (G - back) * CP, !rag);
      for (int c = 0; c < CP; ++c) {
        const int32_t vc = c - a.i_loc;
        if (!pad && static_cast<uint32_t>(vc) < static_cast<uint32_t>(a.i_vc))
          ck.src_run(sbase + vc * a.i_ssc + p0 - back, G, !rag);
        for (int64_t j : {int64_t{0}, G - back - 1})
          ck.same_source(dbase + (p0 + j) * CP + c,
                         pad || static_cast<uint32_t>(vc) >= static_cast<uint32_t>(a.i_vc)
                             ? -1
                             : sbase + vc * a.i_ssc + p0 + j);
      }
    }
    break;
  }
  case kFamPermute: {
    if (a.work64 > (int64_t{1} << 22) || a.work != a.work64)
      bad_launch(dp, "more blocks than one launch takes");
    const int64_t CE = a.p_ce.d, E = a.p_e.d, T = a.p_t, C = CE / E, G = a.p_g, GE = a.p_ge.d;
    const int VI = 16 / win;
    if (G < 1 || C % G != 0 || GE != G * E || a.p_lds != T * GE * wout || a.p_lds > 32768 ||
        int64_t{a.p_run.d} * 16 != T * E * wout || a.vec != VI || GE % VI != 0 ||
        (E * wout) % 16 != 0 || int64_t{a.p_cgt.d} * (C / G) != a.work64)
      bad_launch(dp, "block geometry disagrees with the kernel");
    // a direct launch replaces each division by a shift and mask, and each
    // vector's parameter entry by c & p_cmask
    const int pk = chain_param_stage(a.chain_code);
    const int64_t M = a.p_m;
    if (int64_t{a.p_tiles.d} != ceil_div(M, T) || (M % T && a.p_direct != kPermuteDiv))
      bad_launch(dp, "m-tiles disagree with the box");
    if (a.p_direct == kPermuteShift)
      for (const FastDiv *f : {&a.p_ge, &a.p_e, &a.p_run})
        if (!pow2(f->d) || f->m != 1 || (uint64_t{1} << f->s) != f->d)
          bad_launch(dp, "a direct permute divides by a number that is not a power of two");
    if (a.p_direct) {
      if (a.chain_code == kChainGeneric || (pk >= 0 && a.chain.st[pk].vec != 0) ||
          (a.p_cmask != 0 && a.p_cmask != ~0u))
        bad_launch(dp, "a direct permute with a chain it cannot run");
      for (int j = 0; j + 1 < kBatchLevels; ++j)
        if (a.lv[j].div.d != 1 || a.lv[j].vcnt != 1 || a.lv[j].ss != 0 || a.lv[j].ds != 0)
          bad_launch(dp, "a direct permute over more than one batch level");
      if (a.lv[kBatchLevels - 1].div.d > 1 &&
          (int64_t{a.lv[kBatchLevels - 1].ss} * (a.lv[kBatchLevels - 1].div.d - 1) >= kMaxLaunchWork ||
           int64_t{a.lv[kBatchLevels - 1].ds} * (a.lv[kBatchLevels - 1].div.d - 1) >= kMaxLaunchWork))
        bad_launch(dp, "a direct permute's batch offsets leave 32 bits");
    }
    for (uint32_t t = 0; t < a.work; ++t) {
      // the kernel's own decomposition: group, then batch entry and m-tile
      const uint32_t cg = fdiv(t, a.p_cgt);
      const uint32_t t2 = t - cg * a.p_cgt.d;
      const uint32_t batch = fdiv(t2, a.p_tiles);
      const int64_t m0 = int64_t{t2 - batch * a.p_tiles.d} * T;
      int64_t sbase = a.sbase, dbase = a.dbase;
      if (decompose_rt(kBatchLevels, a.lv, batch, sbase, dbase))
        bad_launch(dp, "a permute block reaches a pad");
      const int64_t rows = std::min(T, M - m0);
      for (int64_t tt = 0; tt < rows; ++tt) {
        const int64_t so = sbase + (m0 + tt) * CE + int64_t{cg} * GE;
        ck.src_run(so, GE, false);
        if ((so * win) % 16 != 0)
          bad_launch(dp, "unaligned source rows");
      }
      for (int64_t cl = 0; cl < G; ++cl) {
        const int64_t c = int64_t{cg} * G + cl;
        ck.dst_run(dbase + c * a.p_dsc + m0 * E, rows * E, false);
        if (((dbase + c * a.p_dsc + m0 * E) * wout) % 16 != 0)
          bad_launch(dp, "unaligned destination runs");
        for (int64_t tt = 0; tt < rows; ++tt)
          for (int64_t e = 0; e < E; e += VI) {
            const int64_t o = dbase + c * a.p_dsc + (m0 + tt) * E + e;
            ck.same_source(o, sbase + (m0 + tt) * CE + c * E + e);
            ck.channels(o, VI);
            if (a.p_direct && pk >= 0 &&
                chan_of(a.chain.st[pk], o) != (static_cast<uint32_t>(c) & a.p_cmask))
              bad_launch(dp, "a direct permute reads another parameter entry");
          }
      }
    }
    break;
  }
  default: {
    const bool element = dp.family == kFamElement;
    if (element && (a.work64 >= kMaxLaunchWork || a.work != a.work64))
      bad_launch(dp, "work above 2^31");
    for (int64_t i = 0; i < a.work64; ++i) {
      int64_t rem = i, dof = 0, sof = 0;
      bool pad = false;
      for (int k = a.rank - 1; k >= 0; --k) {
        const int64_t p = rem % a.box_ext[k] + a.box_lo[k];
        rem /= a.box_ext[k];
        dof += p * a.ds[k];
        const int64_t v = p - a.lo[k];
        if (v < 0 || v >= a.vext[k])
          pad = true;
        else
          sof += v * a.ss[k];
      }
      ck.dst_run(dof, 1, false);
      if (!pad)
        ck.src_run(sof, 1, false);
      if (element) { // the kernel's own arithmetic gives the same element
        int64_t s32 = a.sbase, d32 = a.dbase;
        const bool p32 = decompose_rt(a.nlev, a.lv, static_cast<uint32_t>(i), s32, d32);
        if (p32 != pad || d32 != dof || (!pad && s32 != sof))
          bad_launch(dp, "the levels disagree with the box");
        for (int k = 0; k < a.chain.n; ++k) {
          const DevStage &s = a.chain.st[k];
          if (s.mode == kChanDim && chan_of(s, dof) != (dof / s.ch_rs) % s.ch_re)
            bad_launch(dp, "a 32-bit channel disagrees with its map");
        }
      }
    }
  }
  }
}

namespace {

bool verify_enabled() {
  static const bool on = [] {
    const char *v = std::getenv("RELX_VERIFY_LAUNCHES");
    return v && *v && std::strcmp(v, "0") != 0;
  }();
  return on;
}

} // namespace

int64_t launch_program(const DeviceProgram &dp, int64_t v0, int64_t v1, bool first, bool last,
                       const void *src, void *dst, const float *pf, const int32_t *pi,
                       int32_t *status, hipStream_t s) {
  const bool part = dp.chunk_axis >= 0 && v1 > v0; // else the whole box
  return launch_all(dp, box_launches(dp, v0, v1, first, last), src, dst, pf, pi, status, s,
                    part ? v0 * dp.chunk_stride : 0, part ? v1 * dp.chunk_stride : -1);
}

std::string launch_kernel(const KArgs &a) {
  switch (a.family) {
  case kFamStream:
    return "stream";
  case kFamFlat:
    return "flat";
  case kFamRows:
    return "rows";
  case kFamTranspose:
    return (a.t_flags & kTileKeep) ? "transpose_keep" : "transpose";
  case kFamRaggedTranspose:
    return a.t_wc == kRaggedLargeC ? "ragged_transpose_large" : "ragged_transpose";
  case kFamInterleave:
    return "interleave";
  case kFamRaggedInterleave:
    return "ragged_interleave";
  case kFamPermute:
    return std::string(a.p_direct == kPermuteShift ? "permute_shift "
                       : a.p_direct == kPermuteDiv ? "permute_div "
                                                   : "permute ") +
           std::to_string(a.p_g) + "x" + std::to_string(a.p_t);
  case kFamElement:
    return "element";
  default:
    return "generic";
  }
}

int64_t launch_all(const DeviceProgram &dp, const std::vector<KArgs> &launches, const void *src,
                   void *dst, const float *pf, const int32_t *pi, int32_t *status, hipStream_t s,
                   int64_t wire_lo, int64_t wire_hi) {
  // these families move aligned 16-byte vectors: with buffers that are not
  // 16-byte aligned their boxes run element-wise (the ragged ones and the rows
  // take any alignment)
  const bool aligned = reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(dst) % 16 == 0;
  int64_t n = 0;
  for (const KArgs &laid : launches) {
    KArgs a = laid;
    if (!aligned && (a.family == kFamStream || a.family == kFamFlat || a.family == kFamTranspose ||
                     a.family == kFamInterleave || a.family == kFamPermute)) {
      Box b{};
      std::copy(a.box_lo, a.box_lo + a.rank, b.lo);
      std::copy(a.box_ext, a.box_ext + a.rank, b.ext);
      element_args(dp, b, a);
    }
    if (verify_enabled())
      verify_launch(dp, a, wire_lo, wire_hi);
    a.src = static_cast<const uint8_t *>(src);
    a.dst = static_cast<uint8_t *>(dst);
    a.pf = pf;
    a.pi = pi;
    const hipError_t e = launch_box(a.family, a, status, s);
    if (e != hipSuccess)
      fail("backend_failure", std::string("kernel launch: ") + hipGetErrorString(e));
    ++n;
  }
  return n;
}

} // namespace relx
