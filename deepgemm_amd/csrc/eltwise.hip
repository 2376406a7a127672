// eltwise.hip -- the HBM-bound stages around the GEMMs (gfx950):
//   * the top-k combine as an inverse-index gather (no atomics, fixed slot order):
//     y[t] = bf16(sum_s f32(part[output_index[t,s]])), the reference's reduce
//     (deep_gemm/include/deep_gemm/impls/mega_moe_dcu.cuh:706-760) and baseline gather
//     (csrc/kernels/mega_moe_baseline_hip.cu:98-127);
//   * row gather for the DeepEP-style preprocess, channelwise FP8 cast, Marlin pack.
#include "common.cuh"
#include "kernels.h"
#include "launch.h"

namespace mmoe {

namespace {

constexpr int kEltThreads = 256;
constexpr int kEltWaves = kEltThreads / kWave;

// ---------------------------------------------------------------- requant
// One wave per row: amax = max |y|; a = max(amax, 1e-4); act = e4m3(clip(y * (448/a)));
// act_scale = a/448 (the K2 requant, megamoe/dcu_megamoe_large_opt/K2_fused/
// k2_fused_ext.cu:341-364). A row of up to kRequantGroups*4*64 channels stays in registers
// between the reduction and the quantization; a longer one is read twice. y is GEMM1's SwiGLU
// x route weight output in bf16 (k2_fused_ext.cu:283-340, computed in GEMM1's epilogue and
// rounded as the reference's fused path rounds its activation, mega_moe_dcu_tiles.cuh:530-550).
constexpr int kRequantGroups = 8;  // float4 groups per lane held in registers

struct RequantArgs {
  const uint16_t* src;  // bf16 y [rows, I]
  float* amax;
  int32_t* meta;
  uint8_t* act;
  float* act_scale;
  int inter;
  RowDest dest;
  const int32_t* dual_rows;  // dual launches: the WIDE GEMM1 ran iff *dual_rows >= dual_min_rows
  int dual_min_rows;
};

// Nontemporal accesses for the streams these kernels touch once: y and the partial rows are
// read once, act is written once and read by GEMM2 from HBM anyway at prefill sizes. At c3 the
// requant went from 405 to 379 us and the combine from 427 to 410 us (same box, alternating
// builds); nontemporal stores of the combine's y rows were slower (436 us), so those stay plain.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld_nt(const float4* p) {
  const f32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint2 ld_nt(const uint2* p) {
  const u32x2_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p));
  return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ uint4 ld_nt(const uint4* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// channels 4q .. 4q+3 of row `row`
__device__ __forceinline__ float4 requant_load(const RequantArgs& r, int64_t row, int q) {
  const uint2 b = ld_nt(reinterpret_cast<const uint2*>(r.src + row * r.inter) + q);
  return make_float4(bf16_to_f32(b.x & 0xffff), bf16_to_f32(b.x >> 16), bf16_to_f32(b.y & 0xffff),
                     bf16_to_f32(b.y >> 16));
}

// wide: the WIDE GEMM1 ran (meta[1]); direct: build the direct-write table
__device__ __forceinline__ void requant_rows(const RequantArgs& r, bool wide, bool direct) {
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  const int rows = r.meta[0];
  const int groups = r.inter >> 2;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    r.meta[1] = wide ? 1 : 0;
    if (r.dest.meta_flag != nullptr) *r.dest.meta_flag = direct ? 1 : 0;
  }
  for (int row = blockIdx.x * kEltWaves + wave; row < rows; row += gridDim.x * kEltWaves) {
    const int tok = direct ? r.dest.row_token[row] : 0;
    uint32_t* ar = reinterpret_cast<uint32_t*>(r.act + static_cast<int64_t>(row) * r.inter);
    float m = 0.0f;
    if ((r.inter & 7) == 0 && r.inter <= 8 * (kRequantGroups / 2) * kWave) {
      // 8 channels (16 bytes) a load, their 8 codes one 8-byte store
      const int octs = r.inter >> 3;
      const uint4* src = reinterpret_cast<const uint4*>(r.src + static_cast<int64_t>(row) * r.inter);
      float4 v[kRequantGroups];
#pragma unroll
      for (int j = 0; j < kRequantGroups / 2; ++j) {
        const int o = lane + j * kWave;
        const uint4 b = o < octs ? ld_nt(src + o) : make_uint4(0, 0, 0, 0);
        v[2 * j] = make_float4(bf16_to_f32(b.x & 0xffff), bf16_to_f32(b.x >> 16), bf16_to_f32(b.y & 0xffff),
                               bf16_to_f32(b.y >> 16));
        v[2 * j + 1] = make_float4(bf16_to_f32(b.z & 0xffff), bf16_to_f32(b.z >> 16), bf16_to_f32(b.w & 0xffff),
                                   bf16_to_f32(b.w >> 16));
        m = abs_max4(abs_max4(m, v[2 * j]), v[2 * j + 1]);
      }
      m = wave_max(m);
      const float inv = kE4m3Max / fmaxf(m, kAmaxFloor);
      u32x2_t* dst = reinterpret_cast<u32x2_t*>(r.act + static_cast<int64_t>(row) * r.inter);
#pragma unroll
      for (int j = 0; j < kRequantGroups / 2; ++j) {
        const int o = lane + j * kWave;
        const float4 a = v[2 * j], c = v[2 * j + 1];
        const u32x2_t codes = {pack_e4m3x4(a.x * inv, a.y * inv, a.z * inv, a.w * inv),
                               pack_e4m3x4(c.x * inv, c.y * inv, c.z * inv, c.w * inv)};
        if (o < octs) __builtin_nontemporal_store(codes, dst + o);
      }
    } else if (groups <= kRequantGroups * kWave) {
      float4 v[kRequantGroups];
#pragma unroll
      for (int i = 0; i < kRequantGroups; ++i) {
        const int q = lane + i * kWave;
        v[i] = q < groups ? requant_load(r, row, q) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        m = abs_max4(m, v[i]);
      }
      m = wave_max(m);
      const float inv = kE4m3Max / fmaxf(m, kAmaxFloor);
#pragma unroll
      for (int i = 0; i < kRequantGroups; ++i) {
        const int q = lane + i * kWave;
        if (q < groups) __builtin_nontemporal_store(pack_e4m3x4(v[i].x * inv, v[i].y * inv, v[i].z * inv, v[i].w * inv), ar + q);
      }
    } else {
      for (int q = lane; q < groups; q += kWave) m = abs_max4(m, requant_load(r, row, q));
      m = wave_max(m);
      const float inv = kE4m3Max / fmaxf(m, kAmaxFloor);
      for (int q = lane; q < groups; q += kWave) {
        const float4 v = requant_load(r, row, q);
        __builtin_nontemporal_store(pack_e4m3x4(v.x * inv, v.y * inv, v.z * inv, v.w * inv), ar + q);
      }
    }
    if (direct) {
      // the row's token has exactly one routed slot: GEMM2 writes its output row straight to y
      const int slot_row = lane < r.dest.topk
          ? r.dest.output_index[static_cast<int64_t>(tok) * r.dest.topk + lane] : -1;
      const int routed = __popcll(__ballot(slot_row >= 0));
      if (lane == 0) r.dest.row_dest[row] = routed == 1 ? tok : -1;
    }
    if (lane == 0) {
      r.amax[row] = m;
      r.act_scale[row] = fmaxf(m, kAmaxFloor) / kE4m3Max;
    }
  }
}

// kMode 0: after the 8-wave GEMM1, 1: after the WIDE GEMM1, 2: decided on the device (a dual
// GEMM1 launch; RequantArgs)
template <int kMode>
__global__ __launch_bounds__(kEltThreads) void requant_kernel(RequantArgs r) {
  // (after a dual launch the direct rows go with the WIDE GEMMs only)
  const bool wide = kMode == 1 || (kMode == 2 && *r.dual_rows >= r.dual_min_rows);
  const bool direct = r.dest.row_dest != nullptr && (kMode != 2 || wide);
  requant_rows(r, wide, direct);
}

// ---------------------------------------------------------------- combine
// One wave per (token, piece of V*64 16-byte column groups), grid-stride over those items; the
// next item's slot rows are loaded while the current one is summed, and the partial rows of up
// to 4 (V = 2) or 2 (V = 8) slots are loaded together. Lanes 0..K-1 hold the token's slot rows; every lane owns the 16-byte
// groups lane + 64j of the piece. Slots are summed in ascending order into fp32 accumulators
// that start at +0 (the reference's order); a token without routed slots gets zeros, and with
// skip_single a token with exactly one routed slot is left alone (GEMM2 wrote that row to y).
// V = 8 (whole 4096-column rows) for many tokens; V = 2 spreads few tokens over more waves.
template <int V>
__global__ __launch_bounds__(kEltThreads) void combine_kernel(CombineArgs c) {
  const int lane = lane_id();
  const int tokens = effective_tokens(c.runtime_tokens, c.host_tokens);
  const int nvec = c.hidden >> 3;
  const int parts = (nvec + kWave * V - 1) / (kWave * V);
  const int64_t items = static_cast<int64_t>(tokens) * parts;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kEltWaves;
  int64_t it = static_cast<int64_t>(blockIdx.x) * kEltWaves + threadIdx.x / kWave;
  // lane < K: the row of slot `lane` of item i's token (-1: not routed) and its weight
  auto slot_row = [&](int64_t i, float& w) {
    w = 1.0f;
    if (i >= items || lane >= c.topk) return -1;
    const int64_t route = (i / parts) * c.topk + lane;
    int row = c.output_index[route];
    if (c.topk_ids != nullptr) {
      const int64_t ex = c.ids_i64 ? static_cast<const int64_t*>(c.topk_ids)[route]
                                   : static_cast<const int32_t*>(c.topk_ids)[route];
      if (ex < 0) row = -1;
    }
    if (c.apply_weights) w = c.topk_w[route];
    return row;
  };
  const bool skip_single = c.skip_single != nullptr && *c.skip_single != 0;
  // tokens below zdone without a routed slot: GEMM1 wrote their zero rows (ZeroFill)
  int64_t zdone = 0;
  if (c.zfill_claim != nullptr) {
    const int64_t claimed = *c.zfill_claim;
    const int64_t nchunks = (tokens + kZeroFillTokens - 1) / kZeroFillTokens;
    zdone = (claimed < nchunks ? claimed : nchunks) * kZeroFillTokens;
  }
  float w;
  int row = slot_row(it, w);
  for (; it < items; it += stride) {
    float next_w;
    const int next_row = slot_row(it + stride, next_w);
    const uint64_t routed = __ballot(row >= 0);
    if (!(skip_single && __popcll(routed) == 1) && !(routed == 0 && it / parts < zdone)) {
      const int64_t t = it / parts;
      const int v0 = static_cast<int>(it - t * parts) * kWave * V;
      float sum[V][8];
#pragma unroll
      for (int j = 0; j < V; ++j)
#pragma unroll
        for (int q = 0; q < 8; ++q) sum[j][q] = 0.0f;
      // the routed slots in ascending order, kSlots at a time: their rows' loads go out together
      // (one round trip per batch instead of one per slot), the sums stay in slot order
      constexpr int kSlots = V <= 2 ? 4 : 2;
      for (uint64_t m = routed; m != 0;) {
        uint4 p[kSlots][V];
        float ws[kSlots];
        bool has[kSlots];
#pragma unroll
        for (int b = 0; b < kSlots; ++b) {
          has[b] = m != 0;  // wave-uniform (a ballot)
          const int s = has[b] ? __ffsll(static_cast<unsigned long long>(m)) - 1 : 0;
          m &= m - 1;
          const int r = __shfl(row, s, kWave);
          ws[b] = __shfl(w, s, kWave);
          const uint4* prow = reinterpret_cast<const uint4*>(c.part + static_cast<int64_t>(r) * c.hidden);
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const int v = v0 + j * kWave + lane;
            p[b][j] = has[b] && v < nvec ? ld_nt(prow + v) : make_uint4(0, 0, 0, 0);
          }
        }
#pragma unroll
        for (int b = 0; b < kSlots; ++b) {
          if (!has[b]) break;
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const uint32_t words[4] = {p[b][j].x, p[b][j].y, p[b][j].z, p[b][j].w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float lo = bf16_to_f32(words[q] & 0xffff);
              float hi = bf16_to_f32(words[q] >> 16);
              if (c.apply_weights) { lo *= ws[b]; hi *= ws[b]; }
              sum[j][2 * q] += lo;
              sum[j][2 * q + 1] += hi;
            }
          }
        }
      }
      uint4* yrow = reinterpret_cast<uint4*>(c.y + t * c.hidden);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int v = v0 + j * kWave + lane;
        if (v < nvec)
          yrow[v] = make_uint4(pack_bf16x2(sum[j][0], sum[j][1]), pack_bf16x2(sum[j][2], sum[j][3]),
                               pack_bf16x2(sum[j][4], sum[j][5]), pack_bf16x2(sum[j][6], sum[j][7]));
      }
    }
    row = next_row;
    w = next_w;
  }
}

// Scalar tail of the combine for hidden % 8 != 0 (kept simple; the layer uses H % 128 == 0).
__global__ __launch_bounds__(kEltThreads) void combine_scalar_kernel(CombineArgs c) {
  const int tokens = effective_tokens(c.runtime_tokens, c.host_tokens);
  for (int t = blockIdx.x; t < tokens; t += gridDim.x) {
    for (int h = threadIdx.x; h < c.hidden; h += kEltThreads) {
      float sum = 0.0f;
      for (int s = 0; s < c.topk; ++s) {
        const int64_t route = static_cast<int64_t>(t) * c.topk + s;
        const int row = c.output_index[route];
        if (row < 0) continue;
        if (c.topk_ids != nullptr) {
          const int64_t ex = c.ids_i64 ? static_cast<const int64_t*>(c.topk_ids)[route]
                                       : static_cast<const int32_t*>(c.topk_ids)[route];
          if (ex < 0) continue;
        }
        float v = bf16_to_f32(c.part[static_cast<int64_t>(row) * c.hidden + h]);
        if (c.apply_weights) v *= c.topk_w[route];
        sum += v;
      }
      c.y[static_cast<int64_t>(t) * c.hidden + h] = f32_to_bf16(sum);
    }
  }
}

// ---------------------------------------------------------------- task gather (preprocess)
__global__ __launch_bounds__(kEltThreads) void gather_tasks_kernel(uint8_t* gx, float* gs,
                                                                   const uint8_t* x,
                                                                   const float* x_sf,
                                                                   const int32_t* output_index,
                                                                   int64_t tasks, int topk,
                                                                   int hidden) {
  const int lane = lane_id();
  const int wave = threadIdx.x / kWave;
  for (int64_t task = static_cast<int64_t>(blockIdx.x) * kEltWaves + wave; task < tasks;
       task += static_cast<int64_t>(gridDim.x) * kEltWaves) {
    const int64_t r = output_index[task];
    if (r < 0) continue;
    const int64_t tok = task / topk;
    const uint8_t* src = x + static_cast<int64_t>(tok) * hidden;
    uint8_t* dst = gx + r * hidden;
    if ((hidden & 15) == 0) {
      for (int v = lane; v < (hidden >> 4); v += kWave)
        reinterpret_cast<uint4*>(dst)[v] = reinterpret_cast<const uint4*>(src)[v];
    } else {
      for (int v = lane; v < hidden; v += kWave) dst[v] = src[v];
    }
    if (lane == 0) gs[r] = x_sf[tok];
  }
}

// The rows that the routing may leave out (counts above the tasks' own): weight 0, expert -1.
__global__ __launch_bounds__(kEltThreads) void clear_rows_kernel(float* row_weight, int32_t* m_indices, int rows) {
  // (64-bit: the step past the last row of a count near 2^31 does not fit an int)
  for (int64_t r = blockIdx.x * kEltThreads + threadIdx.x; r < rows; r += gridDim.x * kEltThreads) {
    row_weight[r] = 0.0f;
    m_indices[r] = -1;
  }
}

// ---------------------------------------------------------------- channelwise cast
// scale = max(amax, 1e-4) / 448 and the codes e4m3(clip(x / scale)) of rows of bf16. Every value is
// read from memory once: it stays in registers between the row's maximum and its codes.
//
// The quotient: q0 = x * rcp with rcp = 1 / scale rounded, then one correction step (Markstein),
// q = q0 - (q0 * scale - x) * rcp in two fused multiply-adds: the rounded x / scale for every bf16
// mantissa over every fp32 scale mantissa (all 2^30 pairs compared on the CPU), and a zero keeps its
// sign. Three VALU instructions instead of the ten of the IEEE division. A row with an infinity has
// an infinite scale and takes the division itself. Bound by HBM: against the
// two-pass kernel with 2-byte loads (kept below for rows that the wide loads do not fit) a pass that
// casts 4000 x 4096 tokens, groups them and combines their rows went from 83 to 63 us.
struct RowQuant {
  float scale, rcp;
  bool finite;
  __device__ __forceinline__ explicit RowQuant(float amax)
      : scale(fmaxf(amax, kAmaxFloor) / kE4m3Max), rcp(1.0f / scale), finite(scale < __builtin_inff()) {}
  __device__ __forceinline__ float operator()(float x) const {
    if (!finite) return x / scale;
    const float q0 = x * rcp;
    return __builtin_fmaf(-__builtin_fmaf(q0, scale, -x), rcp, q0);
  }
  // the codes of the eight bf16 values of v
  __device__ __forceinline__ u32x2_t codes(const uint4& v) const {
    const RowQuant& q = *this;
    return u32x2_t{pack_e4m3x4(q(bf16_lo(v.x)), q(bf16_hi(v.x)), q(bf16_lo(v.y)), q(bf16_hi(v.y))),
                   pack_e4m3x4(q(bf16_lo(v.z)), q(bf16_hi(v.z)), q(bf16_lo(v.w)), q(bf16_hi(v.w)))};
  }
  static __device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
  static __device__ __forceinline__ float max8(float m, const uint4& v) {
    m = fmaxf(fmaxf(m, fabsf(bf16_lo(v.x))), fabsf(bf16_hi(v.x)));
    m = fmaxf(fmaxf(m, fabsf(bf16_lo(v.y))), fabsf(bf16_hi(v.y)));
    m = fmaxf(fmaxf(m, fabsf(bf16_lo(v.z))), fabsf(bf16_hi(v.z)));
    return fmaxf(fmaxf(m, fabsf(bf16_lo(v.w))), fabsf(bf16_hi(v.w)));
  }
};

// Rows of up to 8 * 64 * V columns (a multiple of 8, rows 16-byte aligned), a wave a row: V
// 16-byte loads a lane, all in flight together, and 8-byte stores of the codes.
template <int V>
__global__ __launch_bounds__(kEltThreads) void cast_fp8_rows_kernel(uint8_t* out, float* scale,
                                                                    const uint16_t* x,
                                                                    int64_t rows, int cols) {
  const int lane = lane_id();
  const int octs = cols >> 3;
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * kEltWaves + threadIdx.x / kWave; r < rows;
       r += static_cast<int64_t>(gridDim.x) * kEltWaves) {
    const uint4* xr = reinterpret_cast<const uint4*>(x + r * cols);
    uint4 v[V];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int o = lane + j * kWave;
      v[j] = o < octs ? ld_nt(xr + o) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < V; ++j) m = RowQuant::max8(m, v[j]);
    const RowQuant q(wave_max(m));
    if (lane == 0) scale[r] = q.scale;
    u32x2_t* orow = reinterpret_cast<u32x2_t*>(out + r * cols);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int o = lane + j * kWave;
      if (o < octs) orow[o] = q.codes(v[j]);
    }
  }
}

// Any other row (columns not a multiple of 8, unaligned rows, more than 8192 columns): a workgroup
// a row, read twice.
__global__ __launch_bounds__(kEltThreads) void cast_fp8_any_kernel(uint8_t* out, float* scale,
                                                                   const uint16_t* x, int64_t rows,
                                                                   int64_t cols) {
  __shared__ float s_red[kEltWaves];
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const uint16_t* xr = x + r * cols;
    float amax = 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += kEltThreads) amax = fmaxf(amax, fabsf(bf16_to_f32(xr[c])));
    amax = wave_max(amax);
    if (lane_id() == 0) s_red[threadIdx.x / kWave] = amax;
    __syncthreads();
    float m = s_red[0];
    for (int w = 1; w < kEltWaves; ++w) m = fmaxf(m, s_red[w]);
    const RowQuant q(m);
    if (threadIdx.x == 0) scale[r] = q.scale;
    uint8_t* orow = out + r * cols;
    for (int64_t c = threadIdx.x; c < cols; c += kEltThreads) orow[c] = f32_to_e4m3(q(bf16_to_f32(xr[c])));
    __syncthreads();
  }
}

// The cast of bf16 weight rows straight into the Marlin layout (below): a workgroup takes the 16
// rows of a row tile, whose codes are 16 * k contiguous bytes. Lane l of a wave holds row l % 16:
// per step 16 consecutive values of it (32 bytes; four lanes read 128 contiguous bytes of a row),
// whose 16 codes are one 16-byte piece, so that a wave stores 1 KB contiguously. V steps of 512
// columns stay in registers until the rows' maxima have met in LDS. Bound by HBM: 32 experts of
// 4096 x 4096 and 4096 x 2048 (2.4 GB read and written) 523 us, 4.6 TB/s where a plain copy reaches
// 4.9; the cast and the pack one after the other, with the codes through memory, took 2380 us.
constexpr int kPackThreads = 512;
constexpr int kPackWaves = kPackThreads / kWave;

template <int V>
__global__ __launch_bounds__(kPackThreads) void cast_marlin_kernel(uint8_t* out, float* scale,
                                                                   const uint16_t* x,
                                                                   int64_t row_tiles, int k) {
  __shared__ float s_max[kPackWaves][16];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int row = lane & 15;
  const int blocks = k >> 4;                  // 16-column blocks of a row
  const int b0 = wave * 4 + (lane >> 4);      // this lane's block of step 0; + 32 a step
  for (int64_t t = blockIdx.x; t < row_tiles; t += gridDim.x) {
    const uint4* xr = reinterpret_cast<const uint4*>(x + (t * 16 + row) * k);
    uint4 v[V][2];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int b = b0 + j * kPackWaves * 4;
      const bool in = b < blocks;
      v[j][0] = in ? ld_nt(xr + 2 * b) : make_uint4(0, 0, 0, 0);
      v[j][1] = in ? ld_nt(xr + 2 * b + 1) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < V; ++j) m = RowQuant::max8(RowQuant::max8(m, v[j][0]), v[j][1]);
    m = fmaxf(m, __shfl_xor(m, 16, kWave));
    m = fmaxf(m, __shfl_xor(m, 32, kWave));
    if (lane < 16) s_max[wave][row] = m;
    __syncthreads();
    m = s_max[0][row];
#pragma unroll
    for (int w = 1; w < kPackWaves; ++w) m = fmaxf(m, s_max[w][row]);
    __syncthreads();  // (the next tile's maxima are written after these reads)
    const RowQuant q(m);
    if (threadIdx.x < 16) scale[t * 16 + row] = q.scale;
    uint8_t* tile = out + t * 16 * k + row * 16;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int b = b0 + j * kPackWaves * 4;
      const u32x2_t lo = q.codes(v[j][0]), hi = q.codes(v[j][1]);
      if (b < blocks) __builtin_nontemporal_store(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, reinterpret_cast<u32x4_t*>(tile + b * 256));
    }
  }
}

// ---------------------------------------------------------------- Marlin pack
// out[g, r/16, (k/16)*256 + (r%16)*16 + k%16] = in[g, r, k]; one thread per 16-byte block row.
__global__ __launch_bounds__(kEltThreads) void marlin_pack_kernel(uint8_t* out, const uint8_t* in,
                                                                  int64_t groups, int64_t rows,
                                                                  int64_t k) {
  const int64_t kblocks = k >> 4;
  const int64_t total = groups * rows * kblocks;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kEltThreads + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * kEltThreads) {
    const int64_t kb = i % kblocks;
    const int64_t gr = i / kblocks;  // g * rows + r
    const int64_t r = gr % rows;
    const int64_t gidx = gr / rows;
    const uint4 v = *reinterpret_cast<const uint4*>(in + gr * k + kb * 16);
    const int64_t dst = ((gidx * (rows >> 4) + (r >> 4)) * k + kb * 16) * 16 + (r & 15) * 16;
    *reinterpret_cast<uint4*>(out + dst) = v;
  }
}

__global__ __launch_bounds__(kEltThreads) void f32_to_e4m3_kernel(uint8_t* out, const float* in,
                                                                  int64_t n) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kEltThreads + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kEltThreads)
    out[i] = f32_to_e4m3(in[i]);
}

unsigned grid_for(int64_t work_items, int64_t per_block, int64_t cap) {
  int64_t g = (work_items + per_block - 1) / per_block;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

}  // namespace

hipError_t launch_requant(const uint16_t* src, bool wide, float* amax, int32_t* meta, uint8_t* act,
                          float* act_scale, int64_t max_rows, int inter, const RowDest& dest,
                          int num_cus, hipStream_t stream, const int32_t* dual_rows,
                          int dual_min_rows) {
  if (max_rows <= 0) return hipSuccess;
  if (inter % 4) return hipErrorInvalidValue;
  if (dest.row_dest != nullptr && (dest.row_token == nullptr || dest.output_index == nullptr ||
                                   dest.topk < 1 || dest.topk > kWave))
    return hipErrorInvalidValue;
  const RequantArgs r{src, amax, meta, act, act_scale, inter, dest, dual_rows, dual_min_rows};
  // grid of up to 16 workgroups a CU (one row per wave in flight; the hardware keeps what fits
  // resident): 397 us at 195,558 rows vs 470 us with 4 a CU
  const unsigned grid = grid_for(max_rows, kEltWaves, static_cast<int64_t>(num_cus) * 16);
  if (dual_rows != nullptr)
    return launch_kernel(requant_kernel<2>, dim3(grid), dim3(kEltThreads), 0, stream, r);
  if (wide) return launch_kernel(requant_kernel<1>, dim3(grid), dim3(kEltThreads), 0, stream, r);
  return launch_kernel(requant_kernel<0>, dim3(grid), dim3(kEltThreads), 0, stream, r);
}

hipError_t launch_combine(const CombineArgs& c, int num_cus, hipStream_t stream) {
  if (c.host_tokens <= 0) return hipSuccess;
  if (c.topk > 16) return hipErrorInvalidValue;
  if ((c.hidden & 7) == 0) {
    // a wave per item, up to 8 four-wave workgroups a CU in flight; whole rows once there are
    // at least 16 tokens a CU
    const int64_t nvec = c.hidden >> 3;
    if (c.host_tokens >= static_cast<int64_t>(num_cus) * 16) {
      const int64_t items = c.host_tokens * ((nvec + kWave * 8 - 1) / (kWave * 8));
      const unsigned grid = grid_for(items, kEltWaves, static_cast<int64_t>(num_cus) * 8);
      return launch_kernel(combine_kernel<8>, dim3(grid), dim3(kEltThreads), 0, stream, c);
    } else {
      const int64_t items = c.host_tokens * ((nvec + kWave * 2 - 1) / (kWave * 2));
      const unsigned grid = grid_for(items, kEltWaves, static_cast<int64_t>(num_cus) * 8);
      return launch_kernel(combine_kernel<2>, dim3(grid), dim3(kEltThreads), 0, stream, c);
    }
  } else {
    if (c.skip_single != nullptr) return hipErrorInvalidValue;
    const unsigned grid = grid_for(c.host_tokens, 1, static_cast<int64_t>(num_cus) * 16);
    return launch_kernel(combine_scalar_kernel, dim3(grid), dim3(kEltThreads), 0, stream, c);
  }
}

hipError_t launch_clear_rows(float* row_weight, int32_t* m_indices, int rows, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  return launch_kernel(clear_rows_kernel, dim3(grid_for(rows, kEltThreads, 1024)), dim3(kEltThreads), 0,
                       stream, row_weight, m_indices, rows);
}

hipError_t launch_gather_tasks(uint8_t* grouped_x, float* grouped_scale, const uint8_t* x,
                               const float* x_sf, const int32_t* output_index, int64_t tasks,
                               int topk, int hidden, hipStream_t stream) {
  if (tasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(gather_tasks_kernel, dim3(grid_for(tasks, kEltWaves, 8192)),
                     dim3(kEltThreads), 0, stream, grouped_x, grouped_scale, x, x_sf,
                     output_index, tasks, topk, hidden);
  return hipGetLastError();
}

hipError_t launch_cast_fp8_channelwise(uint8_t* out, float* scale, const uint16_t* x,
                                       int64_t rows, int64_t cols, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const auto aligned = [](const void* p, uintptr_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; };
  if (cols % 8 != 0 || cols > kCastMaxCols || !aligned(x, 16) || !aligned(out, 8))
    return launch_kernel(cast_fp8_any_kernel, dim3(grid_for(rows, 1, 65536)), dim3(kEltThreads), 0,
                         stream, out, scale, x, rows, cols);
  const dim3 grid(grid_for(rows, kEltWaves, 65536));
  const int n = static_cast<int>(cols);
  if (cols <= 2048)
    return launch_kernel(cast_fp8_rows_kernel<4>, grid, dim3(kEltThreads), 0, stream, out, scale, x, rows, n);
  if (cols <= 4096)
    return launch_kernel(cast_fp8_rows_kernel<8>, grid, dim3(kEltThreads), 0, stream, out, scale, x, rows, n);
  return launch_kernel(cast_fp8_rows_kernel<16>, grid, dim3(kEltThreads), 0, stream, out, scale, x, rows, n);
}

hipError_t launch_cast_marlin(uint8_t* out, float* scale, const uint16_t* x, int64_t groups,
                              int64_t rows, int64_t k, hipStream_t stream) {
  const int64_t tiles = groups * (rows >> 4);
  if (tiles <= 0) return hipSuccess;
  if (k % 16 != 0 || k <= 0 || k > kCastMaxCols) return hipErrorInvalidValue;
  const dim3 grid(grid_for(tiles, 1, 65536));
  const int n = static_cast<int>(k);
  if (k <= 2048)
    return launch_kernel(cast_marlin_kernel<4>, grid, dim3(kPackThreads), 0, stream, out, scale, x, tiles, n);
  if (k <= 4096)
    return launch_kernel(cast_marlin_kernel<8>, grid, dim3(kPackThreads), 0, stream, out, scale, x, tiles, n);
  return launch_kernel(cast_marlin_kernel<16>, grid, dim3(kPackThreads), 0, stream, out, scale, x, tiles, n);
}

hipError_t launch_marlin_pack(uint8_t* out, const uint8_t* in, int64_t groups, int64_t rows,
                              int64_t k, hipStream_t stream) {
  const int64_t total = groups * rows * (k >> 4);
  if (total <= 0) return hipSuccess;
  hipLaunchKernelGGL(marlin_pack_kernel, dim3(grid_for(total, kEltThreads, 65536)),
                     dim3(kEltThreads), 0, stream, out, in, groups, rows, k);
  return hipGetLastError();
}

hipError_t launch_f32_to_e4m3(uint8_t* out, const float* in, int64_t n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(f32_to_e4m3_kernel, dim3(grid_for(n, kEltThreads, 65536)), dim3(kEltThreads),
                     0, stream, out, in, n);
  return hipGetLastError();
}

}  // namespace mmoe
