// gemm.hip -- grouped FP8 (OCP e4m3) GEMMs of the layer on gfx950 MFMA, over the
// expert-contiguous routed rows.
//
// GEMM1 (gate+up, K = H) gathers its A rows straight from the token matrix through row_token
// (the dispatch "pull" of the reference's K1, megamoe/dcu_megamoe_large_opt/K1_fused/
// k1_fused_ext.cu:479-746), so no grouped copy of x exists:
//   h = bf16(acc * x_sf[token] * w1_sf[e, n])       for the gate and the up column of a channel
// It fuses the K2 stage (megamoe/dcu_megamoe_large_opt/K2_fused/
// k2_fused_ext.cu:254-377) into its epilogue:
//   y = silu(min(h_g, c)) * clamp(h_u, -c, c) * w    (fp32, left to right)
// (each output tile holds matching gate and up channels, so SwiGLU is elementwise in
// registers), on both kernels. The per-row requant (amax = max |y|; a = max(amax, 1e-4);
// act = e4m3(clip(y * 448/a)); act_scale = a/448) needs the whole row and runs as its own small
// kernel: a cross-workgroup hand-off inside GEMM1 would need an agent-scope release per tile,
// which on gfx950 writes back the whole (per-XCD, non-coherent) L2 -- measured 4x slower than
// the kernel boundary.
// GEMM2 (down, K = I) reads act/act_scale and writes the bf16 partial rows for the combine:
//   part[r, n] = bf16((sum_k act[r,k] * w2[e,n,k]) * act_scale[r] * w2_sf[e,n]).
//
// B is the Marlin nt_kpack2 weight (deep_gemm/include/deep_gemm/layout/mega_moe_dcu.cuh:50-66):
// per 16-row tile, each 16-byte k-block of the 16 rows is 256 contiguous bytes.
//
// Two persistent kernels per GEMM; the host picks one (gemm_wide_selected):
//  * the 8-wave kernel (one workgroup per CU) runs two tile engines, each expert's chosen on
//    the device from its routed row count, and can route the tasks itself (decode sizes):
//    - STREAM engine (<= 128 rows on the auto schedule: decode, HBM-bound on the weights).
//      A workgroup tile is (expert, 512 output columns, <= 128 rows: 1, 2 or 4 row tiles of
//      32) over the full K; wave w owns columns
//      [64w, 64w + 64) and streams its weight columns from global memory into a register ring
//      4 steps deep (Marlin gives each lane 16 contiguous k-bytes of one weight row; 16 lanes
//      read 256 contiguous bytes): B never touches LDS. The A rows, the same
//      for the 8 waves, go to LDS once per workgroup in k-chunks of 64 KB loaded as whole
//      128-byte lines, double buffered, one barrier per chunk (1-4 per tile). Loading A per
//      wave in MFMA operand order (32 lines per instruction, re-read by every wave) made the A
//      reads, not the weights, set the pace.
//    - TILE engine (more rows). A 256 x 256 output tile per workgroup, the 8 waves as 2 x 4
//      with 128 x 64 each, K in 128-byte stages through double-buffered LDS (A rows
//      XOR-swizzled, B in Marlin's own 256-byte blocks).
//    Both engines use the 32x32x64 MFMA, let lane l supply k-bytes [32*(l/32), 32*(l/32)+32) of each
//    64-k MFMA step for A and B alike and accumulate the 64-k steps in the same order: the same bits.
//  * the 4-wave WIDE kernel (every expert with many rows: prefill, MFMA-bound): one wave per
//    SIMD with its 256 accumulators in AGPRs, 256 x 256 tiles of 16x16x128 MFMAs, weights straight
//    into registers and only A through LDS; described at wide_tile. Its sums take 128 products a step
//    (nearly always the same bits).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.cuh"
#include "kernels.h"
#include "launch.h"
#include "route_wave.cuh"

namespace mmoe {

namespace {

constexpr int kGemmThreads = 512;  // 8 waves, one workgroup per CU
constexpr int kGemmWaves = kGemmThreads / kWave;
constexpr int kMaxGemmExperts = 256;
// STREAM engine
constexpr int kStreamUnit = 64;     // output columns per wave
constexpr int kStreamRows = 64;     // rows of a decode pipeline GEMM2 item
constexpr int kStreamItemRows = 128;  // rows of a STREAM item of the 8-wave GEMM kernel
constexpr int kStreamAutoMaxRows = kStreamItemRows;  // the auto schedule streams experts up to this
constexpr int kStreamDepth = 4;     // 64-k weight steps in flight per wave
constexpr int kAChunk = 65536;      // bytes of one A chunk buffer (32*MT rows x 2048/MT k)
constexpr int kALoads = kAChunk / 1024 / kGemmWaves;  // 16-byte A loads per lane per chunk
constexpr int kTailDepth = 2;       // the same with a short last chunk (stream_tail)
constexpr int kNarrowDepth = 8;     // weight steps in flight of a narrow item's waves
constexpr int kAChunk4 = kAChunk / 256;  // k-bytes of a chunk of 128 rows in half a buffer
// TILE engine: 256 x 256 output tile, BK = 128, the 8 waves as 2 (M) x 4 (N), each wave 128
// rows x 64 columns (4 x 2 MFMA tiles of 32 x 32)
constexpr int kTileBM = 256, kTileBN = 256, kTileBK = 128;
constexpr int kTileWM = 2, kTileWN = 4;
constexpr int kTileStage = (kTileBM + kTileBN) * kTileBK;  // 64 KB: A rows, then B row-tiles
constexpr int kSmemBytes = 2 * kAChunk;  // == 2 * kTileStage

__device__ __forceinline__ v8i make_v8i(const int4& lo, const int4& hi) {
  v8i r;
  r[0] = lo.x; r[1] = lo.y; r[2] = lo.z; r[3] = lo.w;
  r[4] = hi.x; r[5] = hi.y; r[6] = hi.z; r[7] = hi.w;
  return r;
}

__device__ __forceinline__ v16f mfma_fp8(const v8i& a, const v8i& b, const v16f& c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// c[n] += b[n] a for the four 16-column tiles n of an MFMA group, the accumulators in AGPRs. Inline
// assembly: from the builtin the register allocator moved some of a tile's 64 accumulators through
// VGPRs in the loop. The compiler adds no wait states to instructions that it does not see:
//  * an operand that a VALU instruction has written (a copy that the compiler puts in front of the
//    block) may be read two wait states later at the earliest. The block holds no s_nop for that: with
//    one in front of each group (or MFMA) a layer of 24.7K rows takes 690 us instead of 683 and one of
//    196K rows 4995 instead of 4946, and the operands come straight from memory and LDS;
//  * no accumulator may be read or copied between a group and mfma_settle.
// tests/test_isa_waits.py checks both in the code as built, along every path.
__device__ __forceinline__ void mfma_group(const v8i (&b)[4], const v8i& a, v4f (&c)[4]) {
  asm volatile(
      "v_mfma_f32_16x16x128_f8f6f4 %0, %4, %8, %0\n\t"
      "v_mfma_f32_16x16x128_f8f6f4 %1, %5, %8, %1\n\t"
      "v_mfma_f32_16x16x128_f8f6f4 %2, %6, %8, %2\n\t"
      "v_mfma_f32_16x16x128_f8f6f4 %3, %7, %8, %3"
      : "+a"(c[0]), "+a"(c[1]), "+a"(c[2]), "+a"(c[3])
      : "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(a));
}

// The last MFMA's result (8 passes of 4 cycles) is in its registers before any of c is read. Volatile
// like the groups, so the wait stays behind the last of them; every later read of c then depends on the
// empty blocks, which stay behind the wait.
template <int N>
__device__ __forceinline__ void mfma_settle(v4f (&c)[N][4]) {
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; i += 2)
    asm volatile("" : "+a"(c[i][0]), "+a"(c[i][1]), "+a"(c[i][2]), "+a"(c[i][3]), "+a"(c[i + 1][0]),
                 "+a"(c[i + 1][1]), "+a"(c[i + 1][2]), "+a"(c[i + 1][3]));
}

__device__ __forceinline__ int4 ld16(const uint8_t* p) { return *reinterpret_cast<const int4*>(p); }

// Streaming load for data read exactly once (the STREAM engine's weights): the nontemporal
// hint keeps it from displacing reused lines in L2/MALL; measured 6.85 vs 6.15 TB/s for a
// one-pass read with one 8-wave workgroup per CU.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4 ld16_stream(const uint8_t* p) {
  const i32x4 v = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(p));
  return make_int4(v[0], v[1], v[2], v[3]);
}

__device__ __forceinline__ float bf16_round(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// Where a GEMM finds the token (gather) and the route weight (SwiGLU) of routed row r: the
// routing tables in global memory, or a workgroup's LDS copy of its rows (in-kernel routing),
// entry r - base.
struct RowSrc {
  const int32_t* tok;
  const float* w;
  int base;
  __device__ __forceinline__ int token(int r) const { return tok[r - base]; }
  __device__ __forceinline__ float weight(int r) const { return w[r - base]; }
};

template <bool kGather>
__device__ __forceinline__ float row_scale(const GemmArgs& g, const RowSrc& rs, int row) {
  return kGather ? g.a_scale[rs.token(row)] : g.a_scale[row];
}

template <bool kGather>
__device__ __forceinline__ const uint8_t* a_row_ptr(const GemmArgs& g, const RowSrc& rs, int row) {
  const int64_t src = kGather ? static_cast<int64_t>(rs.token(row)) : row;
  return g.a + src * g.lda;
}

// Weight row (output column of B) of column tile `ct` (32 columns) of n-block `nb`. With the
// SwiGLU epilogue, tile nb holds gate channels [nb*W, nb*W+W) then the same up channels
// (rows I + ...), W = columns per tile / 2.
template <bool kSwiglu>
__device__ __forceinline__ int weight_row(const GemmArgs& g, int nb, int tile_cols, int col) {
  if (!kSwiglu) return nb * tile_cols + col;
  const int half = tile_cols / 2;
  return col < half ? nb * half + col : g.sw.inter + nb * half + (col - half);
}

// SwiGLU of one (row, channel): h rounded to bf16 exactly like the staged K1 output.
__device__ __forceinline__ float swiglu_value(const GemmArgs& g, float gacc, float uacc, float xs,
                                              float wsg, float wsu, float route_w) {
  return swiglu_weighted(bf16_round(gacc * xs * wsg), bf16_round(uacc * xs * wsu), route_w,
                         g.sw.has_clamp, g.sw.clamp);
}

// Thread index for an engine body, opaque to the optimizer: values derived from it are computed
// inside the body instead of being hoisted out of the persistent item loop, where the
// invariants of every engine variant would stay live at once and crowd out the ring.
__device__ __forceinline__ int opaque_tid() {
  int t = static_cast<int>(threadIdx.x);
  asm volatile("" : "+v"(t));
  return t;
}

// ------------------------------------------------------------------ epilogue
// Per-tile scales: row r's A scale (its token's, when gathering) and route weight (SwiGLU), and
// each lane's weight-row scales (GEMM2: its column in both 32-column tiles; SwiGLU: its gate and
// up channel). They are loaded into registers at the start of an item and written into a static
// LDS table just before the barrier that completes the item's first A chunk (or stage): the A
// loads issued after them have landed by then, so that costs no wait of its own, and the
// epilogue reads LDS instead of memory. (Loaded before a tile's last MFMAs instead, the compiler
// sank the loads into the epilogue: a memory round trip after the last MFMA, then a full vmcnt
// wait behind the first output stores.)
struct TileTables {
  float xs[kTileBM];               // row scale of tile row r
  float rw[kTileBM];               // route weight of tile row r (SwiGLU)
  float bs[kGemmWaves][2][kWave];  // wave w, lane l: its two weight-row scales
};

struct TileScaleRegs {
  float xs, rw, b0, b1;
};

// Thread t: tile row t's scales (t < mrows <= 512 threads), and its lane's weight-row scales of
// the 64-column unit `unit` (a valid unit).
template <bool kGather, bool kSwiglu>
__device__ __forceinline__ TileScaleRegs load_tile_scales(const GemmArgs& g, const RowSrc& rs, int e,
                                                          int row0, int mrows, int unit) {
  const int tid = opaque_tid();
  const int rl = tid & 31;
  TileScaleRegs t{0.0f, 0.0f, 0.0f, 0.0f};
  if (tid < mrows) {
    t.xs = row_scale<kGather>(g, rs, row0 + tid);
    if (kSwiglu) t.rw = rs.weight(row0 + tid);
  }
  if (!kSwiglu) {
    t.b0 = g.b_scale[static_cast<int64_t>(e) * g.n + unit * 64 + rl];
    t.b1 = g.b_scale[static_cast<int64_t>(e) * g.n + unit * 64 + 32 + rl];
  } else {
    const int chan = unit * 32 + rl;
    t.b0 = g.b_scale[static_cast<int64_t>(e) * g.n + chan];
    t.b1 = g.b_scale[static_cast<int64_t>(e) * g.n + g.sw.inter + chan];
  }
  return t;
}

__device__ __forceinline__ void publish_tile_scales(TileTables& tt, const TileScaleRegs& t, int mrows) {
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  if (tid < mrows) {
    tt.xs[tid] = t.xs;
    tt.rw[tid] = t.rw;
  }
  tt.bs[wave][0][lane] = t.b0;
  tt.bs[wave][1][lane] = t.b1;
}

// Stores a wave's MT x (32 rows) x 64 columns of accumulators: rows [row0, row0 + mrows) of
// the output (mrows <= 32 * MT; table row trow0 + r holds row r's scales), 64-column unit `unit`
// of the output (SwiGLU: 32 channels).
// kCoherent: the stores go out device-coherent (sc1, written through the XCD's L2): GEMM2's
// partial rows and GEMM1's SwiGLU rows in the decode pipeline, which workgroups of other XCDs read in
// the same launch.
// SwiGLU: y is stored in bf16 (the reference fused path's rounding of the activation before
// its quantization). kPmax (the decode pipeline's GEMM1): the row maxima of the rounded values
// are stored as well.
// The stores go through a buffer descriptor of the tile's mrows rows, whose bounds check drops the
// rows past them: no branch a row (at 4 row tiles 64 of them, which had also kept the compiler
// from inlining the tile in a kernel of many variants).
constexpr int kBufferFlags = 0x00020000;  // raw buffer, 32-bit data format (unused by raw accesses)
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rows(T* p, int64_t first, int64_t count) {
  // (uniform in the wave: the descriptor sits in scalar registers)
  const int64_t at = reinterpret_cast<int64_t>(p + first);
  const int lo = __builtin_amdgcn_readfirstlane(static_cast<int>(at));
  const int hi = __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32));
  const int bytes = __builtin_amdgcn_readfirstlane(static_cast<int>(count < 0 ? 0 : count) * static_cast<int>(sizeof(T)));
  void* base = reinterpret_cast<void*>(static_cast<int64_t>(hi) << 32 | static_cast<uint32_t>(lo));
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, kBufferFlags);
}

template <bool kSwiglu, int MT, bool kPmax = false, bool kCoherent = false>
__device__ __forceinline__ void store_tile(const GemmArgs& g, const v16f (&acc)[MT][2], int row0,
                                           int mrows, int unit, const TileTables& tt, int trow0) {
  constexpr int kAux = kCoherent ? 16 : 0;  // sc1
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const int rl = lane & 31, hk = lane >> 5;
  const float b0 = tt.bs[wave][0][lane], b1 = tt.bs[wave][1][lane];
  const int cols = kSwiglu ? g.sw.inter : g.n;  // of an output row
  const __amdgpu_buffer_rsrc_t out =
      tile_rows(kSwiglu ? g.sw.y : g.c, static_cast<int64_t>(row0) * cols, static_cast<int64_t>(mrows) * cols);
  const int at = (hk * 4 * cols + unit * (kSwiglu ? 32 : 64) + rl) * 2;  // the lane's row 0 and first column
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    // the 16 rows' table entries read at once (rows past mrows read entries never used)
    float xs[16], rw[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = mt * 32 + (v >> 2) * 8 + hk * 4 + (v & 3);
      xs[v] = tt.xs[trow0 + r];
      rw[v] = kSwiglu ? tt.rw[trow0 + r] : 0.0f;
    }
    float pm[16];  // kPmax: |y| of the lane's channel in each of its 16 rows
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int off = at + (mt * 32 + (v >> 2) * 8 + (v & 3)) * cols * 2;
      if (!kSwiglu) {
        __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(acc[mt][0][v] * xs[v] * b0), out, off, 0, kAux);
        __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(acc[mt][1][v] * xs[v] * b1), out, off + 64, 0, kAux);
      } else {
        const float yv = swiglu_value(g, acc[mt][0][v], acc[mt][1][v], xs[v], b0, b1, rw[v]);
        const uint16_t yb = f32_to_bf16(yv);
        __builtin_amdgcn_raw_buffer_store_b16(yb, out, off, 0, kAux);
        if constexpr (kPmax) pm[v] = fabsf(bf16_to_f32(yb));
      }
    }
    if constexpr (kPmax && kSwiglu) {
      // the row maxima over the unit's 32 channels (the lanes of a half-wave); lane 16 + v of
      // each half writes row v of its half
#pragma unroll
      for (int v = 0; v < 16; ++v) pm[v] = half_wave_max_nonneg(pm[v]);
      float mv = pm[0];
#pragma unroll
      for (int v = 1; v < 16; ++v) mv = (rl & 15) == v ? pm[v] : mv;
      const int v = rl & 15;
      const int r = mt * 32 + (v >> 2) * 8 + hk * 4 + (v & 3);
      if (rl >= 16 && r < mrows)
        __hip_atomic_store(g.row_pmax + static_cast<int64_t>(row0 + r) * (g.n / kStreamUnit) + unit, mv,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// ------------------------------------------------------------------ STREAM engine
// The 8 waves of a STREAM tile step together: a bare s_barrier after every 64-k step (each wave
// has issued that step's ring refill before it, so the weight loads stay in flight). Left to
// themselves the waves drift apart -- the memory pipeline does not serve them evenly -- and a
// workgroup's first and last wave finished their streams 15-16 us apart at c1 (median), the
// last one 6-7 us after the median one, with fewer and fewer loads in flight at the end. In
// step, GEMM1 went from 109 to 97 us at c1 (a barrier every 4 steps: 103 us).
__device__ __forceinline__ void step_barrier() { asm volatile("s_barrier" ::: "memory"); }

// Workgroup barrier for the LDS A chunks: this wave's LDS writes are complete, then s_barrier.
// It waits on no global load, so the weight loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// 16-byte piece p of LDS A row r sits at piece (p & ~7) | ((p ^ r) & 7): 8 lanes reading the
// same k of 8 consecutive rows hit 8 distinct 16-byte bank groups.
__device__ __forceinline__ int swizzle_piece(int p, int r) { return (p & ~7) | ((p ^ r) & 7); }

// An A chunk in LDS: 32*MT rows of kc k-bytes, kc <= kMaxK, at a row stride of kMaxK. Piece i of a
// lane is 16 bytes of row row(i, ..) at piece position pos(i, ..): 64 lanes cover a row's 1024
// bytes (MT = 4: two rows' 512), whole 128-byte lines. A position past kc is never read; the piece
// put there is the chunk's last one (src), so that loads and LDS writes need no masks.
template <int MT, int kLoads = kALoads>
struct AChunk {
  static constexpr int kBytes = kLoads * kGemmWaves * 1024;
  static constexpr int kMaxK = kBytes / (32 * MT);
  static constexpr int kPieces = kMaxK / 16;  // piece positions of a row
  static __device__ __forceinline__ int row(int i, int lane, int wave) {
    return (i * kWave + lane) / kPieces * kGemmWaves + wave;
  }
  static __device__ __forceinline__ int pos(int i, int lane) { return (i * kWave + lane) % kPieces; }
  // the piece of the chunk at that position (swizzled by the row)
  static __device__ __forceinline__ int src(int i, int lane, int wave, int kc) {
    return swizzle_piece(min(pos(i, lane), kc / 16 - 1), row(i, lane, wave));
  }
};

// One workgroup tile (expert e, column block nb of `waves` 64-column units, rows [row0, row0 +
// mrows), mrows <= 32*MT) over the full K in chunks of kc k-bytes (GemmArgs::kc: at most 2048/MT, a
// multiple of 64*D that divides K), with a ring of D weight steps a wave.
//
// A chunk c+1 is loaded into registers (kLoads x 16 bytes per lane, AChunk's pieces) right after the
// barrier that opens chunk c, and written to its LDS buffer at the end of chunk c, before the
// next barrier. Plain loads keep the memory counter in order, so every wait the compiler places
// for a weight step or for the staged chunk is exact; the chunk's loads are older than all
// weight loads of chunk c and cost no wait at all by then.
//
// kEarly: the weight ring's first steps go out first, then `before_a` runs (the decode
// pipeline's wait for the item's rows), then the item's scales and A rows are loaded.
// kAResident: before_a also leaves the item's whole A in the LDS chunk buffers (K of at most two
// chunks), so no A rows are loaded here.
// kNarrow: only the first `waves` waves have columns (2 or 4 of the 8); the others help with A
// and leave. A ring of 8 steps then keeps enough bytes in flight, and the few waves need no
// barrier a step.
// kTail: kc need not divide K (both are multiples of 64*D, and kc <= K). A last chunk that is shorter is
// loaded as the last kc bytes of K: its steps are the end of what lies in LDS, and no load is masked.
struct NoHook {
  __device__ __forceinline__ void operator()() const {}
};
template <bool kGather, bool kSwiglu, int MT, int D, bool kEarly = false, bool kAResident = false,
          bool kPmax = false, bool kCoherent = false, bool kNarrow = false, int kLoads = kALoads,
          bool kTail = false, typename Hook = NoHook>
__device__ void stream_tile(const GemmArgs& g, const RowSrc& rs, int e, int row0, int mrows, int nb,
                            int kc, uint8_t* smem, TileTables& tt, const Hook& before_a = Hook{},
                            int waves = kGemmWaves) {
  static_assert(!kAResident || kEarly, "a resident A is staged by the hook");
  using Chunk = AChunk<MT, kLoads>;
  const int spc = kc / 64;  // steps per chunk
  const int nchunks = kTail ? (g.k + kc - 1) / kc : g.k / kc;
  const int last_spc = kTail ? g.k / 64 - (nchunks - 1) * spc : spc;  // steps of the last chunk
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int units = g.n / kStreamUnit;
  const int unit_raw = nb * (kNarrow ? waves : kGemmWaves) + wave;
  const bool active = unit_raw < units;  // a partial column block leaves waves without columns
  const int unit = active ? unit_raw : units - 1;

  const uint8_t* asrc[kLoads];
  auto a_sources = [&]() {  // (reads the row table: after before_a, which may fill it)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = Chunk::row(i, lane, wave);
      asrc[i] = a_row_ptr<kGather>(g, rs, row0 + (r < mrows ? r : 0)) + Chunk::src(i, lane, wave, kc) * 16;
    }
  };
  if constexpr (!kEarly) a_sources();
  int4 astage[kLoads];
  auto load_chunk = [&](int chunk) {
    if constexpr (kAResident) return;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) astage[i] = ld16(asrc[i] + (kTail ? min(chunk * kc, g.k - kc) : static_cast<int64_t>(chunk) * kc));
  };
  auto store_chunk = [&](int chunk) {
    if constexpr (kAResident) return;
    uint8_t* dst = smem + (chunk & 1) * Chunk::kBytes;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      *reinterpret_cast<int4*>(dst + Chunk::row(i, lane, wave) * Chunk::kMaxK + Chunk::pos(i, lane) * 16) = astage[i];
  };
  if constexpr (kNarrow) {
    if (__builtin_amdgcn_readfirstlane(wave) >= waves) {  // no columns: this wave's share of A, in step with the others' barriers
      if constexpr (kEarly) {
        before_a();
        if constexpr (!kAResident) a_sources();
      }
      const TileScaleRegs tsr = load_tile_scales<kGather, kSwiglu>(g, rs, e, row0, kAResident ? 0 : mrows, 0);
      load_chunk(0);
      store_chunk(0);
      publish_tile_scales(tt, tsr, kAResident ? 0 : mrows);
      lds_barrier();
      for (int c = 0; c + 1 < nchunks; ++c) {
        load_chunk(c + 1);
        store_chunk(c + 1);
        lds_barrier();
      }
      return;
    }
  }
  // operand reads: lane l is row l%32 (+32 mt), k-bytes [64j + 32*(l/32), +32) of chunk step j
  const uint8_t* sbase = smem + (lane & 31) * Chunk::kMaxK;
  const int hk = lane >> 5;
  int pc[2][2];  // swizzled byte offset of piece 4v + 2hk + h within its 128-byte group
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int h = 0; h < 2; ++h) pc[v][h] = (((4 * v + 2 * hk + h) ^ lane) & 7) << 4;

  const uint8_t* bp[2];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int n = weight_row<kSwiglu>(g, unit, kStreamUnit, ct * 32 + (lane & 31));
    bp[ct] = g.b + (static_cast<int64_t>(e) * (g.n / 16) + (n >> 4)) * (static_cast<int64_t>(g.k) * 16) +
             (n & 15) * 16 + hk * 512;
  }
  int4 br[D][2][2];  // [ring slot][column tile][16-byte half]
  auto issue = [&](int d, int s) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const uint8_t* p = bp[ct] + static_cast<int64_t>(s) * 1024;
      br[d][ct][0] = ld16_stream(p);
      br[d][ct][1] = ld16_stream(p + 256);
    }
  };
  v16f acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mt][ct][v] = 0.0f;
  // step j of chunk c (j & 1 is a compile-time constant in the unrolled loops below)
  auto compute = [&](int d, int c, int j) {
    const v8i b0 = make_v8i(br[d][0][0], br[d][0][1]);
    const v8i b1 = make_v8i(br[d][1][0], br[d][1][1]);
    const uint8_t* base = sbase + (c & 1) * Chunk::kBytes + (j >> 1) * 128;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint8_t* rb = base + mt * 32 * Chunk::kMaxK;
      const v8i a = make_v8i(*reinterpret_cast<const int4*>(rb + pc[d & 1][0]),
                             *reinterpret_cast<const int4*>(rb + pc[d & 1][1]));
      acc[mt][0] = mfma_fp8(a, b0, acc[mt][0]);
      acc[mt][1] = mfma_fp8(a, b1, acc[mt][1]);
    }
  };
  static_assert(D % 2 == 0, "ring slot d holds steps of d's parity");

  if constexpr (kEarly) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      issue(d, d);
      __builtin_amdgcn_sched_barrier(0);
    }
    before_a();
    if constexpr (!kAResident) a_sources();
  }
  // a resident A's hook also leaves the rows' scales in tt.xs
  const TileScaleRegs tsr = load_tile_scales<kGather, kSwiglu>(g, rs, e, row0, kAResident ? 0 : mrows, unit);
  load_chunk(0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!kEarly) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      issue(d, d);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  store_chunk(0);
  publish_tile_scales(tt, tsr, kAResident ? 0 : mrows);
  lds_barrier();
  for (int c = 0; c + 1 < nchunks; ++c) {
    load_chunk(c + 1);
    __builtin_amdgcn_sched_barrier(0);
    for (int j = 0; j < spc; j += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(d, c, j + d);
        issue(d, c * spc + j + d + D);
        __builtin_amdgcn_sched_barrier(0);
        if (!kNarrow) step_barrier();
      }
    }
    store_chunk(c + 1);  // its buffer was last read in chunk c - 1, before the last barrier
    lds_barrier();
  }
  {
    const int c = nchunks - 1, j0 = spc - last_spc;
    for (int j = 0; j + D < last_spc; j += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(d, c, j0 + j + d);
        issue(d, c * spc + j + d + D);
        __builtin_amdgcn_sched_barrier(0);
        if (!kNarrow) step_barrier();
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) compute(d, c, spc - D + d);
  }

  if (!active) return;
  store_tile<kSwiglu, MT, kPmax, kCoherent>(g, acc, row0, mrows, unit, tt, 0);
}

// ------------------------------------------------------------------ TILE engine
// One 256 x 256 output tile (expert e, 256-column block nb, rows [row0, row0 + mrows)), K in
// BK = 128 stages through double-buffered LDS: the next stage's global loads go out into
// registers before the MFMAs of the current one and are written to the other LDS stage after
// them (one barrier per stage). A stage holds A as 256 rows of 128 bytes, 16-byte piece p of
// row r at piece p ^ (r % 8) (loaded as whole lines: 8 lanes per row), then B in Marlin's own
// blocks (16 row-tiles x 8 k-blocks x 256 bytes: each row-tile's stage is 2 KB contiguous in
// the weight, copied as is). A 32x32x64 operand is two 16-byte LDS reads per lane; 16 lanes
// read 256 contiguous bytes of B, and 8 lanes read 8 distinct 16-byte bank groups of A.
template <bool kGather, bool kSwiglu>
__device__ void tile_tile(const GemmArgs& g, const RowSrc& rs, int e, int row0, int mrows, int nb,
                          uint8_t* smem, TileTables& tt) {
  constexpr int BK = kTileBK;
  constexpr int TM = kTileBM / kTileWM / 32, TN = kTileBN / kTileWN / 32;  // 4 x 2
  constexpr int kALoads = kTileBM * BK / 16 / kGemmThreads;  // 4
  constexpr int kBLoads = kTileBN * BK / 16 / kGemmThreads;  // 4
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int wm = wave / kTileWN, wn = wave % kTileWN;
  const int k_steps = g.k / BK;
  const int units = g.n / kStreamUnit;            // 64-column units of the output
  const int unit = nb * kTileWN + wn;             // this wave's unit
  const int row_tiles = g.n / 16;                 // weight row-tiles of the expert

  // A: load i covers rows i*64 + tid/8, piece tid % 8 (whole 128-byte row lines); stored at
  // piece p ^ ((r / 2) % 8), so 16 consecutive rows at one k hit 16 distinct bank groups
  const uint8_t* a_src[kALoads];
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    const int r = i * (kGemmThreads / 8) + (tid >> 3);
    a_src[i] = a_row_ptr<kGather>(g, rs, row0 + (r < mrows ? r : 0)) + (tid & 7) * 16;
  }
  const int a_key = (tid >> 4) & 7;  // (r / 2) % 8 of every A row this thread stores
  const int a_dst0 = (tid >> 3) * BK + (((tid & 7) ^ a_key) << 4);  // + i * 64 * BK
  // B: load i covers byte q = (i*512 + tid)*16 of the stage's 16 row-tiles x 2 KB
  const uint8_t* b_src[kBLoads];
#pragma unroll
  for (int i = 0; i < kBLoads; ++i) {
    const int q = (i * kGemmThreads + tid) * 16;
    const int rt = q >> 11;  // 2 KB per row-tile per stage
    int n = weight_row<kSwiglu>(g, nb, kTileBN, rt * 16);
    if ((n >> 4) >= row_tiles) n = 0;  // a partial column block: any valid row-tile
    b_src[i] = g.b + (static_cast<int64_t>(e) * row_tiles + (n >> 4)) * (static_cast<int64_t>(g.k) * 16) +
               (q & 2047);
  }
  int4 ra[kALoads], rb[kBLoads];
  auto load_stage = [&](int kt) {
#pragma unroll
    for (int i = 0; i < kALoads; ++i) ra[i] = ld16(a_src[i] + kt * BK);
#pragma unroll
    for (int i = 0; i < kBLoads; ++i) rb[i] = ld16(b_src[i] + static_cast<int64_t>(kt) * BK * 16);
  };
  auto store_stage = [&](int buf) {
    uint8_t* sa = smem + buf * kTileStage;
    uint8_t* sb = sa + kTileBM * BK;
#pragma unroll
    for (int i = 0; i < kALoads; ++i)
      *reinterpret_cast<int4*>(sa + a_dst0 + i * (kGemmThreads / 8) * BK) = ra[i];
#pragma unroll
    for (int i = 0; i < kBLoads; ++i) *reinterpret_cast<int4*>(sb + (i * kGemmThreads + tid) * 16) = rb[i];
  };

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // B column of the wave's column tile tn: without SwiGLU wn*64 + tn*32; with SwiGLU the
  // gate columns (tn = 0) at wn*32 and the matching up columns (tn = 1) at 128 + wn*32.
  auto b_col = [&](int tn) { return kSwiglu ? tn * (kTileBN / 2) + wn * 32 : wn * 64 + tn * 32; };
  const int hk = lane >> 5;
  const int rkey = ((lane & 31) >> 1) & 7;  // (r / 2) % 8 of this lane's A rows
  // Operands are read one MFMA group ahead (double-buffered registers), so the LDS latency of
  // the next A (or the next k-step's B) overlaps the MFMAs of the current one.
  auto read_b = [&](const uint8_t* sb, int ks, v8i (&bv)[TN]) {
    const int p0 = ks * 4 + hk * 2;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int c = b_col(tn) + (lane & 31);
      const uint8_t* bc = sb + (c >> 4) * (BK * 16) + p0 * 256 + (c & 15) * 16;
      bv[tn] = make_v8i(*reinterpret_cast<const int4*>(bc), *reinterpret_cast<const int4*>(bc + 256));
    }
  };
  auto read_a = [&](const uint8_t* sa, int ks, int tm) {
    const int p0 = ks * 4 + hk * 2;
    const uint8_t* ar = sa + (wm * (TM * 32) + tm * 32 + (lane & 31)) * BK;
    return make_v8i(*reinterpret_cast<const int4*>(ar + ((p0 ^ rkey) << 4)),
                    *reinterpret_cast<const int4*>(ar + (((p0 + 1) ^ rkey) << 4)));
  };
  auto compute_stage = [&](int buf) {
    const uint8_t* sa = smem + buf * kTileStage;
    const uint8_t* sb = sa + kTileBM * BK;
    v8i bv[2][TN];
    read_b(sb, 0, bv[0]);
    v8i a_cur = read_a(sa, 0, 0);
#pragma unroll
    for (int ks = 0; ks < BK / 64; ++ks) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        v8i a_next;
        if (tm + 1 < TM) a_next = read_a(sa, ks, tm + 1);
        else if (ks + 1 < BK / 64) {
          read_b(sb, ks + 1, bv[(ks + 1) & 1]);
          a_next = read_a(sa, ks + 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the MFMAs below
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = mfma_fp8(a_cur, bv[ks & 1][tn], acc[tm][tn]);
        __builtin_amdgcn_sched_barrier(0);
        a_cur = a_next;
      }
    }
  };

  // a partial column block leaves waves without columns: their scales come from any valid unit
  const TileScaleRegs tsr =
      load_tile_scales<kGather, kSwiglu>(g, rs, e, row0, mrows, unit < units ? unit : units - 1);
  load_stage(0);
  store_stage(0);
  publish_tile_scales(tt, tsr, mrows);
  __syncthreads();
  for (int kt = 0; kt < k_steps; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < k_steps) load_stage(kt + 1);
    compute_stage(cur);
    if (kt + 1 < k_steps) store_stage(cur ^ 1);
    __syncthreads();
  }
  if (unit >= units) return;
  static_assert(TN == 2 && TM == 4, "a wave's tile is 128 rows x 64 columns");
  const int wrow = row0 + wm * (TM * 32);
  const int wrows = mrows - wm * (TM * 32);
  store_tile<kSwiglu, 2>(g, *reinterpret_cast<const v16f(*)[2][2]>(&acc[0]), wrow, wrows, unit, tt,
                         wm * (TM * 32));
  store_tile<kSwiglu, 2>(g, *reinterpret_cast<const v16f(*)[2][2]>(&acc[2]), wrow + 64, wrows - 64,
                         unit, tt, wm * (TM * 32) + 64);
}

// ------------------------------------------------------------------ WIDE engine
// The TILE engine's 256 x 256 tile for a 4-wave workgroup (one wave per SIMD: 512 registers a
// lane, the 256 accumulators in AGPRs), used when every expert has many rows. Wave w owns the
// 64-column unit nb*4 + w over all 256 rows (16 x 4 MFMA tiles), so each weight column is read
// by one wave only: B goes straight from global memory into MFMA operand registers (Marlin
// gives each lane 16 contiguous k-bytes of a weight row), in a register ring of three 128-k stages,
// and never touches LDS. A goes through LDS in BK = 128 stages: 256 rows of 128 bytes,
// 16-byte piece p of row r at piece p ^ ((r / 2) % 8) (16 consecutive rows at one k hit 16
// distinct 16-byte bank groups), three stages deep, so the first A operand of a stage is read
// before the barrier that ends the previous one and the MFMA pipe does not drain there.
// Tiles are independent (prologue, stages, epilogue): a software pipeline across the
// tiles of a workgroup needed the next tile's offsets live through the stage loop and the
// compiler spilled (measured slower).
//
// The MFMA is 16x16x128. At these sizes the chip is power-bound, and it takes less power for a FLOP
// than 32x32x64: register-only loops over random e4m3 values sustain 4.43 against 4.05 PFLOP/s (over
// zeros 4.97 and 4.96). A layer of 24.7K rows (4096 x 4096, 4096 x 2048) goes from 703 to 689 us, of 49K
// Zipf rows from 1268 to 1256, of 196K rows from 4845 to 4822: more cycles at a higher clock (counters
// at 196K rows: GEMM1 5.5 M at 1.94 GHz, with 32x32x64 4.9 M at 1.75). It adds 128 products a step where the
// 8-wave engines' MFMA adds 64, so a sum can round differently in its last fp32 bit: about one bf16
// partial value in 10^8 is another than theirs. A first version with a two-stage ring (one burst of
// loads a stage) was 1-3% slower than 32x32x64. Where the cycles are, by timing copies at 196K
// rows: GEMM1 5.65 M, without A's and B's loads 4.5 M, without the LDS reads too 4.4 M (prologues and
// epilogues then are 1.25 M of it), 3.15 M of MFMA.
//
// Two shapes (BM = rows of a full tile): BM = 256 with one workgroup per CU (512 registers a
// lane), and BM = 128 with two workgroups per CU (256 registers a lane, 128 AGPR accumulators):
// then each SIMD runs two waves of different tiles, and one tile's prologue and epilogue overlap
// the other's MFMAs. The A operand look-ahead is shallower at BM = 128 (the
// other wave covers the latency).
constexpr int kWideThreads = 256, kWideWaves = 4;
constexpr int kWideBK = 128;
constexpr int kWideBufs = 3;
constexpr int kWideMinRowsPerExpert = kTileBM;  // average routed rows that select it

template <int BM>
struct WideShape {
  static_assert(BM == 256 || BM == 128, "full tile of 256 or 128 rows");
  static constexpr int kStage = BM * kWideBK;  // bytes of one A stage
  // after the A ring, the tile's tables: BM row scales, the 256 weight-row scales (f32), then
  // (GEMM2) BM row addresses (u64)
  static constexpr int kTables = kWideBufs * kStage;
  static constexpr int kColScales = BM * 4;
  static constexpr int kAddrs = kColScales + kWideWaves * kStreamUnit * 4;
  static constexpr int kSmemBytes = kTables + kAddrs + BM * 8;
  static constexpr int kWavesPerSimd = BM == 256 ? 1 : 2;
  static constexpr int kFullTM = BM / 16;
  // the epilogue stages each wave's 64 output rows (8 KB) in the A ring's first bytes
  static_assert(kWideWaves * 8192 <= kTables, "epilogue staging fits the A ring");
};

// Epilogue of a WIDE tile. The MFMAs run transposed (weights as the first operand), so lane
// l holds token row tm*16 + l%16 and, per 16-column tile tn, the 4 consecutive columns 4*(l/16) + v.
// The row scale is then one value per lane and row
// tile, the column scales one 16-byte LDS read per column tile (both from the tile's scale
// table), and every 4 results become one 8-byte bf16 write into the wave's 8 KB slice of a
// free 32 KB A buffer (64 rows x 128 bytes, 16-byte piece p of row r at p ^ ((r / 2) % 8):
// conflict-free both ways); each pass of 64 rows then leaves as whole 16-byte pieces, 8 rows
// per store instruction.
// GEMM2 writes the bf16 partials (-0 as +0) to the row addresses of the tile's table: its part
// row, or for a row whose token has no other routed slot its y row (row_dest).
template <int BM, int TM>
__device__ __forceinline__ void store_wide(const GemmArgs& g, const v4f (&acc)[TM][4], int row0,
                                           int mrows, int unit, uint8_t* stage,
                                           const uint8_t* table) {
  using W = WideShape<BM>;
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1);
  const int rl = lane & 15, q = lane >> 4;
  const float* s_xs = reinterpret_cast<const float*>(table);
  const float* s_bs = reinterpret_cast<const float*>(table + W::kColScales) + (tid / kWave) * kStreamUnit;
  const uint64_t* s_addr = reinterpret_cast<const uint64_t*>(table + W::kAddrs);
  float4 bs[4];
#pragma unroll
  for (int tn = 0; tn < 4; ++tn) bs[tn] = *reinterpret_cast<const float4*>(s_bs + tn * 16 + q * 4);
  uint8_t* wlds = stage + (tid / kWave) * 8192;
  const int piece = lane & 7;
  const int col = unit * 64 + piece * 8;
#pragma unroll
  for (int pass = 0; pass < (TM + 3) / 4; ++pass) {
#pragma unroll
    for (int t4 = 0; t4 < (TM < 4 ? TM : 4); ++t4) {  // (TM = 2: rows 32-63 unused)
      const int tm = pass * 4 + t4;
      const float xs = s_xs[tm * 16 + rl];
      const int r = t4 * 16 + rl;  // row within the pass
      const int rkey = (r >> 1) & 7;
#pragma unroll
      for (int tn = 0; tn < 4; ++tn) {
        const float4 ws = bs[tn];
        // the scale product as fma(., ., +0), the same rounding, but a zero is +0 (the
        // combine's sum from +0 writes +0 too, so a y row written here matches it bitwise)
        auto scaled = [&](float a, float w) { return __builtin_fmaf(a * xs, w, 0.0f); };
        const uint32_t lo = pack_bf16x2(scaled(acc[tm][tn][0], ws.x), scaled(acc[tm][tn][1], ws.y));
        const uint32_t hi = pack_bf16x2(scaled(acc[tm][tn][2], ws.z), scaled(acc[tm][tn][3], ws.w));
        // columns 16tn + 4q .. +4 -> bytes 32tn + 8q: piece 2tn + q/2, half q%2
        const int pc = (2 * tn + (q >> 1)) ^ rkey;
        *reinterpret_cast<uint2*>(wlds + r * 128 + pc * 16 + (q & 1) * 8) = make_uint2(lo, hi);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's LDS writes before its reads
    int4 val[8];
    uint64_t base[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rr = i * 8 + (lane >> 3);
      val[i] = *reinterpret_cast<const int4*>(wlds + rr * 128 + ((piece ^ ((rr >> 1) & 7)) << 4));
      base[i] = s_addr[pass * 64 + rr];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int grow = pass * 64 + i * 8 + (lane >> 3);
      // the row's address from the table (its part row or its token's y row); a global (not
      // flat) store: a flat one would also hold up the LDS counter. Nontemporal: the rows are
      // read once, by the combine (c3 -25 us)
      const i32x4 v = {val[i].x, val[i].y, val[i].z, val[i].w};
      if (grow < mrows)
        __builtin_nontemporal_store(v, (__attribute__((address_space(1))) i32x4*)(base[i] + col * 2));
    }
    // the next pass's LDS writes follow these reads in the wave's own (in-order) LDS queue
  }
}

// Epilogue of a WIDE GEMM1 tile with the SwiGLU: the wave's unit holds the gate channels
// unit*32 + c (column tiles 0, 1) and the up channels of the same c (column tiles 2, 3), so lane l
// has, for token row tm*16 + l%16, two runs of 4 channels 16tn + 4*(l/16) .. + 4 of both. Per channel:
// g = bf16(acc_g * x_scale * w_scale_g) and u = bf16(acc_u * x_scale * w_scale_u) (the staged
// K1 output h, rounded like its stores), then y = SwiGLU(g, u) x route weight (the K2 formula,
// with the activation clamp when kClamp) and y rounded to bf16: bf16 y [rows, I] for the
// requant, half of h's bytes. Each 4-channel run is one 8-byte write into the wave's 4 KB LDS
// slice (64 rows x 64 bytes, 16-byte piece p of row r at p ^ ((r / 4) % 4)); a pass of 64 rows
// leaves as 16-byte pieces, 16 rows per store instruction.
template <bool kClamp, int BM, int TM>
__device__ __forceinline__ void store_wide_swiglu(const GemmArgs& g, const v4f (&acc)[TM][4], int row0,
                                                  int mrows, int unit, uint8_t* stage,
                                                  const uint8_t* table) {
  using W = WideShape<BM>;
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1);
  const int rl = lane & 15, q = lane >> 4;
  const float* s_xs = reinterpret_cast<const float*>(table);
  const float* s_rw = reinterpret_cast<const float*>(table + W::kAddrs);  // route weights
  const float* s_bs = reinterpret_cast<const float*>(table + W::kColScales) + (tid / kWave) * kStreamUnit;
  float4 bs[4];
#pragma unroll
  for (int tn = 0; tn < 4; ++tn) bs[tn] = *reinterpret_cast<const float4*>(s_bs + tn * 16 + q * 4);
  uint8_t* wlds = stage + (tid / kWave) * 4096;
  const int64_t ld = g.sw.inter;
  uint16_t* out = g.sw.y + static_cast<int64_t>(row0) * ld + unit * 32 + (lane & 3) * 8;
  const float cv = g.sw.clamp;
#pragma unroll
  for (int pass = 0; pass < (TM + 3) / 4; ++pass) {
#pragma unroll
    for (int t4 = 0; t4 < (TM < 4 ? TM : 4); ++t4) {  // (TM = 2: rows 32-63 unused)
      const int tm = pass * 4 + t4;
      const float xs = s_xs[tm * 16 + rl];
      const float rw = s_rw[tm * 16 + rl];
      const int r = t4 * 16 + rl;  // row within the pass
      const int rkey = (r >> 2) & 3;
#pragma unroll
      for (int tn = 0; tn < 2; ++tn) {
        const float4 wg = bs[tn], wu = bs[tn + 2];
        const v4f& ag = acc[tm][tn];
        const v4f& au = acc[tm][tn + 2];
        // gate and up of a channel rounded to bf16 together (one conversion for the pair)
        auto y_of = [&](float a_g, float a_u, float w_g, float w_u) {
          const uint32_t h = pack_bf16x2(a_g * xs * w_g, a_u * xs * w_u);
          return swiglu_weighted_c<kClamp>(__uint_as_float(h << 16), __uint_as_float(h & 0xffff0000u), rw, cv);
        };
        const float y0 = y_of(ag[0], au[0], wg.x, wu.x);
        const float y1 = y_of(ag[1], au[1], wg.y, wu.y);
        const float y2 = y_of(ag[2], au[2], wg.z, wu.z);
        const float y3 = y_of(ag[3], au[3], wg.w, wu.w);
        // channels 16tn + 4q .. +4 -> bytes 32tn + 8q of the row: piece 2tn + q/2, half q%2
        *reinterpret_cast<uint2*>(wlds + r * 64 + (((2 * tn + (q >> 1)) ^ rkey) << 4) + (q & 1) * 8) =
            make_uint2(pack_bf16x2(y0, y1), pack_bf16x2(y2, y3));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's LDS writes before its reads
    int4 val[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rr = i * 16 + (lane >> 2);
      val[i] = *reinterpret_cast<const int4*>(wlds + rr * 64 + (((lane & 3) ^ ((rr >> 2) & 3)) << 4));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int grow = pass * 64 + i * 16 + (lane >> 2);
      if (grow < mrows) *reinterpret_cast<int4*>(out + grow * ld) = val[i];
    }
    // the next pass's LDS writes follow these reads in the wave's own (in-order) LDS queue
  }
}

// TM row tiles of 16: BM/16 for a full tile; fewer (8, 4 or 2) for an expert's last tile of
// at most 128, 64 or 32 rows (a fraction of the MFMAs and A traffic for the row remainder).
//
// The stage loop is unrolled by 3, so that the LDS buffer, the B ring slot and the A registers of a
// stage are fixed. At stage kt every even group writes one piece of stage kt + 2's A to LDS and loads,
// into the same registers, the piece 1.5 stages further on; the odd groups of the first half
// load stage kt + 2's weights into the ring slot that stage kt - 1 has left. Spread out like that, the
// loads and LDS writes issue in the gaps between MFMAs instead of stalling the MFMA pipe in
// bursts, and every load has at least a stage and a half (~1.5 us) to arrive.
//
// kBig: the token matrix spans 4 GB or more (GEMM1's gathered rows need 64-bit offsets).
template <bool kGather, bool kSwiglu, int BM, int TM, bool kBig, typename Hook = NoHook>
__device__ void wide_tile(const GemmArgs& g, const RowSrc& rs, int e, int row0, int mrows, int nb,
                          uint8_t* smem, const Hook& before_epilogue = Hook{}) {
  using W = WideShape<BM>;
  using Offset = std::conditional_t<kBig, uint64_t, uint32_t>;
  constexpr int kWideStage = W::kStage;
  constexpr int kWideTables = W::kTables;
  static_assert(TM <= W::kFullTM && TM >= 2, "a tile of at most BM rows");
  constexpr int TN = kStreamUnit / 16;                            // 4
  constexpr int kALoads = TM * 16 * kWideBK / 16 / kWideThreads;  // TM / 2
  constexpr int kRowsPerLoad = kWideThreads / (kWideBK / 16);     // 32
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int stages = g.k / kWideBK;
  const int units = g.n / kStreamUnit;
  const int unit_raw = nb * kWideWaves + wave;
  const bool active = unit_raw < units;
  const int unit = active ? unit_raw : units - 1;  // a partial column block: any valid columns
  const int q = lane >> 4;

  // A: load i covers row i*32 + tid/8, piece tid % 8 (rows past mrows read row 0). GEMM1
  // (gather): the row scales for the epilogue's table are loaded by the same threads, from the
  // same tokens (the eight threads of a row read one word and write one LDS entry with the same
  // value), all the tokens first and then all the scales, with no branch between them, ahead of
  // the stages' loads, so that every wait the compiler places in the prologue is exact (a scale
  // chain of its own, token -> scale, had been sunk behind all the stage loads and made the
  // prologue wait for every one of them). GEMM2 loads one row scale a thread (no chain).
  const uint8_t* const a_base = kGather ? g.a : g.a + static_cast<int64_t>(row0) * g.lda;
  Offset a_off[kALoads];
  float a_rs[kALoads];
  int a_row[kALoads];
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    const int r = i * kRowsPerLoad + (tid >> 3);
    const int row = r < mrows ? r : 0;
    a_row[i] = kGather ? rs.token(row0 + row) : row;
  }
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    a_off[i] = static_cast<Offset>(a_row[i]) * static_cast<Offset>(g.lda) + (tid & 7) * 16;
    a_rs[i] = kGather ? g.a_scale[a_row[i]] : 0.0f;
  }
  const float pre_xs = kGather ? 0.0f : g.a_scale[row0 + min(tid, mrows - 1)];
  const int a_dst0 = (tid >> 3) * kWideBK + (((tid & 7) ^ ((tid >> 4) & 7)) << 4);
  auto fetch_a = [&](int i, int kt) { return ld16(a_base + kt * kWideBK + a_off[i]); };
  // piece i of stage kt in buffer `buf` (kt % 3)
  auto put_a = [&](int buf, int i, const int4& v) {
    *reinterpret_cast<int4*>(smem + buf * kWideStage + a_dst0 + i * kRowsPerLoad * kWideBK) = v;
  };
  // Pieces in flight: piece i of stage kt in slot (kt * kALoads + i) % kSlots, the same for kt and
  // kt + 3. kDelay pieces lie between a slot's LDS write and its next load: 1.5 stages (TM = 2: 2).
  constexpr int kDelay = TM == 2 ? 2 : kALoads + kALoads / 2;
  constexpr int kSlots = TM == 2 ? 3 : kDelay;
  static_assert(3 * kALoads % kSlots == 0, "slots repeat with the unrolled stages");
  int4 ra[kSlots];
  // B: column tile tn (16 columns) of the wave's unit, stage s at + s * 2048: lane l has column l % 16
  // and the 16-byte k-blocks l/16 and l/16 + 4 of the stage's eight (A's operands the same, so the
  // order of k inside the MFMA is the caller's to choose: a load is 1 KB contiguous)
  const uint8_t* bp[TN];
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
    const int n = weight_row<kSwiglu>(g, unit, kStreamUnit, tn * 16);
    bp[tn] = g.b + (static_cast<int64_t>(e) * (g.n / 16) + (n >> 4)) * (static_cast<int64_t>(g.k) * 16);
  }
  int4 br[3][TN][2];
  const uint32_t b_off = lane * 16;
  auto load_b = [&](int slot, int j, int s) {  // half j % 2 of tile j / 2
    br[slot][j / 2][j % 2] = ld16(bp[j / 2] + static_cast<int64_t>(s) * 2048 + (j % 2) * 1024 + b_off);
  };

  v4f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.0f;

  const int rkey = ((lane & 15) >> 1) & 7;
  const uint8_t* const a_read = smem + (lane & 15) * kWideBK + ((q ^ rkey) << 4);
  const uint8_t* const a_read4 = smem + (lane & 15) * kWideBK + (((q ^ rkey) << 4) ^ 64);
  auto read_a = [&](int buf, int tm) {
    const int at = buf * kWideStage + tm * 16 * kWideBK;
    return make_v8i(*reinterpret_cast<const int4*>(a_read + at), *reinterpret_cast<const int4*>(a_read4 + at));
  };
  // A stage = 16 MFMA groups (16 row tiles, 4 MFMAs each). The A operand of group
  // g + 3 is read while group g's MFMAs run (ring of 4 operands; the last groups read the next
  // stage's first operands, whose buffer is complete since the previous barrier), which
  // covers the LDS latency with one wave per SIMD. Order pinned by sched_barrier.
  constexpr int kGroups = TM;
  // one wave a SIMD: read 3 groups ahead; two (BM = 128): 1; TM = 2 has two groups a stage
  constexpr int kAhead = W::kWavesPerSimd == 1 ? (kGroups >= 4 ? 3 : kGroups - 1) : 1;
  static_assert(kGroups % (kAhead + 1) == 0, "operand ring index must repeat per stage");
  v8i abuf[kAhead + 1];
  const int last_stage = stages - 1;
  constexpr int kBGroups = (TM < 8 ? TM : 8) / 2;  // odd groups that load weights
  // stage kt; ph = kt % 3 (a constant)
  auto stage = [&](int kt, int ph) {
#pragma unroll
    for (int gi = 0; gi < kGroups; ++gi) {
      const int ahead = gi + kAhead;
      abuf[ahead % (kAhead + 1)] = read_a((ph + ahead / kGroups) % 3, ahead % kGroups);
      if (gi % 2 == 0) {
        const int i = gi / 2, n = (ph + 2) * kALoads + i;
        put_a((ph + 2) % 3, i, ra[n % kSlots]);
        ra[(n + kDelay) % kSlots] = fetch_a((i + kDelay) % kALoads, min(kt + 2 + (i + kDelay) / kALoads, last_stage));
      } else if (gi / 2 < kBGroups) {
#pragma unroll
        for (int j = gi / 2 * (2 * TN / kBGroups); j < (gi / 2 + 1) * (2 * TN / kBGroups); ++j)
          load_b((ph + 2) % 3, j, min(kt + 2, last_stage));
      }
      __builtin_amdgcn_sched_barrier(0);
      const v8i b[TN] = {make_v8i(br[ph][0][0], br[ph][0][1]), make_v8i(br[ph][1][0], br[ph][1][1]),
                         make_v8i(br[ph][2][0], br[ph][2][1]), make_v8i(br[ph][3][0], br[ph][3][1])};
      mfma_group(b, abuf[gi % (kAhead + 1)], acc[gi]);  // transposed tile
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  };

  // prologue: the epilogue's scales (the row scales loaded with the row tokens above; thread
  // t: the weight-row scale of its wave's column lane), A stages 0 and 1 into LDS, the pieces of the
  // next 1.5 stages into their registers, B stages 0 and 1, the first operands; the loads
  // go out together (stages 0 and 1 through registers of the prologue's own).
  // GEMM2: row tid's output address (its part row, or its token's y row when the token has no
  // other routed slot and direct rows are on); the switch and the row table load side by side.
  // Rows past mrows take the last row's (never stored).
  int pre_dest = -1, pre_on = 0;
  if (!kSwiglu && g.y_direct != nullptr) {
    pre_on = *g.direct_flag;
    pre_dest = g.row_dest[row0 + min(tid, mrows - 1)];
  }
  // GEMM1: row tid's route weight (the SwiGLU epilogue's)
  const float pre_rw = kSwiglu ? g.sw.row_weight[row0 + min(tid, mrows - 1)] : 0.0f;
  const float pre_bs = g.b_scale[static_cast<int64_t>(e) * g.n + weight_row<kSwiglu>(g, unit, kStreamUnit, lane)];
  int4 ra0[2][kALoads];
#pragma unroll
  for (int i = 0; i < kALoads; ++i) ra0[0][i] = fetch_a(i, 0);
#pragma unroll
  for (int i = 0; i < kALoads; ++i) ra0[1][i] = fetch_a(i, min(1, last_stage));
#pragma unroll
  for (int j = 0; j < 2 * TN; ++j) load_b(0, j, 0);
#pragma unroll
  for (int n = 2 * kALoads; n < 2 * kALoads + kDelay; ++n)
    ra[n % kSlots] = fetch_a(n % kALoads, min(n / kALoads, last_stage));
#pragma unroll
  for (int j = 0; j < 2 * TN; ++j) load_b(1, j, min(1, last_stage));
#pragma unroll
  for (int i = 0; i < kALoads; ++i) put_a(0, i, ra0[0][i]);
#pragma unroll
  for (int i = 0; i < kALoads; ++i) put_a(1, i, ra0[1][i]);
  if constexpr (kGather) {
#pragma unroll
    for (int i = 0; i < kALoads; ++i) reinterpret_cast<float*>(smem + kWideTables)[i * kRowsPerLoad + (tid >> 3)] = a_rs[i];
  } else if (tid < BM) {
    reinterpret_cast<float*>(smem + kWideTables)[tid] = pre_xs;
  }
  reinterpret_cast<float*>(smem + kWideTables + W::kColScales)[tid] = pre_bs;
  if (kSwiglu && (BM == kWideThreads || tid < BM)) reinterpret_cast<float*>(smem + kWideTables + W::kAddrs)[tid] = pre_rw;
  if (!kSwiglu && (BM == kWideThreads || tid < BM)) {
    const int prow = row0 + min(tid, mrows - 1);
    reinterpret_cast<uint64_t*>(smem + kWideTables + W::kAddrs)[tid] =
        pre_on != 0 && pre_dest >= 0 ? reinterpret_cast<uint64_t>(g.y_direct + static_cast<int64_t>(pre_dest) * g.n)
                                     : reinterpret_cast<uint64_t>(g.c + static_cast<int64_t>(prow) * g.n);
  }
  lds_barrier();
#pragma unroll
  for (int gi = 0; gi < kAhead; ++gi) abuf[gi] = read_a(gi / kGroups, gi % kGroups);
  // every load is issued unconditionally (past the end it reloads the last stage), which keeps the
  // compiler's load counting exact
  int kt = 0;
  for (; kt + 3 <= stages; kt += 3) {
    stage(kt, 0);
    stage(kt + 1, 1);
    stage(kt + 2, 2);
  }
  if (kt < stages) stage(kt, 0);
  if (kt + 1 < stages) stage(kt + 1, 1);
  // every wave has passed its last LDS read of A (the barrier that ended the last stage)
  before_epilogue();
  mfma_settle(acc);
  if (!active) return;
  if constexpr (kSwiglu) {
    if (g.sw.has_clamp) store_wide_swiglu<true, BM, TM>(g, acc, row0, mrows, unit, smem, smem + kWideTables);
    else store_wide_swiglu<false, BM, TM>(g, acc, row0, mrows, unit, smem, smem + kWideTables);
  } else {
    store_wide<BM, TM>(g, acc, row0, mrows, unit, smem, smem + kWideTables);
  }
}

// ------------------------------------------------------------------ in-kernel routing
// For small task counts GEMM1 routes the tokens itself instead of a separate routing kernel:
// every workgroup counts all tasks with its 8 waves (LDS atomics into per-wave counts; integer
// sums, so order-free and deterministic), keeps each task's expert in an LDS byte table, turns
// the counts into per-wave bases and expert offsets, and plans the items. For an item it then
// ranks only its own expert's tasks (one ballot per 64 tasks from the LDS table, ascending
// task order as in the routing kernels) into an LDS row table of tokens and route weights.
// The workgroup holding column block 0 of a row range writes that range's routing outputs
// (row_token, row_weight, m_indices, output_index) for the later stages; workgroup 0 writes
// counts, offsets, meta, stats and the -1 of the invalid tasks.
constexpr int kFusedPasses = 16;  // 64-task passes per wave
constexpr int kFusedMaxTasks = kGemmWaves * kFusedPasses * kWave;
constexpr int kFusedMaxExperts = 255;  // expert ids in a byte, 255 = invalid task
constexpr int kFusedBatch = 16;        // passes whose loads are in flight together
constexpr int kRowTable = kTileBM;  // LDS row table: one TILE's 256 rows

__device__ __forceinline__ int fused_per_wave(int ntasks) {
  return (ntasks + kGemmWaves * kWave - 1) / (kGemmWaves * kWave) * kWave;
}

// Per-wave counts of all tasks into s_wcnt[wave][e] and each task's expert into s_ev;
// workgroup 0 also marks the invalid tasks.
__device__ void fused_count(const RouteArgs& a, int ntasks, int (*s_wcnt)[kMaxGemmExperts],
                            uint8_t* s_ev, float* s_task_w, bool publisher) {
  const int lane = lane_id();
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int per = fused_per_wave(ntasks);
  const int begin = wave * per;
  const int end = min(begin + per, ntasks);
  for (int b = begin; b < end; b += kFusedBatch * kWave) {
    int ev[kFusedBatch];
    float wv[kFusedBatch];
    wave_load<kFusedBatch>(a, b, end, ev, wv);
#pragma unroll
    for (int p = 0; p < kFusedBatch; ++p) {
      const int task = b + p * kWave + lane;
      if (task < end) {
        s_ev[task] = ev[p] < 0 ? 255 : static_cast<uint8_t>(ev[p]);
        s_task_w[task] = wv[p];
        if (ev[p] >= 0) atomicAdd(&s_wcnt[wave][ev[p]], 1);
        else if (publisher) a.output_index[task] = -1;
      }
    }
  }
}

// Rows [r_lo, r_lo + kRowTable) of expert e (cnt rows): tokens and route weights into the LDS
// row table; rows in [w_lo0, w_hi0) or [w_lo1, w_hi1) are this workgroup's to write out.
// Ends with the table complete (workgroup barrier).
__device__ void fused_rows(const RouteArgs& a, int ntasks, int e, int cnt, int off_e,
                           const int (*s_wcnt)[kMaxGemmExperts], const uint8_t* s_ev,
                           const float* s_task_w, int r_lo, int w_lo0, int w_hi0, int w_lo1,
                           int w_hi1, int* s_task, int* s_tok, float* s_rw) {
  const int lane = lane_id();
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int per = fused_per_wave(ntasks);
  const int begin = wave * per;
  const int end = min(begin + per, ntasks);
  int run = s_wcnt[wave][e];  // rank of the wave's first task of expert e
  for (int b = begin; b < end; b += kWave) {
    const int task = b + lane;
    const int ev = task < end ? s_ev[task] : 255;
    const uint64_t m = __ballot(ev == e);
    if (ev == e) {
      const int rank = run + __popcll(m & lanes_below());
      if (rank >= r_lo && rank < r_lo + kRowTable) {
        s_task[rank - r_lo] = task;
        s_tok[rank - r_lo] = task / a.topk;
      }
    }
    run += __popcll(m);
  }
  __syncthreads();
  const int n = min(kRowTable, cnt - r_lo);
  for (int t = opaque_tid(); t < n; t += kGemmThreads) {  // recomputed, not kept live across items
    const int task = s_task[t];
    const float w = s_task_w != nullptr ? s_task_w[task] : a.topk_w[task];
    s_rw[t] = w;
    const int rank = r_lo + t;
    if ((rank >= w_lo0 && rank < w_hi0) || (rank >= w_lo1 && rank < w_hi1)) {
      const int64_t row = static_cast<int64_t>(off_e) + rank;
      const int out = row < a.row_cap ? static_cast<int>(row) : -1;
      // device-coherent: the decode pipeline's combine reads it from other XCDs
      __hip_atomic_store(&a.output_index[task], out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (out >= 0) {
        a.row_token[out] = s_tok[t];
        if (a.row_weight != nullptr) a.row_weight[out] = w;
        if (a.m_indices != nullptr) a.m_indices[out] = e;
      }
    }
  }
  __syncthreads();
}

// Wave 0: the per-wave counts s_wcnt[w][e] -> per-wave bases (the wave's first rank of each
// expert), the expert totals s_count[e] and their exclusive scan s_off[0..E] (expert offsets).
// The LDS traffic of one wave stays in order, so a plan by the same wave can follow at once.
__device__ void fused_scan(int E, int (*s_wcnt)[kMaxGemmExperts], int* s_count, int* s_off) {
  const int lane = lane_id();
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += kWave) {
    const int e = e0 + lane;
    int run = 0;
    if (e < E) {
      for (int w = 0; w < kGemmWaves; ++w) {
        const int c = s_wcnt[w][e];
        s_wcnt[w][e] = run;
        run += c;
      }
      s_count[e] = run;
    }
    const int inc = wave_inclusive_sum(run);
    if (e < E) s_off[e] = carry + inc - run;
    carry += __shfl(inc, kWave - 1, kWave);
  }
  if (lane == 0) s_off[E] = carry;
}

// ------------------------------------------------------------------ persistent dispatcher
__device__ __forceinline__ int stream_blocks(const GemmArgs& g) {
  return (g.n / kStreamUnit + kGemmWaves - 1) / kGemmWaves;
}

// Wave 0 fills s_prefix[0..E] with the exclusive prefix of the workgroup work items of the
// experts and s_tile[e] with the expert's engine (1 = TILE), from the routed rows s_count[e].
// A STREAM item is one (128-row chunk, 512-column block), an expert's chunks of one column
// block next to each other; a TILE item is one 256 x 256 tile (tile_coords' order).
__device__ void plan_items(const GemmArgs& g, int* s_prefix, int* s_tile, const int* s_count,
                           bool all_tile = false, int tile_rows = kTileBM) {
  const int E = g.num_experts;
  const int lane = lane_id();
  const int stream_nb = stream_blocks(g);
  const int tile_nb = (g.n + kTileBN - 1) / kTileBN;
  if (threadIdx.x < kWave) {
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
      const int e = e0 + lane;
      int items = 0;
      if (e < E) {
        const int cnt = s_count[e];
        const bool tile = all_tile || g.engine == GemmEngine::kTile ||
                          (g.engine == GemmEngine::kAuto && cnt > kStreamAutoMaxRows);
        items = tile ? (cnt + tile_rows - 1) / tile_rows * tile_nb
                     : (cnt + kStreamItemRows - 1) / kStreamItemRows * stream_nb;
        s_tile[e] = tile;
      }
      const int inc = wave_inclusive_sum(items);
      if (e < E) s_prefix[e] = carry + inc - items;
      carry += __shfl(inc, kWave - 1, kWave);
    }
    if (lane == 0) s_prefix[E] = carry;
  }
}

// The expert owning item t: the last e with s_prefix[e] <= t (s_prefix is non-decreasing, so
// that is the count of such e, minus one). One LDS read and one ballot per 64 experts, the
// whole wave at once, instead of a chain of dependent reads.
__device__ __forceinline__ int expert_of_item(const int* s_prefix, int E, int t) {
  const int lane = lane_id();
  int below = 0;
  for (int e0 = 0; e0 < E; e0 += kWave) {
    const int e = e0 + lane;
    below += __popcll(__ballot(e < E && s_prefix[e] <= t));
  }
  return below - 1;
}

// The items of one workgroup. Workgroup b runs on XCD b % 8, so items are dealt to the XCDs
// in contiguous ranges and the workgroups of an XCD share its L2 for the same experts' rows and
// weights (when the grid is not a multiple of 8: one range, the whole grid). A range is dealt
// in rounds of `step` items (its workgroups); in round k the workgroup takes position
// (slot + k) % step. The rotation hands every workgroup every position in turn, so items of
// unequal cost that recur with a period dividing the step (an expert's short last row block)
// spread over all the workgroups instead of landing on the same few; a round is still the same
// set of consecutive items, and each round is a bijection, so every item runs exactly once.
struct ItemDeal {
  int begin, end, step, slot;
  __device__ __forceinline__ int rounds() const { return (end - begin + step - 1) / step; }
  __device__ __forceinline__ int item(int k) const { return begin + k * step + (slot + k) % step; }
};

__device__ __forceinline__ ItemDeal deal_items(int total) {
  const int nwg = static_cast<int>(gridDim.x);
  const int b = static_cast<int>(blockIdx.x);
  if (nwg % 8 != 0) return ItemDeal{0, total, nwg, b};
  const int xcd = b % 8;
  return ItemDeal{static_cast<int>(static_cast<int64_t>(total) * xcd / 8),
                  static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / 8), nwg / 8, b / 8};
}

// Dynamic dealing (WIDE kernel). The same XCD ranges, but only each workgroup's first item is
// fixed (position `slot` of its range); after that it claims the next item of its range from
// the range's counter (one device atomic a tile, issued when the tile starts and read when it
// ends, so its latency hides behind the tile), and when its range runs out, from the other
// XCDs' ranges in turn. Claims follow item order, so the tiles an XCD runs together stay
// neighbours (shared L2 traffic), while fast workgroups take more items than slow ones: tiles of
// unequal cost (an expert's short last row block) and a range that does not divide evenly no
// longer leave some workgroups with a whole extra tile. Every claim only moves a counter
// forward, so the loop ends; the last workgroup to finish resets the counters to zero.
struct Claims {
  int32_t* sched;  // [0..7] claim counters, [8] finished workgroups
  int total, nranges, home, step, slot;
  __device__ __forceinline__ int begin(int r) const { return static_cast<int>(static_cast<int64_t>(total) * r / nranges); }
  __device__ __forceinline__ int end(int r) const { return static_cast<int>(static_cast<int64_t>(total) * (r + 1) / nranges); }
  __device__ __forceinline__ int range(int ri) const { return (home + ri) % nranges; }
  // claimed index c of range r -> the item (the first `step` items are the fixed first items)
  __device__ __forceinline__ int item(int r, int c) const { return begin(r) + step + c; }
  // thread 0: the next item from range index ri on (advancing ri past exhausted ranges), or -1
  __device__ int claim_from(int& ri) const {
    for (; ri < nranges; ++ri) {
      const int r = range(ri);
      const int t = item(r, atomicAdd(&sched[r], 1));
      if (t < end(r)) return t;
    }
    return -1;
  }
};

__device__ __forceinline__ Claims make_claims(int32_t* sched, int total) {
  const int nwg = static_cast<int>(gridDim.x);
  const int b = static_cast<int>(blockIdx.x);
  const int nranges = nwg % 8 == 0 ? 8 : 1;
  return Claims{sched, total, nranges, nranges == 8 ? b % 8 : 0, nwg / nranges, nranges == 8 ? b / 8 : b};
}

// TILE item `local` of an expert with cnt rows -> (row block mt, column block nb): row blocks
// in groups of 4, columns inside a group, so that the consecutive items an XCD runs together
// form 4 x 8 tiles sharing A rows and B columns in its L2.
__device__ __forceinline__ void tile_coords(int local, int cnt, int tile_nb, int& mt, int& nb,
                                            int tile_rows = kTileBM) {
  const int mblocks = (cnt + tile_rows - 1) / tile_rows;
  const int group = local / (4 * tile_nb);
  const int in_group = local - group * 4 * tile_nb;
  const int rows_in_group = min(4, mblocks - group * 4);
  nb = in_group / rows_in_group;
  mt = group * 4 + (in_group - nb * rows_in_group);
}

// kTail (stream_tail): how the STREAM engine cuts K. Kernels of their own, so that a kernel's code (and its
// cold instruction fetches in the one-time prologue) holds one ring for each item height, and because
// the short last chunk costs the ring of 4 ten spilled registers (K = 3072 and 1024, 256 tokens on 32
// experts: 71 -> 76 us a layer).
//   kTailNone: chunks that divide K, rings of 4
//   kTail256: K a multiple of 256; chunks with a short last one and a ring of 2 up to 64 rows, chunks of 256
//     and a ring of 4 above
//   kTailAny: chunks with a short last one and a ring of 2
constexpr int kTailNone = 0, kTail256 = 1, kTailAny = 2;

// A dual launch's kernel that the routed rows do not select returns at once (GemmArgs).
__device__ __forceinline__ bool dual_skips(const GemmArgs& g, bool wide) {
  return g.dual_rows != nullptr && ((*g.dual_rows >= g.dual_min_rows) != wide);
}

template <bool kGather, bool kSwiglu, int kTail>
__global__ __launch_bounds__(kGemmThreads, 1) void grouped_gemm_kernel(GemmArgs g) {
  constexpr int kRing = kTail == kTailNone ? kStreamDepth : kTailDepth;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int s_prefix[kMaxGemmExperts + 1];
  __shared__ int s_tile[kMaxGemmExperts];
  __shared__ int s_count[kMaxGemmExperts];
  __shared__ int s_off[kMaxGemmExperts + 1];
  __shared__ int s_wcnt[kGemmWaves][kMaxGemmExperts];  // in-kernel routing: per-wave counts/bases
  __shared__ int s_tok[kRowTable];
  __shared__ float s_rw[kRowTable];
  __shared__ int s_task[kRowTable];
  __shared__ uint8_t s_ev[kFusedMaxTasks];  // in-kernel routing: expert of each task
  __shared__ TileTables s_tt;                // the current item's scales (epilogue)
  const int E = g.num_experts;
  const RouteArgs& ra = g.route;
  int ntasks = 0;
  bool fused = false;
  if (kSwiglu && g.route_in_kernel) {
    ntasks = effective_tokens(ra.runtime_tokens, ra.host_tokens) * ra.topk;
    fused = g.route_in_kernel == 1 || ntasks <= kFusedMaxTasks;
  }
  // a dual launch: this kernel runs when it routes the live tasks itself (then there are too
  // few rows for WIDE, and the routed-row count is not written yet), else when the routing's
  // row count does not select WIDE
  if (!fused && dual_skips(g, false)) return;
  if (fused) {
    {  // each wave clears its own count row: only that wave adds to it, so no barrier is needed
      const int wave = static_cast<int>(threadIdx.x) / kWave;
      for (int e = lane_id(); e < E; e += kWave) s_wcnt[wave][e] = 0;
    }
    // the route weights stay in the (still unused) dynamic LDS for the first item's row table
    fused_count(ra, ntasks, s_wcnt, s_ev, reinterpret_cast<float*>(smem), blockIdx.x == 0);
    __syncthreads();
    if (threadIdx.x < kWave) {
      fused_scan(E, s_wcnt, s_count, s_off);
      plan_items(g, s_prefix, s_tile, s_count);
    }
    __syncthreads();
    if (blockIdx.x == 0) {  // the routing kernel's outputs that the later stages read
      for (int e = threadIdx.x; e <= E; e += kGemmThreads) ra.offsets[e] = s_off[e];
      for (int e = threadIdx.x; e < E; e += kGemmThreads) {
        ra.counts[e] = s_count[e];
        if (ra.stats != nullptr) ra.stats[e] += s_count[e];
      }
      if (threadIdx.x == 0) {
        ra.meta[0] = s_off[E] < ra.row_cap ? s_off[E] : static_cast<int>(ra.row_cap);
        ra.meta[3] = 0;  // the call's status: no bounded wait on this path
      }
    }
  } else {
    for (int e = threadIdx.x; e <= E; e += kGemmThreads) {
      if (e < E) s_count[e] = g.counts[e];
      s_off[e] = g.offsets[e];
    }
    __syncthreads();
    plan_items(g, s_prefix, s_tile, s_count);
    __syncthreads();
  }
  const int total = s_prefix[E];
  const int tile_nb = (g.n + kTileBN - 1) / kTileBN;
  const ItemDeal deal = deal_items(total);
  // the route weights cached in LDS are valid until the first item's loads overwrite them
  const float* task_w = reinterpret_cast<const float*>(smem);
  bool first_item = true;
  for (int k = 0; k < deal.rounds(); ++k) {
    const int t = deal.item(k);
    if (t >= deal.end) continue;  // the last round's short tail (uniform in the workgroup)
    const float* item_task_w = first_item ? task_w : nullptr;
    first_item = false;
    const int e = expert_of_item(s_prefix, E, t);
    const int local = t - s_prefix[e];
    const int cnt = s_count[e];
    const int off_e = s_off[e];
    if (s_tile[e]) {
      int mt, nb;
      tile_coords(local, cnt, tile_nb, mt, nb);
      RowSrc rs{g.row_token, g.sw.row_weight, 0};
      if (fused) {
        const int r0 = mt * kTileBM;
        fused_rows(ra, ntasks, e, cnt, off_e, s_wcnt, s_ev, item_task_w, r0,
                   nb == 0 ? r0 : 0, nb == 0 ? r0 + kTileBM : 0, 0, 0, s_task, s_tok, s_rw);
        rs = RowSrc{s_tok, s_rw, off_e + r0};
      }
      tile_tile<kGather, kSwiglu>(g, rs, e, off_e + mt * kTileBM, min(kTileBM, cnt - mt * kTileBM),
                                  nb, smem, s_tt);
    } else {
      // An expert's row chunks of one column block (more than one only on the streaming
      // schedule) are neighbouring items, so they run in the same round on the same XCD and
      // read those weight columns from HBM once (through L2).
      const int nch = (cnt + kStreamItemRows - 1) / kStreamItemRows;
      const int nb = local / nch;
      const int mc = local - nb * nch;
      const int mrows = min(kStreamItemRows, cnt - mc * kStreamItemRows);
      const int row0 = off_e + mc * kStreamItemRows;
      RowSrc rs{g.row_token, g.sw.row_weight, 0};
      if (fused) {
        const int r0 = mc * kStreamItemRows;
        fused_rows(ra, ntasks, e, cnt, off_e, s_wcnt, s_ev, item_task_w, r0,
                   nb == 0 ? r0 : 0, nb == 0 ? r0 + kStreamItemRows : 0, 0, 0, s_task, s_tok, s_rw);
        rs = RowSrc{s_tok, s_rw, row0};
      }
      if (mrows > 64) {
        if constexpr (kTail != kTailAny)
          stream_tile<kGather, kSwiglu, 4, kStreamDepth, false, false, false, false, false, kALoads / 2>(g, rs, e, row0, mrows, nb, kAChunk4, smem, s_tt);
        else
          stream_tile<kGather, kSwiglu, 4, kTailDepth, false, false, false, false, false, kALoads, true>(g, rs, e, row0, mrows, nb, g.kc[2], smem, s_tt);
      } else if (mrows > 32) {
        stream_tile<kGather, kSwiglu, 2, kRing, false, false, false, false, false, kALoads, kTail != kTailNone>(g, rs, e, row0, mrows, nb, g.kc[1], smem, s_tt);
      } else {
        stream_tile<kGather, kSwiglu, 1, kRing, false, false, false, false, false, kALoads, kTail != kTailNone>(g, rs, e, row0, mrows, nb, g.kc[0], smem, s_tt);
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ decode pipeline
// GEMM1 (with the in-kernel routing), the requant and GEMM2 of the streaming engine in one
// launch, so that a group of rows goes on to GEMM2 as soon as its own GEMM1 items are done,
// instead of after the slowest XCD's last GEMM1 item, and without the requant's and GEMM2's
// launches and prologues.
//
// Work: an expert's rows are cut into groups, a GEMM1 item is a group and a column block (512
// columns, fewer when there are few groups: PipeShape), and a GEMM2 item a column block and the rows
// of a group or of half of one. All the GEMM1 items in expert order are dealt to the XCDs in equal
// contiguous ranges, and so are the GEMM2 items; the workgroups of an XCD -- found by the hardware XCD id, not
// by launch order -- claim their range of GEMM1 items, then of GEMM2 items, in order. A claim goes
// out one item ahead, so its latency hides behind an item. A workgroup whose range is all claimed
// takes items of the other XCDs' ranges.
//
// Hand-off: a GEMM1 item stores its bf16 SwiGLU rows and their block maxima device-coherent (sc1,
// through its XCD's L2), waits for them (vmcnt 0) and counts itself done for its group. A GEMM2
// item, of any XCD, issues its first weight steps, polls until its group's count is complete,
// invalidates its CU's L1 and requantizes the group's rows straight into its LDS A buffers (the
// requant kernel's arithmetic, so the same bits; the group's first GEMM2 item also writes act
// and amax out). It reads the rows through its own L2, which holds none of their lines: nothing in
// this launch reads a row's line before the row's group is complete (a row is whole lines:
// decode_pipeline_supported). The maxima, whose lines two groups can share, it reads device-coherent. A workgroup starts on GEMM2
// items only when every GEMM1 item is claimed, and a GEMM1 item waits on nothing, so every wait
// ends, also when some XCDs have no workgroups; a wait is also bounded (kPipeSpinLimit polls), and
// one that runs out is counted (the launch's last workgroup leaves the count in meta[3], the call's
// status) instead of hanging.
//
// Combine (PipeArgs::y set): a GEMM2 item stores its partial rows device-coherent (sc1: written
// through the XCD's L2, which other XCDs do not see), drains them and counts itself done for its
// expert. A workgroup out of items combines its share of the tokens, one wave a token: for each
// routed slot (the task's expert from the routing's LDS table) it waits until the expert's
// GEMM1 items are done (its rows' output_index entries are written, also device-coherent) and
// loads the row, then until the expert's GEMM2 items are done, and reads the partial rows with
// device-coherent loads. A workgroup starts to combine only when every GEMM2 item is claimed, so
// every wait ends. The workgroup that leaves last sets the counters back to zero.
__device__ __forceinline__ int hw_xcc_id() {
  int v;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
  return v & 0xf;
}

// This wave's outstanding memory operations (the stores a hand-off publishes) are complete.
__device__ __forceinline__ void vm_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Later loads of this CU miss its L1 (they read the XCD's L2, where the producer's stores are).
__device__ __forceinline__ void l1_invalidate() { asm volatile("buffer_inv sc0" ::: "memory"); }

// Thread-level poll (a vector atomic load: lane-divergent code) until *c >= target, at most
// `limit` polls (false: it ran out).
__device__ __forceinline__ bool wait_count(const int32_t* c, int target, int limit) {
  for (int i = 0; i < limit; ++i) {
    if (__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= target) return true;
    __builtin_amdgcn_s_sleep(2);
  }
  return false;
}

// One 16-byte piece at byte offset off of a buffer, device-coherent (sc1: an L2 line that another
// XCD wrote is not served stale).
__device__ __forceinline__ uint4 ld16_coherent(__amdgpu_buffer_rsrc_t r, int off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16 /* sc1 */);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// The combine of token t in the decode pipeline (one wave, kPipeCombineV * 512 columns at a time):
// the slot-ordered fp32 sum of its routed slots' partial rows from +0, bf16 RNE (the combine
// kernel's arithmetic, so the same bits); a token without routed slots gets zeros.
constexpr int kPipeCombineV = 8;  // 16-byte column groups per lane

__device__ void pipe_combine_token(const PipeArgs& p, int64_t t, const uint8_t* s_ev,
                                   const int* s_prefix1, const int* s_prefix2, int n1, int n2,
                                   const int32_t* done1, const int32_t* done2,
                                   __amdgpu_buffer_rsrc_t part) {
  constexpr int V = kPipeCombineV;
  const RouteArgs& ra = p.g1.route;
  const int lane = lane_id();
  const int hidden = p.g2.n;
  const int nvec = hidden >> 3;
  int row = -1;
  if (lane < ra.topk) {
    const int64_t task = t * ra.topk + lane;
    const int ev = s_ev[task];
    if (ev != 255) {
      bool ok = true;
      for (int grp = s_prefix1[ev]; grp < s_prefix1[ev + 1]; ++grp)
        ok = ok && wait_count(&done1[grp], n1, p.spin_limit);
      row = __hip_atomic_load(&ra.output_index[task], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ok = ok && wait_count(&done2[ev * kPipeDone2Stride], n2 * (s_prefix2[ev + 1] - s_prefix2[ev]),
                            p.spin_limit);
      if (!ok) atomicAdd(&p.pipe[kPipeFailAt], 1);
    }
  }
  const uint64_t routed = __ballot(row >= 0);
  uint4* yrow = reinterpret_cast<uint4*>(p.y + t * hidden);
  for (int v0 = 0; v0 < nvec; v0 += V * kWave) {
    float sum[V][8];
#pragma unroll
    for (int j = 0; j < V; ++j)
#pragma unroll
      for (int q = 0; q < 8; ++q) sum[j][q] = 0.0f;
    // the routed slots in ascending order, two at a time (their loads go out together)
    constexpr int kSlots = 2;
    for (uint64_t m = routed; m != 0;) {
      uint4 pv[kSlots][V];
      bool has[kSlots];
#pragma unroll
      for (int b = 0; b < kSlots; ++b) {
        has[b] = m != 0;  // wave-uniform (a ballot)
        const int s = has[b] ? __ffsll(static_cast<unsigned long long>(m)) - 1 : 0;
        m &= m - 1;
        const int r = __shfl(row, s, kWave);
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const int v = v0 + j * kWave + lane;
          pv[b][j] = has[b] && v < nvec ? ld16_coherent(part, (r * hidden + v * 8) * 2) : make_uint4(0, 0, 0, 0);
        }
      }
#pragma unroll
      for (int b = 0; b < kSlots; ++b) {
        if (!has[b]) break;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const uint32_t words[4] = {pv[b][j].x, pv[b][j].y, pv[b][j].z, pv[b][j].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            sum[j][2 * q] += bf16_to_f32(words[q] & 0xffff);
            sum[j][2 * q + 1] += bf16_to_f32(words[q] >> 16);
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int v = v0 + j * kWave + lane;
      if (v < nvec)
        yrow[v] = make_uint4(pack_bf16x2(sum[j][0], sum[j][1]), pack_bf16x2(sum[j][2], sum[j][3]),
                             pack_bf16x2(sum[j][4], sum[j][5]), pack_bf16x2(sum[j][6], sum[j][7]));
    }
  }
}

// The two kernels of the pipeline: for few tasks (kPipeSmallTasks) chunks of up to 32 rows and items
// of 2, 4 or 8 units, else chunks of up to 128 rows in GEMM1 and of 64 rows in GEMM2 (whose A rows
// are resident in LDS) and whole items.
//
// 64-column units (waves) of an item of the small kernel in a GEMM of n columns when there are G groups:
// the narrowest of 2, 4 and 8 whose items still are one round on the CUs. A CU reads at most ~50 GB/s, so
// few items leave the HBM idle; a second round of narrow items costs more than it gains. At least 2: the
// 64 channels that two units of GEMM1 write to a row of y are one 128-byte line, which then comes from one
// workgroup. Us a layer of 8 rows a group with 2, 4 and 8 units in both GEMMs: H = 4096, I = 2048 47, 53,
// 75 at 8 groups; 73, 56, 76 at 9; 83, 74, 85 at 16; 101, 103, 88 at 17. By each GEMM's own items: H =
// 4096, I = 1536 47 at 9 groups (52, 54, 76), 77 at 21 (88, 81, 89), 89 at 22 (96, 95, 90); H = 7168,
// I = 2048 58 at 5 (64, 73, 110).
template <bool kSmall>
struct PipeShape {
  static constexpr int kRows1 = kSmall ? 32 : kStreamItemRows;  // rows of a GEMM1 item (a group)
  static constexpr int kRows2 = kSmall ? 32 : kStreamRows;      // rows of a GEMM2 item
  static_assert(kRows1 % kRows2 == 0, "a GEMM2 item's rows are one group's");
  static constexpr __host__ __device__ int units(int G, int n) {
    const int all = G * (n / kStreamUnit);
    return !kSmall || all > 4 * kPipeCus ? kGemmWaves : all > 2 * kPipeCus ? 4 : 2;
  }
};
static_assert(PipeShape<true>::units(17, 4096) == 8 && PipeShape<true>::units(16, 4096) == 4 &&
                  PipeShape<true>::units(9, 4096) == 4 && PipeShape<true>::units(8, 4096) == 2,
              "4096 columns: whole items from 17 groups on");
static_assert(PipeShape<true>::units(32, 1024) == 2 && PipeShape<true>::units(10, 7168) == 8 &&
                  PipeShape<true>::units(21, 3072) == 4 && PipeShape<true>::units(22, 3072) == 8,
              "the width follows the items that the GEMM makes, not the groups, and keeps them one round");

// Whole groups to an XCD, one group's items after the other's, when a last round of GEMM1 items keeps at most
// half of the CUs: the others go on to GEMM2 meanwhile, and the groups of the rounds before are complete
// then. Dealt item by item, a group's items can lie in two XCDs' ranges, and column block by column block
// an expert's groups end together: the first GEMM2 items then wait for the last round (1560, 1800 and 2040
// Zipf rows: 198, 197 and 197 us; whole groups 184, 185 and 187). Above half, and when the last round is
// full, the even deal ends the last round earlier (2160, 2400 and 2640 rows: 199, 201 and 200 us; whole
// groups 204, 213 and 217; 64 groups, two full rounds, 3666 and 3634 rows: 214 and 238 against 231 and 246).
constexpr __host__ __device__ bool few_in_last_round(int items) {
  const int last = items % kPipeCus;
  return items > kPipeCus && last != 0 && 2 * last <= kPipeCus;
}
static_assert(few_in_last_round(384) && !few_in_last_round(392) && !few_in_last_round(512) && !few_in_last_round(256) &&
                  few_in_last_round(264),
              "a full last round is not a short one");

// Wave 0: s_prefix[0..E] = exclusive prefix of the experts' chunks of `rows` rows; their number.
__device__ int plan_chunks(int E, int rows, const int* s_count, int* s_prefix) {
  const int lane = lane_id();
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += kWave) {
    const int e = e0 + lane;
    const int n = e < E ? (s_count[e] + rows - 1) / rows : 0;
    const int inc = wave_inclusive_sum(n);
    if (e < E) s_prefix[e] = carry + inc - n;
    carry += __shfl(inc, kWave - 1, kWave);
  }
  if (lane == 0) s_prefix[E] = carry;
  return carry;
}

// The requant of rows [row0, row0 + mrows) of GEMM1's bf16 output y into the LDS A chunk buffers
// of a STREAM GEMM2 tile of MT 32-row tiles (stream_tile's chunk layout; K = I in at most two chunks
// of kc): the row's amax, inv = 448 / max(amax, 1e-4), then 16 e4m3 codes per
// LDS piece -- the requant kernel's arithmetic, so the same bits. The amax is the max of the
// row's 2I/64 partial maxima that GEMM1's epilogue stored (one per 64-column block, exact), eight
// lanes a row. The row scale a/448 goes straight into the tile's LDS scale table (s_xs); with
// write_act the rows' act, act_scale and amax also go out. The y pieces go out kStageBatch at a
// time, the first batch together with the maxima; rows past mrows are neither loaded nor
// quantized (their LDS rows feed only accumulator rows that are never stored).
constexpr int kPipeMaxInter = 2 * kAChunk / kStreamRows;  // I of a group's rows in both A buffers

template <int MT, int kStageBatch>
__device__ void stage_rows_from_y(const PipeArgs& p, int row0, int mrows, int kc, bool write_act,
                                  uint8_t* smem, float* s_inv, float* s_xs) {
  using Chunk = AChunk<MT>;
  constexpr int kUnitsPerLane = 2 * kPipeMaxInter / kStreamUnit / 8;
  static_assert(kStreamRows == kGemmWaves * kWave / 8, "eight lanes per row cover the group");
  static_assert(kALoads % kStageBatch == 0, "whole batches");
  const int inter = p.g1.sw.inter;
  const int units = 2 * inter / kStreamUnit;
  const int nchunks = inter / kc;
  const int tid = opaque_tid();
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const uint16_t* y = p.g1.sw.y;
  const int r8 = tid >> 3;
  float pm[kUnitsPerLane];
#pragma unroll
  for (int j = 0; j < kUnitsPerLane; ++j) {
    const int u = j * 8 + (tid & 7);
    pm[j] = 0.0f;
    if (r8 < mrows && u < units)
      pm[j] = __hip_atomic_load(p.g1.row_pmax + static_cast<int64_t>(row0 + r8) * units + u, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
  }
  // batch b of chunk c: pieces i = b * kStageBatch + h of the chunk: 16 channels, 32 bytes of y
  uint4 v[kStageBatch][2];
  auto valid = [&](int i) { return Chunk::row(i, lane, wave) < mrows; };
  auto source = [&](int c, int i) { return c * kc + Chunk::src(i, lane, wave, kc) * 16; };  // piece i's channel
  auto load_batch = [&](int c, int b) {
#pragma unroll
    for (int h = 0; h < kStageBatch; ++h) {
      const int i = b * kStageBatch + h;
      if (valid(i)) {
        const uint4* src = reinterpret_cast<const uint4*>(
            y + static_cast<int64_t>(row0 + Chunk::row(i, lane, wave)) * inter + source(c, i));
        v[h][0] = src[0];
        v[h][1] = src[1];
      }
    }
  };
  auto lo = [](uint32_t w) { return bf16_to_f32(static_cast<uint16_t>(w & 0xffff)); };
  auto hi = [](uint32_t w) { return bf16_to_f32(static_cast<uint16_t>(w >> 16)); };
  load_batch(0, 0);
  {
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < kUnitsPerLane; ++j) m = fmaxf(m, pm[j]);
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, kWave));
    if ((tid & 7) == 0 && r8 < mrows) {
      s_inv[r8] = kE4m3Max / fmaxf(m, kAmaxFloor);
      s_xs[r8] = fmaxf(m, kAmaxFloor) / kE4m3Max;
      if (write_act) {
        p.act_scale[row0 + r8] = fmaxf(m, kAmaxFloor) / kE4m3Max;
        p.amax[row0 + r8] = m;
      }
    }
  }
  __syncthreads();
  for (int c = 0; c < nchunks; ++c) {
    for (int b = 0; b < kALoads / kStageBatch; ++b) {
      if (c > 0 || b > 0) load_batch(c, b);
#pragma unroll
      for (int h = 0; h < kStageBatch; ++h) {
        const int i = b * kStageBatch + h;
        const int r = Chunk::row(i, lane, wave);
        int4 q = make_int4(0, 0, 0, 0);  // rows past mrows: never stored
        if (valid(i)) {
          const float inv = s_inv[r];
          const uint4 a = v[h][0], b2 = v[h][1];
          q.x = static_cast<int>(pack_e4m3x4(lo(a.x) * inv, hi(a.x) * inv, lo(a.y) * inv, hi(a.y) * inv));
          q.y = static_cast<int>(pack_e4m3x4(lo(a.z) * inv, hi(a.z) * inv, lo(a.w) * inv, hi(a.w) * inv));
          q.z = static_cast<int>(pack_e4m3x4(lo(b2.x) * inv, hi(b2.x) * inv, lo(b2.y) * inv, hi(b2.y) * inv));
          q.w = static_cast<int>(pack_e4m3x4(lo(b2.z) * inv, hi(b2.z) * inv, lo(b2.w) * inv, hi(b2.w) * inv));
          if (write_act)
            *reinterpret_cast<int4*>(p.act + static_cast<int64_t>(row0 + r) * inter + source(c, i)) = q;
        }
        *reinterpret_cast<int4*>(smem + (c & 1) * kAChunk + r * Chunk::kMaxK + Chunk::pos(i, lane) * 16) = q;
      }
    }
  }
}

// The items of one GEMM, `units` pieces of `step` items, dealt to the XCDs in equal contiguous ranges of
// whole pieces. Wave 0 holds in one register (`held`) the workgroup's next claim (lane 0) and what the
// XCDs' counters read when that claim went out (XCD q's in lane kPeekLane + q).
constexpr int kPeekLane = 8;
struct PipeDeal {
  int32_t* claims;  // XCD x's counter at claims[x * kPipeLine]
  int units;
  int step;
  __device__ __forceinline__ int begin(int x) const { return static_cast<int>(static_cast<int64_t>(units) * x / kPipeXcds) * step; }
  __device__ __forceinline__ int size(int x) const { return begin(x + 1) - begin(x); }
  // wave 0: claims the next item of XCD x and peeks at all counters
  __device__ __forceinline__ int claim(int x) const {
    const int lane = lane_id();
    int held = 0;
    if (lane == 0) held = atomicAdd(&claims[x * kPipeLine], 1);
    else if (lane >= kPeekLane && lane < kPeekLane + kPipeXcds)
      held = __hip_atomic_load(&claims[(lane - kPeekLane) * kPipeLine], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return held;
  }
  // wave 0: the XCDs with items left by a peek (claims only grow: an empty mask stays empty)
  __device__ __forceinline__ uint32_t left(int held) const {
    const int q = lane_id() - kPeekLane;
    return static_cast<uint32_t>(__ballot(q >= 0 && q < kPipeXcds && held < size(q & (kPipeXcds - 1))) >> kPeekLane);
  }
};

// The kernel's argument block through a pointer that is opaque to the optimizer, one for each item:
// what an item needs of the 900 bytes is then read (from the scalar cache) in that item. Read
// through the argument itself, all of it was hoisted in front of the item loop and spilled there
// (180 scalar registers).
__device__ __forceinline__ const PipeArgs& item_args() {
  uint64_t at = reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr());
  asm volatile("" : "+s"(at));
  return *(const PipeArgs*)(const __attribute__((address_space(4))) PipeArgs*)(at);
}

template <bool kSmall>
__global__ __launch_bounds__(kGemmThreads, 1) void decode_pipeline_kernel(PipeArgs p) {
  using Shape = PipeShape<kSmall>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int s_prefix1[kMaxGemmExperts + 1];  // the experts' chunks: GEMM1 (groups), GEMM2
  __shared__ int s_prefix2[kMaxGemmExperts + 1];
  __shared__ int s_count[kMaxGemmExperts];
  __shared__ int s_off[kMaxGemmExperts + 1];
  __shared__ int s_wcnt[kGemmWaves][kMaxGemmExperts];
  __shared__ int s_tok[kRowTable];
  __shared__ float s_rw[kRowTable];
  __shared__ int s_task[kRowTable];
  __shared__ uint8_t s_ev[kFusedMaxTasks];
  __shared__ TileTables s_tt;
  __shared__ float s_inv[kStreamRows];
  __shared__ int s_word;    // wave 0 -> the workgroup
  __shared__ int s_claim2;  // the first GEMM2 claim
  __shared__ int s_rows1;   // rows of a group
  const GemmArgs& g1 = p.g1;
  const GemmArgs& g2 = p.g2;
  const RouteArgs& ra = g1.route;
  const int E = g1.num_experts;
  int32_t* const done1 = p.pipe + kPipeDone1At;  // [groups]
  int32_t* const done2 = p.pipe + kPipeDone2At;  // [experts]
  const int home = hw_xcc_id() & (kPipeXcds - 1);
  // wave 0: the first claims of both GEMMs (their latency hides behind the routing; nothing is known
  // to be left then, and a peek of zeros says nothing)
  int held = 0, held2 = 0;
  if (threadIdx.x == 0) {
    held = atomicAdd(&p.pipe[home * kPipeLine], 1);
    held2 = atomicAdd(&p.pipe[home * kPipeLine + kPipeClaim2], 1);
  }
  const int ntasks = effective_tokens(ra.runtime_tokens, ra.host_tokens) * ra.topk;
  {
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    for (int e = lane_id(); e < E; e += kWave) s_wcnt[wave][e] = 0;
  }
  fused_count(ra, ntasks, s_wcnt, s_ev, reinterpret_cast<float*>(smem), blockIdx.x == 0);
  if (threadIdx.x == 0) s_claim2 = held2;
  __syncthreads();
  if (threadIdx.x < kWave) {
    fused_scan(E, s_wcnt, s_count, s_off);
    // groups of GEMM2's rows when they take no more rounds of items than the larger ones: an item of 4
    // row tiles has half the weight steps in flight (three loads of 2046 Zipf rows: 207-216 us in
    // 128-row groups, 186-194 in 64-row ones, both two rounds; 3072 even rows, one round against two: 203
    // and 223)
    const int n = stream_blocks(g1), cus = static_cast<int>(gridDim.x);
    int rows = Shape::kRows1;
    const int chunks1 = plan_chunks(E, rows, s_count, s_prefix1);
    const int chunks2 = plan_chunks(E, Shape::kRows2, s_count, s_prefix2);
    if (Shape::kRows1 != Shape::kRows2 && (chunks2 * n + cus - 1) / cus <= (chunks1 * n + cus - 1) / cus) {
      rows = Shape::kRows2;
      plan_chunks(E, rows, s_count, s_prefix1);
    }
    if (threadIdx.x == 0) s_rows1 = rows;
  }
  __syncthreads();
  if (blockIdx.x == 0) {  // the routing outputs that the later stages read
    for (int e = threadIdx.x; e <= E; e += kGemmThreads) ra.offsets[e] = s_off[e];
    for (int e = threadIdx.x; e < E; e += kGemmThreads) {
      ra.counts[e] = s_count[e];
      if (ra.stats != nullptr) ra.stats[e] += s_count[e];
    }
    if (threadIdx.x == 0) {
      ra.meta[0] = s_off[E] < ra.row_cap ? s_off[E] : static_cast<int>(ra.row_cap);
      p.meta[1] = 0;  // the 8-wave GEMM1
      if (p.direct_flag != nullptr) *p.direct_flag = 0;
    }
  }
  // more groups than counters (the host's task bound rules it out): flagged, and no items
  const bool too_many = s_prefix1[E] > kMaxPipeGroups;
  if (too_many && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&p.pipe[kPipeFailAt], 1);
  const int G = __builtin_amdgcn_readfirstlane(too_many ? 0 : s_prefix1[E]);
  const int waves1 = Shape::units(G, g1.n), waves2 = Shape::units(G, g2.n);
  const int n1 = g1.n / (kStreamUnit * waves1), n2 = g2.n / (kStreamUnit * waves2);
  const bool by_group = few_in_last_round(G * n1) && s_rows1 == Shape::kRows2;
  const float* task_w = reinterpret_cast<const float*>(smem);  // valid until the first item's loads
  bool first_item = true;
  for (int phase = 0; phase < 2; ++phase) {
    const bool gemm1 = phase == 0;
    const int chunks = gemm1 ? G : too_many ? 0 : __builtin_amdgcn_readfirstlane(s_prefix2[E]);
    const int blocks = gemm1 ? n1 : n2;
    const PipeDeal deal{p.pipe + (gemm1 ? 0 : kPipeClaim2), by_group ? chunks : chunks * blocks, by_group ? blocks : 1};
    if (!gemm1) held = threadIdx.x == 0 ? s_claim2 : 0;
    int x = home;
    for (;;) {
      if (threadIdx.x == 0) s_word = held;
      __syncthreads();
      const int c = __builtin_amdgcn_readfirstlane(s_word);
      __syncthreads();
      if (c >= deal.size(x)) {
        // this range is claimed: an XCD with items left, the next one from here on, or the next phase
        if (threadIdx.x < kWave) {
          uint32_t left = deal.left(held);
          while (left != 0) {  // (each round claims an item, or finds one range more claimed out)
            const uint32_t turned = (left | left << kPipeXcds) >> home;
            x = (home + __ffs(static_cast<int>(turned)) - 1) & (kPipeXcds - 1);
            held = deal.claim(x);
            if (__shfl(held, 0, kWave) < deal.size(x)) break;
            left = deal.left(held) & ~(1u << x);
          }
          if (threadIdx.x == 0) s_word = left == 0 ? -1 : x;
        }
        __syncthreads();
        x = __builtin_amdgcn_readfirstlane(s_word);
        __syncthreads();
        if (x < 0) break;
        continue;
      }
      if (threadIdx.x < kWave) held = deal.claim(x);  // the next claim, one item ahead
      const PipeArgs& q = item_args();
      // item t: an expert's items column block by column block, the chunks of a block next to each
      // other, so that they run together and read its weights from HBM once (by_group: chunk by chunk)
      const int t = deal.begin(x) + c;
      const int* s_prefix = gemm1 ? s_prefix1 : s_prefix2;
      const int per = gemm1 ? n1 : n2;
      const int e = expert_of_item(s_prefix, E, t / per);
      const int first = __builtin_amdgcn_readfirstlane(s_prefix[e]);
      const int nch = __builtin_amdgcn_readfirstlane(s_prefix[e + 1]) - first;
      const int local = t - first * per;
      const int nb = by_group ? local % per : local / nch;
      const int ch = by_group ? local / per : local - nb * nch;
      const int rows1 = __builtin_amdgcn_readfirstlane(s_rows1);
      const int rows = gemm1 ? rows1 : Shape::kRows2;
      const int r0 = ch * rows;
      const int cnt = __builtin_amdgcn_readfirstlane(s_count[e]);
      const int off_e = __builtin_amdgcn_readfirstlane(s_off[e]);
      const int mrows = min(rows, cnt - r0);
      const int row0 = off_e + r0;
      const int grp = gemm1 ? first + ch : __builtin_amdgcn_readfirstlane(s_prefix1[e]) + r0 / rows1;
      if (gemm1) {
        // the weights go out first; then the item's rows are ranked into the LDS row table
        const float* item_w = first_item ? task_w : nullptr;
        const auto rank_rows = [&]() {
          fused_rows(q.g1.route, ntasks, e, cnt, off_e, s_wcnt, s_ev, item_w, r0, nb == 0 ? r0 : 0,
                     nb == 0 ? r0 + rows1 : 0, 0, 0, s_task, s_tok, s_rw);
        };
        const RowSrc rs{s_tok, s_rw, row0};
        if (kSmall && waves1 < kGemmWaves)
          stream_tile<true, true, 1, kNarrowDepth, true, false, true, true, true, kALoads / 2>(q.g1, rs, e, row0, mrows, nb, q.narrow_kc1, smem, s_tt, rank_rows, waves1);
        else if (!kSmall && mrows > 64)
          stream_tile<true, true, 4, 2, true, false, true, true, false, kALoads / 2>(q.g1, rs, e, row0, mrows, nb, kAChunk4, smem, s_tt, rank_rows);
        else if (!kSmall && mrows > 32)
          stream_tile<true, true, 2, kStreamDepth, true, false, true, true>(q.g1, rs, e, row0, mrows, nb, q.g1.kc[1], smem, s_tt, rank_rows);
        else
          stream_tile<true, true, 1, kStreamDepth, true, false, true, true>(q.g1, rs, e, row0, mrows, nb, q.g1.kc[0], smem, s_tt, rank_rows);
        vm_drain();  // this wave's y stores are written through to the device-coherent level
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(&q.pipe[kPipeDone1At + grp], 1);
      } else {
        // the weights go out first; then the group's rows, requantized from y into LDS
        const auto stage_rows = [&]() {
          if (threadIdx.x == 0 && !wait_count(&q.pipe[kPipeDone1At + grp], n1, q.spin_limit)) atomicAdd(&q.pipe[kPipeFailAt], 1);
          __syncthreads();
          l1_invalidate();
          // (beside a ring of 8 steps there are registers for two pieces at a time)
          if constexpr (kSmall) stage_rows_from_y<1, 2>(q, row0, mrows, q.g2.kc[0], nb == 0, smem, s_inv, s_tt.xs);
          else if (mrows > 32) stage_rows_from_y<2, 4>(q, row0, mrows, q.g2.kc[1], nb == 0, smem, s_inv, s_tt.xs);
          else stage_rows_from_y<1, 4>(q, row0, mrows, q.g2.kc[0], nb == 0, smem, s_inv, s_tt.xs);
          __syncthreads();
        };
        const RowSrc rs{nullptr, nullptr, 0};
        if (kSmall && waves2 < kGemmWaves)
          stream_tile<false, false, 1, kNarrowDepth, true, true, false, true, true>(q.g2, rs, e, row0, mrows, nb, q.g2.kc[0], smem, s_tt, stage_rows, waves2);
        else if (!kSmall && mrows > 32)
          stream_tile<false, false, 2, kStreamDepth, true, true, false, true>(q.g2, rs, e, row0, mrows, nb, q.g2.kc[1], smem, s_tt, stage_rows);
        else
          stream_tile<false, false, 1, kStreamDepth, true, true, false, true>(q.g2, rs, e, row0, mrows, nb, q.g2.kc[0], smem, s_tt, stage_rows);
        vm_drain();  // this wave's partial rows are written through to the device-coherent level
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(&q.pipe[kPipeDone2At + e * kPipeDone2Stride], 1);
      }
      first_item = false;
      __syncthreads();
    }
  }
  if (p.y != nullptr && !too_many) {
    // the combine: token i goes to wave (i / gridDim.x) % 8 of workgroup i % gridDim.x, so the
    // tokens spread over all workgroups (each wave's tokens are independent of the others')
    const int tokens = effective_tokens(ra.runtime_tokens, ra.host_tokens);
    const int64_t part_bytes = static_cast<int64_t>(ra.row_cap) * g2.n * 2;
    const __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(
        g2.c, 0, static_cast<int>(part_bytes < 0x7fffffff ? part_bytes : 0x7fffffff), 0x00020000);
    const int wave = static_cast<int>(threadIdx.x) / kWave;
    for (int64_t t = blockIdx.x + static_cast<int64_t>(wave) * gridDim.x; t < tokens;
         t += static_cast<int64_t>(gridDim.x) * kGemmWaves)
      pipe_combine_token(p, t, s_ev, s_prefix1, s_prefix2, n1, n2, done1, done2, part);
  }
  // the workgroup that leaves last (every other one has made its last counter access): the
  // count of waits that ran out into meta[3] (the call's status), the counters back to zero
  // for the next launch. Each wave's counter atomics are complete (vmcnt) before its
  // workgroup counts itself out, so the last one reads every failure.
  vm_drain();
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool last = atomicAdd(p.pipe + kPipeExitAt, 1) == static_cast<int>(gridDim.x) - 1;
    if (last) p.meta[3] = __hip_atomic_load(p.pipe + kPipeFailAt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_word = last ? 1 : 0;
  }
  __syncthreads();
  if (s_word != 0) {
    for (int i = threadIdx.x; i < kPipeHeader + G; i += kGemmThreads) p.pipe[i] = 0;
    for (int i = threadIdx.x; i < E; i += kGemmThreads) done2[i * kPipeDone2Stride] = 0;
  }
}

// Persistent dispatcher of the WIDE engine: every expert's rows as BM x 256 tiles, items dealt
// to the XCDs in contiguous ranges like the 8-wave dispatcher's.
template <bool kGather, bool kSwiglu, int BM, bool kBig>
__global__ __launch_bounds__(kWideThreads, WideShape<BM>::kWavesPerSimd) void wide_gemm_kernel(GemmArgs g) {
  if (dual_skips(g, true)) return;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int s_prefix[kMaxGemmExperts + 1];
  __shared__ int s_tile[kMaxGemmExperts];
  __shared__ int s_count[kMaxGemmExperts];
  __shared__ int s_off[kMaxGemmExperts + 1];
  const int E = g.num_experts;
  for (int e = threadIdx.x; e <= E; e += kWideThreads) {
    if (e < E) s_count[e] = g.counts[e];
    s_off[e] = g.offsets[e];
  }
  __syncthreads();
  plan_items(g, s_prefix, s_tile, s_count, true, BM);
  __syncthreads();
  const int total = s_prefix[E];
  const int tile_nb = (g.n + kTileBN - 1) / kTileBN;
  const RowSrc rs{g.row_token, g.sw.row_weight, 0};
  auto run_item = [&](int t, const auto& before_epilogue) {
    const int e = expert_of_item(s_prefix, E, t);
    const int cnt = __builtin_amdgcn_readfirstlane(s_count[e]);
    int mt, nb;
    tile_coords(t - __builtin_amdgcn_readfirstlane(s_prefix[e]), cnt, tile_nb, mt, nb, BM);
    const int mrows = min(BM, cnt - mt * BM);
    const int row0 = __builtin_amdgcn_readfirstlane(s_off[e]) + mt * BM;
    if (BM == 256 && mrows > 128)
      wide_tile<kGather, kSwiglu, BM, BM / 16, kBig>(g, rs, e, row0, mrows, nb, smem, before_epilogue);
    else if (mrows > 64)
      wide_tile<kGather, kSwiglu, BM, 8, kBig>(g, rs, e, row0, mrows, nb, smem, before_epilogue);
    else if (mrows > 32)
      wide_tile<kGather, kSwiglu, BM, 4, kBig>(g, rs, e, row0, mrows, nb, smem, before_epilogue);
    else
      wide_tile<kGather, kSwiglu, BM, 2, kBig>(g, rs, e, row0, mrows, nb, smem, before_epilogue);
  };
  // One item at a time from the static deal or from the claims. Claiming only pays when a
  // workgroup has few items (the last round's granularity is then a large share of its work;
  // 24.7K routed rows: 7 items a workgroup, 5% faster); with many it measured slower (196K rows,
  // 49 items: 1% slower; 49K Zipf rows, 13 items: 1% slower) -- the lockstep rounds of the static
  // deal keep an XCD's concurrent tiles on the same rows and weights, and at those sizes the
  // chip is power-bound, so idle workgroups cost less than the looser L2 sharing.
  constexpr int kClaimMaxItemsPerWg = 10;
  const bool dynamic =
      g.sched != nullptr && total <= kClaimMaxItemsPerWg * static_cast<int>(gridDim.x);
  const ItemDeal deal = deal_items(total);
  const Claims cl = make_claims(g.sched, total);
  __shared__ int s_item;
  int k = 0;   // static: the round
  int ri = 0;  // dynamic, thread 0: index of the range it claims from
  if (threadIdx.x == 0 && dynamic) {
    const int first = cl.begin(cl.home) + cl.slot;
    s_item = first < cl.end(cl.home) ? first : cl.claim_from(ri);
  }
  __syncthreads();
  while (true) {
    int t;
    if (dynamic) {
      t = __builtin_amdgcn_readfirstlane(s_item);
    } else {
      for (t = -1; k < deal.rounds() && t < 0; ++k) {
        const int c = deal.item(k);
        t = c < deal.end ? c : -1;  // the last round's short tail
      }
    }
    if (t < 0) break;
    // thread 0: the claim for the item after this one, issued when the tile's MFMAs are done
    // (its latency hides behind the epilogue; issued at the tile's start, its result stayed live
    // through the tile and was spilled, with a wait for every memory operation in flight)
    int pending = 0;
    run_item(t, [&]() {
      if (dynamic && threadIdx.x == 0 && ri < cl.nranges) pending = atomicAdd(&g.sched[cl.range(ri)], 1);
    });
    if (dynamic && threadIdx.x == 0) {
      int next = -1;
      if (ri < cl.nranges) {
        const int r = cl.range(ri);
        next = cl.item(r, pending);
        if (next >= cl.end(r)) {
          ++ri;
          next = cl.claim_from(ri);
        }
      }
      s_item = next;  // read after the barrier; rewritten only after the next tile's barriers
    }
    __syncthreads();
  }
  if (g.zf.y != nullptr && !dynamic) {
    // out of tiles: the zero y rows of tokens without a valid routed slot, a claimed chunk of
    // kZeroFillTokens tokens at a time (a wave a token), while other workgroups still run tiles
    // (z.idle counts the workgroups out of tiles); the combine writes the chunks left. Only
    // with the static deal (many tiles a workgroup): with claimed tiles the idle end is short,
    // and the zero rows' writes slowed the last tiles by more than the combine saved (c2: +28 us
    // per layer; c3: -60 us).
    const ZeroFill& z = g.zf;
    const int tokens = effective_tokens(z.runtime_tokens, z.host_tokens);
    const int nchunks = (tokens + kZeroFillTokens - 1) / kZeroFillTokens;
    const int lane = lane_id(), wave = static_cast<int>(threadIdx.x) / kWave;
    const int nvec = z.hidden >> 3;
    if (threadIdx.x == 0) atomicAdd(z.idle, 1);
    for (;;) {
      __syncthreads();  // every thread has read s_item
      if (threadIdx.x == 0) {
        const int idle = __hip_atomic_load(z.idle, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_item = idle >= static_cast<int>(gridDim.x) ? nchunks : atomicAdd(z.claim, 1);
      }
      __syncthreads();
      const int c = s_item;
      if (c >= nchunks) break;
      const int t_end = min(tokens, (c + 1) * kZeroFillTokens);
      for (int t = c * kZeroFillTokens + wave; t < t_end; t += kWideWaves) {
        const int v = lane < z.topk ? z.output_index[static_cast<int64_t>(t) * z.topk + lane] : -1;
        if (__ballot(v >= 0) != 0) continue;
        i32x4* row = reinterpret_cast<i32x4*>(z.y + static_cast<int64_t>(t) * z.hidden);
        for (int i = lane; i < nvec; i += kWave) __builtin_nontemporal_store(i32x4{0, 0, 0, 0}, row + i);
      }
    }
  }
  if (dynamic && threadIdx.x == 0) {  // every claim of this workgroup is done: count it out
    if (atomicAdd(&g.sched[8], 1) == static_cast<int>(gridDim.x) - 1) {
      for (int r = 0; r < 8; ++r) atomicExch(&g.sched[r], 0);
      atomicExch(&g.sched[8], 0);
    }
  }
}

// The dynamic-LDS limit of kernel K raised to `bytes` (above the default) once per device of
// the process (the attribute is set for the current device; a bit per device id below 64).
template <auto K>
hipError_t ensure_dynamic_lds(int bytes) {
  static std::atomic<uint64_t> done{0};
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  const uint64_t bit = dev >= 0 && dev < 64 ? (1ull << dev) : 0;
  if (bit != 0 && (done.load(std::memory_order_acquire) & bit) != 0) return hipSuccess;
  err = hipFuncSetAttribute(reinterpret_cast<const void*>(K), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (err == hipSuccess && bit != 0) done.fetch_or(bit, std::memory_order_release);
  return err;
}

template <bool kGather, bool kSwiglu, int BM, bool kBig = false>
hipError_t launch_wide(const GemmArgs& g, int max_rows, int num_cus, hipStream_t stream) {
  using W = WideShape<BM>;
  {  // the dynamic LDS (up to 104 KB) exceeds the default limit
    const hipError_t err = ensure_dynamic_lds<&wide_gemm_kernel<kGather, kSwiglu, BM, kBig>>(W::kSmemBytes);
    if (err != hipSuccess) return err;
  }
  const int64_t bound =
      (static_cast<int64_t>(max_rows) / BM + g.num_experts) * ((g.n + kTileBN - 1) / kTileBN);
  int64_t grid = static_cast<int64_t>(num_cus) * W::kWavesPerSimd;  // workgroups a CU: 1 or 2
  if (grid > bound) grid = bound;
  return launch_kernel(wide_gemm_kernel<kGather, kSwiglu, BM, kBig>, dim3(static_cast<unsigned>(grid)),
                       dim3(kWideThreads), W::kSmemBytes, stream, g);
}

template <bool kGather, bool kSwiglu, int kTail>
hipError_t launch_engines_k(const GemmArgs& g, int max_rows, int num_cus, hipStream_t stream) {
  {  // the 128 KB of dynamic LDS exceeds the default limit
    const hipError_t err = ensure_dynamic_lds<&grouped_gemm_kernel<kGather, kSwiglu, kTail>>(kSmemBytes);
    if (err != hipSuccess) return err;
  }
  // upper bound of the work items over any split of max_rows rows into the experts
  const int64_t stream_nb = (g.n / kStreamUnit + kGemmWaves - 1) / kGemmWaves;
  const int64_t stream_items = (static_cast<int64_t>(max_rows) / kStreamItemRows + g.num_experts) * stream_nb;
  const int64_t tile_items =
      (static_cast<int64_t>(max_rows) / kTileBM + g.num_experts) * ((g.n + kTileBN - 1) / kTileBN);
  const int64_t bound = g.engine == GemmEngine::kStream ? stream_items
                        : g.engine == GemmEngine::kTile ? tile_items
                                                        : std::max(stream_items, tile_items);
  int64_t grid = num_cus;  // one 8-wave workgroup per CU
  if (grid > bound) grid = bound;
  return launch_kernel(grouped_gemm_kernel<kGather, kSwiglu, kTail>, dim3(static_cast<unsigned>(grid)),
                       dim3(kGemmThreads), kSmemBytes, stream, g);
}

// The largest multiple of 64 * ring that divides k and is at most cap; 0: there is none.
int whole_chunk(int k, int cap, int ring) {
  for (int kc = cap / (64 * ring) * (64 * ring); kc > 0; kc -= 64 * ring)
    if (k % kc == 0) return kc;
  return 0;
}

// The chunk of the fewest, about equally long, chunks of k that are at most cap each and whole rings (k
// and cap are multiples of 64 * ring); the last one may be shorter.
int tail_chunk(int k, int cap, int ring) {
  const int unit = 64 * ring, chunks = (k + cap - 1) / cap;
  return (k + chunks * unit - 1) / (chunks * unit) * unit;
}

// The LDS buffer of a chunk of MT = 1 << i row tiles, in k-bytes.
int chunk_cap(int i) { return kAChunk / 32 >> i; }

// The STREAM engine's chunks of K for 1, 2 and 4 row tiles with a ring of 4 weight steps: as long as
// the LDS buffers allow, so that the workgroup's barriers are few. Beside the accumulators of 4 row
// tiles a ring of 4 leaves registers for half the A loads only, so chunks of 256 in half the buffers:
// 2715 rows of 32 experts 181.5 -> 177 us a layer against a ring of 2 and chunks of 512.
void set_stream_chunks(GemmArgs* g) {
  for (int i = 0; i < 2; ++i) g->kc[i] = whole_chunk(g->k, chunk_cap(i), kStreamDepth);
  g->kc[2] = kAChunk4;
}

// A short last chunk where K is not a multiple of 256, or where chunks that divide K are at most half as
// long: a chunk's loads and LDS writes are those of a whole buffer, and every chunk ends in a barrier.
// 256 tokens on 32 experts, top-6 of 128 (I = 1024 where K = H, H = 4096 where K = I), us a layer, chunks
// of 128 or 256 / the kernel here: K = H = 2944 90 / 71, 4352 115 / 104, 5504 203 / 192; K = I = 2176 188 /
// 182.
int stream_tail(const GemmArgs& g) {
  if (g.k % (64 * kStreamDepth) != 0) return kTailAny;
  for (int i = 0; i < 2; ++i)
    if (2 * whole_chunk(g.k, chunk_cap(i), kStreamDepth) <= tail_chunk(g.k, chunk_cap(i), kTailDepth)) return kTail256;
  return kTailNone;
}

template <bool kGather, bool kSwiglu>
hipError_t launch_engines(const GemmArgs& args, int max_rows, int num_cus, hipStream_t stream) {
  GemmArgs g = args;
  const int tail = stream_tail(g);
  if (tail == kTailNone) {
    set_stream_chunks(&g);
    return launch_engines_k<kGather, kSwiglu, kTailNone>(g, max_rows, num_cus, stream);
  }
  for (int i = 0; i < 3; ++i) g.kc[i] = tail_chunk(g.k, chunk_cap(i), kTailDepth);
  return tail == kTail256 ? launch_engines_k<kGather, kSwiglu, kTail256>(g, max_rows, num_cus, stream)
                          : launch_engines_k<kGather, kSwiglu, kTailAny>(g, max_rows, num_cus, stream);
}

}  // namespace

int gemm_route_max_tasks() { return kFusedMaxTasks; }
int gemm_route_max_experts() { return kFusedMaxExperts; }

// Many rows per expert on average: every expert as WIDE tiles (one launch, no per-expert engine
// choice). More tasks than the in-kernel routing takes, so the two never meet; the choice
// depends only on the shape and the row bound, so separate stage calls agree on it.
bool gemm_wide_selected(const GemmArgs& g, int max_rows) {
  return g.engine != GemmEngine::kStream && g.k % (2 * kWideBK) == 0 && g.n % kStreamUnit == 0 &&
         max_rows > kFusedMaxTasks &&
         static_cast<int64_t>(max_rows) >= static_cast<int64_t>(kWideMinRowsPerExpert) * g.num_experts;
}

bool gemm_shape_supported(int n, int k) {
  return n > 0 && k > 0 && n % 128 == 0 && k % 128 == 0;
}

// Full WIDE tile heights. 256 rows (one workgroup a CU) for both GEMMs: with 128-row tiles and
// two workgroups a CU, GEMM1 (weights read twice as often) ran 1.33x slower at the 196K-row
// prefill; GEMM2 ran 7% faster at 24.7K rows but slower at 196K rows, where it also left the
// next layer's GEMM1 2% slower (measured on one box, builds alternated).
constexpr int kWideBM1 = 256;
constexpr int kWideBM2 = 256;

int gemm_wide_min_rows(int num_experts) {
  return std::max(kFusedMaxTasks + 1, kWideMinRowsPerExpert * num_experts);
}

// Eager calls whose row bound selects WIDE only by a small margin: the routed rows may be far
// fewer (an EP share keeps ~1/8 of its slots), so both kernels go out and the routing's largest
// expert row count chooses on the device -- the 8-wave kernels while every expert has at most
// 128 rows (one STREAM item a column block), WIDE from 129.
// Measured (whole eager layers after a read-only cache flush) at T = 256..576 a rank (256 global
// experts, top-6): 188-202 us on the 8-wave kernels (one 128-row item per expert and column
// block: 256 items, one round) against 230-248 us on WIDE. Streaming experts of up to 256 rows
// (two items) and going WIDE only past that was within -4..+3% of this choice at T = 640..1024.
// Auto schedules only (an engine set by the caller keeps its kernels); from 8 x 128 tasks an
// expert (an EP share of 1/8 then routes 128 rows an expert on average, so some expert has
// more) the bound selects WIDE directly (no launches that return at once).
constexpr int kEagerDualMinLargest = kStreamAutoMaxRows + 1;
int gemm_eager_dual_min_largest() { return kEagerDualMinLargest; }
bool gemm_eager_dual(const GemmArgs& g, int max_rows) {
  return g.engine == GemmEngine::kAuto && gemm_wide_selected(g, max_rows) &&
         static_cast<int64_t>(max_rows) < 8ll * kStreamAutoMaxRows * g.num_experts;
}

// Tasks (S * K) up to which the pipeline's small kernel runs. H = 4096, I = 2048, top-6, us on it and on
// the large one, three loads each: 32 of 256 experts local 33-46 against 65-74 at 8 tokens, 43-91 against
// 73-91 at 24, 61-110 against 78-110 at 48; past the bound they tie (64 tokens: 88-118 both). A chunk is 32
// rows here, so a skewed load pays for it: Zipf loads of 28 local experts 66-76 against 82-86 at 8 tokens
// and 107-119 against 112-121 at 24, but at 53 114, 128 and 135 against 118, 122 and 131, and past the
// bound, at 80, 162-177 against 130-138. At H = 7168, top-8, the other side is the separate launches: 51-97
// against 107-126 at 10 tokens, 113-190 against 137-189 at 40; Zipf loads 148-172 against 144-168 at 10
// and 192, 210 and 224 against 202, 203 and 215 at 40.
constexpr int kPipeSmallTasks = 320;
// The groups' counters: a group of the small kernel has a row at least, one of the large kernel is a whole
// chunk of GEMM2's rows or an expert's last.
static_assert(kPipeSmallTasks <= kMaxPipeGroups && kFusedMaxTasks / kStreamRows + kFusedMaxExperts <= kMaxPipeGroups,
              "a counter for every group");

static bool pipe_small(const GemmArgs& g1) {
  return static_cast<int64_t>(g1.route.host_tokens) * g1.route.topk <= kPipeSmallTasks;
}

// The decode pipeline needs rings of 4 weight steps and whole items for both GEMMs, GEMM2's K = I
// in at most two chunks (staged whole by the requant) of an even number of narrow rings, GEMM1's
// in-kernel routing, and the whole MI355X (8 XCDs of 32 CUs: its queues are the hardware XCD ids).
// Past the small kernel's tasks it also wants whole A chunks in both GEMMs: at H = 7168 or I = 1536
// the separate launches are as fast there with few rows an expert (I = 1536, 512 tokens of 128
// experts: 120 us against 116) and faster with many (R = 2139: 204 against 130).
// And y in whole 128-byte lines (a caller's route_scratch can lie anywhere): a line that the last row
// of one group shared with the first row of the next would come into an XCD's L2 with the first group's
// rows, before the second group's are written. The separate launches take any other base.
bool decode_pipeline_supported(const GemmArgs& g1, const GemmArgs& g2, int num_cus) {
  GemmArgs c1 = g1, c2 = g2;
  set_stream_chunks(&c1);
  set_stream_chunks(&c2);
  for (int i = 0; i < 2; ++i)  // (chunks that a ring of 2 steps would not make twice as long)
    if (2 * c1.kc[i] <= whole_chunk(g1.k, chunk_cap(i), 2) || 2 * c2.kc[i] <= whole_chunk(g2.k, chunk_cap(i), 2))
      return false;
  const bool whole_chunks = g1.k % (kAChunk / 32) == 0 && g2.k == kAChunk / 32;
  return num_cus == kPipeCus && g1.engine != GemmEngine::kTile && g2.engine != GemmEngine::kTile &&
         g1.route_in_kernel == 1 && g1.sw.enabled && g1.num_experts <= kFusedMaxExperts &&
         (whole_chunks || pipe_small(g1)) && reinterpret_cast<uintptr_t>(g1.sw.y) % 128 == 0 &&
         whole_chunk(g1.k, kAChunk / 64, kNarrowDepth) > 0 &&
         g2.k <= kPipeMaxInter && c2.kc[0] == g2.k && 2 * c2.kc[1] >= g2.k && g2.k % (64 * kNarrowDepth) == 0 &&
         g1.n == 2 * g1.sw.inter && g2.k == g1.sw.inter && g1.n % (kStreamUnit * kGemmWaves) == 0 &&
         g2.n % (kStreamUnit * kGemmWaves) == 0 && g1.row_token != nullptr && g2.row_token == nullptr &&
         g1.dual_rows == nullptr && g2.dual_rows == nullptr && g2.y_direct == nullptr;
}

hipError_t launch_decode_pipeline(const PipeArgs& args, int num_cus, hipStream_t stream) {
  if (!decode_pipeline_supported(args.g1, args.g2, num_cus) || args.pipe == nullptr ||
      args.g1.row_pmax == nullptr || args.act != args.g2.a || args.act_scale != args.g2.a_scale ||
      args.g2.lda != args.g1.sw.inter)
    return hipErrorInvalidValue;
  const bool small = pipe_small(args.g1);
  const hipError_t err = small ? ensure_dynamic_lds<&decode_pipeline_kernel<true>>(kSmemBytes)
                               : ensure_dynamic_lds<&decode_pipeline_kernel<false>>(kSmemBytes);
  if (err != hipSuccess) return err;
  PipeArgs p = args;
  set_stream_chunks(&p.g1);
  set_stream_chunks(&p.g2);
  p.narrow_kc1 = whole_chunk(p.g1.k, kAChunk / 64, kNarrowDepth);
  return launch_kernel(small ? decode_pipeline_kernel<true> : decode_pipeline_kernel<false>,
                       dim3(static_cast<unsigned>(num_cus)), dim3(kGemmThreads), kSmemBytes, stream, p);
}

static hipError_t launch_wide_gemm(const GemmArgs& g, int max_rows, int num_cus, hipStream_t stream) {
  if (!g.sw.enabled) return launch_wide<false, false, kWideBM2>(g, max_rows, num_cus, stream);
  // 32-bit offsets into the token matrix (8 registers and an addition a load less) up to 4 GB
  return g.a_bytes >= int64_t{1} << 32 ? launch_wide<true, true, kWideBM1, true>(g, max_rows, num_cus, stream)
                                       : launch_wide<true, true, kWideBM1>(g, max_rows, num_cus, stream);
}

hipError_t launch_grouped_gemm(const GemmArgs& g, int max_rows, int num_cus, hipStream_t stream,
                               const int32_t* rows_on_device, bool route_small_in_kernel,
                               int dual_min_rows) {
  if (max_rows <= 0) return hipSuccess;
  if (g.num_experts > kMaxGemmExperts || g.dual_rows != nullptr) return hipErrorInvalidValue;
  const bool wide = gemm_wide_selected(g, max_rows);
  if (wide && g.route_in_kernel) return hipErrorInvalidValue;
  // direct writes to y: the WIDE GEMM2 epilogue only
  if (g.y_direct != nullptr && (!wide || g.sw.enabled || g.row_dest == nullptr || g.direct_flag == nullptr))
    return hipErrorInvalidValue;
  if (g.sw.enabled && (g.row_token == nullptr || g.n != 2 * g.sw.inter)) return hipErrorInvalidValue;
  if (!g.sw.enabled && g.row_token != nullptr) return hipErrorInvalidValue;
  // the 8-wave kernel routes the live tasks itself when they fit (the routing launch of the
  // same call returns at once then): a GEMM1 on device-read tokens only
  if (route_small_in_kernel && (!g.sw.enabled || g.route_in_kernel || rows_on_device == nullptr ||
                                g.num_experts > kFusedMaxExperts))
    return hipErrorInvalidValue;
  GemmArgs eight = g;
  if (route_small_in_kernel) eight.route_in_kernel = 2;
  if (wide && rows_on_device != nullptr) {
    // the bound selects WIDE, but the rows are known on the device only: both kernels go out,
    // and the one the routed rows do not select returns at once (the 8-wave one without the
    // WIDE GEMM2's direct writes, which the requant then leaves switched off)
    GemmArgs d = g;
    d.dual_rows = rows_on_device;
    d.dual_min_rows = dual_min_rows > 0 ? dual_min_rows : gemm_wide_min_rows(g.num_experts);
    // (a smaller threshold than the default only where the 8-wave kernel never routes itself)
    if (d.dual_min_rows <= kFusedMaxTasks && route_small_in_kernel) return hipErrorInvalidValue;
    eight.dual_rows = d.dual_rows;
    eight.dual_min_rows = d.dual_min_rows;
    eight.row_dest = nullptr;
    eight.y_direct = nullptr;
    eight.direct_flag = nullptr;
    const hipError_t err = g.sw.enabled ? launch_engines<true, true>(eight, max_rows, num_cus, stream)
                                        : launch_engines<false, false>(eight, max_rows, num_cus, stream);
    if (err != hipSuccess) return err;
    return launch_wide_gemm(d, max_rows, num_cus, stream);
  }
  if (wide && route_small_in_kernel) return hipErrorInvalidValue;  // (rows_on_device is set)
  if (wide) return launch_wide_gemm(g, max_rows, num_cus, stream);
  return g.sw.enabled ? launch_engines<true, true>(eight, max_rows, num_cus, stream)
                      : launch_engines<false, false>(eight, max_rows, num_cus, stream);
}

}  // namespace mmoe
