// route.hip -- deterministic routing for the grouped expert GEMMs (gfx950).
//
// Semantics (reference): a task (token t, slot s) is routed to local expert e =
// topk_idx[t,s] iff 0 <= e < E and, for the layer, topk_weights[t,s] != 0
// (deep_gemm/include/deep_gemm/impls/mega_moe_dcu.cuh:352). Routed rows are
// expert-contiguous at tight exclusive-scan offsets (csrc/kernels/mega_moe_baseline_hip.cu:
// 37-47). The reference places rows inside an expert by atomicAdd arrival
// (mega_moe_baseline_hip.cu:75, mega_moe_dcu.cuh:359); here the order is the stable one --
// ascending task index -- so counts, rows and output_index are bitwise reproducible.
//
// Ranks come from wave ballots: one ballot per bit of the expert id gives every lane the mask
// of lanes holding the same expert (a match-any in log2(E) votes); a lane's rank is the
// popcount of that mask below it and the group's lowest lane publishes the group size. Per-wave
// counts become per-wave bases through LDS prefix sums.
//
// Two launch shapes, both integer work bound by the topk tables' reads and their latency:
//   * up to 16384 tasks: one launch with a workgroup for each expert, which ranks that expert's tasks;
//   * more: a count kernel (one workgroup per chunk, LDS histogram) and a scatter kernel
//     (one workgroup per chunk) that rebuilds the expert offsets and its chunk base from the
//     per-chunk counts itself, so no grid-wide barrier or separate scan launch is needed.
#include "launch.h"
#include "route_wave.cuh"

namespace mmoe {

namespace {

constexpr int kExpertThreads = 1024;
constexpr int kExpertWaves = kExpertThreads / kWave;
constexpr int kExpertMaxExperts = 256;
// Tasks up to which a workgroup an expert routes: it reads all of them, so its time grows with their
// number, while the chunk kernels' two launches have a floor of 10.5 us. 32 experts, us (one of 8
// slots local / all of them local): 8192 tasks 5.6 / 7.2, 16384 8.3 / 11.6, 24576 10.4 / 16.1, against
// the chunk kernels' 10.5 / 11 at 24576. One workgroup for all experts had taken 16 / 17 at 8192 and
// 27 / 32 at 16384.
constexpr int kExpertPasses = 16;  // of a wave
constexpr int kExpertMaxTasks = kExpertPasses * kExpertThreads;
constexpr int kChunkThreads = 1024;
constexpr int kChunkWaves = kChunkThreads / kWave;
static_assert(kMaxExperts <= kChunkThreads, "the chunk-count reduction needs a thread per expert");
static_assert(kChunkWaves == kRouteWaves, "per-wave counts of a chunk in the workspace");

// Assigns rows to one 64-task pass in task order; base[e] is this wave's running base.
__device__ __forceinline__ void wave_scatter_pass(const RouteArgs& a, int64_t task, bool in_range,
                                                  int e, float w, int id_bits, int* base) {
  const uint64_t m = match_expert(e, id_bits);
  int row = -1;
  if (e >= 0) row = base[e] + __popcll(m & lanes_below());
  __builtin_amdgcn_wave_barrier();
  if (e >= 0 && (m & lanes_below()) == 0ull) base[e] += __popcll(m);
  __builtin_amdgcn_wave_barrier();
  if (row >= 0 && row >= a.row_cap) row = -1;
  if (in_range) a.output_index[task] = row;
  if (row >= 0) {
    a.row_token[row] = static_cast<int32_t>(task / a.topk);
    if (a.row_weight != nullptr) a.row_weight[row] = w;
    if (a.m_indices != nullptr) a.m_indices[row] = e;
  }
}

// Counts then scatters the tasks [begin, end) of this wave, in batches of kBatch passes held
// in registers. `cnt` is the wave's count row (zeroed by the caller); between the two phases
// the caller turns counts into bases (needs a workgroup barrier), passed through `phase_gap`.
constexpr int kBatch = 8;

// Counts of the tasks [begin, end) of this wave into its count row.
__device__ void wave_count_range(const RouteArgs& a, int64_t begin, int64_t end, int* row) {
  int ev[kBatch];
  float wv[kBatch];
  const int id_bits = expert_id_bits(a.num_experts);
  for (int64_t b = begin; b < end; b += kBatch * kWave) {
    wave_load<kBatch>(a, b, end, ev, wv);
#pragma unroll
    for (int p = 0; p < kBatch; ++p) {
      if (b + p * kWave >= end) break;  // (a chunk of 1024 tasks has one pass a wave)
      wave_count_pass(ev[p], id_bits, row);
    }
  }
}

// A wave's first kBatch passes of tasks, loaded ahead.
struct WaveTasks {
  int ev[kBatch];
  float wv[kBatch];
};

// counted: the count rows hold this range's counts already (the count kernel's). `t` holds the
// range's first batch.
template <class Gap>
__device__ void wave_route(const RouteArgs& a, int64_t begin, int64_t end, int* row, WaveTasks& t,
                           Gap phase_gap, bool counted) {
  const int id_bits = expert_id_bits(a.num_experts);
  if (!counted) wave_count_range(a, begin, end, row);
  phase_gap();
  const int lane = lane_id();
  for (int64_t b = begin; b < end; b += kBatch * kWave) {
    if (b > begin) wave_load<kBatch>(a, b, end, t.ev, t.wv);
#pragma unroll
    for (int p = 0; p < kBatch; ++p) {
      if (b + p * kWave >= end) break;
      const int64_t task = b + p * kWave + lane;
      wave_scatter_pass(a, task, task < end, t.ev[p], t.wv[p], id_bits, row);
    }
  }
}

// Expert offsets from totals (exclusive scan, or the caller's counts for the preprocess), by
// wave 0 in 64-expert chunks (DPP scans); fills s_off[0..E], and the writer workgroup
// publishes offsets, counts, stats, the routed row count (meta[0]) and the largest expert's
// row count (meta[4]).
__device__ void publish_offsets(const RouteArgs& a, const int* s_tot, int* s_off, bool writer) {
  if (threadIdx.x < kWave) {
    const int lane = lane_id();
    int carry = 0, routed = 0, largest = 0;
    for (int e0 = 0; e0 < a.num_experts; e0 += kWave) {
      const int e = e0 + lane;
      const int tot = e < a.num_experts ? s_tot[e] : 0;
      const int c = a.given_counts != nullptr ? (e < a.num_experts ? a.given_counts[e] : 0) : tot;
      const int inc = wave_inclusive_sum(c);
      if (e < a.num_experts) s_off[e] = carry + inc - c;
      carry += __shfl(inc, kWave - 1, kWave);
      routed += __shfl(wave_inclusive_sum(tot), kWave - 1, kWave);
      largest = max(largest, wave_max(tot));
    }
    if (lane == 0) {
      s_off[a.num_experts] = carry;
      if (writer) {
        a.meta[0] = static_cast<int32_t>(routed < a.row_cap ? routed : a.row_cap);
        a.meta[3] = 0;  // the call's status: the staged kernels have no bounded waits
        a.meta[4] = largest;
      }
    }
  }
  __syncthreads();
  if (writer) {
    for (int e = threadIdx.x; e <= a.num_experts; e += blockDim.x) a.offsets[e] = s_off[e];
    for (int e = threadIdx.x; e < a.num_experts; e += blockDim.x) {
      a.counts[e] = s_tot[e];
      if (a.stats != nullptr) a.stats[e] += s_tot[e];
    }
  }
}

// A routing launch that GEMM1 stands in for (the live tasks fit its in-kernel routing).
__device__ __forceinline__ bool route_skipped(const RouteArgs& a) {
  return a.fused_max_tasks > 0 &&
         static_cast<int64_t>(effective_tokens(a.runtime_tokens, a.host_tokens)) * a.topk <= a.fused_max_tasks;
}

// The routing launch runs before the GEMMs of a layer: it zeroes their claim counters.
__device__ __forceinline__ void zero_sched(const RouteArgs& a) {
  if (blockIdx.x == 0 && a.zero_ints != nullptr)
    for (int i = threadIdx.x; i < a.zero_count; i += blockDim.x) a.zero_ints[i] = 0;
}

// One launch, a workgroup an expert and one more: workgroup e reads all the tasks, each of its 16
// waves a contiguous range that stays in registers (up to 16 passes of 64 tasks), and counts with two
// ballots a pass the tasks of lower experts (its row offset) and its own (the waves' bases); then
// its own tasks' lanes write their rows. The last workgroup counts every expert, marks the tasks
// without one and publishes counts, offsets, stats and meta. No workgroup waits for another.
//
// kBatch passes of the wave from task `begin` on, 32-bit task numbers: the experts, or -1.
template <typename Id>
__device__ __forceinline__ void expert_load(const RouteArgs& a, const Id* idx, int begin, int end, int* ev) {
  Id id[kBatch];
  float w[kBatch];
#pragma unroll
  for (int p = 0; p < kBatch; ++p) {
    const uint32_t t = min(begin + p * kWave + lane_id(), end - 1);
    id[p] = idx[t];
    w[p] = a.topk_w[t];
  }
#pragma unroll
  for (int p = 0; p < kBatch; ++p)
    ev[p] = begin + p * kWave + lane_id() < end ? valid_expert(a, static_cast<int64_t>(id[p]), w[p]) : -1;
}

__device__ __forceinline__ void expert_load(const RouteArgs& a, int begin, int end, int* ev) {
  if (a.idx_i64) expert_load(a, static_cast<const int64_t*>(a.topk_idx), begin, end, ev);
  else expert_load(a, static_cast<const int32_t*>(a.topk_idx), begin, end, ev);
}

__global__ __launch_bounds__(kExpertThreads) void route_expert_kernel(RouteArgs a) {
  zero_sched(a);  // (also when GEMM1 routes: the WIDE GEMM1 then returns at once, and the
                  // combine reads its zero-fill claim counter as zero)
  if (route_skipped(a)) return;
  __shared__ int s_cnt[kExpertWaves][kExpertMaxExperts];
  __shared__ int s_tot[kExpertMaxExperts];
  __shared__ int s_off[kExpertMaxExperts + 1];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int E = a.num_experts;
  const int e = blockIdx.x;
  const int ntasks = effective_tokens(a.runtime_tokens, a.host_tokens) * a.topk;
  const int per = ((ntasks + kExpertWaves - 1) / kExpertWaves + kWave - 1) / kWave * kWave;
  const int begin = min(wave * per, ntasks);
  const int end = min(begin + per, ntasks);
  if (e == E) {
    for (int i = threadIdx.x; i < kExpertWaves * E; i += kExpertThreads) s_cnt[i / E][i % E] = 0;
    __syncthreads();
    // (LDS atomics into the wave's own row: integer sums, so the order of the lanes is no matter)
    for (int b = begin; b < end; b += kBatch * kWave) {
      int ev[kBatch];
      expert_load(a, b, end, ev);
#pragma unroll
      for (int p = 0; p < kBatch; ++p) {
        const int task = b + p * kWave + lane;
        if (ev[p] >= 0) atomicAdd(&s_cnt[wave][ev[p]], 1);
        else if (task < end) a.output_index[task] = -1;
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < E; i += kExpertThreads) {
      int run = 0;
      for (int w = 0; w < kExpertWaves; ++w) run += s_cnt[w][i];
      s_tot[i] = run;
    }
    __syncthreads();
    publish_offsets(a, s_tot, s_off, true);
    return;
  }
  constexpr int P = kExpertPasses;
  int ev[P];
  int lower = 0, own = 0;
#pragma unroll
  for (int p0 = 0; p0 < P; p0 += kBatch) {
    if (begin + p0 * kWave >= end) break;
    expert_load(a, begin + p0 * kWave, end, ev + p0);
#pragma unroll
    for (int p = p0; p < p0 + kBatch; ++p) {
      own += __popcll(__ballot(ev[p] == e));
      lower += __popcll(__ballot(static_cast<unsigned>(ev[p]) < static_cast<unsigned>(e)));  // (-1: not lower)
    }
  }
  if (lane == 0) {
    s_cnt[wave][0] = own;
    s_cnt[wave][1] = lower;
  }
  if (a.given_counts != nullptr && wave == 0) {  // the caller's counts place the experts
    int given = 0;
    for (int i = lane; i < e; i += kWave) given += a.given_counts[i];
    given = __shfl(wave_inclusive_sum(given), kWave - 1, kWave);
    if (lane == 0) s_off[0] = given;
  }
  __syncthreads();
  int row = a.given_counts != nullptr ? s_off[0] : 0;
#pragma unroll
  for (int w = 0; w < kExpertWaves; ++w)
    row += (a.given_counts != nullptr ? 0 : s_cnt[w][1]) + (w < wave ? s_cnt[w][0] : 0);
#pragma unroll
  for (int p0 = 0; p0 < P; p0 += kBatch) {
    if (begin + p0 * kWave >= end) break;
#pragma unroll
    for (int p = p0; p < p0 + kBatch; ++p) {
      const uint64_t m = __ballot(ev[p] == e);
      if (m == 0) continue;
      if (ev[p] == e) {
        const int task = begin + p * kWave + lane;
        const int r = row + __popcll(m & lanes_below());
        const bool kept = r < a.row_cap;
        a.output_index[task] = kept ? r : -1;
        if (kept) {
          a.row_token[r] = task / a.topk;
          if (a.row_weight != nullptr) a.row_weight[r] = a.topk_w[task];
          if (a.m_indices != nullptr) a.m_indices[r] = e;
        }
      }
      row += __popcll(m);
    }
  }
}

// The tasks of chunk `chunk` that wave `wave` of a chunk workgroup routes: the same split in
// the count and the scatter kernels, so the scatter can take the count kernel's per-wave counts.
struct WaveRange {
  int64_t begin, end;
};
__device__ __forceinline__ WaveRange chunk_wave_range(int64_t ntasks, int chunk, int chunk_tasks, int wave) {
  const int64_t cbegin = static_cast<int64_t>(chunk) * chunk_tasks;
  const int64_t cend = cbegin + chunk_tasks < ntasks ? cbegin + chunk_tasks : ntasks;
  const int64_t per = ((chunk_tasks / kChunkWaves) + kWave - 1) / kWave * kWave;
  const int64_t begin = cbegin + wave * per < cend ? cbegin + wave * per : cend;
  return WaveRange{begin, begin + per < cend ? begin + per : cend};
}

// Per-wave counts of a chunk (each wave's ballot counts of its own task range, no atomics);
// writes the chunk's totals and, when wave_counts is given, the per-wave rows.
__global__ __launch_bounds__(kChunkThreads) void route_count_kernel(RouteArgs a, int chunk_tasks) {
  __shared__ int s_cnt[kChunkWaves][kMaxExperts];
  zero_sched(a);
  if (route_skipped(a)) return;
  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int E = a.num_experts;
  for (int i = tid; i < kChunkWaves * E; i += kChunkThreads) s_cnt[i / E][i % E] = 0;
  __syncthreads();
  const int64_t ntasks =
      static_cast<int64_t>(effective_tokens(a.runtime_tokens, a.host_tokens)) * a.topk;
  const WaveRange wr = chunk_wave_range(ntasks, blockIdx.x, chunk_tasks, wave);
  wave_count_range(a, wr.begin, wr.end, s_cnt[wave]);
  __syncthreads();
  int32_t* dst = a.chunk_counts + static_cast<int64_t>(blockIdx.x) * E;
  for (int e = tid; e < E; e += kChunkThreads) {
    int tot = 0;
#pragma unroll
    for (int w = 0; w < kChunkWaves; ++w) tot += s_cnt[w][e];
    dst[e] = tot;
  }
  if (a.wave_counts != nullptr) {
    int32_t* wdst = a.wave_counts + static_cast<int64_t>(blockIdx.x) * kChunkWaves * E;
    for (int i = tid; i < kChunkWaves * E; i += kChunkThreads) wdst[i] = s_cnt[i / E][i % E];
  }
}


__global__ __launch_bounds__(kChunkThreads) void route_chunk_scatter_kernel(RouteArgs a,
                                                                            int chunk_tasks,
                                                                            int num_chunks) {
  if (route_skipped(a)) return;
  __shared__ int s_wbase[kChunkWaves][kMaxExperts];
  __shared__ int s_tot[kMaxExperts];
  __shared__ int s_off[kMaxExperts + 1];
  __shared__ int s_cbase[kMaxExperts];
  __shared__ int s_part[2 * kChunkThreads];  // 2 * groups * E <= 2 * 1024
  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int E = a.num_experts;
  const int chunk = blockIdx.x;
  // Every load that does not wait for another goes out first: this wave's tasks, the count kernel's
  // per-wave counts of this chunk (same task split; null: count again) and every chunk's counts.
  // Side by side, and without the passes past a wave's range, they took the two launches from 17.2 to
  // 10.9 us at 49,152 tasks and from 21.0 to 18.9 at 1.57 M (32 of 256 experts).
  const int64_t ntasks =
      static_cast<int64_t>(effective_tokens(a.runtime_tokens, a.host_tokens)) * a.topk;
  const WaveRange wr = chunk_wave_range(ntasks, chunk, chunk_tasks, wave);
  WaveTasks tasks;
  wave_load<kBatch>(a, wr.begin, wr.end, tasks.ev, tasks.wv);
  const bool counted = a.wave_counts != nullptr;
  const int32_t* wsrc = counted ? a.wave_counts + static_cast<int64_t>(chunk) * kChunkWaves * E : nullptr;
  for (int i = tid; i < kChunkWaves * E; i += kChunkThreads) s_wbase[i / E][i % E] = counted ? wsrc[i] : 0;
  // Totals and this chunk's base per expert, from every chunk's counts. Thread t sums the
  // chunks g, g + G, g + 2G, ... of expert e = t % E (g = t / E, G = 1024 / E groups), so all
  // threads load at once (consecutive threads, consecutive experts of a chunk row); the G
  // partial sums of an expert then meet in LDS.
  {
    const int groups = kChunkThreads / E;  // >= 1: E <= kMaxExperts == kChunkThreads
    int* s_ptot = s_part;
    int* s_pbase = s_part + groups * E;
    if (tid < groups * E) {
      const int e = tid % E, g = tid / E;
      int tot = 0, base = 0;
      int c = g;
      for (; c + 7 * groups < num_chunks; c += 8 * groups) {  // 8 loads in flight together
        int v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = a.chunk_counts[static_cast<int64_t>(c + j * groups) * E + e];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          tot += v[j];
          base += c + j * groups < chunk ? v[j] : 0;
        }
      }
      for (; c < num_chunks; c += groups) {
        const int v = a.chunk_counts[static_cast<int64_t>(c) * E + e];
        tot += v;
        base += c < chunk ? v : 0;
      }
      s_ptot[g * E + e] = tot;
      s_pbase[g * E + e] = base;
    }
    __syncthreads();
    for (int e = tid; e < E; e += kChunkThreads) {
      int tot = 0, base = 0;
      for (int g = 0; g < groups; ++g) {
        tot += s_ptot[g * E + e];
        base += s_pbase[g * E + e];
      }
      s_tot[e] = tot;
      s_cbase[e] = base;
    }
    __syncthreads();
  }
  publish_offsets(a, s_tot, s_off, chunk == 0);
  wave_route(a, wr.begin, wr.end, s_wbase[wave], tasks, [&]() {
    __syncthreads();
    for (int e = tid; e < E; e += kChunkThreads) {
      int run = s_off[e] + s_cbase[e];
      for (int w = 0; w < kChunkWaves; ++w) {
        const int c = s_wbase[w][e];
        s_wbase[w][e] = run;
        run += c;
      }
    }
    __syncthreads();
  }, counted);
}

}  // namespace

int64_t route_chunk_tasks(int64_t ntasks) {
  // <= 256 chunks (one workgroup each), at least 1024 tasks per chunk, multiple of 1024
  int64_t chunk = (ntasks + 255) / 256;
  chunk = (chunk + kRouteChunk - 1) / kRouteChunk * kRouteChunk;
  return chunk < kRouteChunk ? kRouteChunk : chunk;
}

hipError_t launch_route(const RouteArgs& a, int64_t max_tasks, hipStream_t stream) {
  if (max_tasks <= 0) return hipSuccess;
  if (max_tasks <= kExpertMaxTasks && a.num_experts <= kExpertMaxExperts) {
    return launch_kernel(route_expert_kernel, dim3(static_cast<unsigned>(a.num_experts + 1)),
                         dim3(kExpertThreads), 0, stream, a);
  }
  const int64_t chunk = route_chunk_tasks(max_tasks);
  const int64_t chunks = (max_tasks + chunk - 1) / chunk;
  const hipError_t err = launch_kernel(route_count_kernel, dim3(static_cast<unsigned>(chunks)),
                                       dim3(kChunkThreads), 0, stream, a, static_cast<int>(chunk));
  if (err != hipSuccess) return err;
  return launch_kernel(route_chunk_scatter_kernel, dim3(static_cast<unsigned>(chunks)),
                       dim3(kChunkThreads), 0, stream, a, static_cast<int>(chunk),
                       static_cast<int>(chunks));
}

}  // namespace mmoe
