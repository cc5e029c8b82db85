// Group-offset prefix sum + tile scheduler: one workgroup, everything in LDS.
//
// Produces, bit for bit, what the reference's GroupInfo.create_aligned computes with XLA ops
// (tokamax/_src/ops/ragged_dot/pallas_mosaic_gpu_common.py:119-151), plus the group offsets and
// the number of tasks that belong to non-empty groups. For callers that want those arrays: the GEMM
// kernels work out their tiles themselves (tkx_gemm.hip.h, GroupScan).
#include "tkx_common.h"
#include "tkx_gemm.hip.h"

namespace tkx {
namespace {

constexpr int kThreads = 256;

// Exclusive scan of `partial` (one value per thread) across the workgroup; returns this thread's
// exclusive prefix and writes the grand total to *total. `buf` holds 2*kThreads ints.
__device__ inline int32_t block_exclusive_scan(int32_t v, int32_t* buf, int32_t* total) {
  const int t = threadIdx.x;
  int32_t* a = buf;
  int32_t* b = buf + kThreads;
  a[t] = v;
  __syncthreads();
  for (int d = 1; d < kThreads; d <<= 1) {
    int32_t x = a[t];
    if (t >= d) x += a[t - d];
    b[t] = x;
    __syncthreads();
    int32_t* tmp = a;
    a = b;
    b = tmp;
  }
  int32_t incl = a[t];
  *total = a[kThreads - 1];
  __syncthreads();
  return incl - v;
}

__global__ __launch_bounds__(kThreads) void schedule_kernel(const int32_t* __restrict__ group_sizes, int32_t G,
                                                             int32_t tile, int32_t tid_size, int32_t align_tile,
                                                             int32_t span_width, int32_t* __restrict__ ws,
                                                             int64_t off_offsets, int64_t off_gid, int64_t off_bstart,
                                                             int64_t off_astart, int64_t off_aend, int64_t off_swb,
                                                             int64_t off_asize, int64_t off_sfirst, int64_t off_swidth) {
  extern __shared__ int32_t smem[];
  int32_t* scan_buf = smem;                         // 2*kThreads
  int32_t* starts = smem + 2 * kThreads;            // G+1 : exclusive cumsum of clamped sizes
  int32_t* start_tasks = starts + (G + 1);          // G+1 : exclusive cumsum of blocks per group
  const int t = threadIdx.x;
  const int per = (G + kThreads - 1) / kThreads;
  const int lo = min(t * per, G), hi = min(lo + per, G);

  auto size_of = [&](int g) -> int32_t { return max(group_sizes[g], 0); };
  // pass 1: group starts
  int32_t local = 0;
  for (int g = lo; g < hi; ++g) local += size_of(g);
  int32_t total_rows;
  int32_t run = block_exclusive_scan(local, scan_buf, &total_rows);
  for (int g = lo; g < hi; ++g) {
    starts[g] = run;
    run += size_of(g);
  }
  if (t == 0) starts[G] = total_rows;
  __syncthreads();

  // pass 2: blocks per group -> first task of each group
  auto blocks_of = [&](int g) -> int32_t {
    int32_t sz = size_of(g);
    int32_t aligned = (starts[g] / align_tile) * align_tile;
    return sz == 0 ? 0 : (starts[g] + sz - aligned + tile - 1) / tile;
  };
  local = 0;
  for (int g = lo; g < hi; ++g) local += blocks_of(g);
  int32_t num_tasks;
  run = block_exclusive_scan(local, scan_buf, &num_tasks);
  for (int g = lo; g < hi; ++g) {
    start_tasks[g] = run;
    run += blocks_of(g);
  }
  if (t == 0) {
    start_tasks[G] = num_tasks;
    ws[0] = num_tasks;
    ws[1] = total_rows;
    ws[2] = 0;
  }
  __syncthreads();

  for (int g = t; g <= G; g += kThreads) ws[off_offsets + g] = starts[g];

  // pass 3: tasks. group = #{ j < G-1 : end_task[j] <= task }, end_task[j] == start_tasks[j+1].
  for (int task = t; task < tid_size; task += kThreads) {
    int l = 0, h = G - 1;  // search in start_tasks[1 .. G-1]
    while (l < h) {
      int mid = (l + h) >> 1;
      if (start_tasks[mid + 1] <= task) l = mid + 1; else h = mid;
    }
    const int g = l;
    const int32_t sz = size_of(g);
    const int32_t aligned = (starts[g] / align_tile) * align_tile;
    const int32_t end = starts[g] + sz;
    const int32_t bs = aligned + tile * (task - start_tasks[g]);
    const int32_t vs = max(bs, starts[g]);
    const int32_t ve = min(bs + tile, end);
    ws[off_gid + task] = g;
    ws[off_bstart + task] = bs;
    ws[off_astart + task] = vs;
    ws[off_aend + task] = ve;
    ws[off_swb + task] = vs - bs;
    ws[off_asize + task] = max(0, ve - vs);
    // Span of this task: the group's T tasks are cut into ceil(T / span_width) spans of nearly equal
    // width, so that the tasks that run side by side on an n-panel all use the same group's weights.
    int32_t sfirst = task, swidth = 1;
    // (Sizes that add up to more than m rows make more tasks than slots: spans end with the slots, so that the
    // launch order, which walks whole spans, stays inside the arrays.)
    const int32_t T = min(start_tasks[g + 1], tid_size) - start_tasks[g], idx = task - start_tasks[g];
    if (task < num_tasks && idx < T) {
      const int32_t nspans = (T + span_width - 1) / span_width;
      const int32_t base = T / nspans, extra = T - base * nspans;  // the first `extra` spans are one wider
      const int32_t wide = extra * (base + 1);
      if (idx < wide) {
        swidth = base + 1;
        sfirst = idx / swidth * swidth;
      } else {
        swidth = base;
        sfirst = wide + (idx - wide) / base * base;
      }
      sfirst += start_tasks[g];
    }
    ws[off_sfirst + task] = sfirst;
    ws[off_swidth + task] = swidth;
  }
}

// ---- the tasks of a GEMM launch -----------------------------------------------------------------------
constexpr int kPlanThreads = 256, kPlanWaves = kPlanThreads / 64, kPlanChunks = (int)(kPlanGroups / 256);

// a[0 .. n) += everything in front of it, and `first`: inclusive, saturating at `limit`. One wave.
__device__ __forceinline__ void scan_in_place(int* a, int n, int first, int limit, int lane) {
  for (int i = 0; i < n; i += 64) {
    const int v = min(first + wave_scan(i + lane < n ? a[i + lane] : 0, limit), limit);
    if (i + lane < n) a[i + lane] = v;
    first = __builtin_amdgcn_readlane(v, 63);
  }
}

// What the waves of a GEMM launch otherwise work out one by one (GroupScan), an entry per task: GemmParams::plan. For
// launches with so many groups, or so many workgroups, that the work in every one of them costs more than a kernel in
// front (launch order and row ranges are the same). Every workgroup adds up the groups in chunks of 256, then each wave
// takes 64 tasks. DRHS: the rows of 256 groups per wave instead.
template <int BM, int ALIGN, bool DRHS>
__global__ __launch_bounds__(kPlanThreads) void plan_kernel(const GemmParams p, int32_t unit, int32_t* __restrict__ plan) {
  __shared__ int rows_before[kPlanChunks + 1], tasks_before[kPlanChunks + 1];  // of every chunk
  __shared__ int part[kPlanWaves];
  __shared__ int upto[kPlanWaves][256], starts[kPlanWaves][256], ends[kPlanWaves][256];  // of a wave's current chunk
  typedef GroupScan<BM, ALIGN> Scan;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = DRHS ? p.k_ext : p.m_ext, chunks = (p.num_groups + 255) / 256;
  const int offset = p.group_offset != nullptr ? __builtin_amdgcn_readfirstlane(p.group_offset[0]) : 0;
  // Rows of the groups in front of the first one.
  int rows = 0;
  for (int j = threadIdx.x; j < min(max(offset, 0), p.num_global); j += kPlanThreads) rows = min(rows + min(max(p.group_sizes[j], 0), m), m);
  rows = wave_scan(rows, m);
  if (lane == 63) part[wave] = rows;
  for (int c = wave; c < chunks; c += kPlanWaves) {
    Scan sc;
    sc.scan(p, m, c * 256, offset, lane, 0, 0);
    if (lane == 0) rows_before[c + 1] = sc.rows;
  }
  __syncthreads();
  int lead = 0;
  for (int w = 0; w < kPlanWaves; ++w) lead = min(lead + part[w], m);
  if (wave == 0) {
    if (lane == 0) rows_before[0] = lead;
    scan_in_place(rows_before + 1, chunks, lead, m, lane);
  }
  __syncthreads();
  if constexpr (DRHS) {
    const int c = blockIdx.x * kPlanWaves + wave;
    if (c < chunks) {
      Scan sc;
      sc.scan(p, m, c * 256, offset, lane, rows_before[c], 0);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c * 256 + 4 * lane + e < p.num_groups) plan[c * 256 + 4 * lane + e] = sc.start[e];
      if (c == chunks - 1 && lane == 0) plan[p.num_groups] = sc.rows;
    }
  } else {
    for (int c = wave; c < chunks; c += kPlanWaves) {
      Scan sc;
      sc.scan(p, m, c * 256, offset, lane, rows_before[c], 0);
      if (lane == 0) tasks_before[c + 1] = sc.total;
    }
    __syncthreads();
    if (wave == 0) {
      if (lane == 0) tasks_before[0] = 0;
      scan_in_place(tasks_before + 1, chunks, 0, 0x7fffffff, lane);
    }
    __syncthreads();
    const int total = min(tasks_before[chunks], p.plan_stride);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      plan[0] = total;
      plan[1] = rows_before[chunks];
      plan[2] = lead;
    }
    const int first = (blockIdx.x * kPlanWaves + wave) * 64, last = min(first + 64, total), task = first + lane;
    int32_t* const out = plan + kWsHeader;
    for (int t = first; t < last;) {
      // The chunk that owns task t: the first one that ends behind it.
      int lo = 0, hi = chunks - 1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (tasks_before[mid + 1] > t) hi = mid;
        else lo = mid + 1;
      }
      const int c = __builtin_amdgcn_readfirstlane(lo), before = tasks_before[c], behind = min(tasks_before[c + 1], last);
      Scan sc;
      sc.scan(p, m, c * 256, offset, lane, rows_before[c], before);
      int at = sc.tasks_upto - (sc.tasks[0] + sc.tasks[1] + sc.tasks[2] + sc.tasks[3]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        upto[wave][4 * lane + e] = at += sc.tasks[e];
        starts[wave][4 * lane + e] = sc.start[e];
        ends[wave][4 * lane + e] = sc.end[e];
      }
      __threadfence_block();
      if (task >= t && task < behind) {
        int g = 0, h = 255;  // the first group that ends behind this task
        while (g < h) {
          const int mid = (g + h) >> 1;
          if (upto[wave][mid] > task) h = mid;
          else g = mid + 1;
        }
        const int first_task = g == 0 ? before : upto[wave][g - 1], tasks = upto[wave][g] - first_task, mt = task - first_task;
        const TaskRows r = task_rows<ALIGN>(starts[wave][g], ends[wave][g], tasks, mt, unit);
        int span = 0, width = tasks;
        if (tasks > p.grid_tile_width) {
          const int spans = (tasks + p.grid_tile_width - 1) / p.grid_tile_width;
          const int base = tasks / spans, wide = (tasks - base * spans) * (base + 1);  // the first spans are one task wider
          width = mt < wide ? base + 1 : base;
          span = mt < wide ? mt / width * width : wide + (mt - wide) / width * width;
        }
        out[task] = c * 256 + g;
        out[p.plan_stride + task] = r.row0;
        out[2 * p.plan_stride + task] = r.first;
        out[3 * p.plan_stride + task] = r.end;
        out[4 * p.plan_stride + task] = first_task + span;
        out[5 * p.plan_stride + task] = width;
      }
      __threadfence_block();
      t = behind;
    }
  }
}

__global__ __launch_bounds__(kThreads) void clear_words_kernel(int32_t* __restrict__ words, int32_t count) {
  for (int i = threadIdx.x; i < count; i += kThreads) words[i] = 0;
}

}  // namespace

// (a kernel, not a memset: callers may be capturing a graph)
int32_t launch_clear_words(int32_t* words, int32_t count, hipStream_t stream) {
  clear_words_kernel<<<1, kThreads, 0, stream>>>(words, count);
  TKX_HIP_CHECK(hipGetLastError());
  return TKX_OK;
}

int32_t launch_plan(const GemmParams& p, bool drhs, int32_t block_m, int32_t unit, int32_t align, int32_t* plan, hipStream_t stream) {
  if (p.num_groups > kPlanGroups) return set_error(TKX_ERR_UNSUPPORTED, "too many groups for the task kernel");
  auto go = [&](auto kernel, int64_t items) {
    kernel<<<dim3((unsigned)((items + kPlanThreads - 1) / kPlanThreads)), dim3(kPlanThreads), 0, stream>>>(p, unit, plan);
  };
  if (drhs) {
    go(plan_kernel<1, 1, true>, (int64_t)(p.num_groups + 255) / 256 * 64);  // (a wave per 256 groups)
  } else {
#define TKX_PLAN(BM)                                                            \
  if (block_m == BM) {                                                          \
    if (align == 4) go(plan_kernel<BM, 4, false>, p.plan_stride);               \
    else go(plan_kernel<BM, 1, false>, p.plan_stride);                          \
  } else
    TKX_PLAN(32) TKX_PLAN(64) TKX_PLAN(128) TKX_PLAN(256) return set_error(TKX_ERR_UNSUPPORTED, "no task kernel for block_m=%d", block_m);
#undef TKX_PLAN
  }
  TKX_HIP_CHECK(hipGetLastError());
  return TKX_OK;
}

int32_t launch_schedule(const int32_t* group_sizes, int64_t G, int32_t block_m, int32_t align_tile, int32_t span_width,
                        int32_t* ws, const WsLayout& L, hipStream_t stream) {
  const size_t smem = sizeof(int32_t) * (size_t)(2 * kThreads + 2 * (G + 1));
  if (smem > 64 * 1024) return set_error(TKX_ERR_UNSUPPORTED, "num_groups=%lld too large for the scheduler", (long long)G);
  schedule_kernel<<<1, kThreads, smem, stream>>>(group_sizes, (int32_t)G, block_m, L.tid_size, align_tile,
                                                span_width < 1 ? 1 : span_width, ws, L.offsets, L.task[0], L.task[1],
                                                L.task[2], L.task[3], L.task[4], L.task[5], L.task[6], L.task[7]);
  TKX_HIP_CHECK(hipGetLastError());
  return TKX_OK;
}

}  // namespace tkx
