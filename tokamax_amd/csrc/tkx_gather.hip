// Row gather with optional mask, weight and reduction: the token permute / un-permute steps either
// side of the ragged dot in an MoE layer.
//
//   out[j, :] = sum over r < R of  keep(jR + r) * weight[jR + r] * x[indices[jR + r], :]
//
// R = 1 without weights is a plain gather (ragged_gather/base.py:25-32); with the row range
// [start, end) as the keep test on the index it is ragged_scatter/base.py:26-38; with weights, a
// validity mask and R > 1 it is ragged_gather_reduce/base.py:26-40 (products and sums in f32, one
// rounding to the output type). Bound by HBM: a workgroup moves one output row with 16-byte accesses.
#include "tkx_common.h"
#include "tkx_gemm.hip.h"

namespace tkx {
namespace {

constexpr int kGatherThreads = 256;

struct GatherParams {
  const unsigned char* x;
  const int32_t* indices;
  const float* weights;          // per gathered row, or null
  const unsigned char* valid;    // per gathered row (bytes, nonzero = keep), or null
  const int32_t* start;          // device scalars: keep rows with start <= index < end, or null
  const int32_t* end;
  unsigned char* out;
  int64_t in_rows, out_rows;
  int32_t hidden, reduce, dtype;  // hidden elements per row; rows reduced per output row
};

// R: gathered rows per output row whose index, mask and weight are read once per row and whose pieces are all loaded
// before the first is used (more than R, for R = 8 only: one after the other behind them); U: 16-byte pieces of the
// output row a thread has in flight. Bound by HBM, and for a few rows by the trips to memory in a row: every index, mask
// byte and weight requested together, then every piece, makes three where one after the other made up to 24. Before and
// now, bf16: combine of 4 tokens of 8 experts, hidden 2048, 9.9 -> 6.3 us; of 8192 tokens of 2 experts, hidden 4096,
// 50 -> 36 us (5.5 TB/s); gather of 16384 rows of 4096 50 -> 43 us (4.7 TB/s).
template <int ESZ, int R, int U>
__global__ __launch_bounds__(kGatherThreads) void gather_rows_kernel(const GatherParams p) {
  constexpr int PER = 16 / ESZ;  // elements per 16-byte access
  const int chunks = p.hidden / PER;
  const bool ranged = p.start != nullptr;
  const int lo = ranged ? p.start[0] : 0, hi = ranged ? p.end[0] : 0;
  const int step = kGatherThreads * gridDim.y;  // (a row's pieces over the workgroups along y)
  for (int64_t j = blockIdx.x; j < p.out_rows; j += gridDim.x) {
    // Source row (-1: dropped) of gathered row idx.
    auto source = [&](int idx, bool kept) -> int64_t {
      const bool keep = kept && (!ranged || (idx >= lo && idx < hi));
      // x[indices] as the reference's indexing reads it: a negative index counts from the end, and what is
      // still outside the array after that is clamped to the nearest row.
      const int64_t wrapped = idx < 0 ? (int64_t)idx + p.in_rows : (int64_t)idx;
      return !keep ? -1 : wrapped < 0 ? 0 : wrapped >= p.in_rows ? p.in_rows - 1 : wrapped;
    };
    // (All R indices, mask bytes and weights are requested before the first is looked at; entries past `reduce` repeat
    // the last one and are dropped.)
    int idx[R];
    unsigned char kept[R];
    int64_t rows[R];
    float wts[R];
#pragma unroll
    for (int r = 0; r < R; ++r) idx[r] = p.indices[j * p.reduce + min(r, p.reduce - 1)];
#pragma unroll
    for (int r = 0; r < R; ++r) kept[r] = 1;
    if (p.valid) {
#pragma unroll
      for (int r = 0; r < R; ++r) kept[r] = p.valid[j * p.reduce + min(r, p.reduce - 1)];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) wts[r] = 1.f;
    if (p.weights) {
#pragma unroll
      for (int r = 0; r < R; ++r) wts[r] = p.weights[j * p.reduce + min(r, p.reduce - 1)];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) rows[r] = source(idx[r], kept[r] != 0 && r < p.reduce);
    for (int c0 = blockIdx.y * kGatherThreads + threadIdx.x; c0 < chunks; c0 += U * step) {
      auto load = [&](int64_t row, int c) {
        return *reinterpret_cast<const i32x4*>(p.x + (row * p.hidden + (int64_t)c * PER) * ESZ);
      };
      i32x4 v[U][R];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          v[u][r] = (i32x4){0, 0, 0, 0};
          if (rows[r] >= 0 && c0 + u * step < chunks) v[u][r] = load(rows[r], c0 + u * step);
        }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * step;
        if (c >= chunks) break;
        float acc[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) acc[e] = 0.f;
        auto add = [&](const i32x4& piece, float w) {
#pragma unroll
          for (int e = 0; e < PER; ++e) {
            float f;
            // (Elements go through a scalar first: a bit cast applied straight to a vector subscript
            // was seen to read element 0 whatever the index.)
            const int word = ESZ == 4 ? piece[e] : piece[e >> 1];
            if constexpr (ESZ == 4) f = __builtin_bit_cast(float, word);
            else if (p.dtype == TKX_BF16) f = __builtin_bit_cast(float, (unsigned)(((unsigned)word >> (16 * (e & 1))) << 16));
            else f = (float)__builtin_bit_cast(_Float16, (unsigned short)((unsigned)word >> (16 * (e & 1))));
            acc[e] += w * f;
          }
        };
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (rows[r] >= 0) add(v[u][r], wts[r]);
        for (int r = R; r < p.reduce; ++r) {
          const int64_t g = j * p.reduce + r, row = source(p.indices[g], !p.valid || p.valid[g] != 0);
          if (row >= 0) add(load(row, c), p.weights ? p.weights[g] : 1.f);
        }
        i32x4 o;
        if (p.reduce == 1 && p.weights == nullptr) {
          o = v[u][0];  // a pure copy keeps the bits (a dropped row: zeros)
        } else if constexpr (ESZ == 4) {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = __builtin_bit_cast(int, acc[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            unsigned short h0, h1;
            if (p.dtype == TKX_BF16) {
              h0 = __builtin_bit_cast(unsigned short, (__bf16)acc[2 * e]);
              h1 = __builtin_bit_cast(unsigned short, (__bf16)acc[2 * e + 1]);
            } else {
              h0 = __builtin_bit_cast(unsigned short, (_Float16)acc[2 * e]);
              h1 = __builtin_bit_cast(unsigned short, (_Float16)acc[2 * e + 1]);
            }
            o[e] = (int)((unsigned)h0 | ((unsigned)h1 << 16));
          }
        }
        *reinterpret_cast<i32x4*>(p.out + (j * p.hidden + (int64_t)c * PER) * ESZ) = o;
      }
    }
  }
}

template <int ESZ>
void launch_gather_kernel(const GatherParams& p, hipStream_t stream) {
  // One workgroup per output row, grid-stride beyond 32 rows per CU in flight; fewer rows than 4 per CU are cut into
  // pieces of 256 accesses.
  const int64_t rows = p.out_rows < 256 * 32 ? p.out_rows : 256 * 32;
  const int pieces = (p.hidden / (16 / ESZ) + kGatherThreads - 1) / kGatherThreads;
  const dim3 grid((unsigned)rows, rows < 1024 && pieces > 1 ? (unsigned)(pieces < 64 ? pieces : 64) : 1u);
  if (p.reduce == 1) gather_rows_kernel<ESZ, 1, 2><<<grid, dim3(kGatherThreads), 0, stream>>>(p);
  else if (p.reduce == 2) gather_rows_kernel<ESZ, 2, 2><<<grid, dim3(kGatherThreads), 0, stream>>>(p);
  else gather_rows_kernel<ESZ, 8, 1><<<grid, dim3(kGatherThreads), 0, stream>>>(p);
}

}  // namespace

int32_t launch_gather_rows(const void* x, const int32_t* indices, const float* weights, const unsigned char* valid,
                           const int32_t* start, const int32_t* end, void* out, int64_t in_rows, int64_t out_rows,
                           int64_t hidden, int64_t reduce, int32_t dtype, hipStream_t stream) {
  GatherParams p;
  p.x = static_cast<const unsigned char*>(x);
  p.indices = indices;
  p.weights = weights;
  p.valid = valid;
  p.start = start;
  p.end = end;
  p.out = static_cast<unsigned char*>(out);
  p.in_rows = in_rows;
  p.out_rows = out_rows;
  p.hidden = (int32_t)hidden;
  p.reduce = (int32_t)reduce;
  p.dtype = dtype;
  if (out_rows < 1) return TKX_OK;
  if (dtype == TKX_F32) launch_gather_kernel<4>(p, stream);
  else launch_gather_kernel<2>(p, stream);
  TKX_HIP_CHECK(hipGetLastError());
  return TKX_OK;
}

}  // namespace tkx
