// Absmax quantisation with block scales: the inverse pass of tkx_dequant.hip.
//
//   scale[R, C] = max |x[r, c]| over the tile (R, C) / qmax      (1 where the tile is all zero)
//   q[r, c]     = convert(x[r, c] / scale[r / t_r, c / t_c])
//
// qmax is the largest finite value of the quantised type (127 for int8, 448 for OCP e4m3fn); convert rounds to
// nearest, ties to even, and saturates at +-qmax. This is the symmetric ("absmax") calibration that
// tokamax/_src/quantization.py:65-78 asks of qwix.quantize, in the form the reference states it itself for its fused
// output quantisation (pallas_mosaic_gpu_kernel_sm100_fp8_quant.py:802-822). x is f32, bf16 or f16, row-major.
//
// Three forms, all bound by HBM (the second read of a tile comes from cache where the tile is small):
//   * tiles one row tall (an lhs [m, k] with one scale per row or per (row, t_c columns)): a group of lanes owns a
//     tile, 8 elements per lane and step, keeps it in registers (up to 8192 columns of 16 bits) and reduces with lane
//     shuffles;
//   * tiles several rows tall (weights [g, k, n] as g * k rows with one scale per (group, column) or per
//     (t_r rows, column) or per (t_r x t_c) block): a workgroup owns t_r rows x 256 columns, 8 row slices of 32 lanes x
//     8 columns each, and reduces through LDS;
//   * any other tile several rows tall (one scale for a whole tensor, 512-column blocks, ...): the tile's maximum is
//     collected with an atomic maximum on its bit pattern, then a second pass converts.
#include "tkx_common.h"
#include "tkx_gemm.hip.h"

namespace tkx {
namespace {

constexpr int kQThreads = 256;

template <int EX> struct XVec;
template <> struct XVec<kEF32> { static constexpr int BYTES = 32; };
template <> struct XVec<kEBF16> { static constexpr int BYTES = 16; };
template <> struct XVec<kEF16> { static constexpr int BYTES = 16; };

// 8 consecutive elements of x as they lie in memory, and as f32.
template <int EX> struct Raw8 { i32x4 w[XVec<EX>::BYTES / 16]; };
template <int EX>
__device__ __forceinline__ Raw8<EX> load_raw8(const unsigned char* p) {
  Raw8<EX> r;
#pragma unroll
  for (int h = 0; h < XVec<EX>::BYTES / 16; ++h) r.w[h] = *reinterpret_cast<const i32x4*>(p + 16 * h);
  return r;
}
template <int EX>
__device__ __forceinline__ void widen8(const Raw8<EX>& r, float (&v)[8]) {
  if constexpr (EX == kEF32) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 a = __builtin_bit_cast(f32x4, r.w[h]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * h + e] = a[e];
    }
  } else if constexpr (EX == kEBF16) {
    const bf16x8 a = __builtin_bit_cast(bf16x8, r.w[0]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)a[e];
  } else {
    const f16x8 a = __builtin_bit_cast(f16x8, r.w[0]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)a[e];
  }
}
template <int EX>
__device__ __forceinline__ void load8(const unsigned char* p, float (&v)[8]) { widen8<EX>(load_raw8<EX>(p), v); }

__device__ __forceinline__ float absmax8(const float (&v)[8]) {
  float m = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[e]));
  return m;
}

__device__ __forceinline__ float scale_of(float absmax, QuantRange qr) { return absmax == 0.f ? 1.f : absmax / qr.bound; }

// 8 quotients -> 8 quantised bytes (two dwords).
template <int EQ>
__device__ __forceinline__ i32x2 convert8(const float (&v)[8], QuantRange qr) {
  i32x2 out;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = fminf(fmaxf(v[4 * h + e], qr.lo), qr.hi);
    if constexpr (EQ == kEI8) {
      unsigned w = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) w |= ((unsigned)(int)__builtin_rintf(q[e]) & 0xffu) << (8 * e);
      out[h] = (int)w;
    } else {
      int w = 0;
      w = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], w, false);
      w = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], w, true);
      out[h] = w;
    }
  }
  return out;
}

// 8 values / scale -> 8 quantised bytes.
template <int EQ>
__device__ __forceinline__ i32x2 quantize8(const float (&v)[8], const float (&scale)[8], QuantRange qr) {
  float q[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] = v[e] / scale[e];
  return convert8<EQ>(q, qr);
}

// v / s with the reciprocal r of s, rounded to nearest like s' own division: the product is within two units in the
// last place, the first correction within one, and a quotient that close is rounded correctly by the second (Markstein,
// IBM J. Res. Dev. 34, 1990). Six instructions where a division takes about twice as many. Holds while r and the remainders
// are normal numbers: `has_reciprocal`; a remainder that underflows belongs to a quotient far below the smallest
// quantised value, whose sign is all that counts.
__device__ __forceinline__ bool has_reciprocal(float s) { return s > 0x1p-60f && s < 0x1p60f; }
__device__ __forceinline__ float quotient(float v, float s, float r) {
  float q = v * r;
  q = __builtin_fmaf(__builtin_fmaf(-q, s, v), r, q);
  // (-0 has a remainder of +0, which would take its sign)
  return __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-q, s, v), r, q), v);
}

// 8 values / one scale -> 8 quantised bytes; `near`: every lane's scale has a reciprocal (uniform), r.
template <int EQ>
__device__ __forceinline__ i32x2 quantize8(const float (&v)[8], float s, bool near, float r, QuantRange qr) {
  float q[8];
  if (near) {
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = quotient(v[e], s, r);
  } else {
    asm volatile("");  // (a branch: without it both sides are computed and selected from)
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = v[e] / s;
  }
  return convert8<EQ>(q, qr);
}

// Tiles one row tall. L lanes (a power of two <= 64) own one tile; a wave holds 64 / L tiles of consecutive
// (row, column-tile) pairs. CH > 0: tiles of at most 8 L CH columns, held in registers (every chunk of 8 loaded before
// the first is used), U such sets of tiles at a time: x is read once, with CH * U 16-byte loads of a lane in flight.
// CH == 0: wider tiles, walked twice. Bound by HBM, so the chunks are held as they lie in memory (4 registers per 8
// 16-bit elements; as f32 the 16-chunk form took 217 registers, two waves per SIMD, and lost up to 27 % to walking a tile
// twice). bf16 to fp8, every tile walked twice against this form, caches flushed in front of every pass: 16384 x 7168 per
// row 94.9 -> 62.7 us (5.6 TB/s), per 128 columns 104 -> 76.9 (4.6 TB/s), 16384 x 4096 per row 56.7 -> 37.0 (5.4 TB/s).
template <int EX, int EQ, int CH, int U>
__global__ __launch_bounds__(kQThreads) void quantize_rows_kernel(const unsigned char* __restrict__ x,
                                                                  unsigned char* __restrict__ q, float* __restrict__ scale,
                                                                  int64_t rows, int32_t cols, int32_t t_c, int32_t lanes,
                                                                  QuantRange qmax, bool scale_t) {
  constexpr int XB = XVec<EX>::BYTES;  // bytes of 8 elements of x
  const int L = CH == 1 ? lanes : 64;  // (a tile of more chunks than lanes has a whole wave: constant distances)
  const int lane = threadIdx.x & 63;
  const int tiles_per_row = cols / t_c;
  const int64_t num_tiles = rows * tiles_per_row;
  const int per_wave = 64 / L;
  int64_t wave_id = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) >> 6;
  if constexpr (CH != 1) wave_id = (int64_t)blockIdx.x * (kQThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t num_waves = ((int64_t)gridDim.x * kQThreads) >> 6;
  const int sub = lane / L, l = lane % L;
  const int chunks = t_c / 8;
  for (int64_t t0 = wave_id * per_wave * U; t0 < num_tiles; t0 += num_waves * per_wave * U) {
    float m[U];
    Raw8<EX> held[U][CH > 0 ? CH : 1];
    float v[8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // (Tile t's columns begin at element t * t_c: tiles are one row tall and whole in their rows.)
      const int64_t tile = t0 + u * per_wave + sub;
      const unsigned char* xr = x + tile * t_c * (XB / 8);
      m[u] = 0.f;
      if constexpr (CH > 0) {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          const int c = l + i * L;
          held[u][i] = Raw8<EX>{};
          if (tile < num_tiles && c < chunks) held[u][i] = load_raw8<EX>(xr + (int64_t)c * XB);
        }
      } else if (tile < num_tiles) {
        for (int c = l; c < chunks; c += L) {
          load8<EX>(xr + (int64_t)c * XB, v);
          m[u] = fmaxf(m[u], absmax8(v));
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t tile = t0 + u * per_wave + sub;
      if constexpr (CH > 0) {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          widen8<EX>(held[u][i], v);
          m[u] = fmaxf(m[u], absmax8(v));
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1)
        if (off < L) m[u] = fmaxf(m[u], __shfl_xor(m[u], off));
      const float s = scale_of(m[u], qmax);
      const bool near = __all(has_reciprocal(s));
      const float r = 1.f / s;
      if (tile < num_tiles) {
        if (l == 0) {
          int64_t at = tile;
          if (scale_t) {  // [cols / t_c, rows], the form in which the products with scale blocks along k read them
            const uint32_t row = (uint32_t)tile / (uint32_t)tiles_per_row;  // (fewer than 2^31 tiles)
            at = (int64_t)((uint32_t)tile - row * (uint32_t)tiles_per_row) * rows + row;
          }
          scale[at] = s;
        }
        unsigned char* qr = q + tile * t_c;
        if constexpr (CH > 0) {
#pragma unroll
          for (int i = 0; i < CH; ++i) {
            const int c = l + i * L;
            widen8<EX>(held[u][i], v);
            if (c < chunks) *reinterpret_cast<i32x2*>(qr + c * 8) = quantize8<EQ>(v, s, near, r, qmax);
          }
        } else {
          const unsigned char* xr = x + tile * t_c * (XB / 8);
          for (int c = l; c < chunks; c += L) {
            load8<EX>(xr + (int64_t)c * XB, v);
            *reinterpret_cast<i32x2*>(qr + c * 8) = quantize8<EQ>(v, s, near, r, qmax);
          }
        }
      }
    }
  }
}

// The form of `quantize_rows_kernel` for tiles of `per_lane` chunks a lane: held in registers up to 64 of them (16 chunks
// of 16-bit elements, 8 of f32), more sets of tiles at a time where a tile is short.
template <int EX, int EQ>
void launch_rows(int per_lane, int64_t tiles, int L, const unsigned char* x, unsigned char* q, float* scale, int64_t rows,
                 int32_t cols, int32_t t_c, QuantRange range, bool scale_t, hipStream_t stream) {
  auto go = [&](auto kernel, int sets) {
    const int64_t per_workgroup = (int64_t)(64 / L) * sets * (kQThreads / 64);
    int64_t grid = (tiles + per_workgroup - 1) / per_workgroup;
    if (grid > 256 * 16) grid = 256 * 16;
    if (grid < 1) grid = 1;
    kernel<<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(x, q, scale, rows, cols, t_c, (int32_t)L, range, scale_t);
  };
  // (Four sets at a time need so many tiles that every SIMD still gets waves of its own.)
  const bool many = tiles / (64 / L) >= 256 * 4 * 4 * 4;
  if (per_lane <= 1 && many) go(quantize_rows_kernel<EX, EQ, 1, 4>, 4);
  else if (per_lane <= 1) go(quantize_rows_kernel<EX, EQ, 1, 1>, 1);
  else if (per_lane <= 2) go(quantize_rows_kernel<EX, EQ, 2, 1>, 1);
  else if (per_lane <= 4) go(quantize_rows_kernel<EX, EQ, 4, 1>, 1);
  else if (per_lane <= 8) go(quantize_rows_kernel<EX, EQ, 8, 1>, 1);
  else if (EX != kEF32 && per_lane <= 16) go(quantize_rows_kernel<EX, EQ, EX != kEF32 ? 16 : 8, 1>, 1);
  else go(quantize_rows_kernel<EX, EQ, 0, 1>, 1);
}

// Tiles t_r > 1 rows tall and t_c columns wide (t_c == 1, or a power of two in [8, 256]). A workgroup owns
// (row tile, 256 columns): thread (slice = tid / 32, lane32 = tid % 32) takes columns 8 lane32 .. + 7 of the rows
// slice, slice + 8, ...
template <int EX, int EQ>
__global__ __launch_bounds__(kQThreads) void quantize_blocks_kernel(const unsigned char* __restrict__ x,
                                                                    unsigned char* __restrict__ q, float* __restrict__ scale,
                                                                    int64_t rows, int32_t cols, int32_t t_r, int32_t t_c,
                                                                    QuantRange qmax) {
  constexpr int XB = XVec<EX>::BYTES;
  __shared__ float red[8][256];
  const int tid = threadIdx.x, slice = tid >> 5, l32 = tid & 31;
  const int col_chunks = (cols + 255) / 256;
  const int64_t row_tile = blockIdx.x / col_chunks;
  const int c0 = (int)(blockIdx.x - row_tile * col_chunks) * 256 + 8 * l32;
  const bool live = c0 < cols;  // cols % 8 == 0
  const int64_t r0 = row_tile * t_r;
  float m[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) m[e] = 0.f;
  if (live) {
    for (int r = slice; r < t_r; r += 8) {
      float v[8];
      load8<EX>(x + ((r0 + r) * cols + c0) * (XB / 8), v);
#pragma unroll
      for (int e = 0; e < 8; ++e) m[e] = fmaxf(m[e], fabsf(v[e]));
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[slice][8 * l32 + e] = m[e];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float a = 0.f;
#pragma unroll
    for (int s_ = 0; s_ < 8; ++s_) a = fmaxf(a, red[s_][8 * l32 + e]);
    m[e] = a;
  }
  float s[8];
  if (t_c == 1) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = scale_of(m[e], qmax);
    if (live && slice == 0) {
      float* so = scale + row_tile * cols + c0;
      *reinterpret_cast<f32x4*>(so) = (f32x4){s[0], s[1], s[2], s[3]};
      *reinterpret_cast<f32x4*>(so + 4) = (f32x4){s[4], s[5], s[6], s[7]};
    }
  } else {
    float a = absmax8(m);
    const int lanes = t_c / 8;  // lanes (of the 32 that share a row) whose columns lie in one scale block
#pragma unroll
    for (int off = 16; off > 0; off >>= 1)
      if (off < lanes) a = fmaxf(a, __shfl_xor(a, off));
    const float one = scale_of(a, qmax);
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = one;
    if (live && slice == 0 && (l32 % lanes) == 0) scale[row_tile * (cols / t_c) + c0 / t_c] = one;
  }
  if (live) {
    for (int r = slice; r < t_r; r += 8) {
      float v[8];
      load8<EX>(x + ((r0 + r) * cols + c0) * (XB / 8), v);
      *reinterpret_cast<i32x2*>(q + (r0 + r) * cols + c0) = quantize8<EQ>(v, s, qmax);
    }
  }
}

// Any other tile several rows tall (wider than 256 columns, or not a power of two wide; t_c a multiple of 8): three
// passes over chunks of 8 consecutive elements, which never straddle a tile. (1) The tile's scale slot collects the bit
// pattern of max |x| with an integer atomic maximum (non-negative floats order like their bits; the result does not
// depend on the order of arrival); a wave whose chunks all lie in one tile reduces with shuffles first. (2) The slot
// becomes the scale. (3) The values are divided and converted. The slots are zeroed by the first kernel of the three.
__global__ void tile_slots_clear_kernel(float* __restrict__ scale, int64_t num_tiles) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < num_tiles; t += (int64_t)gridDim.x * blockDim.x) scale[t] = 0.f;
}

__device__ __forceinline__ int64_t tile_of_chunk(int64_t chunk, int32_t chunks_per_row, int32_t t_r, int32_t t_c, int32_t tiles_per_row,
                                                 int64_t* row, int32_t* col) {
  *row = chunk / chunks_per_row;
  *col = (int32_t)(chunk - *row * chunks_per_row) * 8;
  return (*row / t_r) * tiles_per_row + *col / t_c;
}

template <int EX>
__global__ __launch_bounds__(kQThreads) void tile_absmax_kernel(const unsigned char* __restrict__ x, float* __restrict__ scale,
                                                                int64_t rows, int32_t cols, int32_t t_r, int32_t t_c) {
  constexpr int XB = XVec<EX>::BYTES;
  const int32_t chunks_per_row = cols / 8, tiles_per_row = cols / t_c;
  const int64_t chunks = rows * chunks_per_row, stride = (int64_t)gridDim.x * kQThreads;
  // (Every lane of a wave runs the same number of rounds, so that the shuffles below see all 64 lanes.)
  for (int64_t base = (int64_t)blockIdx.x * kQThreads; base < chunks; base += stride) {
    const int64_t chunk = base + threadIdx.x;
    const bool live = chunk < chunks;
    int64_t row;
    int32_t col;
    const int64_t tile = tile_of_chunk(live ? chunk : chunks - 1, chunks_per_row, t_r, t_c, tiles_per_row, &row, &col);
    float m = 0.f;
    if (live) {
      float v[8];
      load8<EX>(x + (row * cols + col) * (XB / 8), v);
      m = absmax8(v);
    }
    const int64_t first = __shfl(tile, 0);
    if (__all(tile == first)) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
      if ((threadIdx.x & 63) == 0) atomicMax(reinterpret_cast<unsigned*>(scale) + tile, __builtin_bit_cast(unsigned, m));
    } else if (live) {
      atomicMax(reinterpret_cast<unsigned*>(scale) + tile, __builtin_bit_cast(unsigned, m));
    }
  }
}

__global__ void tile_scale_kernel(float* __restrict__ scale, int64_t num_tiles, QuantRange qmax) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < num_tiles; t += (int64_t)gridDim.x * blockDim.x)
    scale[t] = scale_of(scale[t], qmax);
}

template <int EX, int EQ>
__global__ __launch_bounds__(kQThreads) void quantize_tiles_kernel(const unsigned char* __restrict__ x, unsigned char* __restrict__ q,
                                                                   const float* __restrict__ scale, int64_t rows, int32_t cols,
                                                                   int32_t t_r, int32_t t_c, QuantRange qmax) {
  constexpr int XB = XVec<EX>::BYTES;
  const int32_t chunks_per_row = cols / 8, tiles_per_row = cols / t_c;
  const int64_t chunks = rows * chunks_per_row, stride = (int64_t)gridDim.x * kQThreads;
  for (int64_t chunk = (int64_t)blockIdx.x * kQThreads + threadIdx.x; chunk < chunks; chunk += stride) {
    int64_t row;
    int32_t col;
    const float s = scale[tile_of_chunk(chunk, chunks_per_row, t_r, t_c, tiles_per_row, &row, &col)];
    const float sv[8] = {s, s, s, s, s, s, s, s};
    float v[8];
    load8<EX>(x + (row * cols + col) * (XB / 8), v);
    *reinterpret_cast<i32x2*>(q + row * cols + col) = quantize8<EQ>(v, sv, qmax);
  }
}

template <int EX>
int32_t launch_for_x(const void* x, void* q, float* scale, int64_t rows, int64_t cols, int64_t t_r, int64_t t_c,
                     int32_t q_dtype, QuantRange qmax, bool scale_t, hipStream_t stream) {
  const auto* xb = static_cast<const unsigned char*>(x);
  auto* qb = static_cast<unsigned char*>(q);
  if (t_r == 1) {
    const int chunks = (int)(t_c / 8);
    const int L = (chunks < 64 && (chunks & (chunks - 1)) == 0) ? chunks : 64;
    const int64_t tiles = rows * (cols / t_c);
    const int per_lane = (chunks + L - 1) / L;
    if (q_dtype == TKX_I8)
      launch_rows<EX, kEI8>(per_lane, tiles, L, xb, qb, scale, rows, (int32_t)cols, (int32_t)t_c, qmax, scale_t, stream);
    else
      launch_rows<EX, kEF8>(per_lane, tiles, L, xb, qb, scale, rows, (int32_t)cols, (int32_t)t_c, qmax, scale_t, stream);
  } else if (t_c != 1 && !((t_c & (t_c - 1)) == 0 && t_c >= 8 && t_c <= 256)) {
    const int64_t num_tiles = (rows / t_r) * (cols / t_c), chunks = rows * (cols / 8);
    int64_t grid = (chunks + kQThreads - 1) / kQThreads;
    if (grid > 256 * 32) grid = 256 * 32;
    int64_t small = (num_tiles + 255) / 256;
    if (small > 1024) small = 1024;
    tile_slots_clear_kernel<<<dim3((unsigned)small), dim3(256), 0, stream>>>(scale, num_tiles);
    tile_absmax_kernel<EX><<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(xb, scale, rows, (int32_t)cols, (int32_t)t_r, (int32_t)t_c);
    tile_scale_kernel<<<dim3((unsigned)small), dim3(256), 0, stream>>>(scale, num_tiles, qmax);
    if (q_dtype == TKX_I8)
      quantize_tiles_kernel<EX, kEI8><<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(xb, qb, scale, rows, (int32_t)cols, (int32_t)t_r, (int32_t)t_c, qmax);
    else
      quantize_tiles_kernel<EX, kEF8><<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(xb, qb, scale, rows, (int32_t)cols, (int32_t)t_r, (int32_t)t_c, qmax);
  } else {
    const int64_t grid = (rows / t_r) * ((cols + 255) / 256);
    if (grid > 0x7fffffffLL) return set_error(TKX_ERR_UNSUPPORTED, "too many tiles");
    if (q_dtype == TKX_I8)
      quantize_blocks_kernel<EX, kEI8><<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(xb, qb, scale, rows, (int32_t)cols, (int32_t)t_r, (int32_t)t_c, qmax);
    else
      quantize_blocks_kernel<EX, kEF8><<<dim3((unsigned)grid), dim3(kQThreads), 0, stream>>>(xb, qb, scale, rows, (int32_t)cols, (int32_t)t_r, (int32_t)t_c, qmax);
  }
  TKX_HIP_CHECK(hipGetLastError());
  return TKX_OK;
}

}  // namespace

int32_t launch_quantize(const void* x, void* q, float* scale, int64_t rows, int64_t cols, int64_t t_r, int64_t t_c,
                        int32_t x_dtype, int32_t q_dtype, QuantRange qmax, bool scale_t, hipStream_t stream) {
  if (x_dtype == TKX_F32) return launch_for_x<kEF32>(x, q, scale, rows, cols, t_r, t_c, q_dtype, qmax, scale_t, stream);
  if (x_dtype == TKX_BF16) return launch_for_x<kEBF16>(x, q, scale, rows, cols, t_r, t_c, q_dtype, qmax, scale_t, stream);
  return launch_for_x<kEF16>(x, q, scale, rows, cols, t_r, t_c, q_dtype, qmax, scale_t, stream);
}

}  // namespace tkx
