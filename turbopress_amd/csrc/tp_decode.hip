// Window decode and generic GEMV over the natural format-v2 streams.
//
// Reference semantics:
//   * window_decode_levels  turbopress/runtime.py:122-139 (+ unpack_le :93-100)
//   * decode_rows           turbopress/runtime.py:291-301
//   * packed GEMV           turbopress/triton_kernel.py:44-157 (row scale
//                           factored out of an fp32 reduction, fp16 output)
//                           then the fp16 bias add of runtime.py:332-333.
//
// These kernels read the streams exactly as the reference stores them (byte-
// granular little-endian field reads), support every bits in [1, 7] and every
// S in {4, 8, 16, 64}, and serve as the bit-exact decode entry points and the
// general fallback GEMV.  The bandwidth-tuned path for k in {2, 3, 4} lives in
// tp_tiled.hip, tp_linear.hip, tp_stack.hip and tp_prefill.hip.
#include "tp_common.h"

namespace tp {

struct DecodeArgs {
  const uint8_t* path;
  int64_t path_stride;
  const uint8_t* member;
  int64_t member_stride;
  int64_t n_rows;
  int64_t d;
  int bits;
  int m;
  uint32_t g0w, g1w;
};

// The 8 columns from c (a multiple of 8) of row r: their path bits are byte
// c / 8 of the row, the up to 6 bits before them the byte before it (zero at
// the row's start), their members the bits - 1 bytes from c / 8 * (bits - 1)
// on.  Both subset bits of all 8 are XORs of the two path bytes shifted by the
// generators' taps (dm0, dm1: bit t set where the subset bit takes the path
// bit t columns back).  level[j] past the row's end is whatever zero stream
// bits decode to.
template <int BITS>
__device__ __forceinline__ void levels_of_8(const DecodeArgs& a, uint32_t dm0, uint32_t dm1, int64_t r, int64_t c,
                                            uint32_t level[8]) {
  const int64_t byte = c >> 3;
  const uint8_t* prow = a.path + r * a.path_stride + byte;
  const uint32_t p = ((uint32_t)prow[0] << 8) | (byte > 0 ? (uint32_t)prow[-1] : 0u);
  uint32_t e0 = 0, e1 = 0;
#pragma unroll
  for (int t = 0; t <= 6; ++t) {
    e0 ^= (p << t) & (0u - ((dm0 >> t) & 1u));
    e1 ^= (p << t) & (0u - ((dm1 >> t) & 1u));
  }
  constexpr int mb = BITS - 1;
  uint64_t mem = 0;  // 8 * mb bits
  if constexpr (mb > 0) {
    const uint8_t* mrow = a.member + r * a.member_stride;
    const int64_t m0 = byte * mb, mend = (a.d * mb + 7) >> 3;
    if (c + 8 <= a.d) {
#pragma unroll
      for (int i = 0; i < mb; ++i) mem |= (uint64_t)mrow[m0 + i] << (8 * i);
    } else {
#pragma unroll
      for (int i = 0; i < mb; ++i) mem |= (uint64_t)(m0 + i < mend ? mrow[m0 + i] : 0) << (8 * i);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t m = mb > 0 ? (uint32_t)(mem >> (j * mb)) & ((1u << mb) - 1u) : 0u;
    level[j] = (m << 2) | (((e1 >> (8 + j)) & 1u) << 1) | ((e0 >> (8 + j)) & 1u);
  }
}

// Decode kernels: a thread per 8 columns, a workgroup along the columns and
// then the rows; 8 weights (16 bytes) or levels (8 bytes) per store where rows
// are aligned for it.  Bound by issue and the output's write: 2560 x 9728,
// k=3, weights 19.7 us (2.5 TB/s written; one thread per weight, each with its
// own byte-wise field reads and 2-byte store: 113.5 us; 1024 x 1024 6.9 -> 3.5 us).
template <int BITS>
__global__ void __launch_bounds__(256)
window_decode_kernel(DecodeArgs a, uint32_t dm0, uint32_t dm1, uint8_t* __restrict__ out, int64_t out_stride,
                     bool wide) {
  const int64_t r = (int64_t)blockIdx.y * blockDim.y + threadIdx.y;
  const int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (r >= a.n_rows || c >= a.d) return;
  uint32_t level[8];
  levels_of_8<BITS>(a, dm0, dm1, r, c, level);
  uint8_t* o = out + r * out_stride + c;
  if (wide && c + 8 <= a.d) {
    uint2 w = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w.x |= level[j] << (8 * j);
      w.y |= level[4 + j] << (8 * j);
    }
    *reinterpret_cast<uint2*>(o) = w;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (c + j < a.d) o[j] = (uint8_t)level[j];
  }
}

template <int BITS>
__global__ void __launch_bounds__(256)
decode_rows_kernel(DecodeArgs a, uint32_t dm0, uint32_t dm1, const uint16_t* __restrict__ scales,
                   const uint16_t* __restrict__ codebook, uint16_t* __restrict__ out, int64_t out_stride,
                   bool wide) {
  __shared__ float cb[256];
  for (int i = threadIdx.y * blockDim.x + threadIdx.x; i < 2 << BITS; i += 256) cb[i] = h2f(codebook[i]);
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.y * blockDim.y + threadIdx.y;
  const int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (r >= a.n_rows || c >= a.d) return;
  uint32_t level[8];
  levels_of_8<BITS>(a, dm0, dm1, r, c, level);
  const float sc = h2f(scales[r]);
  // fp32 product of two fp16 values is exact; one rounding to fp16.
  uint32_t w[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w[j] = (uint32_t)f2h(cb[level[2 * j]] * sc) | ((uint32_t)f2h(cb[level[2 * j + 1]] * sc) << 16);
  uint16_t* o = out + r * out_stride + c;
  if (wide && c + 8 <= a.d) {
    *reinterpret_cast<uint4*>(o) = uint4{w[0], w[1], w[2], w[3]};
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (c + j < a.d) o[j] = (uint16_t)(w[j >> 1] >> (16 * (j & 1)));
  }
}

// GEMV on the natural streams: WPR waves of a workgroup share an output row, a
// lane takes 8 columns at a time (levels_of_8, one 16-byte read of z per batch
// row) for NB batch rows at once; sums over lanes, then over the waves of a
// row through LDS, in a fixed order.  WIDE: rows of z are whole 16-byte groups.
// Bound by issue (decode and conversions, ~15 instructions per weight and lane
// at 4 batch rows) on large linears and by one or two load round trips on
// small ones: at 1 / 4 / 8 batch rows 9728 x 2560 (k=4) 13.3 / 16.1 / 20.9 us,
// 3072 x 1024 (k=3) 5.2 / 6.8 / 9.9 us.  (A thread per weight, fields read byte
// by byte: k=4 gate_proj at batch 1 127 us.)
template <int BITS, int NB, int WPR, bool WIDE>
__device__ __forceinline__ void
gemv_batch_rows(const DecodeArgs& a, uint32_t dm0, uint32_t dm1, const uint16_t* __restrict__ z, int nb,
                const uint16_t* __restrict__ scales, const uint16_t* __restrict__ bias, uint16_t* __restrict__ y,
                int64_t n, const float* cb, float* part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r = (int64_t)blockIdx.x * (4 / WPR) + wave / WPR;
  const int64_t rr = r < n ? r : n - 1;  // (waves past the last row repeat it and write nothing)
  float acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = 0.f;
  for (int64_t c = (int64_t)(wave % WPR) * 512 + lane * 8; c < a.d; c += 512 * WPR) {
    uint4 zw[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint16_t* zb = z + (b < nb ? b : 0) * a.d + c;  // (batch rows past nb: row 0, not written)
      if constexpr (WIDE) {
        zw[b] = *reinterpret_cast<const uint4*>(zb);
      } else {
        uint32_t e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = c + j < a.d ? zb[j] : 0;
        zw[b] = uint4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
      }
    }
    uint32_t level[8];
    levels_of_8<BITS>(a, dm0, dm1, rr, c, level);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      // (past the row's end z is zero, but a zero times an infinite or NaN entry is not)
      const float w = WIDE || c + j < a.d ? cb[level[j]] : 0.f;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t zz = j < 2 ? zw[b].x : j < 4 ? zw[b].y : j < 6 ? zw[b].z : zw[b].w;
        acc[b] += w * h2f((uint16_t)(zz >> (16 * (j & 1))));
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[b] += __shfl_xor(acc[b], off, 64);
  }
  if constexpr (WPR > 1) {
    if (lane == 0) {
#pragma unroll
      for (int b = 0; b < NB; ++b) part[wave * NB + b] = acc[b];
    }
    __syncthreads();
    if (wave % WPR) return;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int w = 1; w < WPR; ++w) acc[b] += part[(wave + w) * NB + b];
  }
  if (lane == 0 && r < n) {
    const float sc = h2f(scales[r]);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b >= nb) continue;
      uint16_t out = f2h(acc[b] * sc);
      if (bias) out = f2h(h2f(out) + h2f(bias[r]));
      y[b * n + r] = out;
    }
  }
}

// NB = 8: batch rows 8 blockIdx.y on, the last 1..7 of them at their own width;
// NB = 1, 4: all of them.
template <int BITS, int NB, int WPR, bool WIDE>
__global__ void __launch_bounds__(256)
generic_gemv_kernel(DecodeArgs a, uint32_t dm0, uint32_t dm1, const uint16_t* __restrict__ z, int64_t batch,
                    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ codebook,
                    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, int64_t n) {
  __shared__ float cb[2 << BITS];
  __shared__ float part[4 * NB];
  for (int i = threadIdx.x; i < 2 << BITS; i += 256) cb[i] = h2f(codebook[i]);
  __syncthreads();
  if constexpr (NB < 8) {
    gemv_batch_rows<BITS, NB, WPR, WIDE>(a, dm0, dm1, z, (int)batch, scales, bias, y, n, cb, part);
  } else {
    const int64_t b0 = (int64_t)blockIdx.y * 8;
    const int nb = (int)(batch - b0 < 8 ? batch - b0 : 8);
    z += b0 * a.d;
    y += b0 * n;
    if (nb > 4) gemv_batch_rows<BITS, 8, WPR, WIDE>(a, dm0, dm1, z, nb, scales, bias, y, n, cb, part);
    else if (nb > 1) gemv_batch_rows<BITS, 4, WPR, WIDE>(a, dm0, dm1, z, nb, scales, bias, y, n, cb, part);
    else gemv_batch_rows<BITS, 1, WPR, WIDE>(a, dm0, dm1, z, nb, scales, bias, y, n, cb, part);
  }
}

// One launch for every batch row (65535 groups of 8 at most per launch).  A
// launch per group of 8 was slower on small linears than the work was: 16 x
// 64, k=5, 33 rows 37.7 us per eager call with the rotation (here 27.0), 2048
// rows 1114 (27.2), and every group waited for the one before it: 3072 x 1024,
// k=5, 64 rows 49 us of GPU time (25.9), 9728 x 2560 at 2048 rows 4924 (3535).
template <int BITS, int NB>
void launch_generic_gemv(const DecodeArgs& a, uint32_t dm0, uint32_t dm1, const uint16_t* z, int64_t batch,
                         const uint16_t* scales, const uint16_t* codebook, const uint16_t* bias, uint16_t* y,
                         int64_t n, hipStream_t s) {
  const bool wide = (a.d & 7) == 0 && ((uintptr_t)z & 15) == 0;
  // four waves per row while a wave per row leaves CUs short of waves
  const bool split = a.d > 1024 && n < (int64_t)16 * device_cu_count();
  auto kern = split ? (wide ? generic_gemv_kernel<BITS, NB, 4, true> : generic_gemv_kernel<BITS, NB, 4, false>)
                    : (wide ? generic_gemv_kernel<BITS, NB, 1, true> : generic_gemv_kernel<BITS, NB, 1, false>);
  const int64_t rows = split ? 1 : 4;
  const int64_t most = (int64_t)65535 * NB;
  for (int64_t b0 = 0; b0 < batch; b0 += most) {
    const int64_t nb = batch - b0 < most ? batch - b0 : most;
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + rows - 1) / rows), (unsigned)((nb + NB - 1) / NB)), dim3(256), 0, s, a,
                       dm0, dm1, z + b0 * a.d, nb, scales, codebook, bias, y + b0 * n, n);
  }
}

template <int BITS>
void generic_gemv(const DecodeArgs& a, uint32_t dm0, uint32_t dm1, const uint16_t* z, int64_t batch,
                  const uint16_t* scales, const uint16_t* codebook, const uint16_t* bias, uint16_t* y, int64_t n,
                  hipStream_t s) {
  if (batch == 1) launch_generic_gemv<BITS, 1>(a, dm0, dm1, z, batch, scales, codebook, bias, y, n, s);
  else if (batch <= 4) launch_generic_gemv<BITS, 4>(a, dm0, dm1, z, batch, scales, codebook, bias, y, n, s);
  else launch_generic_gemv<BITS, 8>(a, dm0, dm1, z, batch, scales, codebook, bias, y, n, s);
}

inline int make_decode_args(const uint8_t* path, int64_t path_stride, const uint8_t* member,
                            int64_t member_stride, int64_t n_rows, int64_t d, int bits,
                            int n_states, DecodeArgs* a) {
  if (!path) return TP_ERR_NULL_POINTER;
  int st = check_bits(bits);
  if (st) return st;
  if (bits > 1 && !member) return TP_ERR_NULL_POINTER;
  TrellisTaps taps;
  st = trellis_taps(n_states, &taps);
  if (st) return st;
  if (n_rows < 0 || d <= 0) return TP_ERR_BAD_DIMS;
  if (path_stride < (d + 7) / 8) return TP_ERR_BAD_DIMS;
  if (bits > 1 && member_stride < (d * (bits - 1) + 7) / 8) return TP_ERR_BAD_DIMS;
  a->path = path;
  a->path_stride = path_stride;
  a->member = member;
  a->member_stride = member_stride;
  a->n_rows = n_rows;
  a->d = d;
  a->bits = bits;
  a->m = taps.m;
  a->g0w = taps.g0w;
  a->g1w = taps.g1w;
  return TP_OK;
}

// Bit t of the result: the subset bit of window generator gw takes the path
// bit t columns back (window bit m - t).
inline uint32_t window_delays(uint32_t gw, int m) {
  uint32_t dm = 0;
  for (int t = 0; t <= m; ++t) dm |= ((gw >> (m - t)) & 1u) << t;
  return dm;
}

// 256 threads over (groups of 8 columns, rows): as many along the columns as
// a row fills, up to a wave (512 columns).
inline dim3 decode_block(int64_t d) {
  unsigned x = 8;
  while (x < 64 && x * 8 < d) x *= 2;
  return dim3(x, 256 / x);
}
inline dim3 decode_grid(int64_t n_rows, int64_t d, dim3 block) {
  return dim3((unsigned)((d + 8 * block.x - 1) / (8 * block.x)), (unsigned)((n_rows + block.y - 1) / block.y));
}

}  // namespace tp

extern "C" int tp_window_decode_levels(const uint8_t* path, int64_t path_stride,
                                       const uint8_t* member, int64_t member_stride,
                                       int64_t n_rows, int64_t d, int bits, int n_states,
                                       uint8_t* levels_out, int64_t out_stride, void* stream) {
  using namespace tp;
  DecodeArgs a;
  int st = make_decode_args(path, path_stride, member, member_stride, n_rows, d, bits, n_states, &a);
  if (st) return st;
  if (!levels_out) return TP_ERR_NULL_POINTER;
  if (out_stride < d) return TP_ERR_BAD_DIMS;
  if (n_rows == 0) return TP_OK;
  if (n_rows > 65535) return TP_ERR_BAD_DIMS;
  const bool wide = (((uintptr_t)levels_out | (uintptr_t)out_stride) & 7) == 0;
  const dim3 block = decode_block(d);
  using Kernel = decltype(&window_decode_kernel<1>);
  static constexpr Kernel kernels[7] = {window_decode_kernel<1>, window_decode_kernel<2>, window_decode_kernel<3>,
                                        window_decode_kernel<4>, window_decode_kernel<5>, window_decode_kernel<6>,
                                        window_decode_kernel<7>};
  hipLaunchKernelGGL(kernels[bits - 1], decode_grid(n_rows, d, block), block, 0, (hipStream_t)stream, a,
                     window_delays(a.g0w, a.m), window_delays(a.g1w, a.m), levels_out, out_stride, wide);
  return launch_status();
}

extern "C" int tp_decode_rows(const uint8_t* path, int64_t path_stride,
                              const uint8_t* member, int64_t member_stride,
                              const uint16_t* scales, const uint16_t* codebook,
                              int64_t n_rows, int64_t d, int bits, int n_states,
                              uint16_t* w_out, int64_t out_stride, void* stream) {
  using namespace tp;
  DecodeArgs a;
  int st = make_decode_args(path, path_stride, member, member_stride, n_rows, d, bits, n_states, &a);
  if (st) return st;
  if (!scales || !codebook || !w_out) return TP_ERR_NULL_POINTER;
  if (out_stride < d) return TP_ERR_BAD_DIMS;
  if (n_rows == 0) return TP_OK;
  if (n_rows > 65535) return TP_ERR_BAD_DIMS;
  const bool wide = (((uintptr_t)w_out | (uintptr_t)out_stride * 2) & 15) == 0;
  const dim3 block = decode_block(d);
  using Kernel = decltype(&decode_rows_kernel<1>);
  static constexpr Kernel kernels[7] = {decode_rows_kernel<1>, decode_rows_kernel<2>, decode_rows_kernel<3>,
                                        decode_rows_kernel<4>, decode_rows_kernel<5>, decode_rows_kernel<6>,
                                        decode_rows_kernel<7>};
  hipLaunchKernelGGL(kernels[bits - 1], decode_grid(n_rows, d, block), block, 0, (hipStream_t)stream, a,
                     window_delays(a.g0w, a.m), window_delays(a.g1w, a.m), scales, codebook, w_out, out_stride, wide);
  return launch_status();
}

extern "C" int tp_tcq_gemv(const uint16_t* z, int64_t batch,
                           const uint8_t* path, int64_t path_stride,
                           const uint8_t* member, int64_t member_stride,
                           const uint16_t* scales, const uint16_t* codebook, const uint16_t* bias,
                           int64_t n, int64_t d, int bits, int n_states,
                           uint16_t* y, void* stream) {
  using namespace tp;
  DecodeArgs a;
  int st = make_decode_args(path, path_stride, member, member_stride, n, d, bits, n_states, &a);
  if (st) return st;
  if (!z || !scales || !codebook || !y) return TP_ERR_NULL_POINTER;
  if (batch < 0) return TP_ERR_BAD_DIMS;
  if (batch == 0 || n == 0) return TP_OK;
  const uint32_t dm0 = window_delays(a.g0w, a.m), dm1 = window_delays(a.g1w, a.m);
  using Gemv = decltype(&generic_gemv<1>);
  static constexpr Gemv gemv[7] = {generic_gemv<1>, generic_gemv<2>, generic_gemv<3>, generic_gemv<4>,
                                   generic_gemv<5>, generic_gemv<6>, generic_gemv<7>};
  gemv[bits - 1](a, dm0, dm1, z, batch, scales, codebook, bias, y, n, (hipStream_t)stream);
  return launch_status();
}
