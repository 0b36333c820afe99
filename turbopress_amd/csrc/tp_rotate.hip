// Randomized-Hadamard activation rotation: z = blockFWHT(x * rot_scale).
//
// Reference semantics: turbopress/runtime.py:192-208 (_fwht/_block_fwht, the
// orthonormal Sylvester transform in natural order, butterflies at distance
// h = 1, 2, 4, ... then one division by sqrt(block)) applied to
// x.f32 * rot_scale.f32 (runtime.py:323), i.e. the fp32 CPU path; the fused
// reference kernel (triton_kernel.py:172-212) computes the same transform with
// fp16 intermediates.  Here every stage is fp32 and z is rounded to fp16 once.
//
// Blocks of at most 4096 columns with rows of a multiple of 4 columns run
// rot_rows_kernel (the tile transform of tp_rotate_tile.h), everything else
// the LDS kernel below it: one workgroup per block of one row, the block in
// LDS as fp32 (block <= 16384 -> 64 KiB), the first log2(EPT) stages in
// registers (each thread owns EPT consecutive elements), one barrier per
// stage for the rest.  Both run the same butterflies in the same order and
// divide exactly, so z does not depend on which one runs.
#include "tp_rotate_tile.h"

#include <algorithm>

namespace tp {

constexpr int kRotMaxBlock = 16384;

// Where the transformed rows go: row-major z [rows][ld], or the MFMA operand
// order the prompt GEMM stages (tp_prefill.hip), `ld` columns per row.
__device__ __forceinline__ size_t rot_out_index(bool packed, int64_t row, int64_t col, int64_t ld) {
  return packed ? prefill_operand_index(row, col, ld >> 7) : (size_t)row * ld + col;
}

struct RotRows {
  const uint16_t* x;
  const uint16_t* pre;   // null: ones
  const uint16_t* post;  // null: ones
  uint16_t* z;
  int64_t rows, groups;  // groups of `rpg` rows
  int32_t d, ld, rpg;
  float div, recip;
  int32_t packed;
};

// One wave transforms 1024 columns of `rpg` consecutive rows, one after the
// other (blocks <= 1024 columns: no barrier anywhere); blocks of 2048 and
// 4096 take the four waves of a workgroup, 4096 columns, together.  The
// scales of its columns stay in registers and the next row loads while this
// one is transformed.  Columns past d load as zeros, are whole blocks, and
// come out as the zeros that pad a row to `ld`.  Row-major it is bound by VALU
// issue (products, butterflies, lane moves): 77 / 83 / 68 % of the SIMD cycles
// of resident workgroups at 2048 x 2560 and 2048 x 9728 (block 512) and 8192 x
// 4096 (block 4096), 8.2 / 21.8 / 37.5 us where a copy takes 3.9 / 12.3 / 19.6.
// In operand order the stores of a wave are 16-byte pieces of 32 cache lines
// and weigh more the larger z is: 12.9 / 39.8 / 66.5 us.  The general kernel (one workgroup per
// block and row, every stage above 8 columns through LDS) took 24.7 us for
// 2048 x 2560 (block 512; here 9.0) and 16.4 us for 199 x 4096 (block 4096;
// here 4.5), and 68.6 us for the load-time fold of a 2560 x 9728 weight
// (here 26.4).
template <int LOGH>
__global__ void __launch_bounds__(kRotThreads) rot_rows_kernel(const RotRows a) {
  constexpr bool kTile = LOGH > 10;
  __shared__ float ex[kTile ? kRotTile : 1];
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m = rot_lane_index(lane), lane4 = 4 * lane;
  const int64_t item = kTile ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
  const int64_t seg = item / a.groups, grp = item - seg * a.groups;
  const int64_t col0 = seg * (kTile ? kRotTile : 1024);
  if (col0 >= a.ld) return;  // (whole workgroups where kTile)
  const int w = kTile ? wave : 0;
  const int64_t r0 = grp * a.rpg;
  const int nr = (int)(a.rows - r0 < a.rpg ? a.rows - r0 : a.rpg);
  const uint32_t rowb = (uint32_t)a.d * 2u;
  const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(a.x + r0 * a.d, (uint32_t)nr * rowb);
  uint32_t off[4];
  u32x2_t xw[4], rw[4], pw[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t col = col0 + rot_col(w, m, 4 * g);
    off[g] = col < a.d ? (uint32_t)col * 2u : kOutOfRange;
    xw[g] = __builtin_amdgcn_raw_buffer_load_b64(xrs, off[g], 0, 0);
    rw[g] = pw[g] = u32x2_t{0x3C003C00u, 0x3C003C00u};
    if (a.pre) rw[g] = __builtin_amdgcn_raw_buffer_load_b64(buffer_rsrc(a.pre, rowb), off[g], 0, 0);
    if (a.post) pw[g] = __builtin_amdgcn_raw_buffer_load_b64(buffer_rsrc(a.post, rowb), off[g], 0, 0);
  }
  for (int r = 0; r < nr; ++r) {
    float v[kRotEPT];
    rot_products<(LOGH > 0)>(xw, rw, v);
    // (past the last row: out of range)
    if (r + 1 < nr) {
#pragma unroll
      for (int g = 0; g < 4; ++g) xw[g] = __builtin_amdgcn_raw_buffer_load_b64(xrs, off[g], (uint32_t)(r + 1) * rowb, 0);
    }
    rot_stages<LOGH>(v, w, m, lane4, ex);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t col = col0 + rot_col(w, m, 4 * g);
      if (col >= a.ld) continue;
      u32x2_t o;
      if (a.post) {
        float q[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float ve = v[4 * g + e];
          q[e] = ((LOGH & 1) ? div_by_block_root_fx(ve, a.div, a.recip) : ve * a.recip) *
                 ((e & 1) ? hhi(pw[g][e >> 1]) : hlo(pw[g][e >> 1]));
        }
        o = u32x2_t{pack_h2(q[0], q[1]), pack_h2(q[2], q[3])};
      } else {
        o = rot_z4<LOGH>(v + 4 * g, a.div, a.recip);
      }
      gst(reinterpret_cast<u32x2_t*>(a.z + rot_out_index(a.packed, r0 + r, col, a.ld)), o);
    }
  }
}

template <int LOGH>
void launch_rot_rows(const RotRows& a, hipStream_t s) {
  const int64_t width = LOGH > 10 ? kRotTile : 1024;
  const int64_t items = (a.ld + width - 1) / width * a.groups;
  const int64_t blocks = LOGH > 10 ? items : (items + 3) / 4;
  hipLaunchKernelGGL((rot_rows_kernel<LOGH>), dim3((unsigned)blocks), dim3(kRotThreads), 0, s, a);
}

// (PACKED a template argument and zr the row's own pointer: with a runtime flag
// and an index per store the row-major launch of a block of 8192 took 0.8 us
// longer)
template <int EPT, bool PACKED>
__global__ void __launch_bounds__(256)
fwht_scale_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ rs,
                  const uint16_t* __restrict__ post, uint16_t* __restrict__ z, int64_t d,
                  int64_t ldz, int block, float inv_norm_div) {
  extern __shared__ float buf[];
  const int64_t row = blockIdx.y;
  const int64_t base = (int64_t)blockIdx.x * block;
  const uint16_t* xr = x + row * d + base;
  const uint16_t* rr = rs ? rs + base : nullptr;
  const uint16_t* pr = post ? post + base : nullptr;
  uint16_t* zr = PACKED ? z : z + row * ldz + base;
  const int nchunks = block / EPT;  // EPT-element chunks, one per thread per pass
  const int t = threadIdx.x;

  for (int c = t; c < nchunks; c += blockDim.x) {
    float v[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      v[e] = h2f(xr[c * EPT + e]);
      if (rr) v[e] *= h2f(rr[c * EPT + e]);
    }
    // In-register stages h = 1 .. EPT/2 (natural order, a+b then a-b).
#pragma unroll
    for (int h = 1; h < EPT; h <<= 1) {
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        if ((e & h) == 0) {
          float a = v[e], b = v[e + h];
          v[e] = a + b;
          v[e + h] = a - b;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e) buf[c * EPT + e] = v[e];
  }
  __syncthreads();
  // Cross-thread stages h = EPT .. block/2 through LDS.
  for (int h = EPT; h < block; h <<= 1) {
    for (int i = t; i < block / 2; i += blockDim.x) {
      int j = (i / h) * (2 * h) + (i % h);
      float a = buf[j], b = buf[j + h];
      buf[j] = a + b;
      buf[j + h] = a - b;
    }
    __syncthreads();
  }
  if constexpr (EPT == 8 && PACKED) {
    // operand order keeps 8 columns together: one 16-byte store for each 8
    // (with a store per column a launch of 24 rows took 4.6 us longer at blocks
    // of 8192, 9.2 us at 16384)
    for (int c = t; c < nchunks; c += blockDim.x) {
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float lo = buf[8 * c + 2 * e] / inv_norm_div, hi = buf[8 * c + 2 * e + 1] / inv_norm_div;
        if (pr) {
          lo *= h2f(pr[8 * c + 2 * e]);
          hi *= h2f(pr[8 * c + 2 * e + 1]);
        }
        w[e] = (uint32_t)f2h(lo) | ((uint32_t)f2h(hi) << 16);
      }
      *reinterpret_cast<uint4*>(z + prefill_operand_index(row, base + 8 * c, ldz >> 7)) = uint4{w[0], w[1], w[2], w[3]};
    }
  } else {
    for (int i = t; i < block; i += blockDim.x) {
      float v = buf[i] / inv_norm_div;
      if (pr) v *= h2f(pr[i]);
      zr[PACKED ? prefill_operand_index(row, base + i, ldz >> 7) : (size_t)i] = f2h(v);
    }
  }
  // The last block of a row also clears the padding columns [d, ldz).
  if (blockIdx.x == gridDim.x - 1) {
    for (int64_t i = d + t; i < ldz; i += blockDim.x) z[rot_out_index(PACKED, row, i, ldz)] = 0;
  }
}

}  // namespace tp

namespace tp {

int block_fwht(const uint16_t* x, const uint16_t* pre, const uint16_t* post, uint16_t* z,
               int64_t rows, int64_t d, int64_t block, int64_t ldz, bool packed, void* stream) {
  if (!x || !z) return TP_ERR_NULL_POINTER;
  if (rows < 0 || d <= 0 || ldz < d) return TP_ERR_BAD_DIMS;
  if (block < 1 || (block & (block - 1)) || d % block || block > kRotMaxBlock) return TP_ERR_BAD_BLOCK;
  if (rows == 0) return TP_OK;
  if (rows > 65535) return TP_ERR_BAD_DIMS;
  // Division by the fp32 value of sqrt(block), as the reference divides an
  // fp32 tensor by math.sqrt(d).
  const float div = (float)__builtin_sqrt((double)block);
  hipStream_t s = (hipStream_t)stream;
  // (8-byte accesses at every group of four columns; d bounded so that a
  // group's rows stay below 2^31 bytes)
  if (block <= kRotTile && ((d | ldz) & 3) == 0 && d <= (1 << 24) && ldz <= (1 << 24) &&
      (((uintptr_t)x | (uintptr_t)z | (uintptr_t)pre | (uintptr_t)post) & 7) == 0) {
    RotRows a;
    a.x = x;
    a.pre = pre;
    a.post = post;
    a.z = z;
    a.rows = rows;
    a.d = (int32_t)d;
    a.ld = (int32_t)ldz;
    a.div = div;
    a.recip = 1.f / div;
    a.packed = packed;
    // rows per wave: one while the launch has fewer than 16 waves per CU
    const int64_t width = block > 1024 ? kRotTile : 1024, per = block > 1024 ? 4 : 1;
    const int64_t waves = (ldz + width - 1) / width * per * rows;
    a.rpg = (int32_t)std::min<int64_t>(8, std::max<int64_t>(1, waves / (16 * device_cu_count())));
    a.groups = (rows + a.rpg - 1) / a.rpg;
    switch (__builtin_ctzll((unsigned long long)block)) {
      case 0: launch_rot_rows<0>(a, s); break;
      case 1: launch_rot_rows<1>(a, s); break;
      case 2: launch_rot_rows<2>(a, s); break;
      case 3: launch_rot_rows<3>(a, s); break;
      case 4: launch_rot_rows<4>(a, s); break;
      case 5: launch_rot_rows<5>(a, s); break;
      case 6: launch_rot_rows<6>(a, s); break;
      case 7: launch_rot_rows<7>(a, s); break;
      case 8: launch_rot_rows<8>(a, s); break;
      case 9: launch_rot_rows<9>(a, s); break;
      case 10: launch_rot_rows<10>(a, s); break;
      case 11: launch_rot_rows<11>(a, s); break;
      default: launch_rot_rows<12>(a, s); break;
    }
    return launch_status();
  }
  const int ept = block >= 8 ? 8 : (int)block;
  const int nchunks = (int)(block / ept);
  const int threads = nchunks < 256 ? (nchunks < 64 ? 64 : nchunks) : 256;
  dim3 grid((unsigned)(d / block), (unsigned)rows);
  const size_t lds = (size_t)block * sizeof(float);
  using Kernel = decltype(&fwht_scale_kernel<8, false>);
  const Kernel kern = ept == 8   ? (packed ? fwht_scale_kernel<8, true> : fwht_scale_kernel<8, false>)
                      : ept == 4 ? (packed ? fwht_scale_kernel<4, true> : fwht_scale_kernel<4, false>)
                      : ept == 2 ? (packed ? fwht_scale_kernel<2, true> : fwht_scale_kernel<2, false>)
                                 : (packed ? fwht_scale_kernel<1, true> : fwht_scale_kernel<1, false>);
  hipLaunchKernelGGL(kern, grid, dim3(threads), lds, s, x, pre, post, z, d, ldz, (int)block, div);
  return launch_status();
}

}  // namespace tp

extern "C" int tp_fwht_scale(const uint16_t* x, const uint16_t* rot_scale, uint16_t* z,
                             int64_t batch, int64_t d, int64_t block, void* stream) {
  if (!rot_scale) return TP_ERR_NULL_POINTER;
  return tp::block_fwht(x, rot_scale, nullptr, z, batch, d, block, d, false, stream);
}

extern "C" int tp_fwht_scale_padded(const uint16_t* x, const uint16_t* rot_scale, uint16_t* z,
                                    int64_t batch, int64_t d, int64_t block, int64_t ldz,
                                    void* stream) {
  if (!rot_scale) return TP_ERR_NULL_POINTER;
  return tp::block_fwht(x, rot_scale, nullptr, z, batch, d, block, ldz, false, stream);
}

extern "C" int tp_block_fwht_rows(const uint16_t* x, const uint16_t* pre_scale,
                                  const uint16_t* post_scale, uint16_t* out,
                                  int64_t rows, int64_t d, int64_t block, void* stream) {
  return tp::block_fwht(x, pre_scale, post_scale, out, rows, d, block, d, false, stream);
}
