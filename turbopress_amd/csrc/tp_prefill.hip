// Packed linear on a whole prompt (more than 32 rows): y = PackedTCQLinear
// .forward(x) (turbopress/runtime.py:304-334 -> triton_kernel.py:235-260
// fwht_scale + :132-157 packed_gemv) as one GEMM whose weight operands are
// decoded on the way into the matrix cores.
//
//   1. the rotation (tp_rotate.hip) writes z in MFMA operand order
//      (prefill_operand_index), so that the GEMM stages it with plain
//      1-KiB copies;
//   2. tcq_prefill_kernel: one workgroup of 8 waves per tile of 32 WM MG
//      weight rows x 64 NG batch rows (WM = 4 waves along the rows, 2 along
//      the batch, MG x NG blocks of v_mfma_f32_32x32x16_f16 per wave).  K runs
//      in steps of 128 columns: lane l decodes row l % 32 of segment l / 32 of
//      the step, which is the A operand layout, from the same words and the
//      same pair table as the decode kernels (tp_tiled_common.h); a step is
//      two half steps, one per path word;
//   3. where the tiles alone leave CUs idle, K is cut into parts whose fp32
//      sums a second launch adds in part order.
//
// Calling the 32-row kernels once per 32 rows decodes every weight again for
// each of them: 1316 us for 2048 rows of a 9728 x 2560 linear (k=3) and 122 us
// for 199 rows of 2560 x 4096, against 125-132 and 23-25 us here.
//
// What bounds the GEMM: at 2048 x 2560 x 9728 the launch takes 112-130 us
// (0.79-0.91 PFLOP/s; a dense fp16 library product of that shape 103-117 us on
// the same card).  While workgroups are resident the matrix cores are busy 61 %
// of the SIMD cycles (128 x 256 tiles; 70 % with 256 x 256 ones, which fill
// fewer CUs here) at the 1.7-1.8 GHz that the power limit leaves, LDS 50 % (pair
// lookups: 4 reads of 4 bytes per lane and A operand; batch operands: one
// 16-byte read per MG MFMAs), other vector instructions 33 %; the rest is each
// tile's table, first loads and output, and the last of 2.4 passes over the
// CUs.  Decode cost per MFMA falls with NG, batch reads with MG; 2 waves per
// SIMD hide both behind the other wave's MFMAs.
#include "tp_slot.h"

#include <algorithm>
#include <type_traits>

namespace tp {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kPreBlkBytes = 1024; // one MFMA B operand: 64 lanes x 16 bytes

struct PrefillArgs {
  const uint32_t* path;
  const uint32_t* member;
  const uint16_t* z;
  const uint16_t* scales;
  const uint16_t* bias;
  const uint16_t* codebook;
  uint16_t* y;
  float* part;              // K parts: [part][tile][wave][g][c][4][64 lanes][4]
  int64_t ldy;
  int32_t n, T, G, U, batch;    // U: K steps of 128 columns
  int32_t rb, cb, kparts, upp;  // row and batch tiles, K parts, K steps per part
};

template <int MW>
struct PreMember;
template <> struct PreMember<2> {
  typedef u32x2_t type;
  static __device__ __forceinline__ type load(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
  }
};
template <> struct PreMember<4> {
  typedef u32x4_t type;
  static __device__ __forceinline__ type load(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
  }
};
template <> struct PreMember<6> {
  typedef MemberWords6 type;
  static __device__ __forceinline__ type load(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    MemberWords6 m;
    m.lo = __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
    m.hi = __builtin_amdgcn_raw_buffer_load_b64(r, v + 16u, s, 0);
    return m;
  }
};

// Wait until at most N vector memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ float lhalf(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)w); }
__device__ __forceinline__ float hhalf(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }

// LDS bytes of one wave's output: 32 NG batch rows of 32 MG halves (+ 16
// bytes, so that the batch rows a store writes start in different banks).
template <int MG, int NG>
constexpr int pre_out_bytes() { return 32 * NG * (64 * MG + 16); }

// Dynamic LDS of a workgroup: the table and three z buffers, then (the same
// bytes) the rows' scales and biases and every wave's output.
template <int WM, int MG, int NG>
constexpr int pre_lds_bytes() {
  const int loop = kTableBytes + 3 * 2 * NG * 4 * kPreBlkBytes, out = 4 * 32 * WM * MG + 2 * WM * pre_out_bytes<MG, NG>();
  return loop > out ? loop : out;
}

// y of MG x NG blocks of 32 rows x 32 batch rows from a wave's MFMA sums
// (lane half h holds rows 32 g + 8 k + 4 h + i in acc[g][c][4 k + i] of batch
// row 32 c + lane % 32): scaled and rounded in registers, transposed through
// the wave's own LDS `wl`, stored along the rows of y.  Stored straight from
// the registers, one store instruction touches 32 rows of y, a cache line
// each: 6.5 us of a 256 x 256 tile's launch.  sr, br: row scales and biases of the wave's
// rows in LDS (br: null without bias); rows and batch rows past the end are
// not written.
template <int MG, int NG>
__device__ __forceinline__ void pre_write(const PrefillArgs& a, const float16_t (&acc)[MG][NG], char* wl,
                                          const uint16_t* sr, const uint16_t* br, int row0, int b0, int lane) {
  constexpr int pitch = 64 * MG + 16;
  const int h = lane >> 5;
#pragma unroll
  for (int g = 0; g < MG; ++g) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = 32 * g + 8 * k + 4 * h;
      const u32x2_t sw = *reinterpret_cast<const u32x2_t*>(sr + r);
      const float s0 = lhalf(sw[0]), s1 = hhalf(sw[0]), s2 = lhalf(sw[1]), s3 = hhalf(sw[1]);
#pragma unroll
      for (int c = 0; c < NG; ++c)
        *reinterpret_cast<u32x2_t*>(wl + (32 * c + (lane & 31)) * pitch + 2 * r) =
            u32x2_t{pack_h2(acc[g][c][4 * k] * s0, acc[g][c][4 * k + 1] * s1),
                    pack_h2(acc[g][c][4 * k + 2] * s2, acc[g][c][4 * k + 3] * s3)};
    }
  }
  wave_lds_fence();
  const int nb = min(32 * NG, a.batch - b0), nr = min(32 * MG, a.n - row0);
  uint16_t* y0 = a.y + (size_t)b0 * a.ldy + row0;
  // 8 rows' sums, rounded, plus their biases
  auto add_bias = [&](u32x4_t w, int r) __attribute__((always_inline)) {
    const u32x4_t bw = *reinterpret_cast<const u32x4_t*>(br + r);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pack_h2(lhalf(w[e]) + lhalf(bw[e]), hhalf(w[e]) + hhalf(bw[e]));
    return w;
  };
  constexpr int chunks = 4 * MG;  // 16-byte chunks of a batch row
  const bool vec = (a.n & 7) == 0 && (a.ldy & 7) == 0 && ((uintptr_t)a.y & 15) == 0;
  for (int i = lane; i < 32 * NG * chunks; i += 64) {
    const int b = i / chunks, r = (i - b * chunks) * 8;
    if (b >= nb || r >= nr) continue;
    u32x4_t w = *reinterpret_cast<const u32x4_t*>(wl + b * pitch + 2 * r);
    if (br) w = add_bias(w, r);
    uint16_t* yp = y0 + (size_t)b * a.ldy + r;
    if (vec) {
      gst(reinterpret_cast<u32x4_t*>(yp), w);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (r + e < nr) gst(yp + e, (uint16_t)(w[e >> 1] >> (16 * (e & 1))));
    }
  }
}

// One tile (see the head of this file).  z is staged by loads straight to LDS
// into three buffers of one half step each, so the loads of half step s + 2
// are in flight during s and s + 1 and each half step has one barrier, in its
// middle, where no wave waits for data it has just asked for.  A operands are
// looked up three MFMA groups ahead, batch operands one.  Measured on the way
// (4096 x 5120 x 4096): one barrier and two z buffers per half step, lookups
// one group ahead, 4 waves of 128 x 128: 1.95 us per half step of 256 x 256;
// this order 1.89, with 8 waves of 64 x 128 1.83.
template <int KB, int NS, int WM, int MG, int NG>
__global__ void __launch_bounds__(128 * WM, 2)
tcq_prefill_kernel(const PrefillArgs a) {
  // the pair table at LDS address 0 (lookups fold the base away), then z
  extern __shared__ __attribute__((aligned(16))) char pre_lds[];
  uint32_t* const table = reinterpret_cast<uint32_t*>(pre_lds);
  char* const zl = pre_lds + kTableBytes;
  constexpr int MW = member_words(KB);
  constexpr int kBuf = 2 * NG * 4 * kPreBlkBytes;  // z of one half step: 2 NG column groups
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int h = lane >> 5, r = lane & 15, tsel = (lane >> 4) & 1;
  const uint32_t laneoff = lane_offsets<KB>(lane);

  // (first of the loads: the table is built while the others are in flight)
  const uint32_t cb_lane = gld(a.codebook + (lane & ((2 << KB) - 1)));

  // tile of this workgroup: each XCD (blockIdx % 8) takes a contiguous run
  const int total = (int)gridDim.x, q8 = total >> 3, r8 = total & 7;
  const int xcd = (int)blockIdx.x & 7;
  int tile = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int per = a.rb * a.cb;
  const int kp = __builtin_amdgcn_readfirstlane(tile / per);
  tile -= kp * per;
  const int cbk = __builtin_amdgcn_readfirstlane(tile / a.rb), rbk = tile - cbk * a.rb;
  const int u0 = kp * a.upp, u1 = min(a.U, u0 + a.upp);

  // weights
  const uint32_t tile_p = (uint32_t)a.G * (kTileRows * 8), tile_m = (uint32_t)a.G * (kTileRows * MW * 4);
  const int g0 = (rbk * WM + wm) * MG;  // first 32-row group of the wave
  __amdgpu_buffer_rsrc_t prs[MG], mrs[MG];
#pragma unroll
  for (int g = 0; g < MG; ++g) {
    const int t = 2 * (g0 + g);
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane(min(max(a.T - t, 0), 2));
    prs[g] = buffer_rsrc(reinterpret_cast<const char*>(a.path) + (size_t)t * tile_p, cnt * tile_p);
    mrs[g] = buffer_rsrc(reinterpret_cast<const char*>(a.member) + (size_t)t * tile_m, cnt * tile_m);
  }
  const uint32_t pv = (uint32_t)tsel * tile_p + (uint32_t)(h * kTileRows + r) * 8u;
  const uint32_t mv = (uint32_t)tsel * tile_m + (uint32_t)(h * kTileRows + r) * (MW * 4u);
  constexpr uint32_t step_p = 2 * kTileRows * 8, step_m = 2 * kTileRows * MW * 4;
  u32x2_t X[MG];
  typename PreMember<MW>::type M[MG];
  uint32_t carry[MG];  // lanes of either half: word 1 of the previous step's second segment
#pragma unroll
  for (int g = 0; g < MG; ++g) {
    X[g] = __builtin_amdgcn_raw_buffer_load_b64(prs[g], pv, (uint32_t)u0 * step_p, 0);
    M[g] = PreMember<MW>::load(mrs[g], mv, (uint32_t)u0 * step_m);
    const uint32_t hv = (uint32_t)tsel * tile_p + (uint32_t)(kTileRows + r) * 8u + 4u;
    carry[g] = __builtin_amdgcn_raw_buffer_load_b32(prs[g], u0 > 0 ? hv : kOutOfRange, (uint32_t)(u0 > 0 ? u0 - 1 : 0) * step_p, 0);
  }

  // z blocks of half step s = 2 u + x: 2 NG column groups x 4 blocks, NG * 2 blocks per wave
  // (buffer loads: a flat global load to LDS in flight makes every LDS wait a full one)
  const uint32_t zcg = (uint32_t)a.U * 8u * kPreBlkBytes;  // bytes per 32-row column group
  const __amdgpu_buffer_rsrc_t zrs =
      buffer_rsrc(reinterpret_cast<const char*>(a.z) + (size_t)(cbk * 2 * NG) * zcg, 2u * NG * zcg);
  const int s1 = 2 * u1;
  auto stage = [&](int s, int buf) __attribute__((always_inline)) {
    const int sc = min(s, s1 - 1);
#pragma unroll
    for (int i = 0; i < 4 * NG / WM; ++i) {
      const int blk = wave * (4 * NG / WM) + i;  // (column group, operand)
      const int cg = blk >> 2, j = blk & 3;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          zrs, (__attribute__((address_space(3))) void*)(zl + buf + blk * kPreBlkBytes), 16, (uint32_t)lane * 16u,
          (uint32_t)cg * zcg + (uint32_t)(sc * 4 + j) * kPreBlkBytes, 0, 0);
    }
  };
  int b0 = 0, b1 = kBuf, b2 = 2 * kBuf;  // LDS buffers of half steps s, s + 1, s + 2
  stage(2 * u0, b0);
  stage(2 * u0 + 1, b1);
  // the row scale and bias this thread keeps for the epilogue
  constexpr int BM = 32 * WM * MG;
  static_assert(BM <= 128 * WM, "a thread per row");
  const int erow = rbk * BM + tid;
  uint16_t srow = 0, brow = 0;
  if (tid < BM && erow < a.n) {
    srow = gld(a.scales + erow);
    if (a.bias) brow = gld(a.bias + erow);
  }

  build_pair_table_lanes<KB>(table, cb_lane, tid, 128 * WM);

  float16_t acc[MG][NG];
#pragma unroll
  for (int g = 0; g < MG; ++g)
#pragma unroll
    for (int c = 0; c < NG; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[g][c][i] = 0.f;

  // Index words of half step x of group g from its loaded words, in three
  // chunks of a few instructions (run between MFMAs; q = 2 is left empty).
  DecodeIndex<KB> idx[2][MG];
  uint32_t prevw = 0, SA = 0, SB = 0;
  auto chunk = [&](auto xc, int g, int q) __attribute__((always_inline)) {
    constexpr int x = decltype(xc)::value;
    if (q == 0) {
      if (x == 0) {
        const auto sw = __builtin_amdgcn_permlane32_swap(X[g][1], X[g][1], false, false);
        const uint32_t halo = h ? sw[0] : carry[g];
        carry[g] = sw[1];
        prevw = ((halo >> 1) & 0x55555555u) | ((X[g][1] << 1) & 0xAAAAAAAAu);
      } else {
        prevw = X[g][0];
      }
    } else if (q == 1) {
      subset_words<NS>(X[g][x], prevw, SA, SB);
    } else if (q == 3) {
      MemberWords<KB> m[2];
      split_members<KB>(M[g], m);
      idx[x][g] = pair_index<KB>(SA, SB, m[x], laneoff);
    }
  };
  using X0 = std::integral_constant<int, 0>;
  using X1 = std::integral_constant<int, 1>;

  half8_t B[2][NG];
  u32x4_t A[4];
  const char* const zw = zl + wn * NG * 4 * kPreBlkBytes + lane * 16;

  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int g = 0; g < MG; ++g)
#pragma unroll
    for (int q = 0; q < 4; ++q) chunk(X0{}, g, q);
#pragma unroll
  for (int c = 0; c < NG; ++c) B[0][c] = *reinterpret_cast<const half8_t*>(zw + b0 + c * 4 * kPreBlkBytes);
#pragma unroll
  for (int k = 0; k < 3; ++k) A[k] = decode_lookup<KB>(idx[0][k % MG], table, k / MG);

  // Half step s = 2 u + x.  Slot (k, c), k = (j, g): the MFMA of row group g
  // and column group c, then a share of the lookups three steps ahead (of
  // the next half step at the end), of the batch operands of j + 1 and of the
  // index words of the next half step.  Halfway the next half step's z is
  // complete (its loads were issued half a step before this one began), every
  // wave has left the previous half step's buffer, and the loads of s + 2 go
  // there.  sched_barrier keeps the order: left alone the scheduler gathers
  // each step's reads right before their use.
  constexpr int S = 4 * MG;                             // steps per half step
  constexpr int CPS = MG >= 4 ? 1 : (MG >= 2 ? 2 : 4);  // index chunks per step
  constexpr int LPG = KB == 4 ? 3 : 2;                  // weight loads per group
  auto half_step = [&](auto xc, int s, uint32_t un) __attribute__((always_inline)) {
    constexpr int x = decltype(xc)::value;
#pragma unroll
    for (int k = 0; k < S; ++k) {
      const int j = k / MG, g = k % MG;
      if (k == S / 2) {
        // weight loads issued after the z loads of s + 1
        constexpr int before = CPS * (S / 2) / 4 < MG ? CPS * (S / 2) / 4 : MG;
        if (x == 0) wait_vm<LPG * before>();
        else wait_vm<LPG * (MG - before)>();
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
        stage(s + 2, b2);
      }
      const half8_t Av = __builtin_bit_cast(half8_t, A[k & 3]);
      const int ka = (k + 3) % S, xa = k + 3 < S ? x : 1 - x;  // lookups of this step
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        acc[g][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Av, B[j & 1][c], acc[g][c], 0, 0, 0);
#pragma unroll
        for (int w = c * (4 / NG); w < (c + 1) * (4 / NG); ++w)
          A[(k + 3) & 3][w] = decode_lookup_word<KB>(idx[xa][ka % MG], table, ka / MG, w);
        if (g == 0)
          B[(j + 1) & 1][c] = *reinterpret_cast<const half8_t*>(zw + (j < 3 ? b0 : b1) + (c * 4 + ((j + 1) & 3)) * kPreBlkBytes);
        if (c == 0) {
#pragma unroll
          for (int q = k * CPS; q < (k + 1) * CPS; ++q) {
            if (q < S) {
              chunk(std::integral_constant<int, 1 - x>{}, q / 4, q % 4);
              if (x == 0 && (q & 3) == 3) {
                X[q / 4] = __builtin_amdgcn_raw_buffer_load_b64(prs[q / 4], pv, un * step_p, 0);
                M[q / 4] = PreMember<MW>::load(mrs[q / 4], mv, un * step_m);
              }
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    const int t = b0;
    b0 = b1;
    b1 = b2;
    b2 = t;
  };

  for (int u = u0; u < u1; ++u) {
    const uint32_t un = (uint32_t)min(u + 1, u1 - 1);
    half_step(X0{}, 2 * u, un);
    half_step(X1{}, 2 * u + 1, un);
  }
  // (no load to LDS may be in flight when the workgroup ends)
  wait_vm<0>();

  // epilogue
  if (a.kparts == 1) {
    __syncthreads();  // every wave is done with the table and z
    uint16_t* rows = reinterpret_cast<uint16_t*>(pre_lds);
    if (tid < BM) {
      rows[tid] = srow;
      rows[BM + tid] = brow;
    }
    __syncthreads();
    pre_write<MG, NG>(a, acc, pre_lds + 4 * BM + wave * pre_out_bytes<MG, NG>(), rows + wm * MG * 32,
                      a.bias ? rows + BM + wm * MG * 32 : nullptr, g0 * 32, (cbk * 2 + wn) * NG * 32, lane);
  } else {
    float* p = a.part + (((size_t)kp * per + tile) * 2 * WM + wave) * (MG * NG * 1024) + lane * 4;
#pragma unroll
    for (int g = 0; g < MG; ++g)
#pragma unroll
      for (int c = 0; c < NG; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          gst(reinterpret_cast<float4_t*>(p + (g * NG + c) * 1024 + 256 * k),
              float4_t{acc[g][c][4 * k], acc[g][c][4 * k + 1], acc[g][c][4 * k + 2], acc[g][c][4 * k + 3]});
  }
}

// Sums the K parts of one 32 x 32 block per wave and writes its y.
template <int WM, int MG, int NG>
__global__ void __launch_bounds__(256) prefill_reduce_kernel(const PrefillArgs a) {
  __shared__ __attribute__((aligned(16))) char red_out[4][pre_out_bytes<1, 1>()];
  __shared__ __attribute__((aligned(16))) uint16_t red_rows[4][64];
  const int lane = threadIdx.x & 63;
  const int per = a.rb * a.cb;
  const int blk = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);  // (tile, wave, g, c)
  if (blk >= per * 2 * WM * MG * NG) return;
  const int c = blk % NG, g = (blk / NG) % MG, w = (blk / (NG * MG)) % (2 * WM), tile = blk / (NG * MG * 2 * WM);
  const int cbk = tile / a.rb, rbk = tile - cbk * a.rb;
  const int row0 = ((rbk * WM + w % WM) * MG + g) * 32, b0 = ((cbk * 2 + w / WM) * NG + c) * 32;
  if (row0 >= a.n || b0 >= a.batch) return;
  const float* p = a.part + (size_t)blk * 1024 + lane * 4;
  float16_t v[1][1];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[0][0][i] = 0.f;
  for (int kp = 0; kp < a.kparts; ++kp, p += (size_t)per * 2 * WM * MG * NG * 1024) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float4_t o = gld(reinterpret_cast<const float4_t*>(p + 256 * k));
#pragma unroll
      for (int i = 0; i < 4; ++i) v[0][0][4 * k + i] += o[i];
    }
  }
  uint16_t* rows = red_rows[threadIdx.x >> 6];
  const int row = row0 + (lane & 31);
  const uint16_t* src = lane < 32 ? a.scales : a.bias;
  rows[lane] = src && row < a.n ? gld(src + row) : (uint16_t)0;
  wave_lds_fence();
  pre_write<1, 1>(a, v, red_out[threadIdx.x >> 6], rows, a.bias ? rows + 32 : nullptr, row0, b0, lane);
}

namespace {

struct PrePlan {
  int mg, ng;                     // tile: 32 WM mg rows x 64 ng batch rows
  int64_t rb, cb, kparts, upp;    // row and batch tiles, K parts, K steps per part
};

constexpr int kPreWM = 4;
constexpr int kPreMaxParts = 16;

// The cheapest of five tiles and 1..16 K parts in a model of the launch: per
// round of one workgroup per CU 7 us (table, first loads, output) plus the
// half steps of a part, and for several parts the second launch, 4 us plus
// its traffic at 4 TB/s.  What decides is the tiles' ratio, not the scale: the
// model's us per half step are 256 x 256 1.70, 384 x 128 1.25, 128 x 256 0.76,
// 128 x 128 0.46, 128 x 64 0.30; the launches alone, 16 x 16 tiles of each, a
// dozen in a row, k=3, take 2.00 / 1.57 / 1.03 / 0.59 / 0.43 and 1-7 us
// besides.  The pick against the fastest of all forced plans (k=3, with the
// rotation): 9728 x 2560 at 2048 rows 128 x 256 125 us (fastest; 384 x 128 133,
// 256 x 256 139, 128 x 128 141), at 1024 rows 384 x 128 67.4 (256 x 256 67.2,
// 128 x 256 79.6); 4096 x 2560 at 2048 rows 128 x 256 55.7 (fastest); 2560 x
// 9728 at 2048 rows 128 x 256 in one part 151 (256 x 256 in 3 parts 145: 160
// workgroups leave 96 CUs idle, and the model takes K parts to cost more than
// they do), at 512 rows 128 x 128 in 3 parts 48.4 (128 x 256 in 6 parts 47.1);
// 2560 x 4096 at 199 rows 128 x 64 in 3 parts 24.4 (fastest; 128 x 128 in 4
// parts 24.9, 128 x 64 in one part 32.5).
PrePlan plan_prefill(int64_t n, int64_t U, int64_t batch, int cus) {
  static constexpr struct {
    int mg, ng;
    double half;
  } tiles[] = {{2, 4, 1.70}, {3, 2, 1.25}, {1, 4, 0.76}, {1, 2, 0.46}, {1, 1, 0.30}};
  PrePlan best{};
  double least = 1e30;
  for (const auto& t : tiles) {
    const int64_t bm = 32 * kPreWM * t.mg, bn = 64 * t.ng;
    const int64_t rb = (n + bm - 1) / bm, cb = (batch + bn - 1) / bn;
    int64_t last = 0;
    for (int64_t want = 1; want <= kPreMaxParts && want <= U; ++want) {
      const int64_t upp = (U + want - 1) / want, kparts = (U + upp - 1) / upp;
      if (kparts == last) continue;
      last = kparts;
      const int64_t wgs = rb * cb * kparts, rounds = (wgs + cus - 1) / cus;
      double cost = (double)rounds * (7.0 + 2.0 * (double)upp * t.half);
      if (kparts > 1) cost += 4.0 + (double)wgs * (double)(bm * bn) * 8.0 / 4e6;
      if (cost < least) {
        least = cost;
        best = PrePlan{t.mg, t.ng, rb, cb, kparts, upp};
      }
    }
  }
  return best;
}

template <int KB, int NS, int WM, int MG, int NG>
void launch_pre(const PrefillArgs& a, hipStream_t s) {
  auto kern = tcq_prefill_kernel<KB, NS, WM, MG, NG>;
  const size_t dyn = pre_lds_bytes<WM, MG, NG>();
  allow_dynamic_lds(reinterpret_cast<const void*>(kern), 0);
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.rb * a.cb * a.kparts)), dim3(128 * WM), dyn, s, a);
  if (a.kparts > 1) {
    const int64_t blks = (int64_t)a.rb * a.cb * 2 * WM * MG * NG;
    hipLaunchKernelGGL((prefill_reduce_kernel<WM, MG, NG>), dim3((unsigned)((blks + 3) / 4)), dim3(256), 0, s, a);
  }
}

template <int KB, int NS>
int launch_pre_tile(const PrefillArgs& a, const PrePlan& p, hipStream_t s) {
  switch (p.mg * 10 + p.ng) {
    case 24: launch_pre<KB, NS, kPreWM, 2, 4>(a, s); break;
    case 32: launch_pre<KB, NS, kPreWM, 3, 2>(a, s); break;
    case 14: launch_pre<KB, NS, kPreWM, 1, 4>(a, s); break;
    case 12: launch_pre<KB, NS, kPreWM, 1, 2>(a, s); break;
    default: launch_pre<KB, NS, kPreWM, 1, 1>(a, s); break;
  }
  return launch_status();
}

// Bytes of z (whole tiles of batch rows; those past the batch are never
// written, and only reach sums that are not stored).
int64_t pre_z_bytes(const PrePlan& p, int64_t U) { return p.cb * 2 * p.ng * U * 8 * kPreBlkBytes; }

int64_t pre_workspace(const PrePlan& p, int64_t U) {
  const int64_t part = (int64_t)32 * kPreWM * p.mg * 64 * p.ng * 4;
  return pre_z_bytes(p, U) + (p.kparts > 1 ? p.kparts * p.rb * p.cb * part : 0);
}

// Sizes the kernel's 32-bit offsets and grid hold (a column group of z below
// 2^31 bytes); rows: what one rotation launch takes.
int pre_geom(int64_t n, int64_t d, int64_t batch, int bits, Geom* g) {
  if (batch < 1 || batch > 65535 || d > (1 << 20) || n > (1 << 24)) return TP_ERR_BAD_DIMS;
  return tiled_geom(n, d, bits, g);
}

}  // namespace
}  // namespace tp

using namespace tp;

extern "C" int64_t tp_prefill_workspace_bytes(int64_t n, int64_t d, int64_t batch, int bits) {
  Geom g;
  if (pre_geom(n, d, batch, bits, &g) != TP_OK) return 0;
  return pre_workspace(plan_prefill(n, 2 * g.G4, batch, device_cu_count()), 2 * g.G4);
}

extern "C" int tp_prefill_plan(int64_t n, int64_t d, int64_t batch, int bits, int cus, int64_t* out) {
  if (!out) return TP_ERR_NULL_POINTER;
  for (int i = 0; i < 4; ++i) out[i] = 0;
  if (cus < 1) return TP_ERR_BAD_DIMS;
  Geom g;
  const int st = pre_geom(n, d, batch, bits, &g);
  if (st) return st;
  const PrePlan p = plan_prefill(n, 2 * g.G4, batch, cus);
  out[0] = 32 * kPreWM * p.mg;
  out[1] = 64 * p.ng;
  out[2] = p.kparts;
  out[3] = p.rb * p.cb * p.kparts;
  return TP_OK;
}

extern "C" int tp_packed_linear_prefill(const uint16_t* x, int64_t batch, const uint16_t* rot_scale, int64_t block,
                                        const uint8_t* path_tiled, const uint8_t* member_tiled,
                                        const uint16_t* scales, const uint16_t* codebook, const uint16_t* bias,
                                        int64_t n, int64_t d, int bits, int n_states, uint16_t* y, int64_t ldy,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  Geom g;
  int st = pre_geom(n, d, batch, bits, &g);
  if (st) return st;
  if (!x || !path_tiled || !member_tiled || !scales || !codebook || !y) return TP_ERR_NULL_POINTER;
  if (n_states != 4 && n_states != 8 && n_states != 16 && n_states != 64) return TP_ERR_UNSUPPORTED_STATES;
  if (ldy < n) return TP_ERR_BAD_DIMS;
  if (((uintptr_t)path_tiled | (uintptr_t)member_tiled) & 15) return TP_ERR_MISALIGNED;
  const int64_t U = 2 * g.G4;
  const PrePlan p = plan_prefill(n, U, batch, device_cu_count());
  if (!workspace || workspace_bytes < pre_workspace(p, U)) return TP_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 15) return TP_ERR_MISALIGNED;
  uint16_t* z = reinterpret_cast<uint16_t*>(workspace);
  st = block_fwht(x, rot_scale, nullptr, z, batch, d, block, U * 128, true, stream);
  if (st) return st;
  PrefillArgs a;
  a.path = reinterpret_cast<const uint32_t*>(path_tiled);
  a.member = reinterpret_cast<const uint32_t*>(member_tiled);
  a.z = z;
  a.scales = scales;
  a.bias = bias;
  a.codebook = codebook;
  a.y = y;
  a.part = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + pre_z_bytes(p, U));
  a.ldy = ldy;
  a.n = (int32_t)n;
  a.T = (int32_t)g.T;
  a.G = (int32_t)g.G;
  a.U = (int32_t)U;
  a.batch = (int32_t)batch;
  a.rb = (int32_t)p.rb;
  a.cb = (int32_t)p.cb;
  a.kparts = (int32_t)p.kparts;
  a.upp = (int32_t)p.upp;
  hipStream_t s = (hipStream_t)stream;
  switch (bits * 100 + n_states) {
    case 204: return launch_pre_tile<2, 4>(a, p, s);
    case 208: return launch_pre_tile<2, 8>(a, p, s);
    case 216: return launch_pre_tile<2, 16>(a, p, s);
    case 264: return launch_pre_tile<2, 64>(a, p, s);
    case 304: return launch_pre_tile<3, 4>(a, p, s);
    case 308: return launch_pre_tile<3, 8>(a, p, s);
    case 316: return launch_pre_tile<3, 16>(a, p, s);
    case 364: return launch_pre_tile<3, 64>(a, p, s);
    case 404: return launch_pre_tile<4, 4>(a, p, s);
    case 408: return launch_pre_tile<4, 8>(a, p, s);
    case 416: return launch_pre_tile<4, 16>(a, p, s);
    case 464: return launch_pre_tile<4, 64>(a, p, s);
    default: return TP_ERR_UNSUPPORTED_STATES;
  }
}
