// TCQ Viterbi encoder (compress time): the minimum-distortion trellis path
// of each row, bit-exact with the reference's fp32 algorithm
// (turbopress/trellis.py:111-179, pipeline.py:209-276).
//
// One wave per row.  The trellis runs in place: the two states p and p + S/2
// that lead to states 2p and 2p + 1 exchange their metrics and keep the
// results, so a lane's state is its index rotated left by the column number
// (inside log2 S bits) and the lanes that exchange at column t differ in one
// lane bit, log2 S - 1 - t mod log2 S: a lane swap or a DPP move instead of two
// shuffles through LDS per column.  (Lanes S and up repeat the first S.)
// Per block of 96 columns:
//   * the squared errors of the nearest member of each of the four subsets are
//     computed once, 16 columns x 4 subsets at a time, one per lane, and go
//     to LDS in pairs (subset, subset of the other predecessor's branch); a
//     lane's two branches have fixed subsets per column phase, so it reads
//     its pair with one 8-byte load;
//   * per column cand = metric + cost in fp32, the branch-1 candidate wins
//     only if strictly smaller (the reference's `cand1 < cand0`); the decision
//     is shifted into the lane's history, which goes to the caller's workspace
//     every 32 columns.
// Floating-point contraction is off in this file: every add and multiply
// rounds separately, as torch's CPU ops do, so the metrics agree bit for bit.
// The end state is the first state of minimum metric (torch.argmin).  The
// backtrack walks the lanes from the end with scalar operations, one history
// read (v_readlane) per column, collecting the lane sequence 32 columns at a
// time into one register (a lane per column); the lanes then emit path bit,
// subset, member and level of their columns in parallel.
// Bound by VALU issue (96 % of the SIMD cycles), 9728 x 2560, k=3, S=64:
// 577 us per search.  (With lane = state, both subset costs computed in every
// lane and two LDS shuffles per column: 1470 us; 2560 x 2560, k=2, S=4: 486 us,
// here 205.)
#pragma clang fp contract(off)

#include "tp_common.h"

#include <type_traits>

namespace tp {

// v_writelane_b32 (the compiler's intrinsic has no builtin): `seq` with lane
// i's value replaced by the wave-uniform `v`.
__device__ int vit_writelane(int v, int i, int seq) __asm("llvm.amdgcn.writelane.i32");

namespace {

constexpr int kVitWaves = 4;  // rows per workgroup

template <int NS>
struct Gen;
template <> struct Gen<4> { static constexpr int m = 2; static constexpr uint32_t g0 = 05, g1 = 07; };
template <> struct Gen<8> { static constexpr int m = 3; static constexpr uint32_t g0 = 015, g1 = 017; };
template <> struct Gen<16> { static constexpr int m = 4; static constexpr uint32_t g0 = 023, g1 = 035; };
template <> struct Gen<64> { static constexpr int m = 6; static constexpr uint32_t g0 = 0133, g1 = 0171; };

// Subset label of the branch from state `prev` on input bit b
// (trellis.py:73-80): x = (b << m) | prev, label = par(x & g1) << 1 | par(x & g0).
template <int NS>
__device__ __forceinline__ int branch_subset(int prev, int b) {
  const uint32_t x = ((uint32_t)b << Gen<NS>::m) | (uint32_t)prev;
  return (int)(((__popc(x & Gen<NS>::g1) & 1) << 1) | (__popc(x & Gen<NS>::g0) & 1));
}

// Member count of one subset at `bits` bits/weight: 2^(bits+1) levels / 4.
template <int BITS>
struct Sub {
  static constexpr int M = 1 << (BITS - 1);
  float thr[M > 1 ? M - 1 : 1];  // midpoints between consecutive members
  float val[M];                  // members, ascending (codebook[j::4])
};

template <int BITS>
__device__ __forceinline__ Sub<BITS> load_subset(const float* __restrict__ cb, int j) {
  Sub<BITS> s;
#pragma unroll
  for (int i = 0; i < Sub<BITS>::M; ++i) s.val[i] = cb[4 * i + j];
#pragma unroll
  for (int i = 0; i + 1 < Sub<BITS>::M; ++i) s.thr[i] = (s.val[i] + s.val[i + 1]) / 2.0f;
  return s;
}

// Nearest member (index = number of thresholds strictly below z) and its
// squared error.
// The member is selected by the comparisons themselves (thresholds ascend,
// so the last one below z names it).  Each candidate value passes through an
// empty asm statement first: a select between two loads of the struct would
// otherwise become a load through a selected address, i.e. a private-memory
// table lookup.
template <int BITS>
__device__ __forceinline__ float subset_cost(const Sub<BITS>& s, float z, int* member) {
  int m = 0;
  float v = s.val[0];
  __asm__("" : "+v"(v));
#pragma unroll
  for (int i = 0; i + 1 < Sub<BITS>::M; ++i) {
    const bool above = s.thr[i] < z;
    float next = s.val[i + 1];
    __asm__("" : "+v"(next));
    m += above ? 1 : 0;
    v = above ? next : v;
  }
  if (member) *member = m;
  const float diff = z - v;
  return diff * diff;
}

constexpr int kVitBlock = 96;  // columns per block: whole history words, whole phase cycles

// The metrics of the two predecessors of this lane's next state, MSB 0 in lo,
// MSB 1 in hi: the lanes of lane bit B clear and set.
template <int B>
__device__ __forceinline__ void vit_exchange(float alpha, float& lo, float& hi) {
  const int x = __builtin_bit_cast(int, alpha);
  int l, h;
  if constexpr (B == 0) {
    l = __builtin_amdgcn_mov_dpp(x, 0xA0, 0xF, 0xF, true);  // quad_perm [0,0,2,2]
    h = __builtin_amdgcn_mov_dpp(x, 0xF5, 0xF, 0xF, true);  // quad_perm [1,1,3,3]
  } else if constexpr (B == 1) {
    l = __builtin_amdgcn_mov_dpp(x, 0x44, 0xF, 0xF, true);  // quad_perm [0,1,0,1]
    h = __builtin_amdgcn_mov_dpp(x, 0xEE, 0xF, 0xF, true);  // quad_perm [2,3,2,3]
  } else if constexpr (B == 2) {
    l = __builtin_amdgcn_update_dpp(x, x, 0x114, 0xF, 0xA, false);  // lanes 4-7, 12-15 of a row: lane - 4
    h = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xF, 0x5, false);  // lanes 0-3, 8-11: lane + 4
  } else if constexpr (B == 3) {
    l = __builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xC, false);  // lanes 8-15: lane - 8
    h = __builtin_amdgcn_update_dpp(x, x, 0x108, 0xF, 0x3, false);  // lanes 0-7: lane + 8
  } else if constexpr (B == 4) {
    const auto r = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
    l = (int)r[0];
    h = (int)r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
    l = (int)r[0];
    h = (int)r[1];
  }
  lo = __builtin_bit_cast(float, l);
  hi = __builtin_bit_cast(float, h);
}

// v rotated left by k (0 <= k < M) inside M bits.
template <int M>
__device__ __forceinline__ int rotl_bits(int v, int k) {
  return ((v << k) | (v >> (M - k))) & ((1 << M) - 1);
}

// Walk 32 whole columns back from lane `lam` through the lanes' histories
// (bit 31 - i = column i's decision); PH = phase of column 0.  Lane i of `seq`
// gets the lane after column i.
template <int M, int PH>
__device__ __forceinline__ int vit_walk32(uint32_t hist, int lam, int& seq) {
#pragma unroll
  for (int i = 31; i >= 0; --i) {
    constexpr int top = M - 1;
    const int bit = 1 << (top - (PH + i) % M);
    seq = vit_writelane(lam, i, seq);
    const uint32_t w = (uint32_t)__builtin_amdgcn_readlane((int)hist, lam);
    lam = ((w >> (31 - i)) & 1u) ? lam | bit : lam & ~bit;
  }
  return lam;
}

template <int NS, int BITS>
__global__ void __launch_bounds__(64 * kVitWaves)
viterbi_kernel(const float* __restrict__ z, int64_t ldz, int64_t n, int d, const float* __restrict__ cb,
               const int32_t* __restrict__ start_state, uint8_t* __restrict__ level, uint8_t* __restrict__ path,
               uint8_t* __restrict__ member, int32_t* __restrict__ end_state, uint64_t* __restrict__ bp_ws) {
  constexpr int m = Gen<NS>::m;
  // subset difference of the branches from p and p + S/2
  constexpr int K = (((Gen<NS>::g1 >> (m - 1)) & 1) << 1) | ((Gen<NS>::g0 >> (m - 1)) & 1);
  static_assert(K == 2 || K == 3, "quad permutes of the pair exchange");
  typedef float f2_t __attribute__((ext_vector_type(2)));
  __shared__ float s_cb[4 * Sub<BITS>::M];
  __shared__ __attribute__((aligned(16))) f2_t s_cost[kVitWaves][kVitBlock * 4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t row = (int64_t)blockIdx.x * kVitWaves + wave;
  for (int i = threadIdx.x; i < 4 * Sub<BITS>::M; i += blockDim.x) s_cb[i] = cb[i];
  __syncthreads();
  if (row >= n) return;  // whole wave leaves together

  const float* zr = z + row * ldz;
  // history words of the row: [32-column chunk][S lanes]
  uint32_t* bp = reinterpret_cast<uint32_t*>(bp_ws + row * (int64_t)d);
  f2_t* const cost = s_cost[wave];
  const int st = lane & (NS - 1);  // this lane's place in the trellis
  // cost reads: the pair of the MSB-0 predecessor's branch at column phase ph
  const f2_t* rd[m];
#pragma unroll
  for (int ph = 0; ph < m; ++ph) {
    const int prev0 = rotl_bits<m>(st, ph) & (NS / 2 - 1);
    rd[ph] = cost + branch_subset<NS>(prev0, (st >> (m - 1 - ph)) & 1);
  }
  const Sub<BITS> mine = load_subset<BITS>(s_cb, lane & 3);
  const int start = start_state ? start_state[row] : 0;
  float alpha = st == start ? 0.0f : __builtin_inff();
  uint32_t hist = 0;

  // ---- forward pass ----------------------------------------------------
  // z of a block: lane l holds columns l and 64 + l (the next block's load meanwhile)
  float z0 = lane < d ? zr[lane] : 0.0f, z1 = 64 + lane < d ? zr[64 + lane] : 0.0f;
  auto block = [&](int tb, auto tail) __attribute__((always_inline)) {
    constexpr bool kTail = decltype(tail)::value;
    const float c0 = z0, c1 = z1;
    if constexpr (!kTail) {
      const int nx = tb + kVitBlock + lane;
      z0 = nx < d ? zr[nx] : 0.0f;
      z1 = lane < 32 && nx + 64 < d ? zr[nx + 64] : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < kVitBlock / 16; ++q) {
      // columns 16 q + lane / 4, subset lane % 4
      const float zv = __shfl(q < 4 ? c0 : c1, (16 * q + (lane >> 2)) & 63, 64);
      const float c = subset_cost<BITS>(mine, zv, nullptr);
      const float o = __builtin_bit_cast(
          float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, c), K == 2 ? 0x4E : 0x1B, 0xF, 0xF, true));
      cost[64 * q + lane] = f2_t{c, o};
    }
    wave_lds_fence();
    f2_t next[m];
#pragma unroll
    for (int ph = 0; ph < m; ++ph) next[ph] = rd[ph][4 * ph];
#pragma unroll
    for (int g = 0; g < kVitBlock / m; ++g) {
      f2_t pair[m];
#pragma unroll
      for (int ph = 0; ph < m; ++ph) pair[ph] = next[ph];
      if (g + 1 < kVitBlock / m) {
#pragma unroll
        for (int ph = 0; ph < m; ++ph) next[ph] = rd[ph][4 * (m * (g + 1) + ph)];
      }
      auto column = [&](auto phc) __attribute__((always_inline)) {
        constexpr int ph = decltype(phc)::value;
        const int c = m * g + ph;
        if (kTail && tb + c >= d) return;
        float a0, a1;
        vit_exchange<m - 1 - ph>(alpha, a0, a1);
        const float cand0 = a0 + pair[ph][0], cand1 = a1 + pair[ph][1];
        const bool take1 = cand1 < cand0;
        alpha = take1 ? cand1 : cand0;
        hist = (hist << 1) | (take1 ? 1u : 0u);
        if ((c & 31) == 31) {
          if (NS == 64 || lane < NS) bp[((tb + c) >> 5) * NS + lane] = hist;
          if (!kTail || c < kVitBlock - 1) hist = 0;
        }
      };
      if constexpr (m > 0) column(std::integral_constant<int, 0>{});
      if constexpr (m > 1) column(std::integral_constant<int, 1 % m>{});
      if constexpr (m > 2) column(std::integral_constant<int, 2 % m>{});
      if constexpr (m > 3) column(std::integral_constant<int, 3 % m>{});
      if constexpr (m > 4) column(std::integral_constant<int, 4 % m>{});
      if constexpr (m > 5) column(std::integral_constant<int, 5 % m>{});
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_lds_fence();  // (before the next block's costs)
  };
  int tb = 0;
  for (; tb + kVitBlock <= d; tb += kVitBlock) block(tb, std::false_type{});
  if (tb < d) block(tb, std::true_type{});

  // ---- end state: first state of minimum metric -------------------------
  float mn = alpha;
#pragma unroll
  for (int w = 1; w < NS; w <<= 1) mn = fminf(mn, __shfl_xor(mn, w, 64));
  // (all metrics NaN: state 0)
  int best = alpha == mn ? rotl_bits<m>(st, d % m) : NS;
#pragma unroll
  for (int w = 1; w < NS; w <<= 1) best = min(best, __shfl_xor(best, w, 64));
  const int state = __builtin_amdgcn_readfirstlane(best == NS ? 0 : best);
  if (lane == 0 && end_state) end_state[row] = state;
  int lam = rotl_bits<m>(state, (m - d % m) % m);

  // ---- backtrack, 32 columns per round ------------------------------------
  // bp must be visible to this wave's own reads below.
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  uint8_t* lr = level + row * (int64_t)d;
  uint8_t* pr = path + row * (int64_t)d;
  uint8_t* mr = member + row * (int64_t)d;
  // Outputs of columns base .. base + cnt - 1 from the lanes after each
  // (seq) and the lane before the first (lam).
  auto emit = [&](int base, int cnt, int seq, int before) __attribute__((always_inline)) {
    int prevl = __shfl(seq, lane - 1, 64);
    prevl = lane == 0 ? before : prevl;
    if (lane < cnt) {
      const int t = base + lane;
      const int ph = t % m;
      const int prev = rotl_bits<m>(prevl, ph);             // state before column t
      const int bit = (seq >> (m - 1 - ph)) & 1;            // the bit that entered
      const int sub = branch_subset<NS>(prev, bit);
      const Sub<BITS> Ss = load_subset<BITS>(s_cb, sub);
      int mem = 0;
      (void)subset_cost<BITS>(Ss, zr[t], &mem);
      pr[t] = (uint8_t)bit;
      mr[t] = (uint8_t)mem;
      lr[t] = (uint8_t)(mem * 4 + sub);
    }
  };
  int chunk = d >> 5;
  const int rem = d & 31;
  uint32_t h = chunk ? bp[(chunk - 1) * NS + st] : 0u;  // (loads while the tail is walked)
  if (rem) {  // the columns after the last whole word: their history is still in `hist`
    int seq = 0;
    for (int i = rem - 1; i >= 0; --i) {
      const int bit = 1 << (m - 1 - (32 * chunk + i) % m);
      seq = lane == i ? lam : seq;
      const uint32_t w = (uint32_t)__builtin_amdgcn_readlane((int)hist, lam);
      lam = ((w >> (rem - 1 - i)) & 1u) ? lam | bit : lam & ~bit;
    }
    emit(32 * chunk, rem, seq, lam);
  }
  for (--chunk; chunk >= 0; --chunk) {
    const uint32_t cur = h;
    if (chunk > 0) h = bp[(chunk - 1) * NS + st];
    int seq = 0;
    const int ph = (32 * chunk) % m;  // 32 % m is 0 (m = 2, 4) or 2 (m = 3, 6): at most three phases
    if constexpr (32 % m == 0) lam = vit_walk32<m, 0>(cur, lam, seq);
    else if (ph == 0) lam = vit_walk32<m, 0>(cur, lam, seq);
    else if (ph == 2) lam = vit_walk32<m, 2 % m>(cur, lam, seq);
    else lam = vit_walk32<m, 4 % m>(cur, lam, seq);
    emit(32 * chunk, 32, seq, lam);
  }
}

template <int NS>
int launch_viterbi(int bits, const float* z, int64_t ldz, int64_t n, int d, const float* cb, const int32_t* start,
                   uint8_t* level, uint8_t* path, uint8_t* member, int32_t* end_state, uint64_t* ws,
                   hipStream_t s) {
  const dim3 grid((unsigned)((n + kVitWaves - 1) / kVitWaves)), block(64 * kVitWaves);
  switch (bits) {
    case 1: hipLaunchKernelGGL((viterbi_kernel<NS, 1>), grid, block, 0, s, z, ldz, n, d, cb, start, level, path, member, end_state, ws); break;
    case 2: hipLaunchKernelGGL((viterbi_kernel<NS, 2>), grid, block, 0, s, z, ldz, n, d, cb, start, level, path, member, end_state, ws); break;
    case 3: hipLaunchKernelGGL((viterbi_kernel<NS, 3>), grid, block, 0, s, z, ldz, n, d, cb, start, level, path, member, end_state, ws); break;
    case 4: hipLaunchKernelGGL((viterbi_kernel<NS, 4>), grid, block, 0, s, z, ldz, n, d, cb, start, level, path, member, end_state, ws); break;
    default: return TP_ERR_UNSUPPORTED_BITS;
  }
  return launch_status();
}

}  // namespace
}  // namespace tp

using namespace tp;

extern "C" int64_t tp_viterbi_workspace_bytes(int64_t n, int64_t d) {
  if (n <= 0 || d <= 0 || n > INT64_MAX / (int64_t)sizeof(uint64_t) / d) return 0;
  return n * d * (int64_t)sizeof(uint64_t);
}

extern "C" int tp_tcq_viterbi(const float* z, int64_t ldz, int64_t n, int64_t d, const float* codebook, int bits,
                              int n_states, const int32_t* start_state, uint8_t* level_codes, uint8_t* path_bits,
                              uint8_t* member_codes, int32_t* end_state, void* workspace, int64_t workspace_bytes,
                              void* stream) {
  if (!z || !codebook || !level_codes || !path_bits || !member_codes || !workspace) return TP_ERR_NULL_POINTER;
  if (bits < 1 || bits > 4) return TP_ERR_UNSUPPORTED_BITS;
  if (n <= 0 || d <= 0 || d > (1 << 24) || ldz < d || n > ((int64_t)1 << 36)) return TP_ERR_BAD_DIMS;
  if (workspace_bytes < tp_viterbi_workspace_bytes(n, d)) return TP_ERR_WORKSPACE;
  if (((uintptr_t)workspace & 7) || ((uintptr_t)z & 3) || ((uintptr_t)codebook & 3)) return TP_ERR_MISALIGNED;
  hipStream_t s = (hipStream_t)stream;
  uint64_t* ws = reinterpret_cast<uint64_t*>(workspace);
  switch (n_states) {
    case 4: return launch_viterbi<4>(bits, z, ldz, n, (int)d, codebook, start_state, level_codes, path_bits, member_codes, end_state, ws, s);
    case 8: return launch_viterbi<8>(bits, z, ldz, n, (int)d, codebook, start_state, level_codes, path_bits, member_codes, end_state, ws, s);
    case 16: return launch_viterbi<16>(bits, z, ldz, n, (int)d, codebook, start_state, level_codes, path_bits, member_codes, end_state, ws, s);
    case 64: return launch_viterbi<64>(bits, z, ldz, n, (int)d, codebook, start_state, level_codes, path_bits, member_codes, end_state, ws, s);
    default: return TP_ERR_UNSUPPORTED_STATES;
  }
}
