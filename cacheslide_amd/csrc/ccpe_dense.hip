// CCPE attention of one request on dense K/V for the element types and head
// sizes the tuned bf16, D = 128 kernel (ccpe_prefill.hip) does not take: f16
// and f32 at D = 64 and 128, bf16 at D = 64.  Default key coordinates
// 0..nk-1, no masks, no policies.
//
// For every query row r (position qpos[r]) and query head h
// (position.py:404-560):
//   logit_j = (q . k_j) / sqrt(D)
//   p_j     = clamp(sum_{j' >= j, j' <= qpos} sigmoid(logit_j'), 0, P-1)
//   bias_j  = QE[floor p] + frac * (QE[min(floor p + 1, P-1)] - QE[floor p])
//   out     = softmax_j(logit_j + bias_j) . V over keys j <= qpos
//
// What bounds it.  f32: the matrix cores (v_mfma_f32_32x32x2_f32, 64 of 64
// cycles for each of the two products of a 32 x 32 tile at D = 128).  16-bit
// types: the position and softmax arithmetic of the VALU beside the MFMAs of 32
// cycles (f16 at D = 128: 8 of Q.K and 40 of P.V a tile), and the latency of a
// tile's loads: the compiler keeps `kr`, and of f32 also `vr`, in scratch memory
// (48 bytes a lane for f16 at D = 128, 80 and 144 for f32, none for 16-bit types
// at D = 64), so that those loads are waited for as they are issued.  Both
// products are contractions, so a wave that computes one (row, head) pair on
// scalar dot products -- the generic kernel -- is two orders of magnitude away:
// at 1000 tokens, 32 query heads over 8 KV heads, D = 128, f16, that kernel
// took 4150 us and this one takes 81; f32 at 2048 tokens, 16 heads over 4, D =
// 128: a whole call 8.6 ms before, 0.54 ms now.
//
// Decomposition, as in ccpe_prefill.hip: a wave owns 32 (row, head) columns
// of one GQA group and walks key tiles of 32 from the right-most causal key
// leftwards; S^T = K Q^T leaves a column's 32 scores on two lanes (n and
// n + 32), where the suffix sum of the gates and the online softmax are
// per-lane scalars.  K and V tiles are staged through LDS by the whole
// workgroup, the next tile's global loads issued before this tile is computed.
// Rows are padded so that the 16-byte K reads of 16 lanes fall in distinct
// banks.  A workgroup has 4 waves at every size, also where a short call leaves
// compute units idle and where the tables (66 KB at P = 128) leave room for one
// workgroup per CU: with 2 waves twice as many workgroups share
// the rows, but each stages its tiles with half the threads, and nothing was
// gained at any size (17 to 4096 tokens, 40 to 300 rows over 3000 keys).  us a
// call with 2 and 4 waves: f16, D = 128, 1000 tokens 142 and 135, 4096 636 and
// 526, P = 128 847 and 690; f32, D = 128, P = 128, 2048 tokens 939 and 692;
// bf16, D = 64, 40 rows over 3000 keys 186 and 153; 17 f16 tokens 72 and 72.
//
// Precision.  Products of the inputs are summed in fp32 and gates in fp64, as
// in the generic kernel, and a probability keeps its fp32 value whatever its
// size: f32 multiplies it in fp32, the 16-bit types as three bf16 terms (24
// bits, the range of fp32) by V in bf16, an f16 V as two bf16 terms, which hold
// it exactly.  (As two f16 terms a probability ends at 2^-25: 40000 keys below
// it, 8e-4 of the softmax, left the output but not its norm.  At 1000
// tokens, 32 heads over 8, D = 128, 2 waves a workgroup, a call took 137 us with
// those, 142 with the bf16 terms; with 4 waves, and each term of P multiplied by
// all of V before the next so that consecutive products are independent, 131.)
// f32 forms gates and exponentials as the generic kernel does; the 16-bit
// types take v_exp_f32 and v_rcp_f32, within a unit in the last place each, of
// a score scaled once, where the generic kernel rounds the logit.  The table QE
// uses fp32 products (f32) or Q and E split into bf16 terms that keep 24 bits
// of their product.  2-norm error against fp64 over 40 .. 2048 tokens: f32
// 1.04e-6 (generic kernel 1.09e-6, lower here at every size), 16-bit types that
// of their output's rounding (2.0e-4 f16, 1.6e-3 bf16, as the generic kernel).
//
// Values whose arithmetic could leave the finite range (a score, a QE entry
// or an output beyond 1e37 in magnitude, or not finite) set
// CS_FLAG_POLICY_GENERIC: the caller then runs the generic kernel, which
// decides between the result and the reference's error.

#include "common.h"

namespace cs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_tr;
#define CS_LDS __attribute__((address_space(3)))

constexpr int kCols = 32;   // (row, head) columns per wave
constexpr int kWaves = 4;   // per workgroup: 128 columns share a staged tile
constexpr int kThreads = 64 * kWaves;
constexpr int kTileN = 32;  // keys per tile
constexpr int kMaxPos = 128;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kHuge = 1e37f;

struct dense_params {
  const char* q;
  const char* k;
  const char* v;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh;  // bytes
  const int64_t* qpos;
  const float* e;  // [D, npos]
  char* out;       // [nq, hq, D] contiguous
  int32_t* flags;
  int32_t nq, nk, hq, hkv, group, rows_per_wg, row_blocks, npos, tab_stride;
};

template <typename T> struct dense_elem;
template <> struct dense_elem<float> {
  static constexpr int kSize = 4, kPad = 32, kVTiles = 1;
};
template <> struct dense_elem<f16_t> {
  static constexpr int kSize = 2, kPad = 16;
  static constexpr int kVTiles = 2;  // V as two bf16 terms, exactly
  using vec = f16x8;
  using scalar = _Float16;
  __device__ static floatx16 mfma(vec a, vec b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct dense_elem<bf16_t> {
  static constexpr int kSize = 2, kPad = 16, kVTiles = 1;
  using vec = bf16x8;
  using scalar = __bf16;
  __device__ static floatx16 mfma(vec a, vec b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// The value of lane l ^ 32.
__device__ inline float other_half(float x, int h) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(h ? r[0] : r[1]);
}
__device__ inline double other_half(double x, int h) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = static_cast<uint32_t>(u), hi = static_cast<uint32_t>(u >> 32);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(h ? b[0] : b[1]) << 32) | (h ? a[0] : a[1]));
}

// a + b + c + ... of x in bf16, each term the rounding of what is left.
template <int N>
__device__ inline void split_bf16(float x, __bf16 (&t)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    t[i] = static_cast<__bf16>(x);
    x -= static_cast<float>(t[i]);
  }
}

// MFMA 32x32 layouts (lane l, n = l % 32, h = l / 32): A holds row n, B column
// n, of k indices 8h .. 8h+7 (16-bit, k = 16) or h (f32, k = 2); C holds
// column n, rows 8 (v / 4) + 4h + v % 4.  Which dims (or keys) stand for the k
// indices is free as long as A and B agree: 16-bit step ks takes dims 16 ks +
// 8h + 0..7; f32 step 4c + i takes dim 8c + 4h + i, so that a lane reads its
// half of a K row in 16-byte pieces; P.V takes the scores as they lie, key
// 8 (v / 4) + 4h + v % 4 for register v.
template <typename T, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
ccpe_dense_kernel(dense_params p) {
  using E = dense_elem<T>;
  constexpr bool kF32 = E::kSize == 4;
  constexpr int kRow = D * E::kSize + E::kPad;      // bytes of a staged row
  constexpr int kChunks = D * E::kSize / 16;        // 16-byte chunks of a row
  constexpr int kLoads = kTileN * kChunks / kThreads;
  constexpr int kDb = D / 32;
  // Scores: f32 keeps logits (scaled and rounded once, as the generic kernel
  // does), the 16-bit types raw products q.k, scaled where they are used.
  constexpr float kInvD = D == 64 ? 0.125f : 0.08838834764831845f;  // 1 / sqrt(D)
  constexpr float kInv = kF32 ? 1.f : kInvD;
  constexpr float kBias = kF32 ? 1.f : (D == 64 ? 8.f : 11.313708498984761f);
  extern __shared__ __align__(16) char smem[];
  char* ks_lds = smem;
  char* vs_lds = smem + kTileN * kRow;
  float* tab = reinterpret_cast<float*>(smem + (1 + E::kVTiles) * kTileN * kRow);  // [cols][tab_stride]
  __shared__ int64_t wg_max_pos;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  // the heaviest (right-most) row blocks first; one KV head's row blocks on
  // one XCD where their count divides by 8
  const int kvh = static_cast<int>(blockIdx.x) % p.hkv;
  const int rb = p.row_blocks - 1 - static_cast<int>(blockIdx.x) / p.hkv;
  const int c = wave * kCols + n;
  const int row = rb * p.rows_per_wg + c / p.group;
  const int head = kvh * p.group + c % p.group;
  const bool row_ok = row < p.nq;
  const int row_c = row_ok ? row : 0;
  const int64_t qp = row_ok ? p.qpos[row_c] : -1;
  bool huge = false;

  if (tid == 0) wg_max_pos = -1;
  __syncthreads();
  int64_t wmax = qp, wmin = row_ok ? qp : INT64_MAX;
  for (int off = 32; off > 0; off >>= 1) {
    const int64_t a = __shfl_xor(wmax, off, 64), d = __shfl_xor(wmin, off, 64);
    wmax = a > wmax ? a : wmax;
    wmin = d < wmin ? d : wmin;
  }
  if (lane == 0 && wmax >= 0)
    atomicMax(reinterpret_cast<long long*>(&wg_max_pos), static_cast<long long>(wmax));

  // ---- Q^T as the B operand
  const char* qrow = p.q + static_cast<int64_t>(row_c) * p.q_st + head * p.q_sh;
  float qf[kF32 ? D / 2 : 1];
  uint4 qb[kF32 ? 1 : D / 16];
  if constexpr (kF32) {
#pragma unroll
    for (int cc = 0; cc < D / 8; ++cc) {
      const floatx4 w = *reinterpret_cast<const floatx4*>(qrow + 32 * cc + 16 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i) qf[4 * cc + i] = row_ok ? w[i] : 0.f;
    }
  } else {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      const uint4 w = *reinterpret_cast<const uint4*>(qrow + 32 * ks + 16 * h);
      qb[ks] = row_ok ? w : make_uint4(0, 0, 0, 0);
    }
  }

  // ---- QE^T = E^T Q^T, straight from E (a few 32 KB tables stay in L2)
  float* tcol = tab + c * p.tab_stride;
  const int p1 = p.npos - 1;
  auto e_at = [&](int dim, int pos) { return pos < p.npos ? p.e[dim * p.npos + pos] : 0.f; };
  for (int pb = 0; 32 * pb < p.npos; ++pb) {
    floatx16 acc = {};
    const int pos = 32 * pb + n;
    if constexpr (kF32) {
#pragma unroll
      for (int g = 0; g < D / 32; ++g) {
        floatx16 part = {};
#pragma unroll
        for (int s = 16 * g; s < 16 * g + 16; ++s)
          part = __builtin_amdgcn_mfma_f32_32x32x2f32(e_at(8 * (s >> 2) + 4 * h + (s & 3), pos), qf[s], part, 0, 0, 0);
        acc += part;
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        bf16x8 e0, e1, e2, q0, q1;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __bf16 t[3];
          split_bf16<3>(e_at(16 * ks + 8 * h + i, pos), t);
          e0[i] = t[0];
          e1[i] = t[1];
          e2[i] = t[2];
        }
        if constexpr (__is_same(T, f16_t)) {
          // an f16 value is the sum of two bf16 values
          const f16x8 qh = __builtin_bit_cast(f16x8, qb[ks]);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            __bf16 t[2];
            split_bf16<2>(static_cast<float>(qh[i]), t);
            q0[i] = t[0];
            q1[i] = t[1];
          }
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e1, q1, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e2, q0, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e0, q1, acc, 0, 0, 0);
        } else {
          q0 = __builtin_bit_cast(bf16x8, qb[ks]);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e2, q0, acc, 0, 0, 0);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e1, q0, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(e0, q0, acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int at = 32 * pb + 8 * (v >> 2) + 4 * h + (v & 3);
      if (!(fabsf(acc[v]) < kHuge)) huge = true;
      if (at < p.npos) tcol[at] = acc[v];
    }
  }
  // Every entry is taken relative to entry P-1, the bias of the saturated
  // keys (softmax is invariant to it), and entry P repeats entry P-1: a
  // saturated key then adds nothing, and a lookup needs no clamp.
  __syncthreads();
  {
    const float top_qe = tcol[p1];
    __syncthreads();  // both lanes of the column have read entry P-1
    for (int at = h; at < p.npos; at += 2) tcol[at] -= top_qe;
    if (h == 0) tcol[p.npos] = 0.f;
  }

  const int64_t wgmax = wg_max_pos;  // written before the barriers above
  const int kend = wgmax < p.nk ? static_cast<int>(wgmax) + 1 : p.nk;  // keys [0, kend); any int64 position
  const int ntiles = (kend + kTileN - 1) / kTileN;
  const int qp32 = qp < 0 ? -1 : static_cast<int>(qp < p.nk ? qp : p.nk);
  const int wmax32 = __builtin_amdgcn_readfirstlane(wmax < 0 ? -1 : static_cast<int>(wmax < p.nk ? wmax : p.nk));
  const int wmin32 = __builtin_amdgcn_readfirstlane(
      wmin > p.nk ? p.nk : (wmin < 0 ? 0 : static_cast<int>(wmin)));

  // ---- tile loads: the workgroup's next K and V tile in registers
  const char* kbase = p.k + kvh * p.k_sh;
  const char* vbase = p.v + kvh * p.v_sh;
  uint4 kr[kLoads], vr[kLoads];
  auto load = [&](int t) {
#pragma unroll
    for (int r = 0; r < kLoads; ++r) {
      const int i = tid + kThreads * r;
      const int key = t * kTileN + i / kChunks;
      const int64_t kc = key < kend ? key : kend - 1;  // past the end: a copy of the last key, masked below
      kr[r] = *reinterpret_cast<const uint4*>(kbase + kc * p.k_st + 16 * (i % kChunks));
      vr[r] = *reinterpret_cast<const uint4*>(vbase + kc * p.v_st + 16 * (i % kChunks));
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int r = 0; r < kLoads; ++r) {
      const int i = tid + kThreads * r;
      const int at = (i / kChunks) * kRow + 16 * (i % kChunks);
      *reinterpret_cast<uint4*>(ks_lds + at) = kr[r];
      if constexpr (__is_same(T, f16_t)) {
        const f16x8 v = __builtin_bit_cast(f16x8, vr[r]);
        bf16x8 v0, v1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          __bf16 t[2];
          split_bf16<2>(static_cast<float>(v[e]), t);
          v0[e] = t[0];
          v1[e] = t[1];
        }
        *reinterpret_cast<bf16x8*>(vs_lds + at) = v0;
        *reinterpret_cast<bf16x8*>(vs_lds + kTileN * kRow + at) = v1;
      } else {
        *reinterpret_cast<uint4*>(vs_lds + at) = vr[r];
      }
    }
  };

  const float top = static_cast<float>(p1);
  double carry = row_ok ? 0.0 : 1e30;
  float m_run = -INFINITY;  // in the units of s
  float l_run = 0.f;
  floatx16 o[kDb];
#pragma unroll
  for (int i = 0; i < kDb; ++i) o[i] = floatx16{};
  const int j16 = lane & 15;
  // this lane's transposed V read: key 4h + j16 / 4, dims 16 (n / 16) + 4 (j16 % 4)
  const char* vrd16 = vs_lds + (4 * h + (j16 >> 2)) * kRow + 2 * (16 * (n >> 4) + 4 * (j16 & 3));
  const char* krd = ks_lds + n * kRow + 16 * h;

  auto compute = [&](int t) {
    const int base = t * kTileN;
    if (base > wmax32) return;  // every column of the wave precedes the tile
    floatx16 s = {};
    if constexpr (kF32) {
      // sums of 32 dims, then their sum: a shorter chain of roundings than the
      // generic kernel's one sum over D
#pragma unroll
      for (int g = 0; g < D / 32; ++g) {
        floatx16 part = {};
#pragma unroll
        for (int cc = 4 * g; cc < 4 * g + 4; ++cc) {
          const floatx4 a = *reinterpret_cast<const floatx4*>(krd + 32 * cc);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], qf[4 * cc + i], part, 0, 0, 0);
        }
        s += part;
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks)
        s = E::mfma(*reinterpret_cast<const typename E::vec*>(krd + 32 * ks),
                    __builtin_bit_cast(typename E::vec, qb[ks]), s);
    }
    if constexpr (kF32) s *= kInvD;
    if constexpr (!__is_same(T, f16_t)) {  // f16 products cannot leave the range
      float big = 0.f;
      bool nan = false;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        big = fmaxf(big, fabsf(s[v]));
        nan = nan || s[v] != s[v];
      }
      huge = huge || nan || big > kHuge;
    }
    // key v of the tile (8 (v/4) + 4h + v%4) is visible when 8 (v/4) + v%4 <= lim
    const int lim = (qp32 < kend - 1 ? qp32 : kend - 1) - base - 4 * h;
    if (base + kTileN - 1 > wmin32 || base + kTileN > kend) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (8 * (v >> 2) + (v & 3) > lim) s[v] = -INFINITY;
    }
    if (!__all(carry >= static_cast<double>(top))) {
      // gates and their suffix sums within runs of 4 keys
      double gsuf[16], run[4], after[4];
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        double acc = 0.0;
#pragma unroll
        for (int i = 3; i >= 0; --i) {
          const int v = 4 * j4 + i;
          float g;
          if constexpr (kF32)
            g = 1.f / (1.f + expf(-s[v]));
          else
            g = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[v] * (-kInv * kLog2e)));
          acc += static_cast<double>(g);  // 0 for a masked key
          gsuf[v] = acc;
        }
        run[j4] = acc;
      }
      // gate mass of the runs with larger keys: (j4, h = 1) follows (j4, h = 0)
      double acc = 0.0;
#pragma unroll
      for (int j4 = 3; j4 >= 0; --j4) {
        const double other = other_half(run[j4], h);
        after[j4] = carry + acc + (h == 0 ? other : 0.0);
        acc += run[j4] + other;
      }
      carry += acc;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float pv = fminf(static_cast<float>(after[v >> 2] + gsuf[v]), top);
        const int lo = static_cast<int>(pv);
        const float frac = __builtin_amdgcn_fractf(pv);
        const float t0 = tcol[lo], t1 = tcol[lo + 1];
        s[v] += kBias * fmaf(frac, t1 - t0, t0);
      }
    }
    // Online softmax against a running max that moves only when a score lies
    // 8 (in log2 units) above it, so that most tiles need no rescale and a
    // probability stays below 2^8.
    float tmax = s[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) tmax = fmaxf(tmax, s[v]);
    tmax = fmaxf(tmax, other_half(tmax, h));
    if (__any(tmax > m_run + 8.f / (kInv * kLog2e))) {
      const float m_new = fmaxf(m_run, tmax);
      float corr = 1.f;
      if (m_new > m_run) corr = kF32 ? expf(m_run - m_new) : __builtin_amdgcn_exp2f((m_run - m_new) * (kInv * kLog2e));
      m_run = m_new;
      l_run *= corr;
#pragma unroll
      for (int d = 0; d < kDb; ++d) o[d] *= corr;
    }
    const float m_ref = m_run == -INFINITY ? 0.f : m_run;
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      if constexpr (kF32)
        s[v] = expf(s[v] - m_ref);
      else
        s[v] = __builtin_amdgcn_exp2f((s[v] - m_ref) * (kInv * kLog2e));
      sum += s[v];
    }
    l_run += sum;
    // O^T += V^T P^T
    if constexpr (kF32) {
      const char* vrd = vs_lds + 4 * h * kRow + 4 * n;
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int db = 0; db < kDb; ++db) {
          const float a = *reinterpret_cast<const float*>(vrd + (8 * (v >> 2) + (v & 3)) * kRow + 128 * db);
          o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, s[v], o[db], 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        // a probability as three bf16 terms, all of its 24 bits at any size
        bf16x8 pb[3];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __bf16 t[3];
          split_bf16<3>(s[8 * ks + i], t);
#pragma unroll
          for (int w = 0; w < 3; ++w) pb[w][i] = t[w];
        }
#pragma unroll
        for (int u = E::kVTiles - 1; u >= 0; --u) {
          bf16x8 va[kDb];
#pragma unroll
          for (int db = 0; db < kDb; ++db) {
            const char* at = vrd16 + u * kTileN * kRow + 16 * ks * kRow + 64 * db;
            const bf16x4_tr lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((CS_LDS bf16x4_tr*)at);
            const bf16x4_tr hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((CS_LDS bf16x4_tr*)(at + 8 * kRow));
            va[db] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          }
          // third term of P times second of V: below 2^-26 of the product
#pragma unroll
          for (int w = 2 - u; w >= 0; --w)
#pragma unroll
            for (int db = 0; db < kDb; ++db)
              o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[db], pb[w], o[db], 0, 0, 0);
        }
      }
    }
  };

  if (ntiles > 0) load(ntiles - 1);
  for (int t = ntiles - 1; t >= 0; --t) {
    __syncthreads();  // the tile before has been read
    store();
    __syncthreads();
    if (t > 0) load(t - 1);
    compute(t);
  }

  const float l_tot = l_run + other_half(l_run, h);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (row_ok) {
    char* orow = p.out + (static_cast<int64_t>(row) * p.hq + head) * (D * E::kSize);
#pragma unroll
    for (int db = 0; db < kDb; ++db)
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        const int dim = 32 * db + 8 * j4 + 4 * h;
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = o[db][4 * j4 + i];
          if (!(fabsf(x) < kHuge)) huge = true;
          w[i] = kF32 ? (l_tot > 0.f ? x / l_tot : 0.f) : x * inv;
        }
        if constexpr (kF32) {
          *reinterpret_cast<floatx4*>(orow + 4 * dim) = floatx4{w[0], w[1], w[2], w[3]};
        } else {
          typedef typename E::scalar x4 __attribute__((ext_vector_type(4)));
          *reinterpret_cast<x4*>(orow + 2 * dim) =
              x4{static_cast<typename E::scalar>(w[0]), static_cast<typename E::scalar>(w[1]),
                 static_cast<typename E::scalar>(w[2]), static_cast<typename E::scalar>(w[3])};
        }
      }
  }
  if (__any(huge && row_ok) && lane == 0) atomicOr(p.flags, CS_FLAG_POLICY_GENERIC);
}

template <typename T, int D>
int launch_dense(dense_params p, hipStream_t s) {
  p.rows_per_wg = kCols * kWaves / p.group;
  const int64_t total = ceil_div(p.nq, p.rows_per_wg) * p.hkv;
  CS_REQUIRE(total < (1ll << 31), "grid too large");
  p.row_blocks = static_cast<int32_t>(total / p.hkv);
  p.tab_stride = (p.npos + 1) | 1;  // entries 0 .. P, an odd number of words
  const size_t smem = (1 + dense_elem<T>::kVTiles) * kTileN * (D * dense_elem<T>::kSize + dense_elem<T>::kPad) +
                      sizeof(float) * kCols * kWaves * static_cast<size_t>(p.tab_stride);
  hipLaunchKernelGGL((ccpe_dense_kernel<T, D>), dim3(static_cast<uint32_t>(total)), dim3(kThreads), smem, s, p);
  CS_LAUNCH_CHECK("ccpe_dense");
  return CS_OK;
}

}  // namespace
}  // namespace cs

using namespace cs;

extern "C" int cs_ccpe_attention_dense(const cs_ccpe_args* a, void* stream) {
  CS_REQUIRE(a != nullptr, "null arguments");
  const cs_view &q = a->q, &k = a->k, &v = a->v, &e = a->e, &out = a->out;
  CS_REQUIRE(q.data && k.data && v.data && e.data && out.data && a->qpos && a->flags, "null arguments");
  CS_REQUIRE(q.ndim == 3 && k.ndim == 3 && v.ndim == 3 && out.ndim == 3, "q, k, v and out must be 3-d");
  CS_REQUIRE(a->kpos == nullptr && !a->attn_mask.data && !a->vis_mask.data && !a->fixed_pos.data &&
                 !a->canonical.data && !a->pos_out.data && !a->sel_rows,
             "the dense MFMA attention takes default key coordinates and no masks or policies");
  const int dt = q.dtype;
  const int64_t d = q.shape[2];
  const bool takes = (dt == CS_F16 || dt == CS_F32 || dt == CS_BF16) && (d == 64 || (d == 128 && dt != CS_BF16));
  if (!takes) {
    set_error("the dense MFMA attention takes f16 and f32 at head size 64 and 128 and bf16 at 64");
    return CS_EUNSUPPORTED;
  }
  const int size = dtype_size(dt);
  CS_REQUIRE(k.dtype == dt && v.dtype == dt && out.dtype == dt && k.shape[2] == d && v.shape[2] == d &&
                 out.shape[2] == d && k.shape[0] == v.shape[0] && k.shape[1] == v.shape[1] &&
                 out.shape[0] == q.shape[0] && out.shape[1] == q.shape[1],
             "q, k, v and out must share dtype, head size and counts");
  CS_REQUIRE(out.stride[2] == 1 && out.stride[1] == d && out.stride[0] == d * q.shape[1],
             "out must be contiguous");
  const cs_view* in[3] = {&q, &k, &v};
  for (const cs_view* x : in) {
    bool ok = x->stride[2] == 1 && (reinterpret_cast<uintptr_t>(x->data) % 16) == 0;
    for (int i = 0; i < 2; ++i) ok = ok && x->stride[i] >= 0 && (x->stride[i] * size) % 16 == 0;
    if (!ok) {
      set_error("the dense MFMA attention needs 16-byte aligned contiguous rows");
      return CS_EUNSUPPORTED;
    }
  }
  CS_REQUIRE(e.dtype == CS_F32 && e.ndim == 2 && e.shape[0] == d && e.stride[1] == 1 && e.stride[0] == e.shape[1],
             "e must be contiguous fp32 [D, P]");
  CS_REQUIRE(k.shape[1] > 0 && q.shape[1] % k.shape[1] == 0, "bad head counts");
  const int64_t group = q.shape[1] / k.shape[1];
  if (e.shape[1] < 2 || e.shape[1] > kMaxPos || group < 1 || kCols % group != 0) {
    set_error("the dense MFMA attention needs 2 <= P <= %d and a GQA group dividing %d", kMaxPos, kCols);
    return CS_EUNSUPPORTED;
  }
  CS_REQUIRE(q.shape[0] < (1ll << 31) && k.shape[0] < (1ll << 31) - 64 && k.shape[0] > 0, "bad row or key count");
  if (q.shape[0] == 0) return CS_OK;
  dense_params p{};
  p.q = static_cast<const char*>(q.data);
  p.k = static_cast<const char*>(k.data);
  p.v = static_cast<const char*>(v.data);
  p.q_st = q.stride[0] * size;
  p.q_sh = q.stride[1] * size;
  p.k_st = k.stride[0] * size;
  p.k_sh = k.stride[1] * size;
  p.v_st = v.stride[0] * size;
  p.v_sh = v.stride[1] * size;
  p.qpos = a->qpos;
  p.e = static_cast<const float*>(e.data);
  p.out = static_cast<char*>(out.data);
  p.flags = a->flags;
  p.nq = static_cast<int32_t>(q.shape[0]);
  p.nk = static_cast<int32_t>(k.shape[0]);
  p.hq = static_cast<int32_t>(q.shape[1]);
  p.hkv = static_cast<int32_t>(k.shape[1]);
  p.group = static_cast<int32_t>(group);
  p.npos = static_cast<int32_t>(e.shape[1]);
  hipStream_t s = as_stream(stream);
  if (dt == CS_F16) return d == 64 ? launch_dense<f16_t, 64>(p, s) : launch_dense<f16_t, 128>(p, s);
  if (dt == CS_BF16) return launch_dense<bf16_t, 64>(p, s);
  return d == 64 ? launch_dense<float, 64>(p, s) : launch_dense<float, 128>(p, s);
}
