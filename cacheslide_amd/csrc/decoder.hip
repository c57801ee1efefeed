// The projections of a decoder layer for one token of each of a few requests
// (PagedDecoder.step), with what surrounds them in the layer fused into them:
// the RMS norm of the input rows, the new token's K and V written to their
// paged records, the SiLU gate and the residual sums (the layer of
// reference.py:177-193; the paged write of paged.py:205-240).
//
// What bounds them: reading the weights once.  As library GEMMs with the
// elementwise steps between them a layer was fifteen launches; at 8 requests,
// hidden 2048, FFN 5632 each of its products of 8 to 46 MB took 11 to 15 us,
// the elementwise launches 2 to 5, and the host more than either.
//
// A workgroup of 8 wavefronts owns 16 (or 32) rows of the weights and every
// request; its wavefronts take 128 of the K dims in turn, products are
// v_mfma_f32_16x16x32_bf16 with the weights as A and the requests as B
// (16 MT columns), and the 8 partial tiles are added in LDS.  A layer is four
// launches beside its attention: at 8 requests, hidden 2048, 16 heads over 4,
// FFN 5632 they take 10 (q/k/v), 5.5, 18 (46 MB) and 10.5 us, the head of
// 32000 tokens 37 us (3.6 TB/s), and a step of four layers 335 us, 760 as
// library calls.  Non-temporal weight loads were slower (20 and 44 us): a
// 128-byte line is read by two loads.
//   A: lane (g, n) holds weight row n, dims 8g .. 8g+7 of a step of 32
//   B: lane (g, n) holds request n, the same dims
//   C: lane (g, n) holds request n, weight rows 4g .. 4g+3
//
// Every value that was a bf16 tensor between the launches is rounded to bf16
// at the same place; sums are fp32.

#include "common.h"

namespace cs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxRows = 32;  // requests of a call

enum epilogue { kPlain, kResidual, kSilu, kQkv };

struct skinny_params {
  const uint16_t* x;       // [m, k] rows
  const uint16_t* w;       // [n, k] (kSilu: [2 n, k], gate rows then up rows)
  const uint16_t* norm_w;  // [k]: x is RMS-normed first (kNorm)
  uint16_t* out;           // [m, n] (kQkv: the q rows [m, q_end])
  int32_t m, n, k;
  float eps;
  // kQkv
  int32_t q_end, k_end;
  char* cache;
  int64_t s_block, s_head, s_off;  // bytes
  int64_t blocks;
  int32_t block_size;
  const int32_t* table;
  int64_t table_stride, table_cols;
  const int64_t* positions;
  int32_t* flags;
};

__device__ inline float round_bf16(float x) { return bf16_to_float(float_to_bf16(x)); }

// RT: 16-row tiles of the weights per workgroup (kSilu: a gate and an up
// tile); MT: 16-request tiles.
template <int RT, int MT, int EPI, bool NORM>
__global__ void __launch_bounds__(kThreads) skinny_kernel(skinny_params p) {
  static_assert(EPI != kSilu || RT == 2, "a gate tile and its up tile");
  __shared__ float red[kWaves][RT * MT][256];
  __shared__ float rstd[16 * MT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, n16 = lane & 15;
  const int n0 = static_cast<int>(blockIdx.x) * (EPI == kSilu ? 16 : 16 * RT);

  const uint16_t* wrow[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    int row = EPI == kSilu ? n0 + n16 + r * p.n : n0 + 16 * r + n16;
    const int rows = EPI == kSilu ? 2 * p.n : p.n;
    row = row < rows ? row : rows - 1;  // past the last row: a copy, not stored
    wrow[r] = p.w + static_cast<int64_t>(row) * p.k;
  }
  // the next group's weights are in flight while a group is multiplied, the
  // first one's also behind the norm's pass over the rows
  auto load_w = [&](u32x4 (&wv)[RT][4], int k0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 32 * s + 8 * g;
#pragma unroll
      for (int r = 0; r < RT; ++r)
        wv[r][s] = k < p.k ? *reinterpret_cast<const u32x4*>(wrow[r] + k) : u32x4{0, 0, 0, 0};
    }
  };
  u32x4 wa[RT][4], wb[RT][4];
  load_w(wa, 128 * wave);

  if constexpr (NORM) {
    for (int m = wave; m < p.m; m += kWaves) {
      const uint16_t* row = p.x + static_cast<int64_t>(m) * p.k;
      float sum = 0.f;
      for (int k = 8 * lane; k < p.k; k += 512) {
        const u32x4 u = *reinterpret_cast<const u32x4*>(row + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a = __uint_as_float(u[i] << 16), b = __uint_as_float(u[i] & 0xffff0000u);
          sum += a * a + b * b;
        }
      }
      sum = wave_sum(sum);
      if (lane == 0) rstd[m] = 1.f / sqrtf(sum / static_cast<float>(p.k) + p.eps);
    }
    __syncthreads();
  }

  const uint16_t* xrow[MT];
  float scale[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + n16;
    xrow[t] = p.x + static_cast<int64_t>(m < p.m ? m : p.m - 1) * p.k;
    scale[t] = NORM && m < p.m ? rstd[m] : 0.f;
  }
  floatx4 acc[RT][MT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[r][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto group = [&](const u32x4 (&wv)[RT][4], int k0) {
    u32x4 xv[MT][4], nv[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 32 * s + 8 * g;
      const bool ok = k < p.k;
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xv[t][s] = ok && 16 * t + n16 < p.m ? *reinterpret_cast<const u32x4*>(xrow[t] + k) : u32x4{0, 0, 0, 0};
      if constexpr (NORM) nv[s] = ok ? *reinterpret_cast<const u32x4*>(p.norm_w + k) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        bf16x8 b = __builtin_bit_cast(bf16x8, xv[t][s]);
        if constexpr (NORM) {
          const bf16x8 nw = __builtin_bit_cast(bf16x8, nv[s]);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            b[i] = static_cast<__bf16>(static_cast<float>(nw[i]) * (scale[t] * static_cast<float>(b[i])));
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[r][s]), b, acc[r][t], 0,
                                                              0, 0);
      }
  };
  constexpr int kStep = 128 * kWaves;
  for (int k0 = 128 * wave; k0 < p.k; k0 += 2 * kStep) {
    load_w(wb, k0 + kStep);
    group(wa, k0);
    if (k0 + kStep >= p.k) break;
    load_w(wa, k0 + 2 * kStep);
    group(wb, k0 + kStep);
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<floatx4*>(&red[wave][r * MT + t][4 * lane]) = acc[r][t];
  __syncthreads();

  // element i = 4 lane + v of a tile: weight row 4 (lane / 16) + v, request lane % 16
  constexpr int kTiles = EPI == kSilu ? MT : RT * MT;
  for (int e = tid; e < 256 * kTiles; e += kThreads) {
    const int tile = e >> 8, i = e & 255;
    const int m = 16 * (tile % MT) + ((i >> 2) & 15);
    const int n = n0 + 16 * (tile / MT) + 4 * (i >> 6) + (i & 3);
    if (m >= p.m || n >= p.n) continue;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) sum += red[w][tile][i];
    const int64_t at = static_cast<int64_t>(m) * p.n + n;
    if constexpr (EPI == kPlain) {
      p.out[at] = float_to_bf16(sum);
    } else if constexpr (EPI == kResidual) {
      p.out[at] = float_to_bf16(round_bf16(sum) + bf16_to_float(p.out[at]));
    } else if constexpr (EPI == kSilu) {
      float up = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) up += red[w][MT + tile][i];
      const float gate = round_bf16(sum);
      p.out[at] = float_to_bf16(round_bf16(gate / (1.f + expf(-gate))) * round_bf16(up));
    } else {
      if (n < p.q_end) {
        p.out[static_cast<int64_t>(m) * p.q_end + n] = float_to_bf16(sum);
      } else {
        const bool is_v = n >= p.k_end;
        const int d = n - (is_v ? p.k_end : p.q_end);
        const int64_t pos = p.positions[m];
        const int64_t col = pos >= 0 ? pos / p.block_size : -1;
        const int64_t blk = col >= 0 && col < p.table_cols ? p.table[m * p.table_stride + col] : -1;
        if (blk >= 0 && blk < p.blocks) {
          char* rec = p.cache + blk * p.s_block + (d >> 7) * p.s_head + (pos % p.block_size) * p.s_off;
          reinterpret_cast<uint16_t*>(rec)[(is_v ? 128 : 0) + (d & 127)] = float_to_bf16(sum);
        } else if (d == 0) {
          atomicOr(p.flags, CS_FLAG_BLOCK_INVALID);
        }
      }
    }
  }
}

__global__ void context_kernel(const int64_t* positions, int32_t n, int32_t* out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = static_cast<int32_t>(positions[i] + 1);
}

template <int RT, int EPI, bool NORM>
int launch_skinny(const skinny_params& p, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>(ceil_div(p.n, EPI == kSilu ? 16 : 16 * RT))), block(kThreads);
  if (p.m <= 16)
    hipLaunchKernelGGL((skinny_kernel<RT, 1, EPI, NORM>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((skinny_kernel<RT, 2, EPI, NORM>), grid, block, 0, s, p);
  CS_LAUNCH_CHECK("decoder projection");
  return CS_OK;
}

bool aligned(std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15) != 0) return false;
  return true;
}

int check_layer(const cs_decoder_layer_args* a) {
  CS_REQUIRE(a != nullptr, "null arguments");
  CS_REQUIRE(a->batch >= 0 && a->batch <= kMaxRows, "the decoder layer takes at most %d requests", kMaxRows);
  CS_REQUIRE(a->heads > 0 && a->kv_heads > 0 && a->hidden == 128 * a->heads && a->ffn > 0 && a->ffn % 32 == 0,
             "the decoder layer needs hidden = heads x 128 and an FFN width that is a multiple of 32");
  return CS_OK;
}

}  // namespace
}  // namespace cs

using namespace cs;

extern "C" int cs_decoder_context(const int64_t* positions, int32_t n, int32_t* out, void* stream) {
  if (n <= 0) return CS_OK;
  CS_REQUIRE(positions && out, "null arguments");
  hipLaunchKernelGGL(context_kernel, dim3(static_cast<uint32_t>(ceil_div(n, 256))), dim3(256), 0, as_stream(stream),
                     positions, n, out);
  CS_LAUNCH_CHECK("decoder_context");
  return CS_OK;
}

extern "C" int cs_decoder_qkv(const cs_decoder_layer_args* a, void* stream) {
  const int st = check_layer(a);
  if (st) return st;
  CS_REQUIRE(aligned({a->residual, a->qkv, a->in_norm, a->q, a->cache}) && a->table && a->positions && a->flags,
             "decoder buffers must be present and 16-byte aligned");
  CS_REQUIRE(a->block_size > 0 && a->blocks >= 0 && a->table_cols > 0, "bad cache shape");
  if (a->batch == 0) return CS_OK;
  skinny_params p{};
  p.x = static_cast<const uint16_t*>(a->residual);
  p.w = static_cast<const uint16_t*>(a->qkv);
  p.norm_w = static_cast<const uint16_t*>(a->in_norm);
  p.out = static_cast<uint16_t*>(a->q);
  p.m = a->batch;
  p.k = a->hidden;
  p.q_end = a->heads * 128;
  p.k_end = p.q_end + a->kv_heads * 128;
  p.n = p.k_end + a->kv_heads * 128;
  p.eps = a->eps;
  p.cache = static_cast<char*>(a->cache);
  p.s_block = 2 * a->s_block;
  p.s_head = 2 * a->s_head;
  p.s_off = 2 * a->s_offset;
  p.blocks = a->blocks;
  p.block_size = a->block_size;
  p.table = a->table;
  p.table_stride = a->table_stride;
  p.table_cols = a->table_cols;
  p.positions = a->positions;
  p.flags = a->flags;
  return launch_skinny<1, kQkv, true>(p, as_stream(stream));
}

extern "C" int cs_decoder_mlp(const cs_decoder_layer_args* a, void* stream) {
  int st = check_layer(a);
  if (st) return st;
  CS_REQUIRE(aligned({a->residual, a->o, a->attn, a->gate_up, a->down, a->post_norm, a->act}),
             "decoder buffers must be present and 16-byte aligned");
  if (a->batch == 0) return CS_OK;
  hipStream_t s = as_stream(stream);
  skinny_params p{};
  p.m = a->batch;
  p.eps = a->eps;
  p.x = static_cast<const uint16_t*>(a->attn);
  p.w = static_cast<const uint16_t*>(a->o);
  p.out = static_cast<uint16_t*>(a->residual);
  p.n = p.k = a->hidden;
  if ((st = launch_skinny<1, kResidual, false>(p, s))) return st;
  p.x = static_cast<const uint16_t*>(a->residual);
  p.w = static_cast<const uint16_t*>(a->gate_up);
  p.norm_w = static_cast<const uint16_t*>(a->post_norm);
  p.out = static_cast<uint16_t*>(a->act);
  p.n = a->ffn;
  if ((st = launch_skinny<2, kSilu, true>(p, s))) return st;
  p.x = static_cast<const uint16_t*>(a->act);
  p.w = static_cast<const uint16_t*>(a->down);
  p.out = static_cast<uint16_t*>(a->residual);
  p.n = a->hidden;
  p.k = a->ffn;
  return launch_skinny<1, kResidual, false>(p, s);
}

extern "C" int cs_decoder_head(const void* x, const void* norm, const void* w, void* out, int32_t batch,
                               int32_t hidden, int32_t vocab, float eps, void* stream) {
  CS_REQUIRE(batch >= 0 && batch <= kMaxRows && hidden > 0 && hidden % 32 == 0 && vocab > 0,
             "the decoder head takes at most %d requests and a hidden size that is a multiple of 32", kMaxRows);
  CS_REQUIRE(aligned({x, norm, w, out}), "decoder buffers must be present and 16-byte aligned");
  if (batch == 0) return CS_OK;
  skinny_params p{};
  p.x = static_cast<const uint16_t*>(x);
  p.w = static_cast<const uint16_t*>(w);
  p.norm_w = static_cast<const uint16_t*>(norm);
  p.out = static_cast<uint16_t*>(out);
  p.m = batch;
  p.n = vocab;
  p.k = hidden;
  p.eps = eps;
  return launch_skinny<2, kPlain, true>(p, as_stream(stream));
}
