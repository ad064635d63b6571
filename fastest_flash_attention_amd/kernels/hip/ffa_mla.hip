// Queries and keys of the MLA module for gfx950 (reference modules/flash_mla.py:129-152):
// q = [q_nope | rope(q_rope)] and k = [k_nope | rope(k_rope)] per head, from the outputs of
// its projections.
//
// Bound by HBM: one pass reads each projection once and writes q and k once, in 16-byte
// chunks, four per thread with their loads issued together (32-bit index math: one chunk
// per thread with 64-bit divisions took 110 us below). Consecutive threads take the chunks
// of a row, then the next token of the same head, so the head-major rows that the attention
// streams are written contiguously and the token-major projections are read in pieces of
// head_dim * 2 bytes (two cache lines at head_dim 128). The rotation is done on the way;
// the pair partner of a rope chunk lies rope_dim / 2 further on, in the same line. On
// MI355X at B 2, S 4096, 32 heads of 128 + 64 dims, bf16 (369 MB): 79 us, 4.7 TB/s, against
// 490 us for the elementwise and concatenation launches that it replaces.

#include "ffa_common.h"
#include "ffa_internal.h"

namespace ffa {
namespace {

struct AssembleParams {
  const uint16_t* q_nope;
  const uint16_t* q_rope;
  const uint16_t* kv;
  const uint16_t* k_rope;
  const void* cos;
  const void* sin;
  uint16_t* q;
  uint16_t* k;
  int64_t q_nope_ss, q_rope_ss, kv_ss, k_rope_ss;  // elements between tokens
  int S, H, hd, R;
  int blocks_per;  // workgroups per (batch, head), for q and for k
};

// Rounds as the tables' type does: with fp32 tables products and sums stay fp32, with
// 16-bit tables each of them is rounded to that type (elementwise ops of that type).
template <typename Tag, bool TAB32>
__device__ inline float as_table(float x) {
  if constexpr (TAB32) {
    return x;
  } else {
    return Elem<Tag>::to_f32(static_cast<uint16_t>(Elem<Tag>::pack2(x, x) & 0xffffu));
  }
}

constexpr int kPerThread = 4;  // chunks per thread, 256 apart

template <typename Tag, bool TAB32>
__global__ __launch_bounds__(256) void mla_assemble_kernel(const AssembleParams p) {
#pragma clang fp contract(off)
  using E = Elem<Tag>;
  // block = kPerThread * 256 consecutive chunks of one (batch, head)'s rows
  const int bh = static_cast<int>(blockIdx.x) / p.blocks_per;
  const int first = (static_cast<int>(blockIdx.x) - bh * p.blocks_per) * (256 * kPerThread);
  const int b = bh / p.H;
  const int h = bh - b * p.H;
  const bool is_k = blockIdx.y != 0;
  const int cpr = (p.hd + p.R) >> 3;  // chunks per output row
  const int n = p.S * cpr;
  const int nope = p.hd >> 3;
  const int half = p.R >> 1;
  const int64_t t0 = static_cast<int64_t>(b) * p.S;
  const int64_t n_ss = is_k ? p.kv_ss : p.q_nope_ss;
  const int64_t r_ss = is_k ? p.k_rope_ss : p.q_rope_ss;
  const uint16_t* const nsrc = (is_k ? p.kv + static_cast<int64_t>(h) * 2 * p.hd
                                     : p.q_nope + static_cast<int64_t>(h) * p.hd) + t0 * n_ss;
  const uint16_t* const rsrc = (is_k ? p.k_rope : p.q_rope + static_cast<int64_t>(h) * p.R) + t0 * r_ss;
  uint16_t* const dst = (is_k ? p.k : p.q) + static_cast<int64_t>(bh) * n * 8;

  // every load first (the nope chunk, or both halves of the rope pair), then the rest
  u32x4 x1[kPerThread], x2[kPerThread];
  int row[kPerThread], col[kPerThread];
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int id = min(first + u * 256 + static_cast<int>(threadIdx.x), n - 1);
    row[u] = id / cpr;
    col[u] = id - row[u] * cpr;
    const int d = 8 * (col[u] - nope);  // dim within the rope part
    const uint16_t* src = d < 0 ? nsrc + row[u] * n_ss + 8 * col[u]
                                : rsrc + row[u] * r_ss + (d < half ? d : d - half);
    x1[u] = *reinterpret_cast<const u32x4*>(src);
    if (d >= 0) x2[u] = *reinterpret_cast<const u32x4*>(src + half);
  }
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int id = first + u * 256 + static_cast<int>(threadIdx.x);
    if (id >= n) return;
    u32x4 out = x1[u];
    const int d = 8 * (col[u] - nope);
    if (d >= 0) {
      const bool upper = d >= half;
      const int64_t tab = static_cast<int64_t>(row[u]) * half + (upper ? d - half : d);
      float cs[8], sn[8];
      if constexpr (TAB32) {
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          const f32x4 c4 = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.cos) + tab + e);
          const f32x4 s4 = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.sin) + tab + e);
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            cs[e + w] = c4[w];
            sn[e + w] = s4[w];
          }
        }
      } else {
        const u32x4 c8 = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.cos) + tab);
        const u32x4 s8 = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.sin) + tab);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          cs[e] = E::to_f32(static_cast<uint16_t>(c8[e >> 1] >> (16 * (e & 1))));
          sn[e] = E::to_f32(static_cast<uint16_t>(s8[e >> 1] >> (16 * (e & 1))));
        }
      }
      float r[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float lo = E::to_f32(static_cast<uint16_t>(x1[u][e >> 1] >> (16 * (e & 1))));
        const float hi = E::to_f32(static_cast<uint16_t>(x2[u][e >> 1] >> (16 * (e & 1))));
        // lo cos - hi sin, hi cos + lo sin: products and sum rounded one by one, never an FMA
        const float m = as_table<Tag, TAB32>((upper ? hi : lo) * cs[e]);
        const float w = as_table<Tag, TAB32>((upper ? lo : hi) * sn[e]);
        r[e] = upper ? m + w : m - w;
      }
      out = u32x4{E::pack2(r[0], r[1]), E::pack2(r[2], r[3]), E::pack2(r[4], r[5]),
                  E::pack2(r[6], r[7])};
    }
    *reinterpret_cast<u32x4*>(dst + static_cast<int64_t>(id) * 8) = out;
  }
}

// cos and sin of position * inv_freq, one entry per thread: four small elementwise launches
// (positions, products, cos, sin) in one. Bound by launch latency: 5 us against 20 on MI355X
// at 4096 positions of 32 frequencies, 1016 against 1034 us for the module's call there.
template <typename Tag, bool TAB32>
__global__ __launch_bounds__(256) void rope_tables_kernel(const ffa_rope_tables_args a) {
#pragma clang fp contract(off)
  using E = Elem<Tag>;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= static_cast<int64_t>(a.seqlen) * a.half) return;
  const int s = static_cast<int>(id / a.half);
  const int i = static_cast<int>(id - static_cast<int64_t>(s) * a.half);
  const float pos = as_table<Tag, false>(static_cast<float>(s));
  if constexpr (TAB32) {
    const float x = pos * static_cast<const float*>(a.inv_freq)[i];
    static_cast<float*>(a.cos)[id] = cosf(x);
    static_cast<float*>(a.sin)[id] = sinf(x);
  } else {
    const float x = as_table<Tag, false>(pos * E::to_f32(static_cast<const uint16_t*>(a.inv_freq)[i]));
    const uint32_t both = E::pack2(cosf(x), sinf(x));
    static_cast<uint16_t*>(a.cos)[id] = static_cast<uint16_t>(both & 0xffffu);
    static_cast<uint16_t*>(a.sin)[id] = static_cast<uint16_t>(both >> 16);
  }
}

}  // namespace

int launch_rope_tables(const ffa_rope_tables_args& a, hipStream_t stream) {
  const int64_t blocks = (static_cast<int64_t>(a.seqlen) * a.half + 255) / 256;
  if (blocks > 0x7fffffff) return FFA_ERR_TOO_LARGE;
  const dim3 grid(static_cast<unsigned>(blocks));
  const bool tab32 = a.table_dtype == FFA_DTYPE_FP32;
  if (a.dtype == FFA_DTYPE_BF16) {
    if (tab32) {
      hipLaunchKernelGGL((rope_tables_kernel<Bf16Tag, true>), grid, dim3(256), 0, stream, a);
    } else {
      hipLaunchKernelGGL((rope_tables_kernel<Bf16Tag, false>), grid, dim3(256), 0, stream, a);
    }
  } else {
    if (tab32) {
      hipLaunchKernelGGL((rope_tables_kernel<F16Tag, true>), grid, dim3(256), 0, stream, a);
    } else {
      hipLaunchKernelGGL((rope_tables_kernel<F16Tag, false>), grid, dim3(256), 0, stream, a);
    }
  }
  return hipGetLastError() == hipSuccess ? FFA_OK : FFA_ERR_LAUNCH;
}

int launch_mla_assemble(const ffa_mla_assemble_args& a, hipStream_t stream) {
  AssembleParams p{};
  p.q_nope = static_cast<const uint16_t*>(a.q_nope);
  p.q_rope = static_cast<const uint16_t*>(a.q_rope);
  p.kv = static_cast<const uint16_t*>(a.kv);
  p.k_rope = static_cast<const uint16_t*>(a.k_rope);
  p.cos = a.cos;
  p.sin = a.sin;
  p.q = static_cast<uint16_t*>(a.q);
  p.k = static_cast<uint16_t*>(a.k);
  p.q_nope_ss = a.q_nope_stride;
  p.q_rope_ss = a.q_rope_stride;
  p.kv_ss = a.kv_stride;
  p.k_rope_ss = a.k_rope_stride;
  p.S = a.seqlen;
  p.H = a.heads;
  p.hd = a.head_dim;
  p.R = a.rope_dim;
  const int64_t chunks = static_cast<int64_t>(a.seqlen) * ((p.hd + p.R) >> 3);  // per (batch, head)
  const int64_t per = (chunks + 256 * kPerThread - 1) / (256 * kPerThread);
  const int64_t blocks = per * a.batch * a.heads;
  if (chunks > 0x7fffff00 || blocks > 0x7fffffff) return FFA_ERR_TOO_LARGE;
  p.blocks_per = static_cast<int>(per);
  const dim3 grid(static_cast<unsigned>(blocks), 2);
  const bool tab32 = a.table_dtype == FFA_DTYPE_FP32;
  if (a.dtype == FFA_DTYPE_BF16) {
    if (tab32) {
      hipLaunchKernelGGL((mla_assemble_kernel<Bf16Tag, true>), grid, dim3(256), 0, stream, p);
    } else {
      hipLaunchKernelGGL((mla_assemble_kernel<Bf16Tag, false>), grid, dim3(256), 0, stream, p);
    }
  } else {
    if (tab32) {
      hipLaunchKernelGGL((mla_assemble_kernel<F16Tag, true>), grid, dim3(256), 0, stream, p);
    } else {
      hipLaunchKernelGGL((mla_assemble_kernel<F16Tag, false>), grid, dim3(256), 0, stream, p);
    }
  }
  return hipGetLastError() == hipSuccess ? FFA_OK : FFA_ERR_LAUNCH;
}

}  // namespace ffa
