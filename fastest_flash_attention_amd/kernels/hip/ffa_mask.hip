// Expansion of a block mask for the prefill kernels on gfx950: the [n_br, n_bc] tile mask
// (reference kernels/cpu_reference.py:220-222) to 64-key bit words per query tile, and the
// number of key tiles the reference loop visits per query tile (cpu_reference.py:215-231).
//
// Bound by launch latency: one workgroup per query tile, a word per thread. On MI355X a
// 125 x 125 mask over 8000 keys takes 4 us in one launch, against 92 us of device time (and
// 140 us of host time) in 23 elementwise launches over [n_br, 64 words] integers.

#include "ffa_common.h"
#include "ffa_internal.h"

namespace ffa {
namespace {

__global__ __launch_bounds__(256) void block_mask_expand_kernel(const ffa_block_mask_args a) {
  __shared__ int count;
  const int i = blockIdx.x;
  const int tid = threadIdx.x;
  if (tid == 0) count = 0;
  __syncthreads();
  const uint8_t* row = a.mask + static_cast<int64_t>(i) * a.mask_stride;
  const int bkv = a.block_kv;
  const int Skv = a.seqlen_kv;
  const int n_bc = (Skv + bkv - 1) / bkv;

  for (int w = tid; w < a.words; w += 256) {
    const int k0 = 64 * w;
    const int k1 = min(k0 + 64, Skv);  // keys past the end, and words of only such, stay clear
    uint64_t bits = 0;
    for (int j = k0 / bkv; k0 < Skv && j < n_bc && j * bkv < k1; ++j) {
      if (row[j] == 0) continue;
      const int lo = max(j * bkv, k0) - k0;
      const int n = min((j + 1) * bkv, k1) - k0 - lo;
      bits |= (n == 64 ? ~uint64_t{0} : (uint64_t{1} << n) - 1) << lo;
    }
    a.key_mask[static_cast<int64_t>(i) * a.words + w] = bits;
  }

  // visited: mask set, not past the causal bound of the tile's last row, not left of its
  // first row's window
  const int64_t q_first = a.q_offset + static_cast<int64_t>(i) * a.block_q;
  const int64_t q_last = a.q_offset + min(static_cast<int64_t>(i + 1) * a.block_q,
                                          static_cast<int64_t>(a.seqlen_q)) - 1;
  int mine = 0;
  for (int j = tid; j < n_bc; j += 256) {
    const int k_first = j * bkv;
    const int k_last = min(k_first + bkv, Skv) - 1;
    const bool ok = row[j] != 0 && (!a.causal || k_first <= q_last) &&
                    (a.window <= 0 || k_last >= q_first - a.window + 1);
    mine += ok ? 1 : 0;
  }
  if (mine != 0) atomicAdd(&count, mine);
  __syncthreads();
  if (tid == 0) a.visited[i] = count;
}

}  // namespace

int launch_block_mask_expand(const ffa_block_mask_args& a, hipStream_t stream) {
  const int n_br = (a.seqlen_q + a.block_q - 1) / a.block_q;
  hipLaunchKernelGGL(block_mask_expand_kernel, dim3(n_br), dim3(256), 0, stream, a);
  return hipGetLastError() == hipSuccess ? FFA_OK : FFA_ERR_LAUNCH;
}

}  // namespace ffa
