// fa_cast.hip — small passes around the attention kernels: fp32 inputs to 16-bit
// operands, and the rows of a packed batch that belong to no sequence.
//
// The reference's launchers cast every input to half with one tensor operation
// each (cuda/flash_attn_fa3_db_full.cu:366-368) and start from zeroed outputs;
// here each of the two is one launch.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "fa_mi355x.h"
#include "fa_tile.hpp"

namespace fa {

template <bool BF16>
__global__ void __launch_bounds__(256) fa_cast_kernel(CastJobs jobs) {
  cast_block<BF16>(jobs, (int)blockIdx.x);
}

// A buffer of `heads` x total rows of `words` 32-bit words.
struct FillBuf {
  uint32_t* p;
  int64_t heads;
  int words;
  uint32_t value;
};

// Rows of the workgroup's chunk that are in no sequence, in every head of
// every buffer. A well-formed cu covers one run of rows, so a workgroup inside
// it leaves after one look at the table (about 3 us for a whole batch; filling
// the outputs whole before the kernels took 45 us of a 686 us training pass
// of 12 sequences, H8 D64). Every workgroup reads the whole table, so of more
// than kCountedSeqs sequences kFillGroups workgroups take several chunks each
// (60000 sequences of 4-12 rows, H2 D64, forward: 2480 us with a workgroup per
// chunk, 2270-2310 so). Only where a sequence is longer than max_seqlen or the table
// falls does each row look for its sequence.
constexpr int kFillRows = 64;
constexpr int kFillGroups = 512;

// Whether a sequence falls or is longer than max_seqlen, the same in every thread.
template <int UNROLL>
__device__ __forceinline__ int odd_table(const Geom& g) {
  int odd = 0;
#pragma unroll UNROLL
  for (int b = threadIdx.x; b < g.B; b += 256) {
    const int c0 = clamp_row(g.cu[b], g.total), c1 = clamp_row(g.cu[b + 1], g.total);
    odd |= c1 < c0 || c1 - c0 > g.N;
  }
  return __syncthreads_or(odd);
}

// Rows r0 .. r0 + kFillRows - 1.
__device__ __forceinline__ void fill_chunk(const Geom& g, const FillBuf& b0, const FillBuf& b1,
                                           const FillBuf& b2, int odd, int r0, uint8_t* inside) {
  const int tid = threadIdx.x;
  const int first = clamp_row(g.cu[0], g.total), last = clamp_row(g.cu[g.B], g.total);
  if (!odd && r0 >= first && min(r0 + kFillRows, g.total) <= last) return;
  if (tid < kFillRows) {
    const int r = r0 + tid;
    bool in = !odd && r >= first && r < last;
    if (odd) {
      // Sequences as the attention kernels take them: up to kCountedSeqs from
      // the running maximum of the bounds on, more of them as they stand.
      int end = 0;
      for (int b = 0; b < g.B; ++b) {
        const int c0 = clamp_row(g.cu[b], g.total), c1 = clamp_row(g.cu[b + 1], g.total);
        const int s0 = g.B <= kCountedSeqs ? max(c0, end) : c0;
        const int s1 = max(s0, c1);
        in |= r >= s0 && r < s0 + min(s1 - s0, g.N);
        end = max(end, s1);
      }
    }
    inside[tid] = in;
  }
  __syncthreads();
  const FillBuf bufs[3] = {b0, b1, b2};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const FillBuf b = bufs[i];
    if (b.p == nullptr) continue;
    for (int64_t h = 0; h < b.heads; ++h) {
      uint32_t* row0 = b.p + (h * g.total + r0) * b.words;
      for (int w = tid; w < kFillRows * b.words; w += 256) {
        const int r = w / b.words;
        if (r0 + r < g.total && !inside[r]) row0[w] = b.value;
      }
    }
  }
}

__global__ void __launch_bounds__(256)
fa_fill_outside_kernel(Geom g, FillBuf b0, FillBuf b1, FillBuf b2) {
  __shared__ uint8_t inside[kFillRows];
  fill_chunk(g, b0, b1, b2, odd_table<1>(g), blockIdx.x * kFillRows, inside);
}

__global__ void __launch_bounds__(256)
fa_fill_outside_many_kernel(Geom g, FillBuf b0, FillBuf b1, FillBuf b2) {
  __shared__ uint8_t inside[kFillRows];
  const int odd = odd_table<4>(g);
  for (int64_t r0 = (int64_t)blockIdx.x * kFillRows; r0 < g.total; r0 += (int64_t)gridDim.x * kFillRows) {
    fill_chunk(g, b0, b1, b2, odd, (int)r0, inside);
    __syncthreads();   // before the next chunk's `inside`
  }
}

}  // namespace fa

extern "C" int fa_cast_f32(const float* const src[3], void* const dst[3], const int64_t n[3],
                           int bf16, void* stream) {
  using namespace fa;
  if (!src || !dst || !n) return FA_ERR_NULL_POINTER;
  int64_t blocks = 0;
  for (int i = 0; i < 3; ++i) {
    if (src[i] == nullptr) continue;
    if (dst[i] == nullptr) return FA_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(src[i]) & 15u) || (reinterpret_cast<uintptr_t>(dst[i]) & 15u))
      return FA_ERR_ALIGNMENT;
    if (n[i] < 0) return FA_ERR_SEQ_LEN;
    blocks += n[i] / 8 / kCastVecs + 1;
    if (blocks > (int64_t(1) << 31) - 1) return FA_ERR_TOO_LARGE;
  }
  const CastJobs jobs = cast_jobs(src, dst, n);
  const unsigned grid = (unsigned)(jobs.blocks[0] + jobs.blocks[1] + jobs.blocks[2]);
  if (grid == 0) return FA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (bf16) hipLaunchKernelGGL(fa_cast_kernel<true>, dim3(grid), dim3(256), 0, s, jobs);
  else hipLaunchKernelGGL(fa_cast_kernel<false>, dim3(grid), dim3(256), 0, s, jobs);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FA_OK : -(int)e;
}

extern "C" int fa_varlen_fill_outside(const int32_t* cu_seqlens, int64_t B, int64_t max_seqlen,
                                      int64_t total, void* const buf[3], const int64_t heads[3],
                                      const int64_t words[3], const uint32_t value[3], void* stream) {
  using namespace fa;
  if (!cu_seqlens || !buf || !heads || !words || !value) return FA_ERR_NULL_POINTER;
  const int64_t most = (int64_t(1) << 31) - 1;
  if (B <= 0) return FA_ERR_BATCH_HEADS;
  if (max_seqlen <= 0 || total < 0) return FA_ERR_SEQ_LEN;
  if (B > most || max_seqlen > most || total > most - kFillRows) return FA_ERR_TOO_LARGE;
  FillBuf b[3];
  for (int i = 0; i < 3; ++i) {
    if (buf[i] != nullptr && (heads[i] <= 0 || words[i] <= 0 || words[i] > 4096)) return FA_ERR_TOO_LARGE;
    if (reinterpret_cast<uintptr_t>(buf[i]) & 3u) return FA_ERR_ALIGNMENT;
    b[i] = FillBuf{(uint32_t*)buf[i], heads[i], (int)words[i], value[i]};
  }
  if (total == 0) return FA_OK;
  const Geom g{cu_seqlens, (int)max_seqlen, 1, FastDiv(1), (int)total, (int)B};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int64_t chunks = (total + kFillRows - 1) / kFillRows;
  if (B > kCountedSeqs && chunks > kFillGroups)
    hipLaunchKernelGGL(fa_fill_outside_many_kernel, dim3(kFillGroups), dim3(256), 0, s, g, b[0], b[1], b[2]);
  else
    hipLaunchKernelGGL(fa_fill_outside_kernel, dim3((unsigned)chunks), dim3(256), 0, s, g, b[0], b[1], b[2]);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FA_OK : -(int)e;
}
