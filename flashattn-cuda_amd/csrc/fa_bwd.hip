// fa_bwd.hip — FlashAttention backward for gfx950 (MI355X): dQ, dK, dV from
// Q, K, V, O, dO and the forward's logsumexp L.
//
// The reference's backward (cuda/flash_attn_kernel.cu:417-503, fp32 math, one
// thread per row) runs three kernels: D_i = rowsum(dO * O) (:173-191), dQ
// (:193-...) and dK/dV, each recomputing P = exp(S - L) from the saved L. This
// file keeps that decomposition — it needs no atomics and no O(N^2) storage —
// and builds each kernel on v_mfma_f32_32x32x16_f16 with fp32 accumulation:
//
//   fa_bwd_di_kernel    D_i = sum_d dO[i][d] * O[i][d] (fp32, stored negated)
//   dK/dV body          a workgroup owns 128 keys (32 per wave, K and V as
//                       register operands) and streams 64-query tiles of Q
//                       and dO (plus L, D_i) through LDS rings: S = Q K^T,
//                       dP = dO V^T, P = exp2(S c - L log2e),
//                       dS = P (dP - D_i), dV^T += dO^T P, dK^T += Q^T dS
//   dQ body             a workgroup owns 128 queries (32 per wave, Q and dO
//                       as register operands) and streams 64-key tiles of K
//                       and V: S^T = K Q^T, dP^T = V dO^T, dS^T as above,
//                       dQ^T += K^T dS^T
//
// The two bodies run as one launch (fa_bwd_fused_kernel: a workgroup takes
// one role by its block index). In each workgroup two wave groups take the
// two 32-row halves of every tile and run one phase apart, so one wave's
// MFMAs overlap the other wave's VALU work on every SIMD.
//
// P and dS are packed to fp16 straight from the score accumulators as the B
// operands of the gradient products (the reduction index is permuted the same
// way in both operands, as in the forward). Tiles are read both as rows (b128)
// and transposed (ds_read_b64_tr_b16) from one copy whose swizzle keeps both
// reads bank-conflict free (t_swz). Two copies, one per kind of read, took
// twice the copy instructions, LDS and L2 traffic (us, two copies -> one: B4
// H16 N4096 D128 causal 1187 -> 1079, B1 H32 over 8 heads N2000 D128 causal
// bf16 187 -> 179, B1 H8 N4096 D64 137.5 -> 135.3).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>


#include <type_traits>

#include "fa_mi355x.h"
#include "fa_probe.h"
#include "fa_tile.hpp"

namespace fa {
namespace bwd {

constexpr int kBQ = 64;     // rows of a streamed tile
// Rows owned by a workgroup of two (TG = 2) or four (TG = 4) waves per 32 rows.
template <int TG>
constexpr int block_rows() { return TG == 2 ? 128 : 64; }

// Per-lane source offset of 1 KiB block b of a 64-row tile (see t_swz).
template <int D>
__device__ __forceinline__ uint32_t block_offset(int b, int lane) {
  const int o = b * 1024 + 16 * lane;
  const int r = o / (2 * D);
  const int slot = (o % (2 * D)) / 16;
  return (uint32_t)(r * 2 * D + (slot ^ t_swz<D>(r)) * 16);
}

// A pointer the caller knows to be the same in every lane, moved to SGPRs
// (buffer resources must be scalar; selects between head pointers otherwise
// leave the compiler unsure of that).
template <typename T>
__device__ __forceinline__ const T* wave_uniform(const T* p) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (const T*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// Copy 1 KiB block `blk` of 64-row tile t of a head (bytes head_bytes; rows
// past the end arrive as zeros) into LDS at dst, with per-lane offset off.
template <int D>
__device__ __forceinline__ void copy_block(const char* head, int head_bytes, int t, uint32_t dst,
                                           uint32_t off) {
  constexpr int TILE = kBQ * D * 2;
  const int done = t * TILE;
  const int bytes = max(0, min(TILE, head_bytes - done));
  dma16(make_rsrc(wave_uniform(head + (bytes > 0 ? done : 0)),
                  __builtin_amdgcn_readfirstlane(bytes)), dst, off);
}

// 64 floats of a row vector (L or D_i) starting at row t*64 into 256 bytes of
// LDS at dst, one per lane (rows >= n arrive as zeros). Dword copies: a head's
// row vector starts at bh*N floats, only 4-byte aligned.
__device__ __forceinline__ void copy_rowvec(const float* base, int n, int t, uint32_t dst,
                                            int lane) {
  const int done = t * kBQ;
  const int bytes = max(0, min(kBQ, n - done)) * 4;
  dma4(make_rsrc(wave_uniform(base + (bytes > 0 ? done : 0)),
                 __builtin_amdgcn_readfirstlane(bytes)), dst, (uint32_t)(4 * lane));
}

// B operand (16 x 32) of a product over D from 32 rows of a [N][D] fp16 head:
// lane l holds row (row0 + l%32), columns 16 kk + 8 (l/32) .. +7 (zeros for
// rows >= n via the buffer range).
template <int D>
__device__ __forceinline__ void load_row_operand(const f16* head, int n, int row0, int lane,
                                                 f16x8 (&out)[D / 16]) {
  const __amdgpu_buffer_rsrc_t r = make_rsrc(head, n * D * 2);
  const int row = row0 + (lane & 31);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(
        r, (uint32_t)(row * D + 16 * kk + 8 * (lane >> 5)) * 2, 0, 0);
    out[kk] = __builtin_bit_cast(f16x8, x);
  }
}

// Store the first NDB blocks of a C-layout accumulator acc[DB] (rows = 32 d of
// each block, columns = 32 rows of the output) as fp32 rows out[row][d], scaled.
template <int D, int NDB>
__device__ __forceinline__ void store_transposed(float* out, int n, int row0, int lane,
                                                 const f32x16 (&acc)[D / 32], float scale) {
  const int row = row0 + (lane & 31);
  if (row >= n) return;
  float* dst = out + (size_t)row * D + 4 * (lane >> 5);
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v = {acc[db][4 * g] * scale, acc[db][4 * g + 1] * scale, acc[db][4 * g + 2] * scale,
                 acc[db][4 * g + 3] * scale};
      *reinterpret_cast<f32x4*>(dst + 32 * db + 8 * g) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Row terms: ND[i] = -D_i = -sum_d dO[i][d] * O[i][d] and NL[i] = -L[i] *
// log2(e), so that P = exp2(S c + NL) takes one fma and dP - D_i = dP + ND
// one add (or an MFMA chain's initial value). 8 lanes per row, one 16-byte
// chunk each per step (coalesced 128-byte runs), reduced with xor shuffles.
// O and dO may come in fp32 (o32, g32; then rounded to the operand type
// first, and dO also stored so): the pass reads them anyway, and the blocks
// after its own convert Q, K and V, so a caller with fp32 tensors needs no
// launches of its own for that (five conversions cost half of a B2 H8 N512
// D64 backward).
// ---------------------------------------------------------------------------
struct RowTermArgs {
  const f16* o;
  f16* g;            // dO: given, or written from g32
  const float* o32;
  const float* g32;
  const float* l;
  float* nd;
  float* nl;
  int64_t rows;
  int blocks;        // 32 rows each; later workgroups convert
};

template <int D, bool BF16>
__global__ void __launch_bounds__(256)
fa_bwd_di_kernel(RowTermArgs a, CastJobs jobs) {
  if ((int)blockIdx.x >= a.blocks) {
    cast_block<BF16>(jobs, (int)blockIdx.x - a.blocks);
    return;
  }
  const int64_t row = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
  const int part = threadIdx.x & 7;
  float acc = 0.f;
  if (row < a.rows) {
#pragma unroll
    for (int i = part; i < D / 8; i += 8) {
      const int64_t at = row * D + 8 * i;
      const f16x8 x = a.o32 != nullptr ? cvt8x<BF16>(a.o32 + at)
                                       : *reinterpret_cast<const f16x8*>(a.o + at);
      f16x8 y;
      if (a.g32 != nullptr) {
        y = cvt8x<BF16>(a.g32 + at);
        *reinterpret_cast<f16x8*>(a.g + at) = y;
      } else {
        y = *reinterpret_cast<const f16x8*>(a.g + at);
      }
      if constexpr (BF16) {
        const bf16x8 xb = __builtin_bit_cast(bf16x8, x), yb = __builtin_bit_cast(bf16x8, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = fmaf((float)xb[e], (float)yb[e], acc);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = fmaf((float)x[e], (float)y[e], acc);
      }
    }
  }
  acc += __shfl_xor(acc, 1, 8);
  acc += __shfl_xor(acc, 2, 8);
  acc += __shfl_xor(acc, 4, 8);
  if (row < a.rows && part == 0) {
    a.nd[row] = -acc;
    a.nl[row] = -a.l[row] * kLog2e;
  }
}

// Accumulator block x of NA arrays of DB blocks, to and from LDS in 16-byte
// accesses (lane-major, conflict-free).
constexpr int kAccBytes = 64 * 16 * 4;   // of a wave's block

__device__ __forceinline__ void put_block(char* at, int lane, const f32x16& a) {
  f32x4* p = reinterpret_cast<f32x4*>(at) + lane;
#pragma unroll
  for (int q = 0; q < 4; ++q) p[64 * q] = f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
}

__device__ __forceinline__ void add_block(const char* at, int lane, f32x16& a) {
  const f32x4* p = reinterpret_cast<const f32x4*>(at) + lane;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 v = p[64 * q];
#pragma unroll
    for (int e = 0; e < 4; ++e) a[4 * q + e] += v[e];
  }
}

// Sums of the partials of the waves that hold the same keys (queries). The two
// groups trade halves, so all eight waves add and store: of the NA x DB blocks
// group 0 ends with the sums of the first half and group 1 with those of the
// second, either in blocks 0 .. HALF - 1 of `a`. (Group 0 adding and storing
// everything, in 4-byte accesses, took B1 H32 N2000 D128 causal 174.9 us, this
// 173.2; long equal units do not notice.) With TG = 4, waves 2 and 3 of a group then send theirs to waves 0
// and 1. True in the waves that hold sums.
template <int TG, int NA, int DB>
__device__ __forceinline__ bool reduce_rows(char* smem, int grp, int wi, int lane,
                                            f32x16 (&a)[NA][DB]) {
  constexpr int HALF = NA * DB / 2;
  char* mine = smem + (grp * 4 + wi) * HALF * kAccBytes;          // written by this wave
  const char* other = smem + ((grp ^ 1) * 4 + wi) * HALF * kAccBytes;
  __syncthreads();   // every wave is done with the staging buffers
  // Selects, not branches: a branch over which block is meant would make the
  // compiler index the accumulators and keep them in scratch.
  static_for<0, HALF>([&](auto xi) {
    constexpr int x = decltype(xi)::value, y = x + HALF;
    f32x16 send;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float lo = a[x / DB][x % DB][r], hi = a[y / DB][y % DB][r];
      send[r] = grp == 0 ? hi : lo;
      a[x / DB][x % DB][r] = grp == 0 ? lo : hi;
    }
    put_block(mine + x * kAccBytes, lane, send);
  });
  __syncthreads();
  static_for<0, HALF>([&](auto xi) {
    constexpr int x = decltype(xi)::value;
    add_block(other + x * kAccBytes, lane, a[x / DB][x % DB]);
  });
  if constexpr (TG == 2) return true;
  __syncthreads();
  if (wi >= 2) {
    static_for<0, HALF>([&](auto xi) {
      constexpr int x = decltype(xi)::value;
      put_block(mine + x * kAccBytes, lane, a[x / DB][x % DB]);
    });
  }
  __syncthreads();
  if (wi >= 2) return false;
  const char* upper = smem + (grp * 4 + wi + 2) * HALF * kAccBytes;
  static_for<0, HALF>([&](auto xi) {
    constexpr int x = decltype(xi)::value;
    add_block(upper + x * kAccBytes, lane, a[x / DB][x % DB]);
  });
  return true;
}

// ---------------------------------------------------------------------------
// dK/dV and dQ bodies (8 waves). A dK/dV workgroup owns 128 keys of one
// (b, h): wave w holds K^T and V^T of keys k0 + 32 (w % 4) .. +31 as register
// B operands, and 64-query tiles of Q and dO stream through LDS (read as rows
// for the score products, transposed for the gradient products), with 64
// floats each of NL and -D_i. A dQ workgroup owns 128 queries the same way
// (Q^T and dO^T as register operands, NL and -D_i lane constants) and streams
// 64-key tiles of K and V.
//
// The two wave groups (waves 0-3 and 4-7) hold the same keys (dK/dV) or
// queries (dQ), each takes one 32-row half of every tile, their partial sums
// are added through LDS at the end (reduce_rows), and they run one phase
// apart. Each tile's work splits into the score products A (S and dP
// MFMAs), the VALU part B (P, dS, packed as B operands) and the gradient
// products C; a group's matrix phase M(j) issues C of its tile j - 1 and A
// of tile j, its softmax phase S(j) runs B of tile j. In every phase one
// group is in M and the other in S, so each SIMD overlaps one wave's MFMAs
// with the other's VALU work:
//
//   phase      2j          2j+1        ...   2T          2T+1
//   group 0    M(j)        S(j)              C(T-1)      -
//   group 1    S(j-1)      M(j)              S(T-1)      C(T-1)
//
// A group reads only its own 32-row half of every tile, so it copies only
// that half, and the row vectors into slots of its own: the groups share no
// staged data, and the barriers keep them one phase apart and sync each
// group's four waves on their copies.
//
// That is TG = 2. With TG = 4 a workgroup owns 64 keys (queries), so a launch
// has twice the workgroups: each group takes whole tiles, group 0 the even and
// group 1 the odd ones, in a ring of its own, two waves hold each 32 keys and
// take a tile's two halves, and four partial sums are added at the end.
//
// D = 64 (rows 32 g .. +31 of each part are its 1 KiB blocks 4 g .. 4 g + 3):
// tile j's stage is read from S(j - 1), which loads tile j's A operands into registers (M(j) then
// issues its score products without LDS waits), to M(j + 1), which reads its
// C operands. S(j) starts the copies of tile j + 3 into the stage of tile
// j - 1 (last read in M(j), before the barrier that starts S(j)) and M(j + 2)
// waits for them, leaving those of S(j + 1) in flight: a ring of 4 stages,
// with the copy issue in the VALU phase.
// ---------------------------------------------------------------------------
constexpr int kPPStages = 4;

template <int D, int TG>
constexpr int dkdv_pp_smem() {
  constexpr int STAGE = 2 * (kBQ * D * 2) + 2048;
  constexpr int RED = 4 * 2 * (D / 32) * 16 * 64 * 4;
  return TG / 2 * kPPStages * STAGE > RED ? TG / 2 * kPPStages * STAGE : RED;
}

template <int D, int TG>
constexpr int dq_pp_smem() {
  constexpr int STAGE = 2 * (kBQ * D * 2);
  constexpr int RED = 4 * (D / 32) * 16 * 64 * 4;
  return TG / 2 * kPPStages * STAGE > RED ? TG / 2 * kPPStages * STAGE : RED;
}

template <int D, bool CAUSAL, bool BF16, int TG>
__device__ __forceinline__ void dkdv_body_pp(const f16* __restrict__ Q, const f16* __restrict__ K,
                                             const f16* __restrict__ V, const f16* __restrict__ dO,
                                             const float* __restrict__ NL,
                                             const float* __restrict__ ND, float* __restrict__ dK,
                                             float* __restrict__ dV, const HeadView& hv, int kb, float c,
                                             float scale, char* smem /* dkdv_pp_smem<D>() bytes */) {
  static_assert(D == 64, "a 32-row half of a tile is 4 blocks, the register budget D = 64's");
  constexpr int TILE = kBQ * D * 2;
  constexpr int BLOCKS = TILE / 1024;
  constexpr int OWN = BLOCKS / 2;              // blocks of a 32-row half
  constexpr int PER = TG == 2 ? OWN / 2 : OWN; // blocks per wave of a group's copies
  constexpr int KSTEPS = D / 16, DB = D / 32;
  constexpr int R = kPPStages;                 // stages of a ring (TG = 4: one per group)
  // Q | dO | row vectors (group g: L at +512 g, D_i at +512 g + 256)
  constexpr int STAGE = 2 * TILE + 2048;
  static_assert(TG / 2 * R * STAGE <= 160 * 1024, "LDS");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave & 3, grp = wave >> 2;
  const int kw = TG == 2 ? wi : wi & 1;        // keys 32 kw .. +31 of the block
  const int qb = TG == 2 ? grp : wi >> 1;      // query half of a tile
  const int hi = lane >> 5;
  const int k0 = kb * block_rows<TG>();
  const int key = k0 + 32 * kw + (lane & 31);

  const int N = hv.n;
  const size_t head = hv.q;
  const int head_bytes = N * D * 2;
  const char* Qh = reinterpret_cast<const char*>(Q + head);
  const char* Gh = reinterpret_cast<const char*>(dO + head);
  const float* Lh = NL + hv.l;
  const float* Dh = ND + hv.l;   // -D_i

  f16x8 kf[KSTEPS], vf[KSTEPS];   // B operands: K^T and V^T of this wave's keys
  load_row_operand<D>(K + hv.kv, N, k0 + 32 * kw, lane, kf);
  load_row_operand<D>(V + hv.kv, N, k0 + 32 * kw, lane, vf);
  f32x16 acc[2][DB];              // [0] = dV^T, [1] = dK^T (unscaled)
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    acc[0][db] = f32x16{};
    acc[1][db] = f32x16{};
  }

  const int n_qt = (N + kBQ - 1) / kBQ;
  const int t0 = CAUSAL ? k0 / kBQ : 0;   // earlier query tiles see none of these keys
  // Steps of this workgroup (>= 1); its groups take a half each of tile j in
  // step j, or (TG = 4) tiles 2 j and 2 j + 1, the last possibly past the end.
  const int T = TG == 2 ? n_qt - t0 : (n_qt - t0 + 1) / 2;
  auto tile_of = [&](int j) { return TG == 2 ? t0 + j : t0 + 2 * j + grp; };

  const uint32_t lds0 = lds_addr(smem);
  const uint32_t half0 = lds0 + qb * 32 * 2 * D;   // this wave's rows of a part
  auto slot_of = [&](int j) { return (TG == 2 ? 0 : grp * R) + j % R; };
  const int rv0 = 2 * TILE + (TG == 2 ? 512 * grp : 0);   // this group's row vectors
  // This group's half (TG = 4: whole) of step j's tile: wave wi copies PER
  // blocks of part wi / 2; waves 0 and 1 also copy the 64-row L and D_i
  // vectors.
  auto issue_own = [&](int j) {
    const uint32_t base = lds0 + slot_of(j) * STAGE;
    const char* src = wi < 2 ? Qh : Gh;
    const int t = tile_of(j);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int b = (TG == 2 ? OWN * grp : 0) + PER * (wi & 1) + i;
      copy_block<D>(src, head_bytes, t, base + (wi >> 1) * TILE + b * 1024, block_offset<D>(b, lane));
    }
    if (wi == 0) copy_rowvec(Lh, N, t, base + rv0, lane);
    if (wi == 1) copy_rowvec(Dh, N, t, base + rv0 + 256, lane);
  };
  // Copies run three tiles ahead: at the end of M phase j tile j + 1 must
  // have landed, and tile j + 2's copies (this wave's last issue) may still
  // be in flight.
  auto wait_next = [&](bool later_in_flight) {
    if (!later_in_flight) wait_vmem();
    else if (wi < 2) wait_vmcnt<PER + 1>();
    else wait_vmcnt<PER>();
  };
  issue_own(0);
  if (T > 1) issue_own(1);
  if (T > 2) issue_own(2);
  wait_next(T > 2);
  __syncthreads();

  f32x16 s = {}, dp = {};   // this wave's scores of its current tile
  f16x8 pb[2], gb[2];       // its packed P and dS (B operands of the two k-steps)
  f16x8 af[KSTEPS][2];      // A operands of its next score products (Q, dO rows)
  auto load_a = [&](int j) {   // of relative tile j
    const uint32_t rb = row_base<D>(half0 + slot_of(j) * STAGE, lane);
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      af[kk][0] = load_row_frag<D>(rb, 0, kk);
      af[kk][1] = load_row_frag<D>(rb, TILE, kk);
    }
  };
  // A: S = Q K^T and dP = dO V^T (C layout: register r holds query
  // qt0 + 32 qb + 8 (r/4) + 4 hi + r%4, lane l key l%32).
  auto mma_a = [&](int kk) {
    s = mma32<BF16>(af[kk][0], kf[kk], kk == 0 ? f32x16{} : s);
    dp = mma32<BF16>(af[kk][1], vf[kk], kk == 0 ? f32x16{} : dp);
  };
  // C of the tile whose column base is cb: dV^T += dO^T P and dK^T += Q^T dS; step
  // kk is k-step kk / DB, d-block kk % DB. Operands (dO^T, Q^T) read two
  // steps ahead.
  auto load_c = [&](uint32_t cb, int kk, f16x8 (&f)[2]) {
    f[0] = load_col_frag<D>(cb, TILE, kk / DB, kk % DB);
    f[1] = load_col_frag<D>(cb, 0, kk / DB, kk % DB);
  };
  auto mma_c = [&](const f16x8 (&f)[2], int kk) {
    const int h = kk / DB, db = kk % DB;
    acc[0][db] = mma32<BF16>(f[0], pb[h], acc[0][db]);
    acc[1][db] = mma32<BF16>(f[1], gb[h], acc[1][db]);
  };
  // M phase of relative tile j (WITH_C: C of tile j - 1; WITH_A: A of tile
  // j); then the wait for the copies this wave started in S(j - 1).
  auto mphase = [&](int j, auto with_c, auto with_a) {
    constexpr bool WC = decltype(with_c)::value, WA = decltype(with_a)::value;
    const uint32_t sc = col_base<D>(half0 + slot_of(j + R - 1) * STAGE, lane);
    f16x8 cf[KSTEPS][2];
    if constexpr (WC) {
      load_c(sc, 0, cf[0]);
      load_c(sc, 1, cf[1]);
    }
    static_for<0, KSTEPS>([&](auto ki) {
      constexpr int kk = decltype(ki)::value;
      if constexpr (WC && kk + 2 < KSTEPS) load_c(sc, kk + 2, cf[kk + 2]);
      if constexpr (WA) mma_a(kk);   // register operands: first, while C's land
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (WC) mma_c(cf[kk], kk);
      __builtin_amdgcn_sched_barrier(0);   // keep every product in this phase
    });
    wait_next(j + 2 < T);
  };
  // S phase of relative tile j: the copies of tile j + 3 (into the stage of
  // tile j - 1, whose last reads were this group's M phase j), P and dS into
  // pb, gb, and tile j + 1's A operands.
  auto sphase = [&](int j) {
    if (j + 3 < T) issue_own(j + 3);
    const int qt0 = tile_of(j) * kBQ;
    const float* ls = reinterpret_cast<const float*>(smem + slot_of(j) * STAGE + rv0);
    const float* nds = ls + 64;
    // Row vectors first (LDS reads return in order), then the next tile's A
    // operands, which land while the VALU work below runs.
    f32x4 lq[4], nd[4];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      lq[r4] = *reinterpret_cast<const f32x4*>(ls + 32 * qb + 8 * r4 + 4 * hi);
      nd[r4] = *reinterpret_cast<const f32x4*>(nds + 32 * qb + 8 * r4 + 4 * hi);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (j + 1 < T) load_a(j + 1);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 p, g;
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = exp2_hw(fmaf(s[r], c, lq[r >> 2][r & 3]));
    const bool edge = (qt0 + 32 * qb + 32 > N) || (CAUSAL && qt0 + 32 * qb < k0 + 32 * kw + 32);
    if (edge) {   // rows past N, and (causal) keys after the row
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int q = qt0 + 32 * qb + 8 * (r >> 2) + 4 * hi + (r & 3);
        p[r] = ((q >= N) || (CAUSAL && key > q)) ? 0.f : p[r];
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) g[r] = p[r] * (dp[r] + nd[r >> 2][r & 3]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      pb[h] = pack_px<BF16>(p, h);
      gb[h] = pack_px<BF16>(g, h);
    }
  };
  // Register-only work stays in its phase (see the forward kernel).
  auto pin_s = [&] { asm volatile("" : "+v"(s), "+v"(dp)); };
  auto pin_p = [&] { asm volatile("" : "+v"(pb[0]), "+v"(pb[1]), "+v"(gb[0]), "+v"(gb[1])); };

  using BT = std::true_type;
  using BF = std::false_type;
  load_a(0);
  if (grp == 1) __syncthreads();   // phase 0: group 1 waits
  mphase(0, BF{}, BT{});
  __syncthreads();
  pin_s();
  sphase(0);
  pin_p();
  __syncthreads();
  for (int j = 1; j < T; ++j) {
    mphase(j, BT{}, BT{});
    __syncthreads();
    pin_s();
    sphase(j);
    pin_p();
    __syncthreads();
  }
  mphase(T, BT{}, BF{});   // C of the last tile
  __syncthreads();
  if (grp == 0) __syncthreads();   // phase 2T + 1: group 0 waits
  if (reduce_rows<TG, 2, DB>(smem, grp, wi, lane, acc)) {
    // group 0 has dV, group 1 dK
    store_transposed<D, DB>((grp == 0 ? dV : dK) + head, N, k0 + 32 * kw, lane, acc[0],
                            grp == 0 ? 1.f : scale);
  }
}

template <int D, bool CAUSAL, bool BF16, int TG>
__device__ __forceinline__ void dq_body_pp(const f16* __restrict__ Q, const f16* __restrict__ K,
                                           const f16* __restrict__ V, const f16* __restrict__ dO,
                                           const float* __restrict__ NL,
                                           const float* __restrict__ ND, float* __restrict__ dQ,
                                           const HeadView& hv, int qblk, float c, float scale,
                                           char* smem /* dq_pp_smem<D>() bytes */) {
  static_assert(D == 64, "a 32-row half of a tile is 4 blocks, the register budget D = 64's");
  constexpr int TILE = kBQ * D * 2;
  constexpr int BLOCKS = TILE / 1024;
  constexpr int OWN = BLOCKS / 2;              // blocks of a 32-row half
  constexpr int PER = TG == 2 ? OWN / 2 : OWN; // blocks per wave of a group's copies
  constexpr int KSTEPS = D / 16, DB = D / 32;
  constexpr int R = kPPStages;
  constexpr int STAGE = 2 * TILE;              // K | V
  static_assert(TG / 2 * R * STAGE <= 160 * 1024, "LDS");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave & 3, grp = wave >> 2;
  const int qw = TG == 2 ? wi : wi & 1;        // queries 32 qw .. +31 of the block
  const int half = TG == 2 ? grp : wi >> 1;    // key half of a tile
  const int hi = lane >> 5;
  const int q0 = qblk * block_rows<TG>();
  const int query = q0 + 32 * qw + (lane & 31);

  const int N = hv.n;
  const size_t head = hv.q;
  const int head_bytes = N * D * 2;
  const char* Kh = reinterpret_cast<const char*>(K + hv.kv);
  const char* Vh = reinterpret_cast<const char*>(V + hv.kv);

  f16x8 qf[KSTEPS], gf[KSTEPS];   // B operands: Q^T and dO^T of this wave's queries
  load_row_operand<D>(Q + head, N, q0 + 32 * qw, lane, qf);
  load_row_operand<D>(dO + head, N, q0 + 32 * qw, lane, gf);
  const bool row_ok = query < N;
  const float nl = row_ok ? NL[hv.l + query] : 0.f;
  // dP^T starts from -D_i (a lane constant), so the chain yields dP - D_i.
  const float ndi = row_ok ? ND[hv.l + query] : 0.f;
  f32x16 acc[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = f32x16{};

  const int kv_end = CAUSAL ? min(N, q0 + block_rows<TG>()) : N;
  const int n_kt = (kv_end + kBQ - 1) / kBQ;   // >= 1
  // Steps: as in the dK/dV body.
  const int T = TG == 2 ? n_kt : (n_kt + 1) / 2;
  auto tile_of = [&](int j) { return TG == 2 ? j : 2 * j + grp; };
  // rows past N (last block only) and, causal, keys after the wave's first query
  const bool rows_edge = q0 + 32 * qw + 32 > N;

  const uint32_t lds0 = lds_addr(smem);
  const uint32_t half0 = lds0 + half * 32 * 2 * D;   // this wave's rows of a part
  auto slot_of = [&](int j) { return (TG == 2 ? 0 : grp * R) + j % R; };
  // This group's half (TG = 4: whole) of step j's tile: wave wi copies PER
  // blocks of part wi / 2.
  auto issue_own = [&](int j) {
    const uint32_t base = lds0 + slot_of(j) * STAGE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int b = (TG == 2 ? OWN * grp : 0) + PER * (wi & 1) + i;
      copy_block<D>(wi < 2 ? Kh : Vh, head_bytes, tile_of(j), base + (wi >> 1) * TILE + b * 1024,
                    block_offset<D>(b, lane));
    }
  };
  // Copies run three tiles ahead (as in the dK/dV body).
  auto wait_next = [&](bool later_in_flight) {
    if (later_in_flight) wait_vmcnt<PER>();
    else wait_vmem();
  };
  issue_own(0);
  if (T > 1) issue_own(1);
  if (T > 2) issue_own(2);
  wait_next(T > 2);
  __syncthreads();

  f32x16 s = {}, dp = {};
  f16x8 gb[2];
  f16x8 af[KSTEPS][2];   // A operands of the next score products (K, V rows)
  auto load_a = [&](int j) {
    const uint32_t rb = row_base<D>(half0 + slot_of(j) * STAGE, lane);
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      af[kk][0] = load_row_frag<D>(rb, 0, kk);
      af[kk][1] = load_row_frag<D>(rb, TILE, kk);
    }
  };
  auto mma_a = [&](int kk) {
    f32x16 dp0;
#pragma unroll
    for (int r = 0; r < 16; ++r) dp0[r] = ndi;
    s = mma32<BF16>(af[kk][0], qf[kk], kk == 0 ? f32x16{} : s);
    dp = mma32<BF16>(af[kk][1], gf[kk], kk == 0 ? dp0 : dp);
  };
  auto load_c = [&](uint32_t cb, int kk) { return load_col_frag<D>(cb, 0, kk / DB, kk % DB); };
  auto mphase = [&](int j, auto with_c, auto with_a) {
    constexpr bool WC = decltype(with_c)::value, WA = decltype(with_a)::value;
    const uint32_t sc = col_base<D>(half0 + slot_of(j + R - 1) * STAGE, lane);
    f16x8 cf[KSTEPS];
    if constexpr (WC) {
      cf[0] = load_c(sc, 0);
      cf[1] = load_c(sc, 1);
    }
    static_for<0, KSTEPS>([&](auto ki) {
      constexpr int kk = decltype(ki)::value;
      if constexpr (WC && kk + 2 < KSTEPS) cf[kk + 2] = load_c(sc, kk + 2);
      if constexpr (WA) mma_a(kk);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (WC) acc[0][kk % DB] = mma32<BF16>(cf[kk], gb[kk / DB], acc[0][kk % DB]);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_next(j + 2 < T);
  };
  auto sphase = [&](int j) {
    if (j + 3 < T) issue_own(j + 3);
    if (j + 1 < T) load_a(j + 1);
    const int kt0 = tile_of(j) * kBQ;
    f32x16 p;
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = exp2_hw(fmaf(s[r], c, nl));
    const bool edge = rows_edge || (kt0 + 32 * half + 32 > N) ||
                      (CAUSAL && kt0 + 32 * half + 31 > q0 + 32 * qw);
    if (edge) {   // keys past N, rows past N, and (causal) keys after the row
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kidx = kt0 + 32 * half + 8 * (r >> 2) + 4 * hi + (r & 3);
        p[r] = ((kidx >= N) || (CAUSAL && kidx > query) || !row_ok) ? 0.f : p[r];
      }
    }
    f32x16 g;
#pragma unroll
    for (int r = 0; r < 16; ++r) g[r] = p[r] * dp[r];
#pragma unroll
    for (int h = 0; h < 2; ++h) gb[h] = pack_px<BF16>(g, h);
  };
  auto pin_s = [&] { asm volatile("" : "+v"(s), "+v"(dp)); };
  auto pin_p = [&] { asm volatile("" : "+v"(gb[0]), "+v"(gb[1])); };

  using BT = std::true_type;
  using BF = std::false_type;
  load_a(0);
  if (grp == 1) __syncthreads();   // phase 0: group 1 waits
  mphase(0, BF{}, BT{});
  __syncthreads();
  pin_s();
  sphase(0);
  pin_p();
  __syncthreads();
  for (int j = 1; j < T; ++j) {
    mphase(j, BT{}, BT{});
    __syncthreads();
    pin_s();
    sphase(j);
    pin_p();
    __syncthreads();
  }
  mphase(T, BT{}, BF{});   // C of the last tile
  __syncthreads();
  if (grp == 0) __syncthreads();   // phase 2T + 1: group 0 waits
  if (reduce_rows<TG, 1, DB>(smem, grp, wi, lane, acc)) {
    // group 1 has the upper half of the columns
    store_transposed<D, DB / 2>(dQ + head + grp * (D / 2), N, q0 + 32 * qw, lane, acc[0], scale);
  }
}

// ---------------------------------------------------------------------------
// D = 128. The phases are those of the D = 64 forms (M(j): C of tile j - 1,
// then A of tile j; S(j): B of tile j; the two groups one phase apart),
// fitted to D = 128's budgets:
//   * registers: the score products' A operands are read from LDS inside
//     the M phase (not prefetched into registers), and the M phase runs all
//     of C(j - 1) before A(j), so the packed P and dS of tile j - 1 are dead
//     before S and dP of tile j are live: the dK/dV body fits the 256 VGPRs
//     of two waves per SIMD without spilling (K^T, V^T and the two
//     accumulators alone take 192);
//   * LDS: a ring of three tiles (99 KiB with the row vectors; the final
//     reduction takes 128). S(j) starts the copies of tile j + 2 into the slot
//     of tile j - 1 (last read in M(j)), and its end waits for those of S(j - 1):
//     every copy has two phases to land, issued from the VALU phase. TG = 4 has
//     two slots per group: S(j) starts and awaits tile j + 1.
// A group copies and reads only its own 32-row half of every part (rows
// 32 g .. +31 are 1 KiB blocks 8 g .. 8 g + 7).
// ---------------------------------------------------------------------------
template <int TG>
constexpr int pp128_slots() { return TG == 2 ? 3 : 4; }   // tiles in LDS (TG = 4: two per group)

template <int D, int TG>
constexpr int dkdv_pp128_smem() {
  constexpr int TILE = kBQ * D * 2;
  constexpr int RING = pp128_slots<TG>() * (2 * TILE + 1024);
  constexpr int RED = 4 * 2 * (D / 32) * 16 * 64 * 4;
  return RING > RED ? RING : RED;
}

template <int D, int TG>
constexpr int dq_pp128_smem() {
  constexpr int TILE = kBQ * D * 2;
  constexpr int RING = pp128_slots<TG>() * (2 * TILE);
  constexpr int RED = 4 * (D / 32) * 16 * 64 * 4;
  return RING > RED ? RING : RED;
}

template <int D, bool CAUSAL, bool BF16, int TG>
__device__ __forceinline__ void dkdv_body_pp128(const f16* __restrict__ Q,
                                                const f16* __restrict__ K,
                                                const f16* __restrict__ V,
                                                const f16* __restrict__ dO,
                                                const float* __restrict__ NL,
                                                const float* __restrict__ ND,
                                                float* __restrict__ dK, float* __restrict__ dV,
                                                const HeadView& hv, int kb, float c, float scale,
                                                char* smem /* dkdv_pp128_smem<D>() bytes */) {
  static_assert(D == 128, "a 32-row half of a tile is 8 blocks");
  constexpr int TILE = kBQ * D * 2;
  constexpr int BLOCKS = TILE / 1024;
  constexpr int OWN = BLOCKS / 2;              // blocks of a 32-row half
  constexpr int PER = TG == 2 ? OWN / 2 : OWN; // blocks per wave of a tile
  constexpr int KSTEPS = D / 16, DB = D / 32;
  constexpr int SLOT = 2 * TILE;               // Q | dO
  constexpr int R = TG == 2 ? 3 : 2;           // slots of a ring (TG = 4: one per group)
  constexpr int R0 = pp128_slots<TG>() * SLOT; // row vectors: group g L at +512 g, -D_i +256
  static_assert(R0 + pp128_slots<TG>() * 1024 <= dkdv_pp128_smem<D, TG>() && dkdv_pp128_smem<D, TG>() <= 160 * 1024,
                "ring inside the buffer, LDS");
  static_assert(2 * KSTEPS == 2 * 2 * DB, "C and A take the same number of steps");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave & 3, grp = wave >> 2;
  const int kw = TG == 2 ? wi : wi & 1;        // keys 32 kw .. +31 of the block
  const int qb = TG == 2 ? grp : wi >> 1;      // query half of a tile
  const int hi = lane >> 5;
  const int k0 = kb * block_rows<TG>();

  const int N = hv.n;
  const size_t head = hv.q;
  const int head_bytes = N * D * 2;
  const char* Qh = reinterpret_cast<const char*>(Q + head);
  const char* Gh = reinterpret_cast<const char*>(dO + head);
  const float* Lh = NL + hv.l;
  const float* Dh = ND + hv.l;   // -D_i

  f16x8 kf[KSTEPS], vf[KSTEPS];   // B operands: K^T and V^T of this wave's keys
  load_row_operand<D>(K + hv.kv, N, k0 + 32 * kw, lane, kf);
  load_row_operand<D>(V + hv.kv, N, k0 + 32 * kw, lane, vf);
  f32x16 acc[2][DB];              // [0] = dV^T, [1] = dK^T (unscaled)
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    acc[0][db] = f32x16{};
    acc[1][db] = f32x16{};
  }

  const int n_qt = (N + kBQ - 1) / kBQ;
  const int t0 = CAUSAL ? k0 / kBQ : 0;   // earlier query tiles see none of these keys
  // Steps of this workgroup (>= 1); its groups take a half each of tile j in
  // step j, or (TG = 4) tiles 2 j and 2 j + 1, the last possibly past the end.
  const int T = TG == 2 ? n_qt - t0 : (n_qt - t0 + 1) / 2;
  auto tile_of = [&](int j) { return TG == 2 ? t0 + j : t0 + 2 * j + grp; };

  const uint32_t lds0 = lds_addr(smem);
  const uint32_t half0 = lds0 + qb * 32 * 2 * D;   // this wave's rows of a part
  auto slot_of = [&](int j) { return (TG == 2 ? 0 : grp * R) + j % R; };
  const int rv0 = R0 + (TG == 2 ? 512 * grp : 0);   // this group's row vectors
  // Wave wi copies PER blocks of part wi >> 1 (Q or dO) of this group's half
  // (TG = 4: whole) of step j's tile, waves 0 and 1 also its row vectors; the
  // per-lane offsets are recomputed per copy (volatile lane id: held across
  // the loop they would take registers the body needs).
  auto issue_tile = [&](int j) {
    int ln;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
    const char* src = wi < 2 ? Qh : Gh;
    const int t = tile_of(j);
    const uint32_t base = lds0 + slot_of(j) * SLOT + (wi >> 1) * TILE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int b = (TG == 2 ? OWN * grp : 0) + PER * (wi & 1) + i;
      copy_block<D>(src, head_bytes, t, base + b * 1024, block_offset<D>(b, ln));
    }
    const uint32_t rv = lds0 + rv0 + slot_of(j) * 1024;
    if (wi == 0) copy_rowvec(Lh, N, t, rv, ln);
    if (wi == 1) copy_rowvec(Dh, N, t, rv + 256, ln);
  };
  // All copies but those of the last tile issued (if `last` was).
  auto wait_for = [&](bool last) {
    if (!last) wait_vmem();
    else if (wi < 2) wait_vmcnt<PER + 1>();
    else wait_vmcnt<PER>();
  };
  constexpr int AHEAD = R - 1;   // S(j) starts the copies of tile j + AHEAD
  issue_tile(0);
  if (AHEAD > 1 && T > 1) issue_tile(1);
  wait_for(AHEAD > 1 && T > 1);
  __syncthreads();

  f32x16 s = {}, dp = {};   // this wave's scores of its current tile
  f16x8 pb[2], gb[2];       // its packed P and dS (B operands of the two k-steps)
  // M phase of relative tile j: C of tile j - 1 (dV^T += dO^T P, dK^T += Q^T
  // dS; step x: k-step x / DB, d-block x % DB), then A of tile j (S = Q K^T,
  // dP = dO V^T; step x: k-step x). Operands two steps ahead.
  auto mphase = [&](int j, auto with_c, auto with_a) {
    constexpr bool WC = decltype(with_c)::value, WA = decltype(with_a)::value;
    constexpr int X0 = WC ? 0 : KSTEPS, X1 = WA ? 2 * KSTEPS : KSTEPS;
    const uint32_t sc = col_base<D>(half0 + slot_of(j + R - 1) * SLOT, lane);   // tile j - 1
    const uint32_t sa = row_base<D>(half0 + slot_of(j) * SLOT, lane);           // tile j
    f16x8 f[2 * KSTEPS][2];
    auto load = [&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (x < KSTEPS) {
        f[x][0] = load_col_frag<D>(sc, TILE, x / DB, x % DB);   // dO^T
        f[x][1] = load_col_frag<D>(sc, 0, x / DB, x % DB);      // Q^T
      } else {
        f[x][0] = load_row_frag<D>(sa, 0, x - KSTEPS);      // Q rows
        f[x][1] = load_row_frag<D>(sa, TILE, x - KSTEPS);   // dO rows
      }
    };
    // Operands two steps ahead within each part; A's first two are loaded
    // where A starts, once C's last operands are consumed (loading them
    // during C measured 2 % slower at config 3).
    auto ahead = [&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (x < X1 && (x < KSTEPS || x >= KSTEPS + 2 || !WC)) load(xi);
    };
    static_for<X0, X0 + 2>(load);   // X1 - X0 >= KSTEPS
    static_for<X0, X1>([&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (WC && WA && x == KSTEPS) static_for<KSTEPS, KSTEPS + 2>(load);
      ahead(std::integral_constant<int, x + 2>{});
      if constexpr (x < KSTEPS) {
        acc[0][x % DB] = mma32<BF16>(f[x][0], pb[x / DB], acc[0][x % DB]);
        acc[1][x % DB] = mma32<BF16>(f[x][1], gb[x / DB], acc[1][x % DB]);
      } else {
        constexpr int kk = x - KSTEPS;
        s = mma32<BF16>(f[x][0], kf[kk], kk == 0 ? f32x16{} : s);
        dp = mma32<BF16>(f[x][1], vf[kk], kk == 0 ? f32x16{} : dp);
      }
      if constexpr (x + 1 == KSTEPS) __builtin_amdgcn_sched_barrier(0);   // C before A
    });
    __builtin_amdgcn_sched_barrier(0);   // keep every product in this phase
  };
  // S phase of relative tile j: the copies of tile j + 2, then P and dS into
  // pb, gb; at the end, the wait for the copies of S(j - 1) (tile j + 1:
  // M(j + 1) reads it).
  auto sphase = [&](int j) {
    const bool more = j + AHEAD < T;
    if (more) issue_tile(j + AHEAD);
    const int qt0 = tile_of(j) * kBQ;
    const float* ls = reinterpret_cast<const float*>(smem + rv0 + slot_of(j) * 1024);
    const float* nds = ls + 64;
    f32x16 p, g;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const f32x4 lq = *reinterpret_cast<const f32x4*>(ls + 32 * qb + 8 * r4 + 4 * hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * r4 + e] = exp2_hw(fmaf(s[4 * r4 + e], c, lq[e]));
    }
    const bool edge = (qt0 + 32 * qb + 32 > N) || (CAUSAL && qt0 + 32 * qb < k0 + 32 * kw + 32);
    if (edge) {   // rows past N, and (causal) keys after the row
      int ln;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
      const int base = qt0 + 32 * qb + 4 * (ln >> 5);
      const int lim_n = N - base, lim_k = k0 + 32 * kw + (ln & 31) - base;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ro = 8 * (r >> 2) + (r & 3);
        p[r] = ((ro >= lim_n) || (CAUSAL && ro < lim_k)) ? 0.f : p[r];
      }
    }
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const f32x4 dq = *reinterpret_cast<const f32x4*>(nds + 32 * qb + 8 * r4 + 4 * hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) g[4 * r4 + e] = p[4 * r4 + e] * (dp[4 * r4 + e] + dq[e]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      pb[h] = pack_px<BF16>(p, h);
      gb[h] = pack_px<BF16>(g, h);
    }
    wait_for(AHEAD > 1 && more);
  };
  auto pin_s = [&] { asm volatile("" : "+v"(s), "+v"(dp)); };
  auto pin_p = [&] { asm volatile("" : "+v"(pb[0]), "+v"(pb[1]), "+v"(gb[0]), "+v"(gb[1])); };

  using BT = std::true_type;
  using BF = std::false_type;
  if (grp == 1) __syncthreads();   // phase 0: group 1 waits
  mphase(0, BF{}, BT{});
  __syncthreads();
  pin_s();
  sphase(0);
  pin_p();
  __syncthreads();
  for (int j = 1; j < T; ++j) {
    mphase(j, BT{}, BT{});
    __syncthreads();
    pin_s();
    sphase(j);
    pin_p();
    __syncthreads();
  }
  mphase(T, BT{}, BF{});   // C of the last tile
  __syncthreads();
  if (grp == 0) __syncthreads();   // phase 2T + 1: group 0 waits
  int ln;   // the lane id again (not held across the loop)
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  if (reduce_rows<TG, 2, DB>(smem, grp, wi, ln, acc)) {
    // group 0 has dV, group 1 dK
    store_transposed<D, DB>((grp == 0 ? dV : dK) + head, N, k0 + 32 * kw, ln, acc[0],
                            grp == 0 ? 1.f : scale);
  }
}

template <int D, bool CAUSAL, bool BF16, int TG>
__device__ __forceinline__ void dq_body_pp128(const f16* __restrict__ Q, const f16* __restrict__ K,
                                              const f16* __restrict__ V,
                                              const f16* __restrict__ dO,
                                              const float* __restrict__ NL,
                                              const float* __restrict__ ND, float* __restrict__ dQ,
                                              const HeadView& hv, int qblk, float c, float scale,
                                              char* smem /* dq_pp128_smem<D>() bytes */) {
  static_assert(D == 128, "a 32-row half of a tile is 8 blocks");
  constexpr int TILE = kBQ * D * 2;
  constexpr int BLOCKS = TILE / 1024;
  constexpr int OWN = BLOCKS / 2;              // blocks of a 32-row half
  constexpr int PER = TG == 2 ? OWN / 2 : OWN; // blocks per wave of a tile
  constexpr int KSTEPS = D / 16, DB = D / 32;
  constexpr int SLOT = 2 * TILE;               // K | V
  constexpr int R = TG == 2 ? 3 : 2;           // slots of a ring (TG = 4: one per group)
  static_assert(pp128_slots<TG>() * SLOT <= dq_pp128_smem<D, TG>() &&
                dq_pp128_smem<D, TG>() <= 160 * 1024, "ring inside the buffer, LDS");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = wave & 3, grp = wave >> 2;
  const int qw = TG == 2 ? wi : wi & 1;        // queries 32 qw .. +31 of the block
  const int half = TG == 2 ? grp : wi >> 1;    // key half of a tile
  const int hi = lane >> 5;
  const int q0 = qblk * block_rows<TG>();
  const int query = q0 + 32 * qw + (lane & 31);

  const int N = hv.n;
  const size_t head = hv.q;
  const int head_bytes = N * D * 2;
  const char* Kh = reinterpret_cast<const char*>(K + hv.kv);
  const char* Vh = reinterpret_cast<const char*>(V + hv.kv);

  f16x8 qf[KSTEPS], gf[KSTEPS];   // B operands: Q^T and dO^T of this wave's queries
  load_row_operand<D>(Q + head, N, q0 + 32 * qw, lane, qf);
  load_row_operand<D>(dO + head, N, q0 + 32 * qw, lane, gf);
  const bool row_ok = query < N;
  const float nl = row_ok ? NL[hv.l + query] : 0.f;
  const float dq_i = row_ok ? ND[hv.l + query] : 0.f;   // -D_i
  f32x16 acc[1][DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[0][db] = f32x16{};

  const int kv_end = CAUSAL ? min(N, q0 + block_rows<TG>()) : N;
  const int n_kt = (kv_end + kBQ - 1) / kBQ;   // >= 1
  // Steps: as in the dK/dV body.
  const int T = TG == 2 ? n_kt : (n_kt + 1) / 2;
  auto tile_of = [&](int j) { return TG == 2 ? j : 2 * j + grp; };
  // rows past N (last block only) and, causal, keys after the wave's first query
  const bool rows_edge = q0 + 32 * qw + 32 > N;

  const uint32_t lds0 = lds_addr(smem);
  const uint32_t half0 = lds0 + half * 32 * 2 * D;   // this wave's rows of a part
  auto slot_of = [&](int j) { return (TG == 2 ? 0 : grp * R) + j % R; };
  // Wave wi copies PER blocks of part wi >> 1 (K or V) of this group's half
  // (TG = 4: whole) of step j's tile.
  auto issue_tile = [&](int j) {
    int ln;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
    const uint32_t base = lds0 + slot_of(j) * SLOT + (wi >> 1) * TILE;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int b = (TG == 2 ? OWN * grp : 0) + PER * (wi & 1) + i;
      copy_block<D>(wi < 2 ? Kh : Vh, head_bytes, tile_of(j), base + b * 1024, block_offset<D>(b, ln));
    }
  };
  auto wait_for = [&](bool last) {   // all copies but those of the last tile issued
    if (last) wait_vmcnt<PER>();
    else wait_vmem();
  };
  constexpr int AHEAD = R - 1;   // S(j) starts the copies of tile j + AHEAD
  issue_tile(0);
  if (AHEAD > 1 && T > 1) issue_tile(1);
  wait_for(AHEAD > 1 && T > 1);
  __syncthreads();

  f32x16 s = {}, dp = {};
  f16x8 gb[2];
  // M phase of tile j: C of tile j - 1 (dQ^T += K^T dS^T; step x: k-step
  // x / DB, d-block x % DB), then A of tile j (S^T = K Q^T, dP^T = V dO^T).
  auto mphase = [&](int j, auto with_c, auto with_a) {
    constexpr bool WC = decltype(with_c)::value, WA = decltype(with_a)::value;
    constexpr int CX = 2 * DB;   // C steps
    constexpr int X0 = WC ? 0 : CX, X1 = WA ? CX + KSTEPS : CX;
    const uint32_t sc = col_base<D>(half0 + slot_of(j + R - 1) * SLOT, lane);   // tile j - 1
    const uint32_t sa = row_base<D>(half0 + slot_of(j) * SLOT, lane);           // tile j
    f16x8 f[CX + KSTEPS][2];
    auto load = [&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (x < CX) {
        f[x][0] = load_col_frag<D>(sc, 0, x / DB, x % DB);   // K^T
      } else {
        f[x][0] = load_row_frag<D>(sa, 0, x - CX);      // K rows
        f[x][1] = load_row_frag<D>(sa, TILE, x - CX);   // V rows
      }
    };
    static_for<X0, X0 + 2 < X1 ? X0 + 2 : X1>(load);
    static_for<X0, X1>([&](auto xi) {
      constexpr int x = decltype(xi)::value;
      if constexpr (x + 2 < X1) load(std::integral_constant<int, x + 2>{});
      if constexpr (x < CX) {
        acc[0][x % DB] = mma32<BF16>(f[x][0], gb[x / DB], acc[0][x % DB]);
      } else {
        constexpr int kk = x - CX;
        s = mma32<BF16>(f[x][0], qf[kk], kk == 0 ? f32x16{} : s);
        dp = mma32<BF16>(f[x][1], gf[kk], kk == 0 ? f32x16{} : dp);
      }
      if constexpr (x + 1 == CX) __builtin_amdgcn_sched_barrier(0);   // C before A
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto sphase = [&](int j) {
    const bool more = j + AHEAD < T;
    if (more) issue_tile(j + AHEAD);
    const int kt0 = tile_of(j) * kBQ;
    f32x16 p;
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = exp2_hw(fmaf(s[r], c, nl));
    const bool edge = rows_edge || (kt0 + 32 * half + 32 > N) ||
                      (CAUSAL && kt0 + 32 * half + 31 > q0 + 32 * qw);
    if (edge) {   // keys past N, rows past N, and (causal) keys after the row
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kidx = kt0 + 32 * half + 8 * (r >> 2) + 4 * hi + (r & 3);
        p[r] = ((kidx >= N) || (CAUSAL && kidx > query) || !row_ok) ? 0.f : p[r];
      }
    }
    f32x16 g;
#pragma unroll
    for (int r = 0; r < 16; ++r) g[r] = p[r] * (dp[r] + dq_i);
#pragma unroll
    for (int h = 0; h < 2; ++h) gb[h] = pack_px<BF16>(g, h);
    wait_for(AHEAD > 1 && more);
  };
  auto pin_s = [&] { asm volatile("" : "+v"(s), "+v"(dp)); };
  auto pin_p = [&] { asm volatile("" : "+v"(gb[0]), "+v"(gb[1])); };

  using BT = std::true_type;
  using BF = std::false_type;
  if (grp == 1) __syncthreads();   // phase 0: group 1 waits
  mphase(0, BF{}, BT{});
  __syncthreads();
  pin_s();
  sphase(0);
  pin_p();
  __syncthreads();
  for (int j = 1; j < T; ++j) {
    mphase(j, BT{}, BT{});
    __syncthreads();
    pin_s();
    sphase(j);
    pin_p();
    __syncthreads();
  }
  mphase(T, BT{}, BF{});   // C of the last tile
  __syncthreads();
  if (grp == 0) __syncthreads();   // phase 2T + 1: group 0 waits
  if (reduce_rows<TG, 1, DB>(smem, grp, wi, lane, acc)) {
    // group 1 has the upper half of the columns
    store_transposed<D, DB / 2>(dQ + head + grp * (D / 2), N, q0 + 32 * qw, lane, acc[0], scale);
  }
}

// dK/dV and dQ in one launch (both bodies take 8 waves and share one LDS
// buffer): the first half of the blocks runs the dK/dV body of a key block,
// the second half the dQ body of a query block, each half longest unit first
// (unit_of). A CU that finished a short dK/dV unit (late keys of a causal
// head) picks up a long dQ unit, and the short dQ units fill the end. The
// halves are not interleaved: a dK/dV unit takes 4/3 of a dQ unit's time, and
// where each CU gets one of both, two dK/dV units on one CU are the longest
// (B1 H8 N4096 D64 non-causal 136 us, interleaved 150).
template <int D, bool CAUSAL, bool BF16, int TG>
__global__ void __launch_bounds__(512)
fa_bwd_fused_kernel(const f16* __restrict__ Q, const f16* __restrict__ K,
                    const f16* __restrict__ V, const f16* __restrict__ dO,
                    const float* __restrict__ NL, const float* __restrict__ ND,
                    float* __restrict__ dK, float* __restrict__ dV, float* __restrict__ dQ,
                    Geom geo, UnitMap um, float c, float scale) {
  // One LDS buffer serves whichever body this workgroup runs.
  constexpr int SK = D == 64 ? dkdv_pp_smem<D, TG>() : dkdv_pp128_smem<D, TG>();
  constexpr int SQ = D == 64 ? dq_pp_smem<D, TG>() : dq_pp128_smem<D, TG>();
  constexpr int ROWS = block_rows<TG>();
  __shared__ __attribute__((aligned(1024))) char smem[SK > SQ ? SK : SQ];
  const int total = um.heads * um.per_head;
  const bool dq_role = (int)blockIdx.x >= total;
  const Unit un = unit_of(dq_role ? blockIdx.x - total : blockIdx.x, um);
  HeadView hv;
  int kb = un.idx;
  if (geo.cu != nullptr) {
    const SeqBlock sb = varlen_block(geo, un.idx, ROWS, threadIdx.x & 63);
    if (sb.n == 0) return;   // the grid is a bound on the units (whole workgroup)
    hv = seq_view<D>(geo, un.head, sb.start, sb.n);
    kb = sb.block;
  } else {
    hv = dense_view<D>(geo, un.head);
  }
  // Causal: the first key blocks and the last query blocks are the longest.
  const int qblk = CAUSAL ? (hv.n + ROWS - 1) / ROWS - 1 - kb : kb;
  if (!dq_role) {
    if constexpr (D == 64) {
      dkdv_body_pp<D, CAUSAL, BF16, TG>(Q, K, V, dO, NL, ND, dK, dV, hv, kb, c, scale, smem);
    } else {
      dkdv_body_pp128<D, CAUSAL, BF16, TG>(Q, K, V, dO, NL, ND, dK, dV, hv, kb, c, scale, smem);
    }
  } else {
    if constexpr (D == 64) {
      dq_body_pp<D, CAUSAL, BF16, TG>(Q, K, V, dO, NL, ND, dQ, hv, qblk, c, scale, smem);
    } else {
      dq_body_pp128<D, CAUSAL, BF16, TG>(Q, K, V, dO, NL, ND, dQ, hv, qblk, c, scale, smem);
    }
  }
}

// GQA: dK (blockIdx.y 0) and dV (1) of KV head hk = sum over its `group` query
// heads of the per-query-head partials (fp32 [B*H, N*D] -> [B*Hkv, N*D]), four
// floats per thread.
__global__ void __launch_bounds__(256)
fa_bwd_group_sum_kernel(const float* __restrict__ part_k, const float* __restrict__ part_v,
                        float* __restrict__ dk, float* __restrict__ dv, int64_t head_elems,
                        int64_t kv_heads, int group) {
  const float* part = blockIdx.y == 0 ? part_k : part_v;
  float* out = blockIdx.y == 0 ? dk : dv;
  const int64_t i4 = (int64_t)blockIdx.x * 256 + threadIdx.x;   // float4 index in out
  const int64_t n4 = kv_heads * head_elems / 4;
  if (i4 >= n4) return;
  const int64_t hk = (i4 * 4) / head_elems;
  const int64_t e = i4 * 4 - hk * head_elems;
  const f32x4* src = reinterpret_cast<const f32x4*>(part + (hk * group) * head_elems + e);
  const int64_t stride4 = head_elems / 4;
  f32x4 acc = src[0];
  for (int j = 1; j < group; ++j) acc += src[j * stride4];
  reinterpret_cast<f32x4*>(out)[i4] = acc;
}

// Inputs of a backward that come in fp32: O and dO (null: 16-bit), and the
// conversions of Q, K and V.
struct Fp32Inputs {
  const float* o;
  const float* g;
  CastJobs qkv;
};

// The three passes (-D_i and -L log2 e, dK/dV, dQ) and, with H_kv < H, the
// group sums. geo is dense (B heads of N rows per head) or varlen (heads of
// geo.total packed rows); `rows` is the number of L rows: B*H*N dense, H*total
// varlen.
template <int D, bool CAUSAL, bool BF16>
static hipError_t launch_bwd(const void* q, const void* k, const void* v, const void* o,
                             const void* dout, const Fp32Inputs& in, const float* lse, float* dq, float* dk, float* dv,
                             float* ws, const Geom& geo, const UnitMap& um, bool rows4, int64_t rows,
                             int64_t out_heads, int64_t head_rows, hipStream_t s) {
  const float scale = (float)(1.0 / sqrt((double)D));
  const float c = scale * kLog2e;
  const f16* Q = (const f16*)q;
  const f16* K = (const f16*)k;
  const f16* V = (const f16*)v;
  const f16* G = (const f16*)dout;
  const int group = (int)geo.group.d;
  float* nd = ws;
  float* nl = ws + rows;
  // GQA: per-query-head dK/dV partials in the workspace, summed per KV head.
  const int64_t part0 = (2 * rows + 3) / 4 * 4;   // 16-byte aligned start of the partials
  float* dk_q = group == 1 ? dk : ws + part0;
  float* dv_q = group == 1 ? dv : ws + part0 + rows * D;
  const RowTermArgs rt{(const f16*)o, (f16*)const_cast<void*>(dout), in.o, in.g, lse, nd, nl, rows,
                       (int)((rows + 31) / 32)};
  hipLaunchKernelGGL((fa_bwd_di_kernel<D, BF16>),
                     dim3((unsigned)(rt.blocks + in.qkv.blocks[0] + in.qkv.blocks[1] + in.qkv.blocks[2])),
                     dim3(256), 0, s, rt, in.qkv);
  // dK/dV and dQ in one launch: with units of one length it measured level
  // with two launches or slightly ahead (D = 128 non-causal, B1 H8 N4096
  // 256.4 -> 254.5 us, B4 H16 N4096 1981.8 -> 1972.3 us; same gradients bit
  // for bit), and a causal head's short and long units even out.
  const dim3 grid(2u * um.heads * um.per_head);
  if (rows4) {
    hipLaunchKernelGGL((fa_bwd_fused_kernel<D, CAUSAL, BF16, 4>), grid, dim3(512), 0, s, Q, K, V, G,
                       nl, nd, dk_q, dv_q, dq, geo, um, c, scale);
  } else {
    hipLaunchKernelGGL((fa_bwd_fused_kernel<D, CAUSAL, BF16, 2>), grid, dim3(512), 0, s, Q, K, V, G,
                       nl, nd, dk_q, dv_q, dq, geo, um, c, scale);
  }
  if (group > 1) {
    // out_heads KV heads of head_rows rows, each the sum of `group`
    // consecutive query heads' partials
    const int64_t head_elems = head_rows * D;
    const int64_t n4 = out_heads * head_elems / 4;
    const dim3 grid((unsigned)((n4 + 255) / 256), 2);
    hipLaunchKernelGGL(fa_bwd_group_sum_kernel, grid, dim3(256), 0, s, dk_q, dv_q, dk, dv,
                       head_elems, out_heads, group);
  }
  return hipGetLastError();
}

}  // namespace bwd
}  // namespace fa

extern "C" int64_t fa_bwd_workspace_floats(int64_t B, int64_t H, int64_t N) {
  if (B <= 0 || H <= 0 || N <= 0) return 0;
  return 2 * B * H * N;   // -D_i, then -L log2(e)
}

extern "C" int64_t fa_bwd_gqa_workspace_floats(int64_t B, int64_t H, int64_t H_kv, int64_t N,
                                               int64_t D) {
  if (B <= 0 || H <= 0 || N <= 0 || H_kv <= 0 || H % H_kv != 0) return 0;
  // -D_i and -L log2(e), then (GQA only, from a 16-byte boundary) the
  // per-query-head dK and dV partials
  if (H_kv == H) return 2 * B * H * N;
  return (2 * B * H * N + 3) / 4 * 4 + 2 * B * H * N * D;
}

namespace fa {
namespace bwd {
// Whether workgroups own 64 rows instead of 128, where `blocks` is the number
// of 128-row blocks (each has a dK/dV and a dQ workgroup): where those fill
// half of the CUs at most, or, causal and of long rows, all of them once (the
// longest block then sets the time). us, 128 -> 64 rows: D = 64 B1 H8 N1024
// 24.8 -> 18.4, B1 H4 N2048 39.0 -> 28.2, causal B1 H8 N2048 40.3 -> 32.7, B1
// H4 N4000 86.2 -> 49.9; D = 128 37.6 -> 29.3, 60.1 -> 44.6, 63.4 -> 50.8, 112.2
// -> 81.3. Beyond: B1 H8 N1500 D = 64 (192 workgroups) 37.0 vs 39.2, causal B2
// H16 N512 (256) 19.3 vs 20.7, B1 H8 N4096 132.9 vs 144.6, causal 84.5 vs 89.1.
static bool narrow_blocks(int64_t blocks, int64_t N, int causal, int cus) {
  const int64_t wide = 2 * blocks;
  return 2 * wide <= cus || (causal && wide <= cus && N >= 1024);
}

template <bool BF16>
static int bwd_run(const void* q, const void* k, const void* v, const void* o, const void* dout,
                   const Fp32Inputs& in, const float* lse, float* dq, float* dk, float* dv, float* workspace,
                   const Geom& geo, int64_t units, int64_t rows, int64_t out_heads,
                   int64_t head_rows, int64_t D, int causal, void* stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const Topology topo = stream_topology(s);
  // Units of a head: its blocks (varlen: a bound on those of its sequences).
  const int64_t heads = geo.cu == nullptr ? units : geo.H;
  auto blocks_of = [&](int br) {
    return geo.cu == nullptr ? (int64_t)(geo.N + br - 1) / br
                             : varlen_units(geo.B, geo.total, geo.N, br);
  };
  const bool rows4 = narrow_blocks(heads * blocks_of(block_rows<2>()), geo.N, causal, topo.cus);
  const int64_t per_head = blocks_of(rows4 ? block_rows<4>() : block_rows<2>());
  if (2 * heads * per_head > (int64_t(1) << 31) - 1) return FA_ERR_TOO_LARGE;
  const UnitMap um = unit_map(heads, per_head, topo, causal != 0 || geo.cu != nullptr);
  hipError_t e;
  if (D == 64) {
    e = causal ? launch_bwd<64, true, BF16>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, um, rows4, rows, out_heads, head_rows, s)
               : launch_bwd<64, false, BF16>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, um, rows4, rows, out_heads, head_rows, s);
  } else {
    e = causal ? launch_bwd<128, true, BF16>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, um, rows4, rows, out_heads, head_rows, s)
               : launch_bwd<128, false, BF16>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, um, rows4, rows, out_heads, head_rows, s);
  }
  return e == hipSuccess ? FA_OK : -(int)e;
}

static int bwd_gqa(bool bf16, const void* q, const void* k, const void* v, const void* o,
                   const void* dout, const float* lse, float* dq, float* dk, float* dv,
                   float* workspace, int64_t B, int64_t H, int64_t H_kv, int64_t N, int64_t D,
                   int causal, void* stream, const Fp32Inputs& in = Fp32Inputs{}) {
  int st = fa_validate_bwd(q, k, v, o, dout, lse, dq, dk, dv, workspace, B, H, N, D);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H % H_kv != 0) return FA_ERR_KV_HEADS;
  // the partials are written and read as 16-byte vectors
  if (H_kv != H && (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0) return FA_ERR_ALIGNMENT;
  const Geom geo{nullptr, (int)N, (int)H, FastDiv(H / H_kv), 0, 0};
  return bf16 ? bwd_run<true>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, B * H,
                              B * H * N, B * H_kv, N, D, causal, stream)
              : bwd_run<false>(q, k, v, o, dout, in, lse, dq, dk, dv, workspace, geo, B * H,
                               B * H * N, B * H_kv, N, D, causal, stream);
}
}  // namespace bwd
}  // namespace fa

extern "C" int fa_probe_bwd_block_rows(int causal, int64_t bh, int64_t N, int cus) {
  using namespace fa::bwd;
  if (bh <= 0 || N <= 0 || cus <= 0) return 0;
  return narrow_blocks(bh * ((N + block_rows<2>() - 1) / block_rows<2>()), N, causal, cus)
             ? block_rows<4>() : block_rows<2>();
}

extern "C" int fa_bwd_f16(const void* q, const void* k, const void* v, const void* o,
                          const void* dout, const float* lse, float* dq, float* dk, float* dv,
                          float* workspace, int64_t B, int64_t H, int64_t N, int64_t D, int causal,
                          void* stream) {
  return fa::bwd::bwd_gqa(false, q, k, v, o, dout, lse, dq, dk, dv, workspace, B, H, H, N, D,
                          causal, stream);
}

extern "C" int fa_bwd_gqa_f16(const void* q, const void* k, const void* v, const void* o,
                              const void* dout, const float* lse, float* dq, float* dk, float* dv,
                              float* workspace, int64_t B, int64_t H, int64_t H_kv, int64_t N,
                              int64_t D, int causal, void* stream) {
  return fa::bwd::bwd_gqa(false, q, k, v, o, dout, lse, dq, dk, dv, workspace, B, H, H_kv, N, D,
                          causal, stream);
}

extern "C" int fa_bwd_bf16(const void* q, const void* k, const void* v, const void* o,
                           const void* dout, const float* lse, float* dq, float* dk, float* dv,
                           float* workspace, int64_t B, int64_t H, int64_t H_kv, int64_t N,
                           int64_t D, int causal, void* stream) {
  return fa::bwd::bwd_gqa(true, q, k, v, o, dout, lse, dq, dk, dv, workspace, B, H, H_kv, N, D,
                          causal, stream);
}

extern "C" int fa_bwd_cast_f32(const float* const f32[5], void* const h16[5], const float* lse,
                               float* dq, float* dk, float* dv, float* workspace, int64_t B,
                               int64_t H, int64_t H_kv, int64_t N, int64_t D, int causal, int bf16,
                               void* stream) {
  using namespace fa;
  if (!f32 || !h16) return FA_ERR_NULL_POINTER;
  // O needs no 16-bit copy: the row terms are its only use.
  const void* o = h16[3] != nullptr ? h16[3] : (const void*)f32[3];
  int st = fa_validate_bwd(h16[0], h16[1], h16[2], o, h16[4], lse, dq, dk, dv, workspace, B, H, N, D);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H % H_kv != 0) return FA_ERR_KV_HEADS;
  for (int i = 0; i < 5; ++i)
    if ((reinterpret_cast<uintptr_t>(f32[i]) & 15u) != 0) return FA_ERR_ALIGNMENT;
  const int64_t nq = B * H * N * D, nkv = B * H_kv * N * D;
  if (nq / 8 / kCastVecs + 2 * (nkv / 8 / kCastVecs) + B * H * N / 32 > (int64_t(1) << 31) - 8)
    return FA_ERR_TOO_LARGE;
  const int64_t n[3] = {nq, nkv, nkv};
  const bwd::Fp32Inputs in{f32[3], f32[4], cast_jobs(f32, h16, n)};
  return bwd::bwd_gqa(bf16 != 0, h16[0], h16[1], h16[2], o, h16[4], lse, dq, dk, dv, workspace, B,
                      H, H_kv, N, D, causal, stream, in);
}

extern "C" int fa_bwd_varlen_f16(const void* q, const void* k, const void* v, const void* o,
                                 const void* dout, const float* lse, float* dq, float* dk,
                                 float* dv, float* workspace, const int32_t* cu_seqlens,
                                 int64_t B, int64_t H, int64_t H_kv, int64_t max_seqlen,
                                 int64_t total, int64_t D, int causal, void* stream) {
  const int st = fa_validate_bwd_varlen(q, k, v, o, dout, lse, dq, dk, dv, workspace, cu_seqlens,
                                        B, H, H_kv, max_seqlen, total, D);
  if (st != FA_OK) return st;
  if (total == 0) return FA_OK;
  if (H_kv != H && (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0) return FA_ERR_ALIGNMENT;
  const fa::Geom geo{cu_seqlens, (int)max_seqlen, (int)H, fa::FastDiv(H / H_kv), (int)total,
                     (int)B};
  return fa::bwd::bwd_run<false>(q, k, v, o, dout, fa::bwd::Fp32Inputs{}, lse, dq, dk, dv, workspace, geo, B * H,
                                 H * total, H_kv, total, D, causal, stream);
}
