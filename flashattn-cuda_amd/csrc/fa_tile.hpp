// fa_tile.hpp — gfx950 building blocks shared by the forward kernel and the
// layout probes: MFMA wrappers, LDS tile layouts, operand loaders, P packing.
//
// Matrix-core conventions (v_mfma_f32_32x32x16_f16, one wave64):
//   A (32 x 16): lane l holds A[l % 32][8*(l/32) + i], i = 0..7
//   B (16 x 32): lane l holds B[8*(l/32) + i][l % 32], i = 0..7
//   C (32 x 32): lane l, register r holds C[8*(r/4) + 4*(l/32) + r%4][l % 32]
// The layout probes in fa_probe.hip check these on the device.
//
// The forward kernel computes S^T = K Q^T (A = K tile from LDS, B = Q held in
// registers), so lane l owns query l%32 and 16 of the 32 keys of a block; row
// statistics are in-lane plus one exchange with lane l^32. It then computes
// O^T = V^T P^T with P^T taken straight from the S^T accumulator (no LDS round
// trip): the PV reduction index is the key, so keys may be visited in any
// order as long as V^T and P^T agree. The order used is the S^T register order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

namespace fa {

typedef _Float16 f16;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Operand registers hold raw 16-bit values; BF16 selects how they are read.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <bool BF16>
__device__ __forceinline__ f32x16 mma32(f16x8 a, f16x8 b, f32x16 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return mfma32(a, b, c);
  }
}

// 2^x on the hardware transcendental unit (v_exp_f32); 2^-inf = 0.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
// log2(x) on v_log_f32.
__device__ __forceinline__ float log2_hw(float x) { return __builtin_amdgcn_logf(x); }

// v_permlane32_swap_b32 with both operands x: element 0 of the result holds,
// in lanes 32..63, x of lane l-32 (lanes 0..31 keep x); element 1 holds, in
// lanes 0..31, x of lane l+32 (lanes 32..63 keep x). So {r0, r1} is
// {x[l], x[l^32]} in some order in every lane.
__device__ __forceinline__ float max_xor32(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float sum_xor32(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Raw buffer resource over `bytes` bytes at `base`: loads at offsets beyond
// `bytes` return zero instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}

// make_rsrc for a wave-uniform range that must sit in SGPRs (the inline
// asm of the LDS copies below takes the descriptor as an SGPR operand): the
// base and length go through readfirstlane, which is free when the compiler
// already holds them in SGPRs.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc_s(const void* base, int bytes) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const void* p = reinterpret_cast<const void*>(((uintptr_t)hi << 32) | lo);
  return make_rsrc(p, __builtin_amdgcn_readfirstlane(bytes));
}

// LDS byte address of a pointer into a __shared__ array.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// 16 bytes per lane from global (rsrc + voffset) straight into LDS at byte
// lds + 16*lane (lds is wave-uniform). Written as inline assembly so the
// compiler does not treat it as an LDS store: it would otherwise wait for
// every DMA in flight before any LDS read it cannot prove disjoint. The
// kernels order these copies themselves (s_waitcnt vmcnt(0) + barrier before
// the data is read), and nothing else in them uses M0.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voffset) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voffset), "s"(r)
               : "memory", "m0");
}

// 4 bytes per lane from global (rsrc + voffset) into LDS at byte lds + 4*lane;
// the dword form needs only 4-byte alignment of the source.
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voffset) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voffset), "s"(r)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt vmcnt(0) through the builtin, so the compiler also knows that its
// own vector-memory loads issued before this point have completed (gfx9
// encoding: vmcnt bits [3:0] and [15:14] = 0, expcnt 7, lgkmcnt 15).
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// f(integral_constant<int, I>) for I = B .. E-1, expanded at compile time
// (a fixed instruction schedule must not depend on the loop unroller).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// s_waitcnt vmcnt(N) (gfx9 encoding: vmcnt[3:0] at bits 3:0, vmcnt[5:4] at
// bits 15:14, expcnt and lgkmcnt left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// ---------------------------------------------------------------------------
// LDS tile layouts. A tile is rows (keys or queries) x D fp16, row stride 2*D
// bytes, stored as 16-byte chunks (8 halves). Chunk c of row r lives at chunk
// slot pos(r, c) of that row; pos is an XOR swizzle chosen so that the
// operand reads below hit distinct LDS banks within each 16-lane group. k_swz
// is that of the forward's K tiles (row reads only; its V tiles are blocks,
// beside its kernel), t_swz below that of the backward's.
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  if constexpr (D == 64) {
    return (r >> 1) & 7;
  } else {
    return r & 15;
  }
}

// XOR swizzles are involutions: slot = c ^ swz(r) and c = slot ^ swz(r).
template <int D>
__device__ __forceinline__ int k_slot(int r, int c) { return c ^ k_swz<D>(r); }

template <int D>
__device__ __forceinline__ int k_off(int r, int c) { return r * (2 * D) + k_slot<D>(r, c) * 16; }

// LDS pointers for the pipelined kernel's operand reads: arithmetic on them
// stays in the 32-bit LDS address space, so constant offsets fold into the
// DS instructions' offset field.
typedef const __attribute__((address_space(3))) char* lds_cp;

// A lane's base address in LDS, opaque to the optimiser: every read of the
// step is then this base plus a constant, instead of a separately hoisted
// loop-invariant offset plus the step's slot base per read.
__device__ __forceinline__ lds_cp lds_lane_base(uint32_t a) {
  asm("" : "+v"(a));
  return (lds_cp)(size_t)a;
}

__device__ __forceinline__ f16x8 lds_b128(lds_cp p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) f16x8*>(p);
}

// ds_read_b64_tr_b16: within each group of 16 lanes, lane s supplies the
// address of 4 consecutive halves M[s][0..3]; it receives
// out[e] = M[4*e + s/4][s%4]. If lane s points at row (k0 + s/4),
// columns (d0 + 4*(s%4)) .. +3 of a row-major [key][d] tile, lane s receives
// the column d0 + s for keys k0 .. k0+3.
__device__ __forceinline__ f16x4 lds_tr16(lds_cp p) {
  typedef __attribute__((address_space(3))) fp16x4_t lds_fp16x4;
  fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_fp16x4*)(p));
  return __builtin_bit_cast(f16x4, v);
}

// A operand of S^T = K Q^T for key block kb (32 keys) and k-step kk (16 of D).
// The K swizzle depends on the row only modulo 16, so block kb is the block-0
// fragment shifted by 32 rows: k_frag_off(kk, lane) + 32 * kb * 2D.
template <int D>
__device__ __forceinline__ int k_frag_off(int kk, int lane) {
  return k_off<D>(lane & 31, 2 * kk + (lane >> 5));
}

template <int D>
__device__ __forceinline__ f16x8 load_k_frag(const char* ks, int kb, int kk, int lane) {
  return *reinterpret_cast<const f16x8*>(ks + 32 * kb * 2 * D + k_frag_off<D>(kk, lane));
}

// One layout for both reads (the backward's tiles, read as rows and
// transposed): chunk c of row r at slot c ^ t_swz(r). Row reads (b128: 16
// lanes take one chunk of 16 consecutive rows, 256 bytes = every bank once)
// need t_swz one to one over 16 rows at D = 128, over 8 row pairs at D = 64.
// Transposed reads (32 lanes take 64 bytes of 4 consecutive rows) need its
// top bits (64-byte column blocks) to differ between rows of the same bank
// half: over r % 4 at D = 128, over (r / 2) % 2 at D = 64. Putting the row's
// low bits on top gives both, so a tile is copied and kept once.
template <int D>
__device__ __forceinline__ int t_swz(int r) {
  if constexpr (D == 64) {
    return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
  } else {
    return ((r & 3) << 2) | ((r >> 2) & 3);
  }
}

// Byte address of a lane's first row read (rows 0 .. 31, k-step 0) and first
// transposed read (rows 0 .. 15, column block 0) of a tile at LDS address
// `tile` (1 KiB aligned). The other reads flip bits of it or add constants, so
// a phase needs one base of each kind; opaque, or the compiler keeps a
// loop-invariant offset for every flip (21 spilled registers in the D = 128
// backward).
template <int D>
__device__ __forceinline__ uint32_t row_base(uint32_t tile, int lane) {
  const int r = lane & 31;
  uint32_t a = tile + r * 2 * D + ((lane >> 5) ^ t_swz<D>(r)) * 16;
  asm("" : "+v"(a));
  return a;
}

template <int D>
__device__ __forceinline__ uint32_t col_base(uint32_t tile, int lane) {
  const int s = lane & 15;
  const int r = 4 * (lane >> 5) + (s >> 2);
  const int c = 2 * ((lane >> 4) & 1) + ((s & 3) >> 1);
  uint32_t a = tile + r * 2 * D + (c ^ t_swz<D>(r)) * 16 + 8 * (s & 1);
  asm("" : "+v"(a));
  return a;
}

// Rows 0 .. 31 of the tile as an A operand (k-step kk of D), `off` bytes on
// (a constant): as load_k_frag.
template <int D>
__device__ __forceinline__ f16x8 load_row_frag(uint32_t base, int off, int kk) {
  return lds_b128((lds_cp)(size_t)(base ^ (32 * kk)) + off);
}

// Columns 32 db .. + 31 of rows 16 j .. + 15 as an A operand (transposed),
// `off` bytes on: slot i of lane l holds column 32 db + l % 32 of row
// 16 j + 8 (i / 4) + 4 (l / 32) + i % 4, the row order of the score
// accumulators (see pack_p). Eight rows up, t_swz differs in its bit 1, address
// bit 5.
template <int D>
__device__ __forceinline__ f16x8 load_col_frag(uint32_t base, int off, int j, int db) {
  const f16x4 lo = lds_tr16((lds_cp)(size_t)(base ^ (64 * db)) + off + 16 * j * 2 * D);
  const f16x4 up = lds_tr16((lds_cp)(size_t)(base ^ (64 * db + 32)) + off + (16 * j + 8) * 2 * D);
  return f16x8{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
}

// Key index (within a 64-key tile) held by register r of key block kb in lane l.
__device__ __forceinline__ int st_key(int kb, int r, int lane) {
  return 32 * kb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}

// fp32 -> fp16 round-to-nearest-even, two at a time (v_cvt_pk_f16_f32).
__device__ __forceinline__ f16x2 cvt2(float a, float b) {
  return f16x2{(f16)a, (f16)b};
}

// fp32 -> 16-bit operand pair: fp16 (v_cvt_pk_f16_f32) or, with BF16,
// bfloat16 round-to-nearest-even (v_cvt_pk_bf16_f32), as raw bits.
template <bool BF16>
__device__ __forceinline__ f16x2 cvt2x(float a, float b) {
  if constexpr (BF16) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(f16x2, __builtin_convertvector(f32x2_t{a, b}, bf16x2));
  } else {
    return cvt2(a, b);
  }
}

// Eight fp32 values as 16-bit operands (round to nearest even), raw bits.
template <bool BF16>
__device__ __forceinline__ f16x8 cvt8x(const float* __restrict__ src) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
  const f16x2 x0 = cvt2x<BF16>(a[0], a[1]), x1 = cvt2x<BF16>(a[2], a[3]);
  const f16x2 x2 = cvt2x<BF16>(b[0], b[1]), x3 = cvt2x<BF16>(b[2], b[3]);
  return f16x8{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
}

// Up to three fp32 tensors to convert in one launch, `vecs` groups of eight
// values each (16-byte aligned on both sides) and `tail` values more. Workgroups
// of 256 threads take kCastVecs groups: first src[0]'s, then src[1]'s, then
// src[2]'s.
constexpr int kCastVecs = 512;
struct CastJobs {
  const float* src[3];
  f16* dst[3];
  int64_t vecs[3];
  int tail[3];
  int blocks[3];   // of each
};

inline CastJobs cast_jobs(const float* const src[3], void* const dst[3], const int64_t n[3]) {
  CastJobs j;
  for (int i = 0; i < 3; ++i) {
    j.src[i] = src[i];
    j.dst[i] = (f16*)dst[i];
    j.vecs[i] = src[i] != nullptr ? n[i] / 8 : 0;
    j.tail[i] = src[i] != nullptr ? (int)(n[i] % 8) : 0;
    j.blocks[i] = (int)((j.vecs[i] + (j.tail[i] > 0) + kCastVecs - 1) / kCastVecs);
  }
  return j;
}

template <bool BF16>
__device__ __forceinline__ void cast_block(const CastJobs& j, int block) {
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    if (block >= 0 && block < j.blocks[t]) {
#pragma unroll
      for (int i = 0; i < kCastVecs / 256; ++i) {
        const int64_t v = (int64_t)block * kCastVecs + 256 * i + threadIdx.x;
        if (v < j.vecs[t]) reinterpret_cast<f16x8*>(j.dst[t])[v] = cvt8x<BF16>(j.src[t] + 8 * v);
        if (v == j.vecs[t])
          for (int e = 0; e < j.tail[t]; ++e)
            j.dst[t][8 * v + e] = cvt2x<BF16>(j.src[t][8 * v + e], 0.f)[0];
      }
    }
    block -= j.blocks[t];
  }
}

// B operand (P^T) of PV k-step j from the S^T accumulators p[2] of a tile.
__device__ __forceinline__ f16x8 pack_p(const f32x16& p, int half_sel) {
  const int b = 8 * half_sel;
  f16x2 x0 = cvt2(p[b + 0], p[b + 1]);
  f16x2 x1 = cvt2(p[b + 2], p[b + 3]);
  f16x2 x2 = cvt2(p[b + 4], p[b + 5]);
  f16x2 x3 = cvt2(p[b + 6], p[b + 7]);
  return f16x8{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
}

// pack_p with the operand format chosen by BF16 (bfloat16 bits in the same
// register layout).
template <bool BF16>
__device__ __forceinline__ f16x8 pack_px(const f32x16& p, int half_sel) {
  const int b = 8 * half_sel;
  f16x2 x0 = cvt2x<BF16>(p[b + 0], p[b + 1]);
  f16x2 x1 = cvt2x<BF16>(p[b + 2], p[b + 3]);
  f16x2 x2 = cvt2x<BF16>(p[b + 4], p[b + 5]);
  f16x2 x3 = cvt2x<BF16>(p[b + 6], p[b + 7]);
  return f16x8{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
}

// Division of 0 <= n < 2^31 by a launch constant d >= 1: n * ceil(2^(31+s) / d)
// >> (31+s) with 2^s >= d (the rounding adds less than 2^s to the numerator's
// 2^(31+s), so the quotient is exact). A few scalar instructions where a
// division by a kernel argument takes about forty vector ones; a workgroup's
// address waits for several (B1 H8 N1024 D64: 8.20 -> 8.54 us with plain
// divisions in unit_of).
struct FastDiv {
  uint32_t d, mul, shift;
  FastDiv() = default;
  explicit FastDiv(int64_t divisor) : d((uint32_t)divisor), shift(31) {
    while ((uint64_t(1) << (shift - 31)) < d) ++shift;
    mul = (uint32_t)(((uint64_t(1) << shift) + d - 1) / d);
  }
  __host__ __device__ __forceinline__ int div(int n) const {
    return (int)(((uint64_t)(uint32_t)n * mul) >> shift);
  }
};

// Where the heads of one launch live. Dense: Q/O [B, H, N, D], K/V
// [B, H/group, N, D], L [B, H, N]. Varlen (cu != nullptr): sequences packed
// head-major, Q/O [H, total, D], K/V [H/group, total, D], L [H, total];
// sequence b is rows cu[b] .. cu[b+1] of every head and N is the grid's
// maximum length. Query head h reads KV head h / group (GQA / MQA).
struct Geom {
  const int32_t* cu;
  int N;
  int H;
  FastDiv group;
  int total;
  int B;       // varlen: number of sequences
};

// Workgroup g of a 1-D grid of `total` lands on XCD g % nxcd (the dispatcher
// deals consecutive workgroups to the XCDs in turn). Map it to a logical index
// so that each XCD gets one contiguous range of logical indices: the units of
// a row block then share one XCD's L2, which serves their K/V after the first
// fetch. nxcd <= 1 (one XCD, or a partition of one) is the identity.
__device__ __forceinline__ int xcd_remap(int g, int total, int nxcd) {
  if (nxcd <= 1) return g;
  const int q = total / nxcd, r = total % nxcd;
  const int xcd = g % nxcd, slot = g / nxcd;
  return (xcd < r) ? xcd * (q + 1) + slot : r * (q + 1) + (xcd - r) * q + slot;
}

// The units of a launch: `heads` heads of `per_head` units, unit 0 of a head
// the longest where lengths differ. One workgroup per unit. See unit_of and,
// for the fields, unit_map.
struct UnitMap {
  int heads, per_head;
  FastDiv nxcd;
  int whole;             // whole heads of an XCD
  FastDiv rem;           // heads that do not divide over the XCDs (at least 1)
  int dealt;             // their units
  FastDiv set_units;     // units of a set of heads an XCD works on at a time
  FastDiv width, last;   // heads of a set, and of the last one
  int sets;
};

struct Unit {
  int head, idx;
};

// The unit of workgroup g. Workgroup g runs on XCD g % nxcd, and each XCD
// starts its workgroups in order, so this decides what shares an L2 and what
// is left for the end:
//   * an XCD gets heads / nxcd whole heads (their K/V then live in its L2),
//     one set of them at a time, level by level: unit i of each of them before
//     unit i + 1 of any. The longest units of several heads start first and
//     the short ones fill the end; one head after the other leaves the last
//     head's long units to a few CUs.
//   * heads that do not divide over the XCDs are dealt out unit by unit,
//     first. A contiguous half of a causal head would give one XCD the long
//     half of the triangle and its neighbour the short one, 3 : 1.
// A permutation of the units for every argument.
__host__ __device__ __forceinline__ Unit unit_of(int g, const UnitMap& m) {
  const int nx = (int)m.nxcd.d;
  int s = m.nxcd.div(g);
  const int x = g - s * nx;
  Unit u;
  if (m.dealt > 0) {
    const int mine = m.nxcd.div(m.dealt + nx - 1 - x);   // this XCD's share of them
    if (s < mine) {
      const int v = s * nx + x;
      u.idx = m.rem.div(v);
      u.head = m.whole * nx + (v - u.idx * (int)m.rem.d);
      return u;
    }
    s -= mine;
  }
  const int set = m.set_units.div(s);
  s -= set * (int)m.set_units.d;
  const FastDiv& w = set + 1 < m.sets ? m.width : m.last;
  u.idx = w.div(s);
  u.head = x * m.whole + set * (int)m.width.d + (s - u.idx * (int)w.d);
  return u;
}

// Compute units and XCDs of a device: read once per device from the runtime
// (hipDeviceAttributeMultiprocessorCount, hipDeviceAttributeNumberOfXccs) and
// kept for later calls. A partitioned MI355X reports its own share (e.g. 32
// CUs on one XCD per partition), so the kernel choices and the XCD remap
// follow the device the launch actually runs on.
struct Topology {
  int cus;
  int xcds;
};

inline Topology device_topology(int dev) {
  constexpr int kMaxDev = 64;
  static std::atomic<int> cache[kMaxDev];   // cus << 8 | xcds, 0 = not read yet
  const bool cacheable = dev >= 0 && dev < kMaxDev;
  if (cacheable) {
    const int v = cache[dev].load(std::memory_order_relaxed);
    if (v != 0) return Topology{v >> 8, v & 0xff};
  }
  int cus = 0, xcds = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;   // MI355X, if the runtime cannot say
  if (hipDeviceGetAttribute(&xcds, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess || xcds <= 0)
    xcds = 1;
  if (xcds > 255) xcds = 255;
  if (cacheable) cache[dev].store(cus << 8 | xcds, std::memory_order_relaxed);
  return Topology{cus, xcds};
}

// Topology of the device that runs work queued on `stream`.
inline Topology stream_topology(hipStream_t stream) {
  int dev = 0;
  if (hipStreamGetDevice(stream, &dev) != hipSuccess && hipGetDevice(&dev) != hipSuccess) dev = 0;
  return device_topology(dev);
}

// Inclusive scan over the wave's 64 lanes of x >= 0 (DPP row shifts and row
// broadcasts): op is + or max; lanes without a source see 0.
template <typename Op>
__device__ __forceinline__ int wave_scan(int x, Op op) {
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));   // row_shr:1
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));   // row_shr:2
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));   // row_shr:4
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));   // row_shr:8
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));   // row_bcast:15
  x = op(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));   // row_bcast:31
  return x;
}

__device__ __forceinline__ int scan_sum(int x) {
  return wave_scan(x, [](int a, int b) { return a + b; });
}

__device__ __forceinline__ int scan_max(int x) {
  return wave_scan(x, [](int a, int b) { return max(a, b); });
}

// Bounds read from cu are clamped into [0, total], so a malformed table never
// moves a head's buffer range outside its own rows.
__device__ __forceinline__ int clamp_row(int r, int total) { return min(max(r, 0), total); }

// Batches of up to kCountedSeqs sequences have their units counted (varlen_block).
constexpr int kCountedSeqs = 512;

// Blocks of `rows` rows per head in a varlen grid: sequence b has
// ceil(n_b / rows) of them, and the host knows only that the n_b are at most
// max_seqlen and sum to at most `total`. B of them where max_seqlen <= rows.
inline int64_t varlen_units(int64_t B, int64_t total, int64_t max_seqlen, int rows) {
  const int64_t by_max = B * ((max_seqlen + rows - 1) / rows);
  const int64_t by_total = total / rows + B;
  return B > kCountedSeqs || by_max < by_total ? by_max : by_total;
}

struct SeqBlock {
  int start, n;   // rows of the sequence; n = 0: there is no such unit
  int block;
};

// Unit u of a head's varlen units: the blocks of the sequences longer than half
// of max_seqlen, sequence by sequence, then those of the others. The short
// sequences then fill the end of the launch, and an XCD works through one or
// two sequences at a time (units of equal length of all sequences together
// keep more K/V in use than an L2 holds). `block` counts from 0 within the
// sequence. Every wave finds it from two wave scans of the block counts (lane l
// takes sequences l, l + 64, ...). A full sort by length, with a binary search
// for the length of unit u, cost a workgroup over 1 us and 4-6 % of a launch
// with sequences of 2048 rows.
// Sequence b + 1 starts no earlier than sequence b ends, also where cu
// decreases, so the units never exceed varlen_units().
template <int J>
__device__ __forceinline__ SeqBlock counted_block(const Geom& g, int u, int rows, int lane) {
  const int half = ((g.N + rows - 1) / rows) / 2;
  int c0[J], c1[J];
  bool falls = false;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int b = 64 * j + lane;
    c0[j] = c1[j] = 0;
    if (b < g.B) {
      c0[j] = clamp_row(g.cu[b], g.total);
      c1[j] = clamp_row(g.cu[b + 1], g.total);
      falls |= c1[j] < c0[j];
    }
  }
  if (__any(falls)) {   // malformed: from the running maximum on
    int end = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      c0[j] = scan_max(max(c0[j], end));
      c1[j] = max(c0[j], c1[j]);
      end = __builtin_amdgcn_readlane(c1[j], 63);
    }
  }
  int n[J], big[J], small[J];   // blocks; their scans over the two kinds
  int nbig = 0, nsmall = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    n[j] = (min(c1[j] - c0[j], g.N) + rows - 1) / rows;
    big[j] = nbig + scan_sum(n[j] > half ? n[j] : 0);
    small[j] = nsmall + scan_sum(n[j] > half ? 0 : n[j]);
    nbig = __builtin_amdgcn_readlane(big[j], 63);
    nsmall = __builtin_amdgcn_readlane(small[j], 63);
  }
  const bool in_big = u < nbig;
  const int v = in_big ? u : u - nbig;
  SeqBlock out{0, 0, 0};
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int sum = in_big ? big[j] : small[j];
    const uint64_t m = __ballot((n[j] > half) == in_big && sum > v);
    if (m != 0 && out.n == 0) {
      const int l = __ffsll((unsigned long long)m) - 1;
      out.start = __builtin_amdgcn_readlane(c0[j], l);
      out.n = min(__builtin_amdgcn_readlane(c1[j], l) - out.start, g.N);
      out.block = v - (__builtin_amdgcn_readlane(sum, l) - __builtin_amdgcn_readlane(n[j], l));
    }
  }
  return out;
}

// The same where no sequence is longer than a block: unit u is sequence u's,
// which starts at the largest of the bounds up to it. One scan, two bounds a
// load: the two scans and the search of counted_block made forwards of 256
// sequences of 64 rows, H32 over 8 D64, 10 % slower (us: in sequence order,
// without a look at the other bounds, 173; counted 191; so 170; of 500
// sequences 338, 363, 338; with a bound a load 354).
template <int J>
__device__ __forceinline__ SeqBlock single_block(const Geom& g, int u, int lane) {
  typedef int pair __attribute__((ext_vector_type(2), aligned(4)));
  const int next = g.cu[u + 1];
  int c = 0;
#pragma unroll
  for (int j = 0; j < (J + 1) / 2; ++j) {
    const int b = 128 * j + 2 * lane;
    if (b <= u) {   // cu[b + 1] is there: u < B
      const pair x = *reinterpret_cast<const pair*>(g.cu + b);
      c = max(c, x[0]);
      if (b < u) c = max(c, x[1]);
    }
  }
  c = clamp_row(c, g.total);
  const int start = __builtin_amdgcn_readlane(scan_max(c), 63);
  return SeqBlock{start, min(max(start, clamp_row(next, g.total)) - start, g.N), 0};
}

template <int J>
__device__ __forceinline__ SeqBlock scanned_block(const Geom& g, int u, int rows, int lane) {
  return g.N <= rows ? single_block<J>(g, u, lane) : counted_block<J>(g, u, rows, lane);
}

__device__ __forceinline__ SeqBlock varlen_block(const Geom& g, int u, int rows, int lane) {
  if (g.B <= 64) return scanned_block<1>(g, u, rows, lane);
  if (g.B <= 256) return scanned_block<4>(g, u, rows, lane);
  if (g.B <= kCountedSeqs) return scanned_block<kCountedSeqs / 64>(g, u, rows, lane);
  const int nbmax = (g.N + rows - 1) / rows;   // more: sequence by sequence
  const int b = u / nbmax, i = u - b * nbmax;
  const int s0 = clamp_row(g.cu[b], g.total);
  const int s1 = max(s0, clamp_row(g.cu[b + 1], g.total));
  const int n = min(s1 - s0, g.N);
  return i * rows < n ? SeqBlock{s0, n, i} : SeqBlock{0, 0, 0};
}

// The map of heads * per_head units onto `topo`. Units of one length run head
// by head: the K/V of one head then fill the L2. `uneven` ones (causal,
// ragged) run in sets of as many heads as give every CU of an XCD a unit (a
// head of 32 blocks alone on MI355X), so that each set's short units meet the
// next set's long ones; wider sets only take more of the L2 (B4 H16 N4096 D128
// causal forward: 303 us with sets of one head, 314 with sets of two).
// Measured, one contiguous range of the head-by-head order per XCD before ->
// now: bf16 causal forward and cache write of B2 H32 (8 KV heads) N1777 D128,
// 14 blocks a head, 78.5 -> 72.5 us; bf16 causal backward B1 H32 (8) N2000
// D128 210 -> 187 us; 12 ragged sequences of up to 4096 rows, H8 D64 causal,
// forward and backward 702 -> 686 us; 60 of up to 400 rows, forward 50 -> 34
// us, backward 150 -> 101 us (fewer empty workgroups).
inline UnitMap unit_map(int64_t heads, int64_t per_head, const Topology& topo, bool uneven) {
  const int64_t nx = topo.xcds > 1 ? topo.xcds : 1;
  const int64_t whole = heads / nx, rem = heads % nx;
  int64_t sets = whole > 0 ? whole : 1;
  if (uneven && whole > 1 && per_head > 0) {
    const int64_t cus = (topo.cus + nx - 1) / nx;
    const int64_t want = (cus + per_head - 1) / per_head;
    sets = whole / want > 1 ? whole / want : 1;
  }
  const int64_t width = whole > 0 ? (whole + sets - 1) / sets : 1;   // sets of about equal width
  sets = whole > 0 ? (whole + width - 1) / width : 1;
  UnitMap m;
  m.heads = (int)heads;
  m.per_head = (int)per_head;
  m.nxcd = FastDiv(nx);
  m.whole = (int)whole;
  m.rem = FastDiv(rem > 0 ? rem : 1);
  m.dealt = (int)(rem * per_head);
  m.set_units = FastDiv(width * per_head > 0 ? width * per_head : 1);
  m.width = FastDiv(width);
  m.last = FastDiv(whole > 0 ? whole - (sets - 1) * width : 1);
  m.sets = (int)sets;
  return m;
}

// One (b, h): element offsets of its Q/O and K/V rows, of its L row, and its
// length.
struct HeadView {
  size_t q, kv, l;
  int n;
};

// Head bh of a dense launch, or head h of sequence b of a packed one.
template <int D>
__device__ __forceinline__ HeadView dense_view(const Geom& g, int bh) {
  HeadView v;
  v.n = g.N;
  v.q = (size_t)bh * g.N * D;
  v.kv = (size_t)g.group.div(bh) * g.N * D;
  v.l = (size_t)bh * g.N;
  return v;
}

template <int D>
__device__ __forceinline__ HeadView seq_view(const Geom& g, int h, int start, int n) {
  HeadView v;
  v.n = n;
  v.q = ((size_t)h * g.total + start) * D;
  v.kv = ((size_t)g.group.div(h) * g.total + start) * D;
  v.l = (size_t)h * g.total + start;
  return v;
}

}  // namespace fa
