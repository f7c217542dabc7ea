// Internal device-side building blocks of the libsas forward kernels
// (sas_fwd.hip): constants, the kernel parameter block, element and MFMA
// helpers, LDS-DMA and wait helpers, the slot resolution every kernel starts
// with, and the split partial merge.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>

#include "../../include/sas.h"
#include "sas_common.h"

#include <atomic>

#define LDS_AS __attribute__((address_space(3)))

namespace sas {

constexpr int kDV = 512;          // output / V channels
constexpr int kMaxSlots = 1280;   // slot range one workgroup may own
constexpr int kRoundsMax = kMaxSlots / 256;  // slot rounds at 256 threads
constexpr int kMaxWaves = 8;
constexpr int kRow656 = 656;      // fp8 cache row bytes
constexpr int kChunksMax = 72;    // 16-byte chunks of a 576-channel bf16 row
constexpr int kLdsRows = 128;     // rows of ring storage per workgroup
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kLazyLog2 = 8.f;   // O / l rescale threshold (log2 units)

// Compute units of the current device (one forward workgroup each): the
// grid planners fill them. Queried once per device; 256 (MI355X) when no
// device answers, e.g. a plan query on a host without a GPU.
inline int device_cus() {
  constexpr int kMaxDev = 64, kDefault = 256;
  static std::atomic<int> cached[kMaxDev] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) {
    (void)hipGetLastError();
    return kDefault;
  }
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return kDefault;
  }
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

// XCDs of the current device: a launch deals its workgroups to them
// round-robin (workgroup b runs on XCD b % XCDs), and the grids place each
// token's workgroups on one XCD by that rule. Queried once per device; 8
// (MI355X) when no device answers. The count only places work: any value
// gives the same results.
inline int device_xcds() {
  constexpr int kMaxDev = 64, kDefault = 8;
  static std::atomic<int> cached[kMaxDev] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) {
    (void)hipGetLastError();
    return kDefault;
  }
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess || n <= 0 || n > 64) {
    (void)hipGetLastError();
    return kDefault;
  }
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

// Loads of cache rows whose addresses are held as integers (the compacted
// row lists): through global-address-space pointers, so they compile to
// global loads, counted by vmcnt only. Through generic pointers they become
// flat loads, which count against lgkmcnt as well, so every LDS wait issued
// while they are in flight waits for them too.
#define SAS_GLOBAL __attribute__((address_space(1)))
typedef unsigned u32x4g __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 gld16(uint64_t a) {
  return __builtin_bit_cast(uint4, *reinterpret_cast<const SAS_GLOBAL u32x4g*>(a));
}
__device__ __forceinline__ float gldf(uint64_t a) { return *reinterpret_cast<const SAS_GLOBAL float*>(a); }

static __shared__ __attribute__((aligned(16))) uint4 lds_ring[kLdsRows * kChunksMax];  // 147,456 B
// compacted rows of the workgroup: the byte address of each cache row
// (+ kRowPad entries past the compacted rows: copies of the last one, so a
// streaming step's row lookups need no clamp)
constexpr int kRowPad = 64;
static __shared__ uint64_t lds_rows[kMaxSlots + kRowPad];
static __shared__ int lds_cnt[kRoundsMax][kMaxWaves];
static __shared__ float lds_ml[kMaxWaves][2][16];
static __shared__ int lds_tok[3];   // resolve(): the token's batch, padded flag and causal threshold
// fp8 rows: the fp32 scale of each ring row's four 128-channel latent groups
// ([group][ring row]; the ring holds the unscaled e4m3 values, exact in bf16)
static __shared__ __attribute__((aligned(16))) float lds_fsc[4][kLdsRows];

struct FwdParams {
  const uint8_t* q;
  const uint8_t* ori_kv;
  const int32_t* ori_bt;
  const uint8_t* cmp_kv;
  const int32_t* cmp_bt;
  const int32_t* cmp_idx;
  const int32_t* q_prefix;
  const int32_t* act_q;   // NULL: q_prefix holds B + 1 entries (cu_seqlens_q)
  const int32_t* act_kv;
  const float* sinks;
  uint8_t* out;
  float* lse;
  uint8_t* part_o;    // [T, S, H, 512] PartT: unnormalised O x 2^e per 256-channel half
  float* part_ml;     // [T, S, H, 4]: running max (log2 units), running sum, e of each half
  int T, B, H;
  int ori_bs, ori_bt_stride, ori_nblocks;
  int cmp_bs, cmp_bt_stride, cmp_nblocks;
  int K, scenario, cmp_ratio, win_left;
  float scale_log2;
  int nsplit, slots_per_split, nhg;
  int nxcd;      // XCDs the grid is dealt over (device_xcds())
  int part_nt;   // 1: split partials go out with non-temporal stores
  int out_nt;    // 1: the output (one split) goes out with non-temporal stores
};

// ---------------------------------------------------------------------------
// element helpers
// ---------------------------------------------------------------------------

// Two floats rounded to nearest-even 16-bit values, a in the low half
// (one v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
template <typename QT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef QT v2 __attribute__((ext_vector_type(2)));
  const v2 v = {(QT)a, (QT)b};
  return __builtin_bit_cast(uint32_t, v);
}

// Four OCP e4m3fn bytes (one dword, byte 0 first) as bf16 pairs, unscaled:
// lo = bytes 0-1, hi = bytes 2-3. gfx950's v_cvt_scalef32_pk_bf16_fp8
// converts two OCP e4m3fn bytes (bias 7, subnormals m * 2^-9) straight to a
// bf16 pair; with scale 1 the result is exact (every e4m3fn value is a bf16
// value). 0x7f / 0xff (NaN) are never written by the cache writer, which
// saturates at 448.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void e4m3x4_to_bf16(uint32_t w, uint32_t& lo, uint32_t& hi) {
  lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
  hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true));
}

// 16x16x32: A = 8 values of row l%16 (k = 8*(l/16)..), B likewise by column
template <typename QT>
__device__ __forceinline__ f32x4 mfma32k(const uint4& a, const uint4& b, const f32x4& c);
template <>
__device__ __forceinline__ f32x4 mfma32k<__bf16>(const uint4& a, const uint4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma32k<_Float16>(const uint4& a, const uint4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// 16x16x16: A = 4 values of row l%16 (k = 4*(l/16)..), B likewise by column
template <typename QT>
__device__ __forceinline__ f32x4 mfma16k(const uint2& a, const uint2& b, const f32x4& c);
template <>
__device__ __forceinline__ f32x4 mfma16k<__bf16>(const uint2& a, const uint2& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                   __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16k<_Float16>(const uint2& a, const uint2& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                               __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
}

// Row swizzle of 16-byte chunks for LDS tiles whose rows are RC chunks long:
// row r keeps logical chunk c at c ^ swz<RC>(r). gfx950 LDS has 64 banks of
// 4 bytes (a 256-byte period, 16 chunk positions). A ds_read_b128 serves each
// half-wave in two cycles, one per set of 16 lanes whose lane-id bits 2..4
// have equal parity; ds_read_b64_tr_b16 serves 32 lanes (256 bytes) per
// cycle. The QK^T operand read (lane l: row l & 15 of a 16-row tile, logical
// chunk 4 ks + l / 16) and the transposed PV read (lane l: row
// 4 (l / 16) + (l & 15) / 4, chunks 2t, 2t + 1) then touch every bank once
// per cycle.
//  RC = 0 mod 16: XOR inside aligned 16-chunk groups with 2 (r & 7).
//  RC = 8 mod 16: odd rows start half a period later, so XOR inside aligned
//                 8-chunk groups with r & 6 (the last 8-chunk group of a
//                 72-chunk row has no 16-chunk partner).
template <int RC>
__device__ __forceinline__ int swz(int r) {
  static_assert(RC % 8 == 0, "rows of whole 8-chunk groups");
  if constexpr (RC % 16 == 0) return (r & 7) << 1;
  else return r & 6;
}
// chunks per aligned XOR group of swz<RC>
template <int RC>
inline constexpr int kSwzGroup = RC % 16 == 0 ? 16 : 8;

// Max / sum over the 4 rows (16-lane groups) of a wave, leaving the result in
// every lane: v_permlane16_swap / v_permlane32_swap exchange rows inside the
// VALU (no LDS round trip as a ds_bpermute-based shuffle would take).
__device__ __forceinline__ float rows_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float m = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// 16 bytes per lane global -> LDS (lane i lands at lds_addr + 16 i). Issued
// as inline asm so the compiler does not track it: its LDS-DMA tracking
// cannot tell the slots apart for transposed LDS reads and would wait for
// every load in flight. Completion is ordered explicitly with wait_vm<>()
// (loads return in order, so the compiler's own vmcnt waits for its loads
// stay conservative).
__device__ __forceinline__ void dma16(const void* src, uint32_t lds_addr) {
  asm volatile(
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off"
      :
      : "v"(src), "s"(lds_addr)
      : "memory", "m0");
}

// dma16 from a wave-uniform base and a 32-bit lane offset
__device__ __forceinline__ void dma16s(uint32_t off, const void* base, uint32_t lds_addr) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, %1"
      :
      : "v"(off), "s"(base), "s"(lds_addr)
      : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_addr_of(const void* p) {
  return (uint32_t)(uintptr_t)(const LDS_AS void*)p;
}

// s_waitcnt vmcnt(N) leaving expcnt / lgkmcnt alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void wait_lgkm0() {
  __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4) | (0 << 8));  // lgkmcnt(0)
}
// N 16-byte chunks from global memory into LDS by NT threads: every load is
// issued (at a clamped, in-range index) before the first LDS write, so the
// copy costs one round trip. (A strided copy loop compiled to load, wait,
// write per pass: nine round trips for a 64-head query tile.)
template <int N, int NT, typename Put>
__device__ __forceinline__ void stage_chunks(const uint4* src, int tid, Put&& put) {
  constexpr int NIT = (N + NT - 1) / NT;
  uint4 v[NIT];
#pragma unroll
  for (int j = 0; j < NIT; ++j) v[j] = src[min(tid + j * NT, N - 1)];
#pragma unroll
  for (int j = 0; j < NIT; ++j) {
    const int i = tid + j * NT;
    if (N % NT == 0 || i < N) put(i, v[j]);
  }
}

// LDS reads done, then a workgroup barrier (no memory fence: in-flight LDS
// DMA of other slots keeps streaming across it).
__device__ __forceinline__ void lds_barrier() {
  wait_lgkm0();
  __builtin_amdgcn_s_barrier();
}

// Split-partial O element type: fp16 under bf16 outputs (scaled by a power
// of two per 256-channel half, 8x finer than the output's rounding), fp32
// under fp16 outputs (fp16 would round as coarsely as the output does).
template <typename QT> struct PartSel { using T = _Float16; };
template <> struct PartSel<_Float16> { using T = float; };
template <typename QT> using PartT = typename PartSel<QT>::T;

// Channels per combine thread (4: 8-byte fp16 partial loads, 8: 16-byte)
#ifndef SAS_COMBINE_CPT
#define SAS_COMBINE_CPT 8
#endif
constexpr int kCombineCpt = SAS_COMBINE_CPT;

// Merge the nsplit partials of (token t, heads [h0, h0 + nh)) with the sink
// into out / lse: M = max(sink, m_i), L = 2^(sink-M) + sum_i l_i 2^(m_i-M),
// out = sum_i 2^(m_i-M) O_i / L, lse = (M ln 2) + ln L (a running merge over
// i, kB splits' loads in flight together). Partial O_i is stored as values
// O_i 2^e_i (PartT: fp16, or fp32 with e_i = 0) with one exponent e_i per
// 256-channel half, so it is recovered exactly as ldexp(value, -e_i). A
// thread owns kCombineCpt consecutive channels of one head. A negative l
// marks a padded token (out = 0, lse = 0). The output goes out with
// non-temporal stores: nothing of it is read again by the kernel, and the
// lines leave before the L2 writeback at the kernel's end (32-token decode
// call 19.3-19.6 -> 18.9-19.1 µs, 31-token 128-head decode 28.7-29.0 ->
// 28.2-28.3 µs).
template <typename QT>
__device__ __forceinline__ void merge_partials(const FwdParams& p, int t, int h0, int nh, int tid,
                                               int nthreads) {
  constexpr int kB = 4, CPT = kCombineCpt, NG = kDV / CPT;   // channel groups per head
  const int S = p.nsplit;
  using PT = PartT<QT>;
  typedef PT vc __attribute__((ext_vector_type(CPT)));
  const vc* po = reinterpret_cast<const vc*>(p.part_o) + (size_t)t * S * p.H * NG;
  const float* pm = p.part_ml + (size_t)t * S * p.H * 4;
  for (int e = tid; e < nh * NG; e += nthreads) {
    const int h = h0 + e / NG, cg = e % NG;
    const int half = cg >= NG / 2;
    float M = p.sinks[h] * kLog2e, L = 1.f;
    float o[CPT];
#pragma unroll
    for (int c = 0; c < CPT; ++c) o[c] = 0.f;
    bool pad = false;
    for (int s0 = 0; s0 < S; s0 += kB) {
      float4 ml[kB];
      vc v[kB];
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        const size_t row = (size_t)min(s0 + j, S - 1) * p.H + h;
        ml[j] = *reinterpret_cast<const float4*>(pm + row * 4);
        v[j] = po[row * NG + cg];
      }
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        if (s0 + j >= S) break;
        pad |= ml[j].y < 0.f;
        if (ml[j].x > M) {
          const float a = exp2f(M - ml[j].x);
          L *= a;
#pragma unroll
          for (int c = 0; c < CPT; ++c) o[c] *= a;
          M = ml[j].x;
        }
        const float w = ml[j].x == -INFINITY ? 0.f : exp2f(ml[j].x - M);
        const int ne = -(int)(half ? ml[j].w : ml[j].z);
        L += w * ml[j].y;
#pragma unroll
        for (int c = 0; c < CPT; ++c) o[c] += ldexpf(w * (float)v[j][c], ne);
      }
    }
    const float inv = pad ? 0.f : 1.f / L;
    uint32_t w[CPT / 2];
#pragma unroll
    for (int c = 0; c < CPT / 2; ++c) w[c] = pack2<QT>(o[2 * c] * inv, o[2 * c + 1] * inv);
    uint16_t* dst = reinterpret_cast<uint16_t*>(p.out) + ((size_t)t * p.H + h) * kDV + cg * CPT;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    if constexpr (CPT == 8) __builtin_nontemporal_store(u32x4{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4*>(dst));
    else __builtin_nontemporal_store(u32x2{w[0], w[1]}, reinterpret_cast<u32x2*>(dst));
    if (cg == 0) p.lse[(size_t)t * p.H + h] = pad ? 0.f : M * kLn2 + logf(L);
  }
}

// ---------------------------------------------------------------------------
// shared prologue: slot resolution
// ---------------------------------------------------------------------------

struct Tok {
  int t, hg, sp;     // token, head group, KV split
  int b, nvalid;     // batch, compacted row addresses in lds_rows
  int thr;           // compressed rows below the token's causal position
  bool padded;       // (b, position) outside the batch's query length
};

// Work item of this workgroup, or -1 for a padding workgroup. Tokens are
// dealt round-robin to the device's XCDs (blockIdx % nxcd is the XCD), latest
// token first; all head groups and splits of a token go to one XCD and share its
// L2. Every XCD then gets the same mix of long and short token rows (causal
// prefill: rows grow with the position), and the longest items start first.
__device__ __forceinline__ int item_index(const FwdParams& p) {
  const unsigned nx = (unsigned)p.nxcd;
  const int x = (int)(blockIdx.x % nx), l = (int)(blockIdx.x / nx);
  const int per_tok = p.nhg * p.nsplit;
  const int q = l / per_tok, sub = l - q * per_tok;
  const int t = p.T - 1 - (q * p.nxcd + x);
  return t >= 0 ? t * per_tok + sub : -1;
}

__device__ __forceinline__ Tok item_of(const FwdParams& p, int item) {
  Tok k;
  const int per_tok = p.nhg * p.nsplit;
  k.t = item / per_tok;
  k.hg = (item % per_tok) / p.nsplit;
  k.sp = item % p.nsplit;
  k.b = 0; k.nvalid = 0; k.thr = 0; k.padded = true;
  return k;
}

// Resolve the item's slot range to cache rows and compact the valid ones, in
// slot order, into lds_rows[0, nvalid) as row byte addresses (ROWB bytes per
// row), so the streaming loops only add a chunk offset. The first NT threads
// (waves 0 .. NT/64 - 1, the older wave of each SIMD when the workgroup has
// 8) do the slot work; the others only run `mid` and join the compaction
// barriers. With all 8 waves resolving, the table reads of waves 4-7 came
// back 1-2 µs after those of waves 0-3 and the compaction waited for them
// (4K prefill 580 -> 573 µs with 4 resolving waves). `mid` runs after the
// block-table loads are issued (a caller can put its own loads behind them
// there).
template <int NT, int ROWB, typename Mid>
__device__ __forceinline__ void resolve(const FwdParams& p, Tok& k, int tid, int lane, int wave, Mid&& mid) {
  constexpr int NWV = NT / 64;
  constexpr int kRounds = (kMaxSlots + NT - 1) / NT;
  static_assert(kRounds <= kRoundsMax && NWV <= kMaxWaves, "resolve geometry");
  const bool worker = tid < NT;   // wave-uniform
  const int t = k.t;
  const int wincap = p.win_left + 1;
  const int nslots = wincap + (p.scenario >= SAS_CFA ? p.K : 0);
  const int s0 = k.sp * p.slots_per_split;
  const int s1 = min(s0 + p.slots_per_split, nslots);
  const int nr = (s1 - s0 + NT - 1) / NT;   // slot rounds of NT (<= kRounds)

  uint64_t rad[kRounds];
  bool val[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) { rad[r] = 0; val[r] = false; }
  if (worker) {
    // ---- round trip 1: top-k indices and batch scalars ----------------------
    int idxv[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      idxv[r] = -1;
      const int j = s0 + r * NT + tid;
      if (r < nr && p.scenario == SAS_SCFA && j < s1 && j >= wincap)
        idxv[r] = p.cmp_idx[(size_t)t * p.K + (j - wincap)];
    }
    // act_q == NULL: q_prefix is cu_seqlens_q [B + 1] and a query length is
    // the difference of two entries (loaded in the same round trip)
    const bool cu = p.act_q == nullptr;
    int qp0 = INT_MAX, aq0 = 0, akv0 = 0;
    if (lane < p.B) { qp0 = p.q_prefix[lane]; aq0 = cu ? p.q_prefix[lane + 1] : p.act_q[lane]; akv0 = p.act_kv[lane]; }
    // token -> (batch, position): largest b with q_prefix[b] <= t (q_prefix is
    // non-decreasing), one ballot per 64 batches
    int b = 0, aq = 0, akv = 0, qpb = 0;
    {
      uint64_t m = __ballot(qp0 <= t);
      int n = __popcll(m);
      if (n) { b = n - 1; qpb = __shfl(qp0, n - 1); aq = __shfl(aq0, n - 1); akv = __shfl(akv0, n - 1); }
      for (int c = 64; n == 64 && c < p.B; c += 64) {
        const int i = c + lane;
        int qpi = INT_MAX, aqi = 0, akvi = 0;
        if (i < p.B) { qpi = p.q_prefix[i]; aqi = cu ? p.q_prefix[i + 1] : p.act_q[i]; akvi = p.act_kv[i]; }
        m = __ballot(qpi <= t);
        n = __popcll(m);
        if (n) { b = c + n - 1; qpb = __shfl(qpi, n - 1); aq = __shfl(aqi, n - 1); akv = __shfl(akvi, n - 1); }
      }
    }
    if (cu) aq -= qpb;   // end of the batch's tokens -> its query length
    const int spos = t - qpb;
    const bool padded = spos < 0 || spos >= aq;
    const int sg = akv - aq + spos;                              // causal position
    const int nwin = (padded || sg < 0) ? 0 : min(sg, p.win_left) + 1;
    const int wlo = sg - nwin + 1;                               // = max(sg - win_left, 0)
    const int thr = (padded || sg + 1 <= 0) ? 0 : (sg + 1) / p.cmp_ratio;
    if (tid == 0) { lds_tok[0] = b; lds_tok[1] = padded; lds_tok[2] = thr; }

    // ---- round trip 2: block tables -----------------------------------------
    // Every table read is issued unconditionally at a clamped, in-range
    // address (validity is kept apart), so the reads of all rounds are in
    // flight together and retire with one wait.
    const int32_t* obt = p.ori_bt + (size_t)b * p.ori_bt_stride;
    const int32_t* cbt = p.cmp_bt ? p.cmp_bt + (size_t)b * p.cmp_bt_stride : obt;
    int phys[kRounds], off[kRounds];
    bool ok[kRounds], ori[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      phys[r] = -1; ok[r] = false; ori[r] = true; off[r] = 0;
      if (r >= nr) continue;   // uniform
      const int j = s0 + r * NT + tid;
      const bool live = j < s1 && !padded;
      int blk;
      if (j < wincap) {
        const int pos = wlo + j;
        blk = pos / p.ori_bs;
        off[r] = pos - blk * p.ori_bs;
        ok[r] = live && j < nwin && blk < p.ori_bt_stride;
      } else {
        const int idx = p.scenario == SAS_SCFA ? idxv[r] : j - wincap;
        const int ic = max(idx, 0);
        blk = ic / p.cmp_bs;
        off[r] = ic - blk * p.cmp_bs;
        ori[r] = false;
        ok[r] = live && idx >= 0 && idx < thr && blk < p.cmp_bt_stride;
      }
      phys[r] = (ori[r] ? obt : cbt)[ok[r] ? blk : 0];
    }
    // the caller's loads go behind the table reads, so waiting for the
    // tables leaves them in flight
    asm volatile("" ::: "memory");
    mid();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      const bool inb = phys[r] >= 0 && phys[r] < (ori[r] ? p.ori_nblocks : p.cmp_nblocks);
      val[r] = ok[r] && inb;
      const int row = val[r] ? phys[r] * (ori[r] ? p.ori_bs : p.cmp_bs) + off[r] : 0;
      rad[r] = reinterpret_cast<uint64_t>(ori[r] ? p.ori_kv : p.cmp_kv) + (uint64_t)(uint32_t)row * ROWB;
    }
  } else {
    mid();
  }
  // ---- compaction (ballot + per-wave counts) -------------------------------
  uint64_t vmask[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    vmask[r] = __ballot(val[r]);
    if (worker && r < nr && lane == 0) lds_cnt[r][wave] = __popcll(vmask[r]);
  }
  __syncthreads();
  int nvalid = 0;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    if (r >= nr) break;
    int wpre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const int cw = lds_cnt[r][w];
      wpre += w < wave ? cw : 0;
      tot += cw;
    }
    if (val[r])
      lds_rows[nvalid + wpre + __popcll(vmask[r] & ((1ull << lane) - 1ull))] = rad[r];
    nvalid += tot;
  }
  k.b = lds_tok[0];
  k.padded = lds_tok[1] != 0;
  k.thr = lds_tok[2];
  __syncthreads();
  k.nvalid = nvalid;
}

}  // namespace sas
