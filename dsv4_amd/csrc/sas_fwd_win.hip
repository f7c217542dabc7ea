// Window-only forward over runs of consecutive tokens, MI355X (gfx950).
//
// A prefill's neighbouring tokens share all but one window row. The
// one-workgroup-per-token kernel gathers every token's window anew and spends
// most of a token's time on round trips (tables, rows, query, output) with
// nothing beside them: 12.7 us per token and CU for 64 heads, D = 512,
// against 6.6 us that the query and output bytes alone take at the card's
// copy rate. Here a workgroup walks a run of consecutive tokens of one batch
// with the window rows resident in an LDS ring (position p in slot p mod NS):
// kGroup tokens at a time need win_left + kGroup rows, so a group loads
// kGroup new rows and the waves then work without a barrier until the next.
// A wave's unit is (token, 16 heads), all keys and channels: S over the whole
// window first, then P against the final maximum (as the exact schedule
// rounds it), then P.V; the next unit's query is loaded under P.V. 8192 tokens,
// 64 heads, D = 512: 247 us against 406 (copy-rate floor 210: query and
// output, 1.08 GB).

#include "sas_fwd_win.h"

namespace sas {
namespace {

// A workgroup's run of tokens [r0, r1) of batch b. A batch owns the tokens from
// its start (batch 0: from 0) to the next batch's, valid or padded; group i is
// the i-th run over all batches.
struct Run { int b, r0, r1, qp, aq, akv; };
__device__ __forceinline__ bool find_run(const FwdParams& p, int run, int grp, int lane, Run& o) {
  const bool cu = p.act_q == nullptr;
  int base = 0;
  for (int c = 0; c < p.B; c += 64) {
    const int i = c + lane;
    int s = 0, e = 0, qpi = 0, aqi = 0, kvi = 0;
    if (i < p.B) {
      qpi = p.q_prefix[i];
      s = i == 0 ? 0 : min(max(qpi, 0), p.T);
      e = i + 1 < p.B ? min(max(p.q_prefix[i + 1], s), p.T) : p.T;
      aqi = cu ? p.q_prefix[i + 1] - qpi : p.act_q[i];
      kvi = p.act_kv[i];
    }
    const int n = (e - s + run - 1) / run;
    int x = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) { const int v = __shfl_up(x, d); x += lane >= d ? v : 0; }
    const uint64_t m = __ballot(base + x > grp);
    if (m) {
      const int j = __ffsll((unsigned long long)m) - 1;
      const int k = grp - base - (__shfl(x, j) - __shfl(n, j));
      const int r0 = __shfl(s, j) + k * run;
      o.b = __builtin_amdgcn_readfirstlane(c + j);
      o.r0 = __builtin_amdgcn_readfirstlane(r0);
      o.r1 = __builtin_amdgcn_readfirstlane(min(r0 + run, __shfl(e, j)));
      o.qp = __builtin_amdgcn_readfirstlane(__shfl(qpi, j));
      o.aq = __builtin_amdgcn_readfirstlane(__shfl(aqi, j));
      o.akv = __builtin_amdgcn_readfirstlane(__shfl(kvi, j));
      return true;
    }
    base += __shfl(x, 63);
  }
  return false;
}

// 16 heads x 512 channels of a wave (lane (g, c16): channels 16 i + 4 g .. + 3
// of head c16), scaled by inv, staged PT channel tiles at a time in the wave's
// own LDS rows and stored as whole runs of a head's row. The output leaves
// with non-temporal stores: nothing reads it again here.
template <int PT, typename QT>
__device__ __forceinline__ void store_out(const f32x4 (&acc)[kDV / 16], float inv, uint8_t* sb, uint8_t* ob, int lane) {
  constexpr int SRB = PT * 32 + 16, CPR = PT * 2;          // staged row bytes, its 16-byte chunks
  static_assert(16 * CPR % 64 == 0, "whole store instructions");
  const int c16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int c = 0; c < kDV / 16; c += PT) {
#pragma unroll
    for (int i = 0; i < PT; ++i)
      *reinterpret_cast<uint2*>(sb + c16 * SRB + (i * 16 + 4 * g) * 2) =
          make_uint2(pack2<QT>(acc[c + i][0] * inv, acc[c + i][1] * inv), pack2<QT>(acc[c + i][2] * inv, acc[c + i][3] * inv));
#pragma unroll
    for (int i = 0; i < 16 * CPR / 64; ++i) {
      const int e = i * 64 + lane, r = e / CPR, k = e - r * CPR;
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 w = *reinterpret_cast<const u32x4*>(sb + r * SRB + k * 16);
      __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(ob + (size_t)r * kDV * 2 + c * 32 + k * 16));
    }
  }
}
__device__ __forceinline__ void store_zero(uint8_t* ob, int lane) {
  uint4* o = reinterpret_cast<uint4*>(ob);
#pragma unroll
  for (int i = 0; i < 16 * kDV * 2 / 16 / 64; ++i) o[i * 64 + lane] = make_uint4(0, 0, 0, 0);
}

constexpr int kWinMax = 128;   // window rows a unit holds: 8 key tiles

template <int D> struct WinCfg {
  static constexpr int CH = D / 8;                       // 16-byte chunks per row
  static constexpr int NS = D == 576 ? 136 : 144;        // ring slots (a multiple of 8: the swizzle follows the position)
  static constexpr int kGroup = NS - kWinMax;            // tokens per group
  static constexpr int PT = D == 576 ? 2 : 4;            // channel tiles staged at a time on the way out
  static constexpr int SRB = PT * 32 + 16;               // staged row bytes
};

template <int D, typename QT>
__global__ void __launch_bounds__(256) sas_fwd_win_kernel(const FwdParams p, const int run) {
  using C = WinCfg<D>;
  constexpr int CH = C::CH, NS = C::NS, KS = D / 32, NT = kDV / 16;
  constexpr int XK = kSwzGroup<CH> / 4;                  // k-steps per swizzle group
  constexpr int XV = kSwzGroup<CH> / 2;                  // channel tiles per swizzle group
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * CH * 16];
  __shared__ __attribute__((aligned(16))) uint8_t stage[4][16 * C::SRB];
  __shared__ uint64_t radr[NS];                          // this group's new rows: address (0: no such row)
  __shared__ int bad[NS];                                // per slot: 1 if its row is missing

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int c16 = lane & 15, g = lane >> 4;
  // workgroup -> (batch, run)
  Run rn;
  if (!find_run(p, run, (int)blockIdx.x, lane, rn)) return;
  const int b = rn.b, r0 = rn.r0, r1 = rn.r1, qp = rn.qp, aq = rn.aq, akv = rn.akv;
  const int sg0 = akv - aq - qp;                 // causal position of token t: t + sg0
  const int v0 = max(r0, qp), v1 = (int)min((long long)r1, (long long)qp + max(aq, 0));   // its valid tokens
  const int nhg = p.H / 16;
  const int32_t* bt = p.ori_bt + (size_t)b * p.ori_bt_stride;

  uint4 qf[KS];
  auto load_q = [&](int t, int hg) {
    const uint4* q = reinterpret_cast<const uint4*>(p.q + ((size_t)t * p.H + hg * 16 + c16) * D * 2) + g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = q[ks * 4];
  };
  int loaded = INT_MIN;                          // positions below are in the ring (or behind it)
  int any_bad = 0;
  if (tid < NS) bad[tid] = 0;
  for (int t0 = r0; t0 < r1; t0 += C::kGroup) {
    const int t1 = min(t0 + C::kGroup, r1);
    // rows of the group's valid tokens
    const int w0 = max(t0, v0), w1 = min(t1, v1);          // valid tokens of the group
    const int hi = w0 < w1 ? w1 - 1 + sg0 : -1;            // last position
    const int lo = w0 < w1 ? max(max(w0 + sg0 - p.win_left, 0), loaded) : 0;
    const int n = hi - lo + 1;                             // new rows (<= NS)
    __syncthreads();                                       // every wave is done with the slots they take
    if (n > 0) {
      if (tid < n) {
        const int pos = lo + tid, blk = pos / p.ori_bs;
        uint64_t a = 0;
        if (blk < p.ori_bt_stride) {
          const int ph = bt[blk];
          if (ph >= 0 && ph < p.ori_nblocks)
            a = reinterpret_cast<uint64_t>(p.ori_kv) + (uint64_t)(uint32_t)(ph * p.ori_bs + pos - blk * p.ori_bs) * (D * 2);
        }
        radr[tid] = a;
        bad[pos % NS] = a == 0;
      }
      any_bad |= __syncthreads_or(tid < n && radr[tid] == 0);
      for (int i = wave; i < n; i += 4) {                  // wave-uniform
        const uint64_t a = radr[i];
        const uint64_t src = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                             (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
        const int slot = (lo + i) % NS, sw = swz<CH>(slot);
        const uint32_t dst = lds_addr_of(ring) + slot * CH * 16;
        // a missing row is zero bytes: masked out, and finite for P.V
        if (src == 0) {
          *reinterpret_cast<uint4*>(ring + slot * CH * 16 + lane * 16) = make_uint4(0, 0, 0, 0);
          if (CH > 64 && lane < CH - 64) *reinterpret_cast<uint4*>(ring + slot * CH * 16 + (64 + lane) * 16) = make_uint4(0, 0, 0, 0);
          continue;
        }
        dma16s((uint32_t)((lane ^ sw) * 16), reinterpret_cast<const void*>(src), __builtin_amdgcn_readfirstlane(dst));
        if (CH > 64 && lane < CH - 64)
          dma16s((uint32_t)((64 + (lane ^ sw)) * 16), reinterpret_cast<const void*>(src), __builtin_amdgcn_readfirstlane(dst + 1024));
      }
      loaded = hi + 1;
    }
    const int items = (t1 - t0) * nhg;
    int it = wave;
    if (it < items) load_q(t0 + it / nhg, it % nhg);
    __builtin_amdgcn_s_waitcnt(0);                         // my rows (and the query)
    __builtin_amdgcn_s_barrier();
    for (; it < items; it += 4) {
      const int t = t0 + it / nhg, hg = it % nhg;
      const bool padded = t < qp || t - qp >= aq;
      const int sg = t + sg0, nwin = padded || sg < 0 ? 0 : min(sg, p.win_left) + 1;
      const int nx = it + 4 < items ? it + 4 : it;         // (the last unit's query again)
      const float sink2 = p.sinks[hg * 16 + c16] * kLog2e;
      float* lse = p.lse + (size_t)t * p.H + hg * 16;
      if (nwin == 0) {
        store_zero(p.out + ((size_t)t * p.H + hg * 16) * kDV * 2, lane);
        if (g == 0) lse[c16] = padded ? 0.f : sink2 * kLn2;
        load_q(t0 + nx / nhg, nx % nhg);
        continue;
      }
      const int s0 = (sg - nwin + 1) % NS;                 // slot of the window's first row
      auto slot_of = [&](int r) {                          // window row r (past the end: the last one)
        const int s = s0 + min(r, nwin - 1);
        return s >= NS ? s - NS : s;
      };
      // S^T: key tile i, rows 16 i + c16 of the window; logical chunk 4 ks + g
      f32x4 s[8];
      uint32_t ka[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int sl = slot_of(16 * i + c16);
        ka[i] = (uint32_t)(sl * CH * 16 + ((g ^ swz<CH>(sl)) * 16));
      }
      auto kfrag = [&](int ks, int i) {
        return *reinterpret_cast<const uint4*>(ring + ((ka[i] ^ (uint32_t)((ks % XK) * 64)) + (ks / XK) * (kSwzGroup<CH> * 16)));
      };
      {
        uint4 a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = kfrag(0, i);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const uint4 ai = a[i];
            if (ks + 1 < KS) a[i] = kfrag(ks + 1, i);
            s[i] = mfma32k<QT>(ai, qf[ks], s[i]);
          }
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
        for (int j = 0; j < KS * 8; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (j < KS * 8 - 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
      load_q(t0 + nx / nhg, nx % nhg);
      // lane (g, c16): keys 16 i + 4 g + j of head c16
      float m = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] *= p.scale_log2;
      if (nwin < kWinMax || any_bad) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int r = 16 * i + 4 * g + j;
            if (r >= nwin || (any_bad && bad[slot_of(r)])) s[i][j] = -INFINITY;
          }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) m = fmaxf(m, fmaxf(fmaxf(s[i][0], s[i][1]), fmaxf(s[i][2], s[i][3])));
      m = fmaxf(rows_max(m), sink2);
      const float mb = m == -INFINITY ? 0.f : m;           // no sink and no row present: every P is 0
      float l = 0.f;
      uint32_t pk[8][2];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { s[i][j] = __builtin_amdgcn_exp2f(s[i][j] - mb); l += s[i][j]; }
        pk[i][0] = pack2<QT>(s[i][0], s[i][1]);
        pk[i][1] = pack2<QT>(s[i][2], s[i][3]);
      }
      l = rows_sum(l) + __builtin_amdgcn_exp2f(sink2 - mb);
      // O^T[channel][head] += V^T . P^T over 32 keys at a time
      f32x4 acc[NT];
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (32 * k >= nwin) break;                         // uniform
        uint32_t va[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int sl = slot_of(32 * k + 16 * h + 4 * g + (c16 >> 2));
          va[h] = (uint32_t)(sl * CH * 16 + ((((c16 & 3) >> 1) ^ swz<CH>(sl)) * 16) + (c16 & 1) * 8);
        }
        auto vfrag = [&](int ct) {
          uint2 u[2];
#pragma unroll
          for (int h = 0; h < 2; ++h)
            u[h] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (LDS_AS i16x4*)(ring + ((va[h] ^ (uint32_t)((ct % XV) * 32)) + (ct / XV) * (kSwzGroup<CH> * 16)))));
          return make_uint4(u[0].x, u[0].y, u[1].x, u[1].y);
        };
        const uint4 pf = make_uint4(pk[2 * k][0], pk[2 * k][1], pk[2 * k + 1][0], pk[2 * k + 1][1]);
        constexpr int PV = 4;
        uint4 v[PV];
#pragma unroll
        for (int i = 0; i < PV; ++i) v[i] = vfrag(i);
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          const uint4 a = v[ct % PV];
          if (ct + PV < NT) v[ct % PV] = vfrag(ct + PV);
          acc[ct] = mfma32k<QT>(a, pf, acc[ct]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * PV, 1);
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
          if (ct + PV < NT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        }
      }
      store_out<C::PT, QT>(acc, 1.f / l, stage[wave], p.out + ((size_t)t * p.H + hg * 16) * kDV * 2, lane);
      if (g == 0) lse[c16] = m * kLn2 + logf(l);
    }
  }
}

// ---------------------------------------------------------------------------
// dense compressed scenario (window + every compressed row below the causal
// threshold)
// ---------------------------------------------------------------------------
//
// A workgroup (64 heads, 4 waves) walks a run of tokens of one batch, one token
// at a time, in 32-row steps through two LDS slots whose DMA runs a step
// ahead, across tokens: no token waits for its tables (the run's row addresses
// are looked up once, into LDS) or its first rows. A wave holds 16 heads over
// all keys and channels; online softmax seeded by the sink, O and l rescaled
// when a row's maximum rises by more than 2^8. A step is ~4500 clk of mostly
// serial work (scores 1200, softmax 1300, P.V 1350) and a token's output
// stores another 5400, so two workgroups share each CU (80 KB of LDS and 256
// registers a wave each, 14 to 17 of them spilled): one, with four slots and a
// deeper DMA lead, took 520 us for 8192 tokens, 64 heads, D = 512, ratio 128;
// two take 364, the one-workgroup-per-token kernel 452.
__device__ const uint4 kZeroRow[576 * 2 / 16] = {};   // a missing row's bytes: finite, whatever the caller's hold

template <int D, typename QT>
__global__ void __launch_bounds__(256, 2) sas_fwd_dense_kernel(const FwdParams p, const int run) {
  // slot: the 32 rows' latent chunks [32][64] (chunk c of row r at c ^
  // swz<64>(r)), then, D = 576, their rope chunks [32][8] (at c ^ (r >> 1)):
  // a latent row is one DMA instruction, eight rows' rope another
  constexpr int KS = D / 32, NT = kDV / 16, LCH = 64, ROPE = D > kDV, RI = 8 + ROPE;
  constexpr int LAT = 32 * LCH * 16, SLOT = LAT + ROPE * 32 * 128, PT = ROPE ? 2 : 4;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[2 * SLOT];
  __shared__ __attribute__((aligned(16))) uint8_t stage[4][16 * (PT * 32 + 16)];
  // row addresses (0: no such row): window rows, then compressed ones
  __shared__ uint64_t tab[kDenseWinRows + kDenseCmpRows];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int c16 = lane & 15, g = lane >> 4;
  const int hb = (int)(blockIdx.x % (unsigned)p.nhg), hq = hb * 64 + wave * 16;
  Run rn;
  if (!find_run(p, run, (int)(blockIdx.x / (unsigned)p.nhg), lane, rn)) return;
  const int sg0 = rn.akv - rn.aq - rn.qp;                  // causal position of token t: t + sg0
  const int v0 = max(rn.r0, rn.qp), v1 = (int)min((long long)rn.r1, (long long)rn.qp + max(rn.aq, 0));
  // the run's window and compressed row addresses
  const int wlo = max(0, v0 + sg0 - p.win_left);
  auto thr_of = [&](int sg) { return sg + 1 <= 0 ? 0 : min((sg + 1) / p.cmp_ratio, p.K); };
  const int ncmp = v0 < v1 ? thr_of(v1 - 1 + sg0) : 0;
  int missing = 0;
  for (int i = tid; i < kDenseWinRows + ncmp; i += 256) {
    const bool ori = i < kDenseWinRows;
    const int pos = ori ? wlo + i : i - kDenseWinRows, bs = ori ? p.ori_bs : p.cmp_bs, blk = pos / bs;
    uint64_t a = 0;
    const bool want = !ori || (v0 < v1 && pos <= v1 - 1 + sg0);
    if (want && blk < (ori ? p.ori_bt_stride : p.cmp_bt_stride)) {
      const int ph = (ori ? p.ori_bt + (size_t)rn.b * p.ori_bt_stride : p.cmp_bt + (size_t)rn.b * p.cmp_bt_stride)[blk];
      if (ph >= 0 && ph < (ori ? p.ori_nblocks : p.cmp_nblocks))
        a = reinterpret_cast<uint64_t>(ori ? p.ori_kv : p.cmp_kv) + (uint64_t)(uint32_t)(ph * bs + pos - blk * bs) * (D * 2);
    }
    missing |= want && a == 0;
    tab[i] = a;
  }
  const bool any_bad = __syncthreads_or(missing);

  // a token's rows: window rows from tab[wb], then the compressed ones
  struct Rows { int wb, nwin, n, steps; };
  auto rows_of = [&](int t) {
    Rows r;
    const int sg = t + sg0;
    const bool ok = t >= v0 && t < v1 && sg >= 0;
    r.nwin = ok ? min(sg, p.win_left) + 1 : 0;
    r.wb = sg - r.nwin + 1 - wlo;
    r.n = ok ? r.nwin + thr_of(sg) : 0;
    r.steps = (r.n + 31) >> 5;
    return r;
  };
  const uint64_t spare = reinterpret_cast<uint64_t>(kZeroRow);
  auto row_addr = [&](const Rows& r, int j) {
    j = max(min(j, r.n - 1), 0);
    return tab[j < r.nwin ? r.wb + j : kDenseWinRows + j - r.nwin];
  };
  // producer: step ps of token pt goes to slot pi % 2; a wave moves the rows
  // 8 wave .. + 7 of every step in RI instructions
  int pt = rn.r0, ps = 0, pi = 0;
  Rows pr = rows_of(pt);
  uint64_t pl = 0, pp = 0;   // address of row 8 wave + (lane & 7) / + (lane >> 3) of the step
  auto prep = [&] {
    while (pt < rn.r1 && ps >= pr.steps) {                 // uniform
      ++pt;
      ps = 0;
      pr = rows_of(pt < rn.r1 ? pt : rn.r1 - 1);
    }
    // (past the run, and for a missing row: zero bytes, masked out)
    pl = row_addr(pr, ps * 32 + 8 * wave + (lane & 7));
    if (ROPE) pp = row_addr(pr, ps * 32 + 8 * wave + (lane >> 3));
    if (pt >= rn.r1) pl = pp = 0;
    if (pl == 0) pl = spare;
    if (pp == 0) pp = spare;
    ++ps;
  };
  const uint32_t ol = (uint32_t)lane * 16, orp = 1024 + (uint32_t)(((lane & 7) ^ (((8 * wave + (lane >> 3)) >> 1) & 7)) * 16);
  auto fire = [&](int m) {
    const uint32_t slot = lds_addr_of(ring + (pi & 1) * SLOT);
    if (m < 8) {
      const uint64_t a = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(pl >> 32), m) << 32) |
                         (uint32_t)__builtin_amdgcn_readlane((int)pl, m);
      dma16s(ol ^ (uint32_t)(swz<LCH>(m) * 16), reinterpret_cast<const void*>(a),
             __builtin_amdgcn_readfirstlane(slot + (8 * wave + m) * 1024));
    } else {
      dma16(reinterpret_cast<const void*>(pp + orp), __builtin_amdgcn_readfirstlane(slot + LAT + 8 * wave * 128));
    }
  };
  uint4 qf[KS];
  auto load_q = [&](int t) {
    const uint4* q = reinterpret_cast<const uint4*>(p.q + ((size_t)t * p.H + hq + c16) * D * 2) + g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = q[ks * 4];
  };
  const float sink2 = p.sinks[hq + c16] * kLog2e;
  load_q(rn.r0);
  prep();
#pragma unroll
  for (int m = 0; m < RI; ++m) fire(m);
  ++pi;
  const uint32_t ka = (uint32_t)(c16 * 1024 + ((g ^ swz<LCH>(c16)) * 16));
  const uint32_t kr = (uint32_t)(LAT + c16 * 128 + ((g ^ (c16 >> 1)) * 16));   // rope: rows 16 apart share the xor
  const int vr = 4 * g + (c16 >> 2);
  const uint32_t va = (uint32_t)(vr * 1024 + ((((c16 & 3) >> 1) ^ swz<LCH>(vr)) * 16) + (c16 & 1) * 8);
  int ci = 0;                                              // consumer's step
  constexpr int kTokStores = 17;   // a token's stores (output 16, lse), issued behind the next query's loads
  __builtin_amdgcn_s_waitcnt(0);
  for (int t = rn.r0; t < rn.r1; ++t) {
    const Rows r = rows_of(t);
    const int tn = min(t + 1, rn.r1 - 1);
    uint8_t* ob = p.out + ((size_t)t * p.H + hq) * kDV * 2;
    float* lse = p.lse + (size_t)t * p.H + hq;
    if (r.steps == 0) {                                    // padded, or before the first row: the sink alone
      store_zero(ob, lane);
      if (g == 0) lse[c16] = t >= v0 && t < v1 ? sink2 * kLn2 : 0.f;
      load_q(tn);
      __builtin_amdgcn_s_waitcnt(0);
      continue;
    }
    f32x4 acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = sink2, l = 0.f;                              // l: this lane's keys
    const uint8_t* kt;
    f32x4 s[2];
    int st = 0;
    auto scores = [&]() __attribute__((always_inline)) {
      if (st) wait_vm<0>();   // my DMA of this step (a token's first: waited for with its query)
      lds_barrier();
      kt = ring + (ci & 1) * SLOT;
      prep();
      s[0] = s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
      {
        auto kfrag = [&](int ks, int mt) {
          return *reinterpret_cast<const uint4*>(
              kt + (ks < 16 ? (ka ^ (uint32_t)((ks & 3) * 64)) + (ks >> 2) * 256 + mt * 16 * 1024
                            : (kr ^ (uint32_t)((ks & 1) * 64)) + mt * 16 * 128));
        };
        constexpr int PF = 2;
        uint4 a[PF][2];
#pragma unroll
        for (int i = 0; i < PF; ++i) { a[i][0] = kfrag(i, 0); a[i][1] = kfrag(i, 1); }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const uint4 a0 = a[ks % PF][0], a1 = a[ks % PF][1];
          if (ks + PF < KS) { a[ks % PF][0] = kfrag(ks + PF, 0); a[ks % PF][1] = kfrag(ks + PF, 1); }
          s[0] = mfma32k<QT>(a0, qf[ks], s[0]);
          s[1] = mfma32k<QT>(a1, qf[ks], s[1]);
          if (ks % 2 == 1 && ks / 2 < RI) fire(ks / 2);
        }
        ++pi;
      }
    };
    auto softmax_pv = [&]() __attribute__((always_inline)) {
      // the step's rows that count, bit k for row k
      const int nk = r.n - st * 32;
      uint32_t ok = nk >= 32 ? 0xffffffffu : (1u << nk) - 1u;
      if (any_bad) ok &= ~(uint32_t)__ballot(lane < 32 && row_addr(r, st * 32 + (lane & 31)) == 0);
      const uint32_t okl = ok >> (4 * g);
      float mx = -INFINITY;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[mt][j] = okl >> (16 * mt + j) & 1u ? s[mt][j] * p.scale_log2 : -INFINITY;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) mx = fmaxf(mx, fmaxf(fmaxf(s[mt][0], s[mt][1]), fmaxf(s[mt][2], s[mt][3])));
      mx = rows_max(mx);
      if (__ballot(mx > m + kLazyLog2)) {
        const float mn = fmaxf(m, mx), al = m == mn ? 1.f : __builtin_amdgcn_exp2f(m - mn);
        l *= al;
        m = mn;
#pragma unroll
        for (int i = 0; i < NT; ++i)   // in place: written as a product, the accumulators are copied on both paths
          asm volatile("v_mul_f32 %0, %4, %0\n\tv_mul_f32 %1, %4, %1\n\tv_mul_f32 %2, %4, %2\n\tv_mul_f32 %3, %4, %3"
                       : "+v"(acc[i][0]), "+v"(acc[i][1]), "+v"(acc[i][2]), "+v"(acc[i][3]) : "v"(al));
      }
      const float mb = m == -INFINITY ? 0.f : m;           // no sink and no row present yet: every P is 0
      uint32_t pk[4];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { s[mt][j] = __builtin_amdgcn_exp2f(s[mt][j] - mb); l += s[mt][j]; }
        pk[2 * mt] = pack2<QT>(s[mt][0], s[mt][1]);
        pk[2 * mt + 1] = pack2<QT>(s[mt][2], s[mt][3]);
      }
      const uint4 pf = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      auto vfrag = [&](int ct) {
        const uint8_t* b0 = kt + ((va ^ (uint32_t)((ct & 7) * 32)) + (ct >> 3) * 256);
        const uint2 u0 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0)));
        const uint2 u1 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0 + 16 * 1024)));
        return make_uint4(u0.x, u0.y, u1.x, u1.y);
      };
      constexpr int PV = 4;
      uint4 v[PV];
#pragma unroll
      for (int i = 0; i < PV; ++i) v[i] = vfrag(i);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        const uint4 a = v[ct % PV];
        if (ct + PV < NT) v[ct % PV] = vfrag(ct + PV);
        acc[ct] = mfma32k<QT>(a, pf, acc[ct]);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * PV, 1);
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
        if (ct + PV < NT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
      }
    };
    // The query is known to be here before the step loop, and the next one's
    // loads are issued after it: a load the compiler tracks inside the loop
    // makes it wait for every row DMA in flight at each step.
    __builtin_amdgcn_s_waitcnt((kTokStores & 15) | (7 << 4) | (15 << 8) | ((kTokStores >> 4) << 14));   // vmcnt(kTokStores)
    for (; st < r.steps; ++st, ++ci) {
      scores();
      softmax_pv();
    }
    load_q(tn);
    l = rows_sum(l) + __builtin_amdgcn_exp2f(sink2 - (m == -INFINITY ? 0.f : m));
    store_out<PT, QT>(acc, l == 0.f ? 0.f : 1.f / l, stage[wave], ob, lane);   // (0: no sink, no row)
    if (g == 0) lse[c16] = m * kLn2 + logf(l);
  }
  wait_vm<0>();   // the spare steps' DMA
}

template <int D, typename QT>
int launch(const FwdParams& fp, int run, hipStream_t st) {
  const int nb = fp.T / run + fp.B;
  if (fp.scenario == SAS_CFA) hipLaunchKernelGGL((sas_fwd_dense_kernel<D, QT>), dim3((unsigned)nb * fp.nhg), dim3(256), 0, st, fp, run);
  else hipLaunchKernelGGL((sas_fwd_win_kernel<D, QT>), dim3(nb), dim3(256), 0, st, fp, run);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(SAS_ELAUNCH, "sas_fwd_win launch: %s", hipGetErrorString(e));
  return SAS_OK;
}

}  // namespace

int launch_fwd_win(const FwdParams& fp, int D, int q_dtype, int run, hipStream_t st) {
  if (q_dtype == SAS_DT_BF16) return D == 576 ? launch<576, __bf16>(fp, run, st) : launch<512, __bf16>(fp, run, st);
  return D == 576 ? launch<576, _Float16>(fp, run, st) : launch<512, _Float16>(fp, run, st);
}

}  // namespace sas
