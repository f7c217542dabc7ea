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
// 64 heads, D = 512: 247 us against 447 (copy-rate floor 210: query and
// output, 1.08 GB).

#include "sas_fwd_win.h"

namespace sas {
namespace {

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
  // workgroup -> (batch, run): a batch owns the tokens from its start (batch
  // 0: from 0) to the next batch's, valid or padded
  const bool cu = p.act_q == nullptr;
  int b = -1, r0 = 0, r1 = 0, qp = 0, aq = 0, akv = 0;
  {
    int base = 0;
    for (int c = 0; c < p.B && b < 0; c += 64) {
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
      const uint64_t m = __ballot(base + x > (int)blockIdx.x);
      if (m) {
        const int j = __ffsll((unsigned long long)m) - 1;
        b = c + j;
        const int k = (int)blockIdx.x - base - (__shfl(x, j) - __shfl(n, j));
        r0 = __shfl(s, j) + k * run;
        r1 = min(r0 + run, __shfl(e, j));
        qp = __shfl(qpi, j); aq = __shfl(aqi, j); akv = __shfl(kvi, j);
      }
      base += __shfl(x, 63);
    }
  }
  if (b < 0) return;
  b = __builtin_amdgcn_readfirstlane(b);
  r0 = __builtin_amdgcn_readfirstlane(r0);
  r1 = __builtin_amdgcn_readfirstlane(r1);
  qp = __builtin_amdgcn_readfirstlane(qp);
  aq = __builtin_amdgcn_readfirstlane(aq);
  akv = __builtin_amdgcn_readfirstlane(akv);
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
  // 16 heads x PT tiles staged, then stored as whole runs of a head's row
  auto store_zero = [&](int t, int hg) {
    uint4* o = reinterpret_cast<uint4*>(p.out + ((size_t)t * p.H + hg * 16) * kDV * 2);
#pragma unroll
    for (int i = 0; i < 16 * kDV * 2 / 16 / 64; ++i) o[i * 64 + lane] = make_uint4(0, 0, 0, 0);
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
        store_zero(t, hg);
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
      float l = 0.f;
      uint32_t pk[8][2];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { s[i][j] = __builtin_amdgcn_exp2f(s[i][j] - m); l += s[i][j]; }
        pk[i][0] = pack2<QT>(s[i][0], s[i][1]);
        pk[i][1] = pack2<QT>(s[i][2], s[i][3]);
      }
      l = rows_sum(l) + __builtin_amdgcn_exp2f(sink2 - m);
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
      const float inv = 1.f / l;
      uint8_t* sb = stage[wave];
      uint8_t* ob = p.out + ((size_t)t * p.H + hg * 16) * kDV * 2;
#pragma unroll
      for (int c = 0; c < NT; c += C::PT) {
#pragma unroll
        for (int i = 0; i < C::PT; ++i)
          *reinterpret_cast<uint2*>(sb + c16 * C::SRB + (i * 16 + 4 * g) * 2) =
              make_uint2(pack2<QT>(acc[c + i][0] * inv, acc[c + i][1] * inv), pack2<QT>(acc[c + i][2] * inv, acc[c + i][3] * inv));
        constexpr int CPR = C::PT * 2;                     // 16-byte chunks per staged row
#pragma unroll
        for (int i = 0; i < 16 * CPR / 64 + (16 * CPR % 64 != 0); ++i) {
          const int e = i * 64 + lane, r = e / CPR, k = e - r * CPR;
          typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
          const u32x4 w = *reinterpret_cast<const u32x4*>(sb + r * C::SRB + k * 16);
          __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(ob + (size_t)r * kDV * 2 + c * 32 + k * 16));
        }
      }
      if (g == 0) lse[c16] = m * kLn2 + logf(l);
    }
  }
}

template <int D, typename QT>
int launch(const FwdParams& fp, int run, hipStream_t st) {
  const int nb = fp.T / run + fp.B;
  hipLaunchKernelGGL((sas_fwd_win_kernel<D, QT>), dim3(nb), dim3(256), 0, st, fp, run);
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
