// sparse_attn_sharedkv backward for prefills on MI355X (gfx950): two kernels
// without per-(token, row) atomics.
//
//  sas_bwd_dq_kernel    token-major: dq and Delta of one token and head group
//                       (the forward's key set; no row gradients);
//  sas_bwd_keys_kernel  key-major: a tile of 64 cache rows stays with its
//                       workgroup, which streams the tokens of one segment
//                       that attend any of them and sums the rows' gradients
//                       in registers; one fp32 add per (row, channel,
//                       segment, 32-head group) at the end.
//
// Per-token row-gradient adds cost one fp32 atomic per (token, row, 64-head
// group, channel), and the device executes ~325 G of them a second: 1.77 ns
// per (token, row) pair and 64 heads at D = 576, whatever the MFMA work. The
// key-major pass costs MFMA work for every (token, row) pair of its tiles,
// selected or not. Window rows are keys of consecutive tokens, and the
// compressed rows below a token's causal threshold are all keys (dense
// compressed) or up to K of them (top-k); a token's membership in the tile
// comes from its index list, counted into LDS.
//
// Forward + backward of a 4096-token, 64-head, top-k 512 step: 4.35 ms with
// per-token adds (the window rows key-major beside them), 2.12 ms here (dq
// 0.78, rows 1.11 ms); the backward of 2726 packed tokens with 128 heads 2.61
// against 1.21 ms.

#include "sas_bwd.h"

namespace sas {
namespace {

// ---------------------------------------------------------------------------
// dq, token-major
// ---------------------------------------------------------------------------
//
// 2 NG waves, wave w = 2 g + hh: 16-head group g, channel half hh. Q^T and
// dO^T of the group live in registers for the wave's half of the k-steps, so
// each K fragment read from LDS feeds the S and the dP MFMA. Rows stream in
// chunks of 32 (one 16x16x32 MFMA per dq tile; 16-row chunks take the K = 16
// MFMA at half the rate) through two LDS slots by LDS-DMA. Per chunk: S^T and
// dP^T over the wave's channels, the pair adds the halves through LDS (own +
// other: the same bits in both, and in sas_bwd64_kernel), dS^T packed in registers is the B operand of
// dq^T[channel x head] += K^T . dS^T, K^T by transposed reads of the row tile.
template <int D, typename QT, int NG>
__global__ void __launch_bounds__(128 * NG) sas_bwd_dq_kernel(const BwdParams bp) {
  constexpr int NW = 2 * NG, NT = 64 * NW, TR = 32;
  constexpr int CH = D / 8;                   // 16-byte chunks per row
  constexpr int KSH = D / 64;                 // S k-steps per channel half
  constexpr int VSH = kDV / 64;               // dP k-steps per channel half
  constexpr int DQT = D / 32;                 // dq tiles per wave
  constexpr int RI = CH / 8;                  // DMA instructions per 8 rows (9 or 8)
  constexpr int NP = 8 / NW;                  // of which a wave takes NP in each 8 rows
  constexpr int OPS = 4 * NP + (RI == 9);     // and waves 0-3 one of the left-over ones
  constexpr int SG = kSwzGroup<CH>;
  constexpr int kRing = 2 * TR * CH;          // chunks
  constexpr int kX = NW * 4 * 64;             // exchange chunks
  constexpr int SRB = DQT * 16 * 2 + 16;      // staged dq row bytes
  static_assert(NW * 16 * SRB <= (kRing + kX) * 16, "dq staging fits");
  static_assert(2 * TR <= kRowPad, "a chunk past the last stays in the padded row list");
  __shared__ __attribute__((aligned(16))) uint4 lds_b[kRing + kX];
  __shared__ float lds_dl[16 * NG];

  const FwdParams& p = bp.f;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int item = item_index(p);
  if (item < 0) return;
  Tok k = item_of(p, item);
  const int g = wave >> 1, hh = wave & 1, c16 = lane & 15, g4 = lane >> 4;
  const int t = k.t, h = k.hg * 16 * NG + 16 * g + c16;
  const size_t th = (size_t)t * p.H + h;

  // Delta = dO . O: 8 threads per head, 64 channels each
  {
    const int hd = tid >> 3, part = tid & 7;
    const size_t at = ((size_t)t * p.H + k.hg * 16 * NG + hd) * kDV * 2 + part * 128;
    const uint32_t* dog = reinterpret_cast<const uint32_t*>(bp.dout + at);
    const uint32_t* og = reinterpret_cast<const uint32_t*>(bp.out + at);
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) d = dot2<QT>(dog[i], og[i], d);
    d += __shfl_xor(d, 1);
    d += __shfl_xor(d, 2);
    d += __shfl_xor(d, 4);
    if (part == 0) lds_dl[hd] = d;
  }
  uint4 qf[KSH], of[VSH];
  {
    const uint4* qg = reinterpret_cast<const uint4*>(p.q + th * D * 2);
    const uint4* dg = reinterpret_cast<const uint4*>(bp.dout + th * kDV * 2);
#pragma unroll
    for (int ks = 0; ks < KSH; ++ks) qf[ks] = qg[(hh * KSH + ks) * 4 + g4];
#pragma unroll
    for (int ks = 0; ks < VSH; ++ks) of[ks] = dg[(hh * VSH + ks) * 4 + g4];
  }
  const float lse2 = p.lse[th] * kLog2e;
  float dl = 0.f;
  // the token's non-finite marks: q (0 times it) or dO (Delta). Stored last: the
  // chunk loop's first wait would include it
  auto mark = [&] {
    float z[2] = {dl, 0.f};
#pragma unroll
    for (int ks = 0; ks < KSH; ++ks)
      z[ks & 1] = dot2<QT>(qf[ks].w, 0, dot2<QT>(qf[ks].z, 0, dot2<QT>(qf[ks].y, 0, dot2<QT>(qf[ks].x, 0, z[ks & 1]))));
    const bool nf = __ballot(!(fabsf(z[0] + z[1]) < INFINITY)) != 0;
    if (lane == 0) bp.nonfinite[(size_t)t * (p.H / 8) + (k.hg * NG + g) * 2 + hh] = nf;
  };

  f32x4 acc[DQT];
#pragma unroll
  for (int j = 0; j < DQT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float scale = p.scale_log2 / kLog2e;
  const int ksw = swz<CH>(c16);
  // transposed reads: dq tile j at voff[j % TPG], whole swizzle groups apart
  constexpr int TPG = SG / 2;
  const int vr = 4 * g4 + (c16 >> 2), vsw = swz<CH>(vr), vb = (c16 & 3) >> 1;
  int voff[TPG];
#pragma unroll
  for (int q = 0; q < TPG; ++q) {
    const int L = 2 * (hh * DQT + q) + vb;
    voff[q] = (vr * CH + ((L & -SG) | ((L & (SG - 1)) ^ vsw))) * 16 + (c16 & 1) * 8;
  }
  // DMA: a chunk's layout repeats every 8 rows (RI instructions); the wave's
  // lanes keep one (row, column) per instruction it takes of them
  int prow[NP + 1];
  uint32_t pcol[NP + 1];
#pragma unroll
  for (int i = 0; i <= NP; ++i) {
    const int P = (i < NP ? wave + NW * i : 8) * 64 + lane, r = P / CH;
    prow[i] = r;
    pcol[i] = (uint32_t)((P - r * CH) ^ swz<CH>(r)) * 16;
  }

  for (int pass = 0; pass < bp.npass; ++pass) {
    k.sp = pass;
    resolve<256, D * 2>(p, k, tid, lane, wave, [] {});
    if (pass == 0) {
      dl = lds_dl[16 * g + c16];   // behind resolve()'s barriers
      if (k.thr > bp.dense_thr) {         // the per-token kernel's token
        mark();
        return;
      }
      if (hh == 0 && g4 == 0) bp.delta[th] = k.padded ? 0.f : dl;
    }
    const int nvalid = __builtin_amdgcn_readfirstlane(k.nvalid);
    if (nvalid == 0) continue;
    if (tid < kRowPad) lds_rows[nvalid + tid] = lds_rows[nvalid - 1];
    __syncthreads();
    // chunk c's DMA instruction o, from row address ra (chunk nch reads the
    // padding: the last row again); the next instruction's address is read
    // behind it
    auto row_addr = [&](int c, int o) {
      const uint32_t rb = __builtin_amdgcn_readfirstlane(lds_addr_of(lds_rows + c * TR));
      const int j = o < 4 * NP ? o & 3 : wave & 3;   // 8-row group
      return *reinterpret_cast<const LDS_AS uint64_t*>((size_t)(rb + 8u * (uint32_t)(prow[o >> 2] + 8 * j)));
    };
    uint64_t ra;
    auto dma_fire = [&](int c, int o) {
      if (o == 4 * NP && wave >= 4) return;   // wave-uniform
      const int j = o < 4 * NP ? o & 3 : wave & 3, m = o < 4 * NP ? wave + NW * (o >> 2) : 8;
      dma16(reinterpret_cast<const void*>(ra + pcol[o >> 2]),
            __builtin_amdgcn_readfirstlane(lds_addr_of(lds_b + (c & 1) * TR * CH) + (j * RI + m) * 1024));
      if (o + 1 < OPS) ra = row_addr(c, o + 1);
    };
    const int nch = (nvalid + TR - 1) / TR;
    ra = row_addr(0, 0);
#pragma unroll
    for (int o = 0; o < OPS; ++o) dma_fire(0, o);
    for (int c = 0; c < nch; ++c) {
      const int nr = nvalid - c * TR;
      const uint4* kt = lds_b + (c & 1) * TR * CH;
      __builtin_amdgcn_s_waitcnt(0);   // known to the compiler: no wait of its own behind the DMA
      __builtin_amdgcn_s_barrier();
      ra = row_addr(c + 1, 0);
      // S^T and dP^T of the chunk's two 16-row tiles over this wave's channels
      f32x4 s[2], dp[2];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) { s[mt] = f32x4{0.f, 0.f, 0.f, 0.f}; dp[mt] = s[mt]; }
      // channel half HH: fragments HH VSH + i; S takes k-steps HH KSH ..,
      // which start OFF fragments later
      auto half = [&](auto HHC) __attribute__((always_inline)) {
        constexpr int HH = decltype(HHC)::value, OFF = HH * (KSH - VSH), NF = KSH + OFF, PF = 3;
        auto kfrag = [&](int i, int mt) {
          const int L = 4 * (HH * VSH + i) + g4;
          return kt[(mt * 16 + c16) * CH + ((L & -SG) | ((L & (SG - 1)) ^ ksw))];
        };
        uint4 a[PF][2];
#pragma unroll
        for (int i = 0; i < PF; ++i)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) a[i][mt] = kfrag(i, mt);
#pragma unroll
        for (int i = 0; i < NF; ++i) {
          const uint4 a0 = a[i % PF][0], a1 = a[i % PF][1];
          if (i + PF < NF) { a[i % PF][0] = kfrag(i + PF, 0); a[i % PF][1] = kfrag(i + PF, 1); }
          if (i >= OFF) {
            s[0] = mfma32k<QT>(a0, qf[i - OFF], s[0]);
            s[1] = mfma32k<QT>(a1, qf[i - OFF], s[1]);
          }
          if (i < VSH) {
            dp[0] = mfma32k<QT>(a0, of[i], dp[0]);
            dp[1] = mfma32k<QT>(a1, of[i], dp[1]);
          }
          // the next chunk's DMA between the MFMAs (see sas_bwd_keys_kernel)
          constexpr int EV = OPS > 5 ? 1 : 2;
          if (i % EV == EV - 1 && i / EV < OPS) dma_fire(c + 1, i / EV);
        }
#pragma unroll
        for (int o = NF / (OPS > 5 ? 1 : 2); o < OPS; ++o) dma_fire(c + 1, o);
      };
      if (hh) half(std::integral_constant<int, 1>{});
      else half(std::integral_constant<int, 0>{});
      f32x4* x = reinterpret_cast<f32x4*>(lds_b + kRing);
      x[(wave * 4 + 0) * 64 + lane] = s[0];
      x[(wave * 4 + 1) * 64 + lane] = s[1];
      x[(wave * 4 + 2) * 64 + lane] = dp[0];
      x[(wave * 4 + 3) * 64 + lane] = dp[1];
      lds_barrier();
      uint32_t pk[4];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        s[mt] += x[((wave ^ 1) * 4 + mt) * 64 + lane];
        dp[mt] += x[((wave ^ 1) * 4 + 2 + mt) * 64 + lane];
        float ds[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pr = __builtin_amdgcn_exp2f(s[mt][i] * p.scale_log2 - lse2);
          ds[i] = mt * 16 + 4 * g4 + i < nr ? pr * (dp[mt][i] - dl) * scale : 0.f;
        }
        pk[2 * mt] = pack2<QT>(ds[0], ds[1]);
        pk[2 * mt + 1] = pack2<QT>(ds[2], ds[3]);
      }
      const uint4 bds = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      // dq^T: A = K^T of keys 4 g4 .. + 3 and 16 + 4 g4 .. + 3, the order of bds
      auto vfrag = [&](int j) {
        const char* b0 = reinterpret_cast<const char*>(kt) + voff[j % TPG] + (j / TPG) * SG * 16;
        const uint2 u0 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0)));
        const uint2 u1 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0 + 16 * CH * 16)));
        return make_uint4(u0.x, u0.y, u1.x, u1.y);
      };
      constexpr int PV = 4;
      uint4 v[PV];
#pragma unroll
      for (int j = 0; j < PV; ++j) v[j] = vfrag(j);
#pragma unroll
      for (int j = 0; j < DQT; ++j) {
        const uint4 a = v[j % PV];
        if (j + PV < DQT) v[j % PV] = vfrag(j + PV);
        acc[j] = mfma32k<QT>(a, bds, acc[j]);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * PV, 2);
#pragma unroll
      for (int j = 0; j < DQT; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 2);
        if (j + PV < DQT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 2);
      }
    }
    wait_vm<0>();      // the spare chunk's DMA
    __syncthreads();   // the row list and the slots are free
  }
  // lane (g4, c16): channels 16 ct + 4 g4 .. + 3 of head c16
  if (bp.dq_direct) {
    // staged in LDS so a store covers whole runs of a head's row
    uint8_t* sb = reinterpret_cast<uint8_t*>(lds_b) + wave * 16 * SRB;
#pragma unroll
    for (int j = 0; j < DQT; ++j)
      *reinterpret_cast<uint2*>(sb + c16 * SRB + (j * 16 + 4 * g4) * 2) =
          make_uint2(pack2<QT>(acc[j][0], acc[j][1]), pack2<QT>(acc[j][2], acc[j][3]));
    uint8_t* dst = reinterpret_cast<uint8_t*>(bp.dq) + (((size_t)t * p.H + k.hg * 16 * NG + 16 * g) * D + hh * DQT * 16) * 2;
    constexpr int CPR = DQT * 2;   // 16-byte chunks per staged row
#pragma unroll
    for (int i = 0; i < 16 * CPR / 64; ++i) {
      const int q = i * 64 + lane, r = q / CPR, c = q - r * CPR;
      *reinterpret_cast<uint4*>(dst + (size_t)r * D * 2 + c * 16) = *reinterpret_cast<const uint4*>(sb + r * SRB + c * 16);
    }
  } else if (!k.padded) {
    float* dst = bp.dq + th * D + hh * DQT * 16 + 4 * g4;
#pragma unroll
    for (int j = 0; j < DQT; ++j) *reinterpret_cast<f32x4*>(dst + j * 16) = acc[j];
  }
  mark();
}

// ---------------------------------------------------------------------------
// row gradients, key-major
// ---------------------------------------------------------------------------
//
// Workgroup = (segment of key_seg consecutive tokens of one batch, 32-head
// group, tile of 64 window or compressed rows), 8 waves. Its unit is one token
// (32 heads): q and dO reach LDS by DMA (two buffers, 139 KB), then
//   S[head][row] = Q . K^T and dP = dO . V^T   (16x16x32 MFMA; wave w: rows
//     16 (w & 3) .., heads 16 (w >> 2) ..; K in registers for the whole
//     segment), P and dS, masked and rounded to the query dtype, to an LDS
//     table [row][head];
//   dkv[row][ch] += dS^T . Q + P^T . dO        (16x16x32 MFMA over the unit's
//     32 heads; wave w: V channel tiles w, w + 8, w + 16, w + 24 for all four
//     row tiles, and a share of the rope tiles; q / dO by transposed reads).
// Every q / dO element is read from LDS by four waves for S and by one for
// dkv. All tiles of a (segment, head group) run on one XCD next to each
// other, so the tokens' q / dO stream through its L2 once.
//
// A unit's products run over every row of the tile, those the token does not
// attend with P = dS = 0. A NaN or Inf in q or dO would reach them as 0 x Inf:
// in a segment that holds one (by sas_bwd_dq_kernel's marks) such elements are
// cleared in LDS before the dkv products, and the rows the token does attend
// get their NaN through P and dS alone. The marks take 0.8 % of the 4096-token
// step (looked for unit by unit instead, in S and dP: 1.5 %).
template <typename QT>
__device__ __forceinline__ uint32_t finite2(uint32_t w) {   // two packed values, non-finite ones as 0
  constexpr uint32_t E = std::is_same<QT, __bf16>::value ? 0x7f80u : 0x7c00u;   // exponent all ones
  if ((w & E) == E) w &= 0xffff0000u;
  if ((w >> 16 & E) == E) w &= 0xffffu;
  return w;
}

template <int D, typename QT>
__global__ void __launch_bounds__(512) sas_bwd_keys_kernel(const BwdParams bp) {
  constexpr int CH = D / 8, OCH = kDV / 8;     // 16-byte chunks per q / dO row
  constexpr int KS = D / 32, VS = kDV / 32;
  static_assert(CH % 8 == 0 && (CH / 8 == 8 || CH / 8 == 9), "q DMA split");
  constexpr int SGQ = kSwzGroup<CH>, SGO = kSwzGroup<OCH>;
  constexpr int TS = 80;                       // table row bytes: 32 heads + 16
  constexpr bool ROPE = D > kDV;
  constexpr int kIdx = 4;                      // index registers: top-k lists up to 2048 entries
  __shared__ __attribute__((aligned(16))) uint4 lds_q[2][32 * CH];
  __shared__ __attribute__((aligned(16))) uint4 lds_o[2][32 * OCH];
  __shared__ __attribute__((aligned(16))) uint8_t lds_t[2][kKeyRows * TS];   // dS, P
  __shared__ __attribute__((aligned(16))) float lds_h[2][2][32];             // per buffer: lse (log2 units), Delta
  __shared__ int lds_c[2][kKeyRows];           // per buffer: how often the token lists each row
  __shared__ uint64_t lds_r[kKeyRows];         // row addresses (0: invalid row)

  const FwdParams& p = bp.f;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int c16 = lane & 15, g4 = lane >> 4;
  const int nhg = p.H / 32, ntile = bp.cmp_tiles + bp.win_tiles_seg;
  // (batch, segment) group gi on XCD (gi nhg + hg) % nxcd, its tiles adjacent there
  const unsigned nx = (unsigned)p.nxcd;
  const int x = (int)(blockIdx.x % nx), l = (int)(blockIdx.x / nx);
  const int gh = (l / ntile) * p.nxcd + x, tile = l % ntile;
  const int gi = gh / nhg, hg = gh - gi * nhg, h0 = hg * 32;
  if (gi >= bp.seg_groups) return;
  // group -> (batch, segment): scan of the batches' segment counts (a token
  // belongs to the last batch that starts at or before it, as in resolve())
  const bool cu = p.act_q == nullptr;
  int b = -1, seg = 0, qp = 0, aq = 0, aqe = 0, akv = 0;
  {
    int base = 0;
    for (int c = 0; c < p.B && b < 0; c += 64) {
      const int i = c + lane;
      int qpi = 0, aqi = 0, ae = 0, kvi = 0;
      if (i < p.B) {
        qpi = p.q_prefix[i];
        const int nxt = i + 1 < p.B ? p.q_prefix[i + 1] : p.T;
        aqi = cu ? p.q_prefix[i + 1] - qpi : p.act_q[i];
        kvi = p.act_kv[i];
        ae = qpi < 0 ? 0 : max(0, min(aqi, min(nxt, p.T) - qpi));
      }
      const int n = (ae + bp.key_seg - 1) / bp.key_seg;
      int s = n;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) { const int v = __shfl_up(s, d); s += lane >= d ? v : 0; }
      const uint64_t m = __ballot(base + s > gi);
      if (m) {
        const int j = __ffsll((unsigned long long)m) - 1;
        b = c + j;
        seg = gi - base - (__shfl(s, j) - __shfl(n, j));
        qp = __shfl(qpi, j); aq = __shfl(aqi, j); aqe = __shfl(ae, j); akv = __shfl(kvi, j);
      }
      base += __shfl(s, 63);
    }
  }
  if (b < 0) return;
  b = __builtin_amdgcn_readfirstlane(b);
  seg = __builtin_amdgcn_readfirstlane(seg);
  qp = __builtin_amdgcn_readfirstlane(qp);
  aq = __builtin_amdgcn_readfirstlane(aq);
  aqe = __builtin_amdgcn_readfirstlane(aqe);
  akv = __builtin_amdgcn_readfirstlane(akv);
  const int sg0 = akv - aq;                     // causal position of the batch's first token
  // token offsets [a0, a1) of the segment in the batch
  int a0 = seg * bp.key_seg, a1 = min(a0 + bp.key_seg, aqe);
  if (a0 + sg0 < 0) a0 = min(a1, -sg0);         // tokens before position 0 attend no row
  const bool cmp = tile < bp.cmp_tiles;
  int p0;                                       // the tile's first position
  if (cmp) {
    p0 = tile * kKeyRows;
    // thr = (sg + 1) / ratio in (p0, dense_thr]
    const long long lo = ((long long)p0 + 1) * p.cmp_ratio - 1 - sg0;
    const long long hi = ((long long)bp.dense_thr + 1) * p.cmp_ratio - 1 - sg0;
    if (lo > a0) a0 = (int)min(lo, (long long)a1);
    if (hi < a1) a1 = (int)max(hi, (long long)a0);
    if (p.scenario == SAS_CFA && p0 >= p.K) return;
  } else {
    const int first = max(0, sg0 + a0 - p.win_left) / kKeyRows;
    p0 = (first + tile - bp.cmp_tiles) * kKeyRows;
    // sg in [p0, p0 + 63 + win_left]
    a0 = max(a0, p0 - sg0);
    a1 = (int)min((long long)a1, (long long)p0 + kKeyRows + p.win_left - sg0);
  }
  if (a0 >= a1) return;   // uniform

  const int32_t* bt = (cmp ? p.cmp_bt + (size_t)b * p.cmp_bt_stride : p.ori_bt + (size_t)b * p.ori_bt_stride);
  if (tid < kKeyRows) {
    const int bs = cmp ? p.cmp_bs : p.ori_bs, pos = p0 + tid, blk = pos / bs;
    uint64_t a = 0;
    if (blk < (cmp ? p.cmp_bt_stride : p.ori_bt_stride)) {
      const int phys = bt[blk];
      if (phys >= 0 && phys < (cmp ? p.cmp_nblocks : p.ori_nblocks))
        a = reinterpret_cast<uint64_t>(cmp ? p.cmp_kv : p.ori_kv) + (uint64_t)(uint32_t)(phys * bs + pos - blk * bs) * (D * 2);
    }
    lds_r[tid] = a;
    lds_c[0][tid] = 0;
    lds_c[1][tid] = 0;
  }
  // (a segment has fewer tokens than the workgroup threads)
  const bool nf = __syncthreads_or(
      tid < a1 - a0 && reinterpret_cast<const uint32_t*>(bp.nonfinite)[((size_t)qp + a0 + tid) * nhg + hg] != 0);
  const int rt = wave & 3, ht = wave >> 2;
  uint4 kf[KS];
  const uint64_t ra = lds_r[16 * rt + c16];
  const bool rok = ra != 0;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kf[ks] = rok ? gld16(ra + (32 * ks + 8 * g4) * 2) : make_uint4(0, 0, 0, 0);

  // A unit's (lse, Delta) and top-k entries are loaded two units ahead into
  // registers and put into LDS one unit ahead; its q and dO one unit ahead by
  // DMA.
  const bool list = cmp && p.scenario == SAS_SCFA;
  const int nidx = list ? (p.K + 511) >> 9 : 0;   // entries per thread
  const bool list_reg = nidx <= kIdx;
  float hv = 0.f;
  int iv[kIdx];
#pragma unroll
  for (int i = 0; i < kIdx; ++i) iv[i] = -1;
  auto load_small = [&](int a) {
    const size_t t = (size_t)qp + a;
    if (wave == 0) hv = (lane < 32 ? p.lse : bp.delta)[t * p.H + h0 + (lane & 31)];
    if (list_reg) {
      const int32_t* ix = p.cmp_idx + t * p.K;
#pragma unroll
      for (int i = 0; i < kIdx; ++i) {
        if (i >= nidx) break;   // uniform
        iv[i] = ix[min(i * 512 + tid, p.K - 1)];
      }
    }
  };
  auto put_small = [&](int a, int buf) {
    if (wave == 0) lds_h[buf][lane >> 5][lane & 31] = lane < 32 ? hv * kLog2e : hv;
    if (list) {
      const unsigned top = (unsigned)min((sg0 + a + 1) / p.cmp_ratio - p0, kKeyRows);   // >= 1: rows below the threshold
      if (list_reg) {
#pragma unroll
        for (int i = 0; i < kIdx; ++i) {
          if (i >= nidx) break;   // uniform
          const unsigned r = (unsigned)(iv[i] - p0);
          if (r < top && i * 512 + tid < p.K) atomicAdd(&lds_c[buf][r], 1);
        }
      } else {
        for (int i = tid; i < p.K; i += 512) {
          const unsigned r = (unsigned)(p.cmp_idx[((size_t)qp + a) * p.K + i] - p0);
          if (r < top) atomicAdd(&lds_c[buf][r], 1);
        }
      }
    }
  };
  // DMA: the q tile repeats its swizzle every 8 rows (RI instructions), the dO
  // tile's rows are one instruction each, so a wave takes instructions RI
  // apart (8 apart for dO) and its lanes keep one offset for all of them; the
  // q instructions that are left over (D = 576: RI = 9) go to waves 0-3.
  constexpr int RI = CH / 8;
  const int Pq = wave * 64 + lane, rq = Pq / CH, Px = 8 * 64 + lane, rx = Px / CH;
  const uint32_t oq = (uint32_t)(rq * CH + ((Pq - rq * CH) ^ swz<CH>(rq))) * 16;
  const uint32_t ox = (uint32_t)(rx * CH + ((Px - rx * CH) ^ swz<CH>(rx))) * 16;
  const uint32_t oo = (uint32_t)(wave * OCH + (lane ^ swz<OCH>(wave))) * 16;
  auto dma = [&](int a, int buf, int i) {   // instruction i < 9 of the wave
    const size_t t = (size_t)qp + a;
    const uint8_t* qs = p.q + (t * p.H + h0) * D * 2;
    const uint8_t* os = bp.dout + (t * p.H + h0) * kDV * 2;
    const uint32_t qb = lds_addr_of(lds_q[buf]) + wave * 1024, ob = lds_addr_of(lds_o[buf]) + wave * 1024;
    const int j = i >> 1;
    if (i < 8 && !(i & 1)) dma16s(oq, qs + j * 8 * D * 2, __builtin_amdgcn_readfirstlane(qb + j * RI * 1024));
    if (i < 8 && (i & 1)) dma16s(oo, os + j * 8 * kDV * 2, __builtin_amdgcn_readfirstlane(ob + j * 8 * 1024));
    if (i == 8 && RI == 9 && wave < 4)
      dma16s(ox, qs + wave * 8 * D * 2, __builtin_amdgcn_readfirstlane(lds_addr_of(lds_q[buf]) + (8 + 9 * wave) * 1024));
  };

  f32x4 acc[4][4], accr[2];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[m][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  accr[0] = accr[1] = acc[0][0];
  const float scale = p.scale_log2 / kLog2e;
  const int qsw = swz<CH>(c16), osw = swz<OCH>(c16);
  const int vr = 4 * g4 + (c16 >> 2), vqs = swz<CH>(vr), vos = swz<OCH>(vr), vb = (c16 & 3) >> 1;
  // transposed read of channel tile ct0 + 8 m (tiles 8 apart are whole swizzle
  // groups apart)
  auto trbase = [&](auto RC, int vsw, int ct0) {
    constexpr int rc = decltype(RC)::value, SG = kSwzGroup<rc>;
    const int L = 2 * ct0 + vb;
    return (vr * rc + ((L & -SG) | ((L & (SG - 1)) ^ vsw))) * 16 + (c16 & 1) * 8;
  };
  auto trfrag = [&](const uint4* base, auto RC, int off) {
    constexpr int rc = decltype(RC)::value;
    const char* b0 = reinterpret_cast<const char*>(base) + off;
    const uint2 u0 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0)));
    const uint2 u1 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS i16x4*)(b0 + 16 * rc * 16)));
    return make_uint4(u0.x, u0.y, u1.x, u1.y);
  };
  const std::integral_constant<int, CH> QC;
  const std::integral_constant<int, OCH> OC;
  const int tq0 = trbase(QC, vqs, wave), to0 = trbase(OC, vos, wave), tr0 = trbase(QC, vqs, kDV / 16 + (wave & 3));

  load_small(a0);
  put_small(a0, 0);
  load_small(min(a0 + 1, a1 - 1));
#pragma unroll
  for (int i = 0; i < 9; ++i) dma(a0, 0, i);
  for (int a = a0; a < a1; ++a) {
    const int buf = (a - a0) & 1;
    // the builtin, not asm: every load the compiler tracks (the rows, the
    // unit's small loads) is then known to be done, and it adds no wait of
    // its own behind the DMA issued below
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    // (past the last unit it is staged again, into the spare buffer)
    const int an = min(a + 1, a1 - 1);
    const uint4* tq = lds_q[buf];
    const uint4* to = lds_o[buf];
    {
      auto qfrag = [&](int ks) {
        const int L = 4 * ks + g4;
        return tq[(16 * ht + c16) * CH + ((L & -SGQ) | ((L & (SGQ - 1)) ^ qsw))];
      };
      auto ofrag = [&](int ks) {
        const int L = 4 * ks + g4;
        return to[(16 * ht + c16) * OCH + ((L & -SGO) | ((L & (SGO - 1)) ^ osw))];
      };
      const f32x4 l2 = *reinterpret_cast<const f32x4*>(&lds_h[buf][0][16 * ht + 4 * g4]);
      const f32x4 dl = *reinterpret_cast<const f32x4*>(&lds_h[buf][1][16 * ht + 4 * g4]);
      const int cnt = lds_c[buf][16 * rt + c16];
      f32x4 sc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}, dc[2] = {sc[0], sc[0]};
      // two chains, one per channel half, as the wave pairs of the per-token
      // kernels sum them: the same bits
      constexpr int PF = 4;
      auto kq = [](int i) { return (i & 1) * (KS / 2) + i / 2; };
      auto ko = [](int i) { return (i & 1) * (VS / 2) + i / 2; };
      uint4 qa[PF], oa[PF];
#pragma unroll
      for (int i = 0; i < PF; ++i) { qa[i] = qfrag(kq(i)); oa[i] = ofrag(ko(i)); }
      put_small(an, buf ^ 1);
      load_small(min(a + 2, a1 - 1));
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const uint4 qv = qa[i % PF];
        if (i + PF < KS) qa[i % PF] = qfrag(kq(i + PF));
        sc[i & 1] = mfma32k<QT>(qv, kf[kq(i)], sc[i & 1]);
        if (i < VS) {
          const uint4 ov = oa[i % PF];
          if (i + PF < VS) oa[i % PF] = ofrag(ko(i + PF));
          dc[i & 1] = mfma32k<QT>(ov, kf[ko(i)], dc[i & 1]);
        }
        // the next unit's DMA, an instruction every few MFMAs: issued at once
        // they fill the CU's memory pipeline and hold every wave ahead of its
        // MFMAs (unit 6100 clk against 4900; in the dkv phase instead they
        // land too late). The asm also keeps the reads PF fragments ahead,
        // where the scheduler would sink each one to its MFMA.
        if (i % 2 == 1) dma(an, buf ^ 1, i / 2);
      }
      const f32x4 s_ = sc[0] + sc[1], d_ = dc[0] + dc[1];
      // lane (g4, c16): heads 16 ht + 4 g4 .. + 3 of row 16 rt + c16
      const int pos = p0 + 16 * rt + c16, sg = sg0 + a;
      int n = cnt;
      if (list) {}
      else if (cmp) n = pos < (sg + 1) / p.cmp_ratio && pos < p.K;
      else n = pos <= sg && pos >= sg - p.win_left;
      if (!rok) n = 0;
      float pr[4], ds[4];
      const float w = (float)n;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[i] = n ? w * __builtin_amdgcn_exp2f(s_[i] * p.scale_log2 - l2[i]) : 0.f;
        ds[i] = n ? pr[i] * (d_[i] - dl[i]) * scale : 0.f;
      }
      // table position of head 16 ht + 4 g4 + i: 8 g4 + 4 ht + i, the k order
      // of the transposed q / dO reads
      const int to_ = (16 * rt + c16) * TS + (8 * g4 + 4 * ht) * 2;
      *reinterpret_cast<uint2*>(lds_t[0] + to_) = make_uint2(pack2<QT>(ds[0], ds[1]), pack2<QT>(ds[2], ds[3]));
      *reinterpret_cast<uint2*>(lds_t[1] + to_) = make_uint2(pack2<QT>(pr[0], pr[1]), pack2<QT>(pr[2], pr[3]));
    }
    lds_barrier();
    if (list && tid < kKeyRows) lds_c[buf][tid] = 0;
    if (nf) {
      auto clear = [&](uint4* b, int n) {
#pragma unroll 1
        for (int i = tid; i < n; i += 512) {
          const uint4 v = b[i];
          b[i] = make_uint4(finite2<QT>(v.x), finite2<QT>(v.y), finite2<QT>(v.z), finite2<QT>(v.w));
        }
      };
      clear(lds_q[buf], 32 * CH);
      clear(lds_o[buf], 32 * OCH);
      lds_barrier();
    }
    {
      uint4 ads[4], ap[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ads[r] = *reinterpret_cast<const uint4*>(lds_t[0] + (16 * r + c16) * TS + g4 * 16);
        ap[r] = *reinterpret_cast<const uint4*>(lds_t[1] + (16 * r + c16) * TS + g4 * 16);
      }
      uint4 bq = trfrag(tq, QC, tq0), bo = trfrag(to, OC, to0);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint4 nq = bq, no = bo;
        if (m < 3) { nq = trfrag(tq, QC, tq0 + (m + 1) * 256); no = trfrag(to, OC, to0 + (m + 1) * 256); }
        else if (ROPE) nq = trfrag(tq, QC, tr0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] = mfma32k<QT>(ads[r], bq, acc[m][r]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] = mfma32k<QT>(ap[r], bo, acc[m][r]);
        bq = nq; bo = no;
      }
      if constexpr (ROPE) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint4 ar = *reinterpret_cast<const uint4*>(lds_t[0] + (16 * (2 * (wave >> 2) + i) + c16) * TS + g4 * 16);
          accr[i] = mfma32k<QT>(ar, bq, accr[i]);
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 12, 1);
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
          if (m < 3 || ROPE) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        }
      if (ROPE) __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
    }
  }
  wait_vm<0>();   // the spare unit's DMA
  // lane (g4, c16): rows 16 r + 4 g4 + i, channel 16 ct + c16
  const uint64_t lo = reinterpret_cast<uint64_t>(cmp ? p.cmp_kv : p.ori_kv);
  float* db = cmp ? bp.d_cmp : bp.d_ori;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t ad = lds_r[16 * r + 4 * g4 + i];
      if (!ad) continue;
      float* gr = db + (ad - lo) / 2 + c16;
#pragma unroll
      for (int m = 0; m < 4; ++m) atomicAdd(gr + (wave + 8 * m) * 16, acc[m][r][i]);
    }
  if constexpr (ROPE) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint64_t ad = lds_r[16 * (2 * (wave >> 2) + j) + 4 * g4 + i];
        if (ad) atomicAdd(db + (ad - lo) / 2 + kDV + (wave & 3) * 16 + c16, accr[j][i]);
      }
  }
}

// d_sinks[h] -= sum over tokens of exp(sink - lse) Delta: one workgroup per
// 64 heads and token range, one add per head. (One add per token and head
// from the per-token kernel serialises on a few cache lines.)
__global__ void __launch_bounds__(256) sas_bwd_sink_kernel(const BwdParams bp) {
  __shared__ float part[4][64];
  const FwdParams& p = bp.f;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = blockIdx.y * 64 + lane;
  float s = 0.f;
  if (h < p.H) {
    const float sk = p.sinks[h] * kLog2e;
    for (int t0 = (blockIdx.x * 4 + wave) * 4; t0 < p.T; t0 += gridDim.x * 16) {
      float d[4], l[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const size_t a = (size_t)min(t0 + i, p.T - 1) * p.H + h;
        d[i] = bp.delta[a];
        l[i] = p.lse[a] * kLog2e;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) s += t0 + i < p.T && d[i] != 0.f ? __builtin_amdgcn_exp2f(sk - l[i]) * d[i] : 0.f;
    }
  }
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && h < p.H) atomicAdd(bp.d_sinks + h, -(part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane]));
}

template <int D, typename QT>
int launch(const BwdParams& bp, hipStream_t st) {
  const FwdParams& p = bp.f;
  const long long nx = p.nxcd;
  const int nhg = p.H / bwd_dq_heads(p.H);
  BwdParams b = bp;
  b.f.nhg = nhg;
  b.f.nsplit = 1;
  const long long nb = (p.T + nx - 1) / nx * nx * nhg;
  const long long kb = ((long long)bp.seg_groups * (p.H / 32) + nx - 1) / nx * nx * (bp.cmp_tiles + bp.win_tiles_seg);
  if (nb > INT_MAX || kb > INT_MAX) return set_error(SAS_EINVAL, "bwd: %lld workgroups beyond one launch", std::max(nb, kb));
  if (bwd_dq_heads(p.H) == 64) hipLaunchKernelGGL((sas_bwd_dq_kernel<D, QT, 4>), dim3((unsigned)nb), dim3(512), 0, st, b);
  else hipLaunchKernelGGL((sas_bwd_dq_kernel<D, QT, 2>), dim3((unsigned)nb), dim3(256), 0, st, b);
  hipLaunchKernelGGL((sas_bwd_keys_kernel<D, QT>), dim3((unsigned)kb), dim3(512), 0, st, b);
  hipLaunchKernelGGL(sas_bwd_sink_kernel, dim3(std::min(256, (p.T + 15) / 16), (p.H + 63) / 64), dim3(256), 0, st, b);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(SAS_ELAUNCH, "sas_bwd prefill launch: %s", hipGetErrorString(e));
  return SAS_OK;
}

}  // namespace

int launch_bwd_prefill(const BwdParams& bp, int D, int q_dtype, hipStream_t st) {
  if (q_dtype == SAS_DT_BF16) return D == 576 ? launch<576, __bf16>(bp, st) : launch<512, __bf16>(bp, st);
  return D == 576 ? launch<576, _Float16>(bp, st) : launch<512, _Float16>(bp, st);
}

}  // namespace sas
