// fp32 arithmetic path of the multi-LoRA linear: every operand, product and sum in
// IEEE float32 on the gfx950 fp32 matrix core (v_mfma_f32_32x32x2_f32).
//
// This is the reference's `precision='fp32'` mode: the native model runs without
// autocast (training/single_device.py:77-80), so TrainableLowRankLinear sees fp32
// x, W, lora_a, lora_b and computes base(x) + s·F.linear(F.linear(x, A), B) in fp32
// (training/low_rank.py:26-28), and autograd's backward in fp32.
//
//   shrink      h[m, j]  = s_a · Σ_k P[m,k]·Op_a(j,k)          (X·Aᵀ, s·dY·B)
//   gemm_fwd    Y[m, n]  = Σ_k X[m,k]·W[n,k] + b[n] + Σ_j h[m,j]·B_a[n,j]
//   gemm_dx     dX[m, k] = Σ_n dY[m,n]·W[n,k] + Σ_j g[m,j]·A_a[j,k]
//   seg_outer   D_a[c, j] = Σ_{m ∈ rows of a} P[m,c]·H[m,j]      (dB_a, dA_aᵀ)
//
// One tile engine (F32Tile) serves all four: a BM x BN output tile whose contraction
// runs over a fixed, ordered list of (P, Q) sources, so the result is deterministic and
// the LoRA term is more contraction in the same accumulators. An operand is either
// contraction-contiguous (O(r, k) = base[r·ld + k]: X, W in the forward, A) or natural
// (O(r, k) = base[k·ld + r]: W and A in dX, dY / X / h in the reductions); indices outside
// the source read as zero.
//
// gfx950 mapping. An fp32 MFMA (4096 flops, 64 cycles) needs one register per operand,
// so the matrix pipe, not the LDS, sets the pace as long as the loads stay ahead of it.
// Operand tiles of 32 contraction elements (KS of them per step, one per wave group) go
// to a ring of LDS stages with direct-to-LDS loads (16 bytes a lane), one barrier per step.
//   * contraction-contiguous tiles keep 128-byte rows with the chunk swizzle of the bf16
//     kernels: one ds_read_b128 gives a lane the 4 contraction elements of 4 MFMAs (lane
//     half h takes elements 8s + 4h + e of substep s);
//   * natural tiles keep their rows (contraction index k), chunk c of row k at slot
//     c ^ 8·((k / 4) % 2), so that the two lane halves, which read rows 4 apart, use different
//     halves of the 64 banks.
// KS > 1: the waves of a workgroup split the contraction of small output tiles and add their
// sums through LDS in wave order.
// Operands that 16-byte loads cannot take (a pointer, pitch or extent not a multiple of 4
// floats, pitches of 2^21 and more) are loaded element by element through registers into the same
// LDS layout (DIRECT = false).
#include "mlora_common.h"
#include "mlora_host.h"

#include <type_traits>

namespace mlora {

// Pitch (floats) below which direct-to-LDS loads address a whole tile with 31-bit byte offsets.
constexpr int64_t kDirectLd = (int64_t)1 << 21;

// One contraction source. K-contiguous P: rows [p_lo, p_hi) are valid; natural operands:
// columns [0, p_hi) / [0, q_hi). klen contraction elements.
struct F32Src {
  const float *P, *Q;
  int64_t ldp, ldq;
  int32_t p_lo, p_hi, q_hi, klen;
};

template <int TM_, int TN_, int WM_, int WN_, int KS_, bool PN_, bool QN_, bool DIRECT_, int STAGES_>
struct F32Cfg {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, KS = KS_;
  static constexpr bool PN = PN_, QN = QN_, DIRECT = DIRECT_;
  static constexpr int STAGES = DIRECT ? STAGES_ : 2;
  static constexpr int NW = WM * WN * KS, THREADS = 64 * NW;
  static constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
  static constexpr int BK = 32 * KS;  // contraction per step
  // LDS columns of an operand tile (natural tiles: at least 64, so that a row spans the banks)
  static constexpr int PWID = PN && BM < 64 ? 64 : BM, QWID = QN && BN < 64 ? 64 : BN;
  static constexpr int P_SUB = PWID * 128, Q_SUB = QWID * 128;  // bytes of one 32-deep tile
  static constexpr int STAGE_BYTES = KS * (P_SUB + Q_SUB);
  static constexpr int P_BLK = KS * P_SUB / 1024, Q_BLK = KS * Q_SUB / 1024;
  static_assert(P_BLK % NW == 0 && Q_BLK % NW == 0, "whole 1 KB loads per wave");
  static constexpr int P_LPW = P_BLK / NW, Q_LPW = Q_BLK / NW, LPW = P_LPW + Q_LPW;
  static constexpr int RED_BYTES = KS > 1 ? NW * TM * TN * 4096 : 0;
  static constexpr int RING_BYTES = STAGES * STAGE_BYTES;
  static constexpr int LDS_BYTES = RING_BYTES > RED_BYTES ? RING_BYTES : RED_BYTES;
  static_assert(LDS_BYTES <= 163840, "the ring fits the LDS");
  static_assert((STAGES - 2) * LPW < 64, "vmcnt field");
  // The bytes from a tile's first row (or contraction index) to the end of its last: the widest, 256
  // rows of a shrink's operand above rank 128, ends 4080 bytes before kOOB.
  static constexpr int64_t ROWS = BM > BN ? (BM > BK ? BM : BK) : (BN > BK ? BN : BK);
  static_assert(ROWS * 4 * (kDirectLd - 4) < kOOB, "offsets stay in range at any pitch taken");
  static constexpr int WG_PER_CU = 163840 / LDS_BYTES;
  static constexpr int WAVES_PER_SIMD = NW * WG_PER_CU / 4 > 4 ? 4 : (NW * WG_PER_CU + 3) / 4;
};

// Direct-to-LDS loads of one operand tile. NAT: natural; WID: LDS columns; BLK: the first of the
// wave's LPW blocks is `wave`, then every NW-th.
template <bool NAT, int WID, int KS, int NW, int LPW>
struct F32Loader {
  __amdgpu_buffer_rsrc_t rs;
  const float *base;
  int64_t ld;
  int32_t ld_b, r0, r_lo, klen;
  int32_t voff[2], vk[2];  // lane offset (natural: kOOB past the columns); contraction index of the chunk

  __device__ __forceinline__ void init(const float *src, int64_t ld_, int r0_, int lo, int hi, int klen_, int lane) {
    ld = ld_;
    ld_b = (int32_t)(4 * ld_);
    r0 = r0_;
    r_lo = lo;
    klen = klen_;
    if constexpr (NAT) {
      base = src + r0;
      constexpr int CPR = WID / 4;
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        const int c = (lane % CPR) ^ (8 * par);
        voff[par] = r0 + 4 * c < hi ? (lane / CPR) * ld_b + 16 * c : kOOB;
      }
    } else {
      base = src;
      rs = make_rsrc(src + (int64_t)r0 * ld, (int64_t)(hi - r0) * 4 * ld);
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        const int c = (lane & 7) ^ (lane >> 3) ^ par;
        vk[par] = 4 * c;
        voff[par] = (lane >> 3) * ld_b + 16 * c;
      }
    }
  }
  // A step whose rows (from r0 on) and contraction indices are all inside the source: no masks
  // but the lane's own (columns past a natural operand; rows past a K-contiguous one end its
  // resource), and one scalar offset per load.
  __device__ __forceinline__ void issue_plain(MLORA_LDS char *dst, int k0, int wave) const {
    constexpr int SB = WID / 8;
    const __amdgpu_buffer_rsrc_t r = NAT ? make_rsrc(base + (int64_t)k0 * ld, kOOB) : rs;
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int b = i * NW + wave, sub = b / SB, q = b % SB;
      MLORA_LDS void *d = dst + b * 1024;
      constexpr int RPB = NAT ? 256 / WID : 8;
      const bool odd = NAT ? ((RPB * q) >> 2) & 1 : q & 1;
      const int32_t soff = NAT ? (32 * sub + RPB * q) * ld_b : 8 * q * ld_b + (k0 + 32 * sub) * 4;
      const int32_t off = odd ? voff[1] : voff[0];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, d, 16, off, soff, 0, 0);
    }
  }
  __device__ __forceinline__ void issue(MLORA_LDS char *dst, int k0, bool live, int wave, int lane) {
    constexpr int SB = WID / 8;  // blocks of one 32-deep tile
    if constexpr (NAT)           // (re-based per step: a natural operand may exceed 2 GB)
      rs = make_rsrc(base + (int64_t)k0 * ld, live ? (int64_t)(klen - k0) * 4 * ld : 0);
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int b = i * NW + wave;  // wave-uniform
      const int sub = b / SB, q = b % SB;
      MLORA_LDS void *d = dst + b * 1024;
      if constexpr (NAT) {
        constexpr int RPB = 256 / WID;  // contraction rows per load
        const int32_t off = ((RPB * q) >> 2) & 1 ? voff[1] : voff[0];
        const int32_t soff = (32 * sub + RPB * q) * ld_b;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, d, 16, off, soff, 0, 0);
      } else {
        int32_t off = q & 1 ? voff[1] : voff[0];
        const int32_t k = k0 + 32 * sub + (q & 1 ? vk[1] : vk[0]);
        if (r0 + 8 * q + (lane >> 3) < r_lo || k >= klen || !live) off = kOOB;
        const int32_t soff = 8 * q * ld_b + (k0 + 32 * sub) * 4;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, d, 16, off, soff, 0, 0);
      }
    }
  }
};

// The same tile through registers, element by element (any alignment, pitch and extent).
template <bool NAT, int WID, int KS, int THREADS>
struct F32RegLoader {
  static constexpr int E = KS * WID * 32 / THREADS;
  float v[E];
  const float *base;
  int64_t ld;
  int32_t r0, lo, hi, klen;
  __device__ __forceinline__ void init(const float *src, int64_t ld_, int r0_, int lo_, int hi_, int klen_) {
    base = src, ld = ld_, r0 = r0_, lo = lo_, hi = hi_, klen = klen_;
  }
  __device__ __forceinline__ static void coords(int e, int tid, int &sub, int &r, int &k) {
    const int idx = tid + THREADS * e;
    sub = idx / (WID * 32);
    const int rem = idx % (WID * 32);
    if constexpr (NAT) k = rem / WID, r = rem % WID;
    else r = rem / 32, k = rem % 32;
  }
  __device__ __forceinline__ void load(int k0, bool live, int tid) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      int sub, rl, kl;
      coords(e, tid, sub, rl, kl);
      const int r = r0 + rl, k = k0 + 32 * sub + kl;
      const bool ok = live && r >= lo && r < hi && k < klen;
      v[e] = ok ? base[NAT ? (int64_t)k * ld + r : (int64_t)r * ld + k] : 0.f;
    }
  }
  __device__ __forceinline__ void store(MLORA_LDS char *dst, int tid) const {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      int sub, r, k;
      coords(e, tid, sub, r, k);
      const int a = NAT ? k * WID * 4 + 16 * ((r >> 2) ^ (8 * ((k >> 2) & 1))) + 4 * (r & 3)
                        : r * 128 + 16 * ((k >> 2) ^ swz(r)) + 4 * (k & 3);
      *(MLORA_LDS float *)(dst + sub * WID * 128 + a) = v[e];
    }
  }
};

// Byte address (within a 32-deep tile) of lane l's first fragment of 32-wide tile t; substeps and
// elements are constant offsets (K-contiguous: one address per substep s).
template <bool NAT, int WID>
__device__ __forceinline__ int32_t f32_frag_addr(int t, int s, int lane) {
  const int l = lane & 31, h = lane >> 5;
  if constexpr (NAT) return (4 * h) * WID * 4 + (t ^ h) * 128 + 4 * l;
  else return (32 * t + l) * 128 + 16 * ((2 * s + h) ^ swz(l));
}

// The tile engine: contracts every source that `next` yields into acc. MFMA 32x32x2: lane l gives
// A[row l % 32][k l / 32] and B[k l / 32][col l % 32]; acc register v of lane l is
// C[8(v / 4) + 4(l / 32) + v % 4][l % 32]. SWAP: the transposed tile (rows <- Q, columns <- P).
template <class C, bool SWAP, class Next>
__device__ __forceinline__ void f32_contract(f32x16 (&acc)[C::TM][C::TN], MLORA_LDS char *lds, int i0, int j0, int tid,
                                             Next &&next) {
  const int lane = tid & 63, wave = wave_id();
  const int ks = wave % C::KS, wi = wave / C::KS / C::WN, wj = wave / C::KS % C::WN;
  F32Src src;
  bool more = next(src);
  if (!more) return;
  int k_next = 0;  // first contraction index of the tile to load next
  int n_real = 0;  // tiles with data so far
  using PL = std::conditional_t<C::DIRECT, F32Loader<C::PN, C::PWID, C::KS, C::NW, C::P_LPW>,
                                F32RegLoader<C::PN, C::PWID, C::KS, C::THREADS>>;
  using QL = std::conditional_t<C::DIRECT, F32Loader<C::QN, C::QWID, C::KS, C::NW, C::Q_LPW>,
                                F32RegLoader<C::QN, C::QWID, C::KS, C::THREADS>>;
  PL pl;
  QL ql;
  int whole = 0;  // steps that end at or before this index need no masks
  auto point = [&]() {
    whole = C::PN || src.p_lo <= i0 ? src.klen : 0;
    if constexpr (C::DIRECT) {
      pl.init(src.P, src.ldp, i0, src.p_lo, src.p_hi, src.klen, lane);
      ql.init(src.Q, src.ldq, j0, 0, src.q_hi, src.klen, lane);
    } else {
      pl.init(src.P, src.ldp, i0, src.p_lo, src.p_hi, src.klen);
      ql.init(src.Q, src.ldq, j0, 0, src.q_hi, src.klen);
    }
  };
  point();
  // first contraction index of the next tile (moving to the next source where one ends); live:
  // false once every source is done
  auto advance = [&](bool &live) -> int {
    if (more && k_next >= src.klen) {
      more = next(src);
      k_next = 0;
      whole = 0;
      if (more) point();
    }
    live = more;
    const int k0 = k_next;
    if (more) k_next += C::BK, ++n_real;
    return k0;
  };
  int32_t pa[C::PN ? C::TM : 4], qa[C::QN ? C::TN : 4];
#pragma unroll
  for (int s = 0; s < (C::PN ? C::TM : 4); ++s)
    pa[s] = ks * C::P_SUB + f32_frag_addr<C::PN, C::PWID>(C::PN ? wi * C::TM + s : wi * C::TM, s, lane);
#pragma unroll
  for (int s = 0; s < (C::QN ? C::TN : 4); ++s)
    qa[s] = C::KS * C::P_SUB + ks * C::Q_SUB +
            f32_frag_addr<C::QN, C::QWID>(C::QN ? wj * C::TN + s : wj * C::TN, s, lane);
  struct Frag {
    float a[C::TM][4], b[C::TN][4];
  };
  auto read = [&](const MLORA_LDS char *base, int s, Frag &f) {
#pragma unroll
    for (int t = 0; t < C::TM; ++t) {
      if constexpr (C::PN) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f.a[t][e] = *(const MLORA_LDS float *)(base + pa[t] + (8 * s + e) * C::PWID * 4);
      } else {
        const f32x4 v = *(const lds_f4 *)(base + pa[s] + 4096 * t);
#pragma unroll
        for (int e = 0; e < 4; ++e) f.a[t][e] = v[e];
      }
    }
#pragma unroll
    for (int t = 0; t < C::TN; ++t) {
      if constexpr (C::QN) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f.b[t][e] = *(const MLORA_LDS float *)(base + qa[t] + (8 * s + e) * C::QWID * 4);
      } else {
        const f32x4 v = *(const lds_f4 *)(base + qa[s] + 4096 * t);
#pragma unroll
        for (int e = 0; e < 4; ++e) f.b[t][e] = v[e];
      }
    }
  };
  // the fragments of substep s + 1 are read between the MFMAs of substep s
  auto compute = [&](auto st_c) {
    const MLORA_LDS char *base = lds + decltype(st_c)::value * C::STAGE_BYTES;
    constexpr int NM = 4 * C::TM * C::TN, NR = (C::PN ? 4 * C::TM : C::TM) + (C::QN ? 4 * C::TN : C::TN);
    Frag f[2];
    read(base, 0, f[0]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s < 3) read(base, s + 1, f[(s + 1) & 1]);
      const Frag &x = f[s & 1];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int ti = 0; ti < C::TM; ++ti)
#pragma unroll
          for (int tj = 0; tj < C::TN; ++tj)
            acc[ti][tj] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x2f32(x.b[tj][e], x.a[ti][e], acc[ti][tj], 0, 0, 0)
                               : __builtin_amdgcn_mfma_f32_32x32x2f32(x.a[ti][e], x.b[tj][e], acc[ti][tj], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);  // substep 0's reads
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int g = 0; g < NM; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
        const int n = s < 3 ? ((g + 1) * NR) / NM - (g * NR) / NM : 0;
#pragma unroll
        for (int r = 0; r < n; ++r) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
  };
  constexpr int S = C::STAGES;
  int t = 0;
  if constexpr (C::DIRECT) {
    auto issue = [&](auto st_c) {
      MLORA_LDS char *base = lds + decltype(st_c)::value * C::STAGE_BYTES;
      if (k_next + C::BK <= whole) {
        pl.issue_plain(base, k_next, wave);
        ql.issue_plain(base + C::KS * C::P_SUB, k_next, wave);
        k_next += C::BK;
        ++n_real;
        return;
      }
      bool live;
      const int k0 = advance(live);
      pl.issue(base, k0, live, wave, lane);
      ql.issue(base + C::KS * C::P_SUB, k0, live, wave, lane);
    };
    // tile t in stage t % S; S - 1 tiles ahead, loads past the last one move no data but keep the
    // wait counts constant
    static_for<S - 1>([&](auto p) {
      issue(p);
      return true;
    });
    auto step = [&](auto cur) -> bool {
      if (t >= n_real) return false;
      constexpr int refill = (decltype(cur)::value + S - 1) % S;
      wait_vmcnt<(S - 2) * C::LPW>();  // this wave's loads of tile t
      lds_pipeline_barrier();          // everyone's; everyone is done with tile t - 1
      issue(std::integral_constant<int, refill>{});
      compute(cur);
      ++t;
      return true;
    };
    while (t < n_real) static_for<S>(step);
    wait_vmcnt<0>();  // nothing may still write LDS after the loop
  } else {
    bool live;
    int k0 = advance(live);
    pl.load(k0, live, tid);
    ql.load(k0, live, tid);
    pl.store(lds, tid);
    ql.store(lds + C::KS * C::P_SUB, tid);
    auto step = [&](auto cur) -> bool {
      if (t >= n_real) return false;
      constexpr int nxt = decltype(cur)::value ^ 1;
      __syncthreads();  // tile t stored; everyone is done with tile t - 1
      k0 = advance(live);
      pl.load(k0, live, tid);
      ql.load(k0, live, tid);
      compute(cur);
      pl.store(lds + nxt * C::STAGE_BYTES, tid);
      ql.store(lds + nxt * C::STAGE_BYTES + C::KS * C::P_SUB, tid);
      ++t;
      return true;
    };
    while (t < n_real) static_for<2>(step);
  }
}

template <class C>
__device__ __forceinline__ void f32_zero(f32x16 (&acc)[C::TM][C::TN]) {
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}

// out(ti, tj, acc) for every 32x32 tile of the workgroup, once per tile. KS > 1: the wave
// groups' sums of a tile are added in wave order by the wave that owns it (tile % KS).
template <class C, class Out>
__device__ __forceinline__ void f32_finish(f32x16 (&acc)[C::TM][C::TN], MLORA_LDS char *lds, int tid, Out &&out) {
  if constexpr (C::KS == 1) {
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
      for (int j = 0; j < C::TN; ++j) out(i, j, acc[i][j]);
  } else {
    const int lane = tid & 63, wave = wave_id(), ks = wave % C::KS, g0 = wave - ks;
    constexpr int NT = C::TM * C::TN;
    __syncthreads();  // the stages are free
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16 &s = acc[n / C::TN][n % C::TN];
        *(lds_f4 *)(lds + ((wave * NT + n) * 4 + q) * 1024 + 16 * lane) =
            f32x4{s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      if (n % C::KS != ks) continue;  // wave-uniform
      f32x16 sum;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 v = *(const lds_f4 *)(lds + ((g0 * NT + n) * 4 + q) * 1024 + 16 * lane);
#pragma unroll
        for (int k = 1; k < C::KS; ++k) v += *(const lds_f4 *)(lds + (((g0 + k) * NT + n) * 4 + q) * 1024 + 16 * lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[4 * q + e] = v[e];
      }
      out(n / C::TN, n % C::TN, sum);
    }
  }
}

// ---------------------------------------------------------------- linear (GEMM + LoRA term), shrink

struct F32LinArgs {
  const float *P;  // [M, Kc] row-major (pitch ldp)
  int64_t ldp;
  const float *Q;  // GEMM: main operand, [Ncols, Kc] or natural [Kc, Ncols] (pitch ldq)
  int64_t ldq;
  const float *E;  // GEMM: LoRA rows [M, >= r] (pitch lde)
  int64_t lde;
  const float *bias;
  float *C;
  int64_t ldc;
  int32_t M, Ncols, Kc;
  int32_t tiles_m, tiles_n;
  const float *qe[kMaxAdapters];  // the adapters' operands
  int64_t qe_ld[kMaxAdapters];
  int32_t rank[kMaxAdapters];
  float scale[kMaxAdapters];
  int32_t tile_start[kMaxSeg + 1];  // shrink: first row tile of each segment
  SegTable seg;
};

// Tile order: XCD-contiguous ids, walked in groups of kF32GroupM row tiles.
constexpr int kF32GroupM = 4;

template <class C>
__global__ __launch_bounds__(C::THREADS, C::WAVES_PER_SIMD) void f32_gemm_kernel(const F32LinArgs a) {
  __shared__ f32x4 smem[C::LDS_BYTES / 16];
  MLORA_LDS char *lds = (MLORA_LDS char *)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int id = xcd_contiguous(blockIdx.x, gridDim.x);
  const int per_group = kF32GroupM * a.tiles_n;
  const int first_m = id / per_group * kF32GroupM;
  const int gsize = min(a.tiles_m - first_m, kF32GroupM);
  const int i0 = (first_m + id % per_group % gsize) * C::BM, j0 = id % per_group / gsize * C::BN;
  f32x16 acc[C::TM][C::TN];
  f32_zero<C>(acc);
  const int iend = min(i0 + C::BM, a.M);
  int s = -1;  // -1: the main term; then the segments
  f32_contract<C, false>(acc, lds, i0, j0, tid, [&](F32Src &src) -> bool {
    if (s < 0) {
      s = a.E != nullptr ? seg_of_row(a.seg, i0) : a.seg.n;
      if (a.Kc > 0) {
        src = F32Src{a.P, a.Q, a.ldp, a.ldq, 0, a.M, a.Ncols, a.Kc};
        return true;
      }
    }
    while (s < a.seg.n && a.seg.off[s] < iend) {
      const int ad = a.seg.aid[s], lo = a.seg.off[s], hi = a.seg.off[s + 1];
      ++s;
      if (ad < 0 || a.rank[ad] == 0 || hi <= i0 || hi == lo) continue;
      src = F32Src{a.E, a.qe[ad], a.lde, a.qe_ld[ad], lo, hi, a.Ncols, a.rank[ad]};
      return true;
    }
    return false;
  });
  const int wi = wave / C::KS / C::WN, wj = wave / C::KS % C::WN;
  f32_finish<C>(acc, lds, tid, [&](int ti, int tj, const f32x16 &v) {
    const int j = j0 + 32 * (C::TN * wj + tj) + (lane & 31);
    if (j >= a.Ncols) return;
    const float b = a.bias ? a.bias[j] : 0.f;
    const int ib = i0 + 32 * (C::TM * wi + ti) + 4 * (lane >> 5);
    float *c = a.C + (int64_t)ib * a.ldc + j;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = 8 * (r >> 2) + (r & 3);
      if (ib + i < a.M) gp(c)[(int64_t)i * a.ldc] = v[r] + b;
    }
  });
}

// One workgroup per BM rows of one segment (blockIdx.x) and BN columns (blockIdx.y): rows without
// an adapter and columns past the rank are written as zeros.
template <class C>
__global__ __launch_bounds__(C::THREADS, C::WAVES_PER_SIMD) void f32_shrink_kernel(const F32LinArgs a) {
  __shared__ f32x4 smem[C::LDS_BYTES / 16];
  MLORA_LDS char *lds = (MLORA_LDS char *)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int bid = blockIdx.x;
  int lo = 0, hi = a.seg.n - 1;  // the last segment whose first tile is <= bid (empty ones have no tile)
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.tile_start[mid] <= bid) lo = mid; else hi = mid - 1;
  }
  const int s = lo, ad = a.seg.aid[s];
  const int i0 = a.seg.off[s] + (bid - a.tile_start[s]) * C::BM, iend = a.seg.off[s + 1];
  const int j0 = blockIdx.y * C::BN;
  const int r = ad < 0 ? 0 : a.rank[ad];
  f32x16 acc[C::TM][C::TN];
  f32_zero<C>(acc);
  bool first = j0 < r && a.Kc > 0;
  f32_contract<C, false>(acc, lds, i0, j0, tid, [&](F32Src &src) -> bool {
    if (!first) return false;
    first = false;
    src = F32Src{a.P, a.qe[ad], a.ldp, a.qe_ld[ad], 0, iend, r, a.Kc};
    return true;
  });
  const int wi = wave / C::KS / C::WN, wj = wave / C::KS % C::WN;
  const float scale = ad < 0 ? 0.f : a.scale[ad];
  f32_finish<C>(acc, lds, tid, [&](int ti, int tj, const f32x16 &v) {
    const int j = j0 + 32 * (C::TN * wj + tj) + (lane & 31);
    if (j >= a.Ncols) return;
    const int ib = i0 + 32 * (C::TM * wi + ti) + 4 * (lane >> 5);
    float *c = a.C + (int64_t)ib * a.ldc + j;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int i = 8 * (q >> 2) + (q & 3);
      if (ib + i < iend) gp(c)[(int64_t)i * a.ldc] = j < r ? v[q] * scale : 0.f;
    }
  });
}

// ---------------------------------------------------------------- segmented outer product

// Work item: 128 columns of P x BN columns of H x one split of an adapter's rows (its segments one
// after another, `chunk_rows` rows per split). An adapter of one split is written to its output;
// otherwise every split leaves a partial sum in the output's own layout, and the reduction adds
// them in split order.
struct F32OuterArgs {
  const float *P;  // [M, Ci] (pitch ldp)
  int64_t ldp;
  const float *H;  // [M, >= r] (pitch ldh)
  int64_t ldh;
  int32_t Ci, cblocks;
  int32_t chunk_rows;
  int32_t n_adapters;
  float *ws;
  float *out[kMaxAdapters];
  int64_t ws_off[kMaxAdapters];  // floats
  int32_t rank[kMaxAdapters], splits[kMaxAdapters];
  int32_t item_start[kMaxAdapters + 1];
  SegTable seg;
};

// OL: the output layout, 0: D_a [Ci, r_a]; 1: D_a [r_a, Ci] (the tile is computed transposed, so
// that the lanes of a store run along the output's rows either way).
template <class C, int OL>
__global__ __launch_bounds__(C::THREADS, C::WAVES_PER_SIMD) void f32_outer_kernel(const F32OuterArgs a) {
  __shared__ f32x4 smem[C::LDS_BYTES / 16];
  MLORA_LDS char *lds = (MLORA_LDS char *)smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int item = xcd_contiguous(blockIdx.x, gridDim.x);
  int ad = 0;
  while (ad + 1 < a.n_adapters && a.item_start[ad + 1] <= item) ++ad;
  const int r = a.rank[ad], local = item - a.item_start[ad];
  const int jbs = (r + C::BN - 1) / C::BN;
  const int i0 = local % a.cblocks * C::BM, j0 = local / a.cblocks % jbs * C::BN, split = local / (a.cblocks * jbs);
  const int64_t v0 = (int64_t)split * a.chunk_rows, v1 = split + 1 < a.splits[ad] ? v0 + a.chunk_rows : INT64_MAX;
  f32x16 acc[C::TM][C::TN];
  f32_zero<C>(acc);
  int s = 0;
  int64_t v = 0;  // rows of the adapter before segment s
  f32_contract<C, OL == 1>(acc, lds, i0, j0, tid, [&](F32Src &src) -> bool {
    while (s < a.seg.n && v < v1) {
      const int off = a.seg.off[s], len = a.seg.off[s + 1] - off;
      const bool mine = a.seg.aid[s++] == ad;
      if (!mine) continue;
      const int64_t b0 = v0 > v ? v0 - v : 0, b1 = v1 - v < len ? v1 - v : len;
      v += len;
      if (b0 >= b1) continue;
      const int64_t row = off + b0;
      src = F32Src{a.P + row * a.ldp, a.H + row * a.ldh, a.ldp, a.ldh, 0, a.Ci, r, (int32_t)(b1 - b0)};
      return true;
    }
    return false;
  });
  float *o = a.splits[ad] > 1 ? a.ws + a.ws_off[ad] + (int64_t)split * a.Ci * r : a.out[ad];
  const int wi = wave / C::KS / C::WN, wj = wave / C::KS % C::WN;
  f32_finish<C>(acc, lds, tid, [&](int ti, int tj, const f32x16 &t) {
    const int ct = i0 + 32 * (C::TM * wi + ti), jt = j0 + 32 * (C::TN * wj + tj);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int i = 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
      const int c = ct + (OL == 0 ? i : lane & 31), j = jt + (OL == 0 ? lane & 31 : i);
      if (c < a.Ci && j < r) gp(o)[OL == 0 ? (int64_t)c * r + j : (int64_t)j * a.Ci + c] = t[q];
    }
  });
}

// Sums the partials of the adapters of more than one split, in split order: four consecutive
// outputs per thread, the loads of up to 8 splits issued together.
__global__ __launch_bounds__(256) void f32_outer_reduce_kernel(const F32OuterArgs a) {
  const int ad = blockIdx.y, n = a.splits[ad];
  const int64_t total = (int64_t)a.Ci * a.rank[ad], i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (a.rank[ad] == 0 || n <= 1 || i >= total) return;
  const MLORA_GLOBAL float *p = gp(a.ws) + a.ws_off[ad] + i;
  const int live = total - i < 4 ? (int)(total - i) : 4;
  const bool vec = total % 4 == 0;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < n; k += 8) {
    float v[8][4];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const MLORA_GLOBAL float *q = p + (int64_t)(k + u) * total;
      if (vec && k + u < n) {
        const f32x4 w = *(const MLORA_GLOBAL f32x4 *)q;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = w[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = k + u < n && e < live ? q[e] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < n)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += v[u][e];
  }
  MLORA_GLOBAL float *o = gp(a.out[ad]) + i;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (e < live) o[e] = sum[e];
}

// ---------------------------------------------------------------- host side

static bool aligned4(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }

// fp32 row-major matrix [rows, cols], pitch ld (elements).
static int check_f32_matrix(const void *p, int64_t ld, int64_t rows, int64_t cols) {
  if (rows == 0 || cols == 0) return MLORA_OK;
  if (p == nullptr || ld < cols) return MLORA_ERR_INVALID;
  if (!aligned4(p)) return MLORA_ERR_UNSUPPORTED;
  return MLORA_OK;
}

// 16-byte direct-to-LDS loads can read the matrix: whole chunks of 4, and the byte offsets of a
// tile (up to 256 rows, F32Cfg) stay below the out-of-range one.
static bool direct_ok(const void *p, int64_t ld, int64_t cols) {
  return aligned16(p) && ld % 4 == 0 && cols % 4 == 0 && ld < kDirectLd;
}

// Adapter operands for the fp32 kernels: any rank in [0, kMaxRank] (no padding). direct: cleared
// when a used operand (pitch and columns: op_cols, or the rank when 0) does not allow 16-byte loads.
static int f32_adapters(F32LinArgs &a, const void *const *ptrs, const int32_t *ranks, const float *scales, int32_t n,
                        int64_t op_cols, bool &direct) {
  if (n < 0) return MLORA_ERR_INVALID;
  if (n > kMaxAdapters) return MLORA_ERR_LIMIT;
  if (n > 0 && ranks == nullptr) return MLORA_ERR_INVALID;
  for (int i = 0; i < kMaxAdapters; ++i) {
    a.qe[i] = nullptr;
    a.rank[i] = 0;
    a.scale[i] = 0.f;
    a.qe_ld[i] = 0;
  }
  for (int i = 0; i < n; ++i) {
    if (ranks[i] < 0) return MLORA_ERR_INVALID;
    if (ranks[i] > kMaxRank) return MLORA_ERR_LIMIT;
    a.rank[i] = ranks[i];
    a.scale[i] = scales ? scales[i] : 1.f;
    a.qe_ld[i] = op_cols > 0 ? op_cols : ranks[i];
    if (ranks[i] > 0 && adapter_used(a.seg, i)) {
      if (ptrs == nullptr || ptrs[i] == nullptr) return MLORA_ERR_INVALID;
      if (!aligned4(ptrs[i])) return MLORA_ERR_UNSUPPORTED;
      a.qe[i] = static_cast<const float *>(ptrs[i]);
      direct = direct && direct_ok(ptrs[i], a.qe_ld[i], a.qe_ld[i]) && ranks[i] % 4 == 0;
    }
  }
  return MLORA_OK;
}

static int f32_max_rank(const F32LinArgs &a) {
  int r = 0;
  for (int s = 0; s < a.seg.n; ++s) {
    const int ad = a.seg.aid[s];
    if (ad >= 0 && a.seg.off[s + 1] > a.seg.off[s] && a.rank[ad] > r) r = a.rank[ad];
  }
  return r;
}

static bool f32_dims_ok(int64_t M, int64_t K, int64_t N) {
  return M >= 0 && K >= 0 && N >= 0 && M <= INT32_MAX - 128 && K <= INT32_MAX - 128 && N <= INT32_MAX - 128;
}

template <class C>
static int launch_f32_gemm(F32LinArgs &a, hipStream_t stream) {
  const int64_t tm = ((int64_t)a.M + C::BM - 1) / C::BM, tn = ((int64_t)a.Ncols + C::BN - 1) / C::BN;
  if (tm == 0 || tn == 0) return MLORA_OK;
  if (tm * tn > INT32_MAX || tn > INT32_MAX / kF32GroupM) return MLORA_ERR_LIMIT;
  a.tiles_m = (int32_t)tm;
  a.tiles_n = (int32_t)tn;
  hipLaunchKernelGGL(f32_gemm_kernel<C>, dim3((unsigned)(tm * tn)), dim3(C::THREADS), 0, stream, a);
  return launch_status();
}

// Tile choice, measured on MI355X (NT and NN within 3% of each other, two adapters of rank 64;
// the figures include ~8 us of launch and event time). The fp32 MFMA rate bounds every tile, so
// small tiles that fill the chip evenly win over large ones:
//   9360 x 1536 x 1536: 128x64 359 us, 64x64 375, 128x128 407 (torch's library 322, without the
//     LoRA term); 4680 rows: 64x64 187, 128x64 212, 128x128 222;
//   512 x 1536 x 1536 (192 tiles of 64x64): two wave groups splitting the contraction 36 us, one 38.
// Before (128x128 tiles, element loads, k-tiles of 16): 1160 us at 9360 rows.
// Element loads of the same call (one rank off a multiple of 4 sends the base there too): 690 us at 9360
// rows (direct 390 on that box, the kernels before 1070), 335 at 4680 (209, 560).
template <bool QN, bool DIRECT>
static int dispatch_f32_gemm(F32LinArgs &a, hipStream_t stream) {
  const int64_t wide = (((int64_t)a.M + 127) / 128) * (((int64_t)a.Ncols + 63) / 64);
  const int64_t tiles = (((int64_t)a.M + 63) / 64) * (((int64_t)a.Ncols + 63) / 64);
  if (tiles <= 256) return launch_f32_gemm<F32Cfg<1, 1, 2, 2, 2, false, QN, DIRECT, 2>>(a, stream);
  if (wide < 1536) return launch_f32_gemm<F32Cfg<1, 1, 2, 2, 1, false, QN, DIRECT, 2>>(a, stream);
  return launch_f32_gemm<F32Cfg<2, 1, 2, 2, 1, false, QN, DIRECT, 2>>(a, stream);
}

template <class C>
static int launch_f32_shrink(F32LinArgs &a, hipStream_t stream) {
  int64_t n = 0;
  for (int s = 0; s < a.seg.n; ++s) {
    a.tile_start[s] = (int32_t)n;
    n += ((int64_t)a.seg.off[s + 1] - a.seg.off[s] + C::BM - 1) / C::BM;
  }
  a.tile_start[a.seg.n] = (int32_t)n;
  const int64_t cols = ((int64_t)a.Ncols + C::BN - 1) / C::BN;
  if (n == 0 || cols == 0) return MLORA_OK;
  if (n > INT32_MAX || cols > 65535) return MLORA_ERR_LIMIT;
  hipLaunchKernelGGL(f32_shrink_kernel<C>, dim3((unsigned)n, (unsigned)cols), dim3(C::THREADS), 0, stream, a);
  return launch_status();
}

// 32-row tiles (so that a few thousand rows fill the chip), the contraction split over two wave
// groups up to rank 128, two LDS stages for two or three workgroups per CU. Cold launches at
// 9360 x 1536, rank 64: 31 us (three stages 32, one wave per 64 columns and four groups 42,
// 128x128 tiles 510); 4000 x 3072, rank 128: 56 us (four waves of two tiles 62).
template <bool QN, bool DIRECT>
static int dispatch_f32_shrink(F32LinArgs &a, int rmax, hipStream_t stream) {
  if (rmax <= 64) return launch_f32_shrink<F32Cfg<1, 1, 1, 2, 2, false, QN, DIRECT, 2>>(a, stream);
  if (rmax <= 128) return launch_f32_shrink<F32Cfg<1, 1, 1, 4, 2, false, QN, DIRECT, 2>>(a, stream);
  return launch_f32_shrink<F32Cfg<1, 2, 1, 4, 1, false, QN, DIRECT, 2>>(a, stream);
}

// ---- reduction plan
constexpr int kOuterC = 128;  // P columns per work item

static int f32_outer_bn(int rmax) { return rmax <= 64 ? 64 : 128; }

// Splits of every adapter's rows: 768 work items (three 48 KB workgroups per CU at ranks <= 64),
// of at least 256 rows. Returns the partial sums' floats. Measured with the reduction, cold
// launches: two adapters of rank 64 over 9360 x 1536 27 us (693 us unsplit, one workgroup per
// 128 columns and adapter); 30000 x 1536 at rank 32 57 us with 768 items, 75 with 512; at 4680
// rows 256-row splits 20.5 us, 128-row ones 22.8.
static int64_t plan_f32_outer(F32OuterArgs &a, int rmax, bool split) {
  const int bn = f32_outer_bn(rmax);
  int64_t rows[kMaxAdapters] = {}, total = 0;
  for (int s = 0; s < a.seg.n; ++s)
    if (a.seg.aid[s] >= 0) rows[a.seg.aid[s]] += a.seg.off[s + 1] - a.seg.off[s];
  a.cblocks = (a.Ci + kOuterC - 1) / kOuterC;
  for (int i = 0; i < a.n_adapters; ++i)
    if (a.rank[i] > 0) total += rows[i] * a.cblocks * ((a.rank[i] + bn - 1) / bn);  // rows x tiles to stream
  int64_t cr = (total / 768 + 31) / 32 * 32;
  if (cr < 256) cr = 256;
  if (cr > ((int64_t)1 << 20)) cr = (int64_t)1 << 20;
  a.chunk_rows = (int32_t)cr;
  int64_t ws = 0, items = 0;
  for (int i = 0; i < a.n_adapters; ++i) {
    a.splits[i] = a.rank[i] == 0 ? 0 : (!split || rows[i] <= cr) ? 1 : (int32_t)((rows[i] + cr - 1) / cr);
    a.item_start[i] = (int32_t)items;
    items += (int64_t)a.splits[i] * a.cblocks * ((a.rank[i] + bn - 1) / bn);
    a.ws_off[i] = ws;
    if (a.splits[i] > 1) ws += ((int64_t)a.splits[i] * a.Ci * a.rank[i] + 3) / 4 * 4;
  }
  a.item_start[a.n_adapters] = (int32_t)(items > INT32_MAX ? -1 : items);
  return ws;
}

// Everything of a reduction but the pointers: the routing, the ranks and the plan.
static int f32_outer_setup(F32OuterArgs &a, int64_t M, int64_t C, const int32_t *ranks, int32_t n_adapters,
                           const int64_t *seg_offsets, const int32_t *adapter_ids, int32_t n_segments, bool split,
                           int &rmax, int64_t &ws_floats) {
  if (!f32_dims_ok(M, C, 0)) return MLORA_ERR_LIMIT;
  int st = build_segtable(a.seg, M, seg_offsets, adapter_ids, n_segments, n_adapters);
  if (st) return st;
  if (n_adapters < 0) return MLORA_ERR_INVALID;
  if (n_adapters > kMaxAdapters) return MLORA_ERR_LIMIT;
  if (n_adapters > 0 && ranks == nullptr) return MLORA_ERR_INVALID;
  rmax = 0;
  for (int i = 0; i < kMaxAdapters; ++i) a.rank[i] = 0;
  for (int i = 0; i < n_adapters; ++i) {
    if (ranks[i] < 0) return MLORA_ERR_INVALID;
    if (ranks[i] > kMaxRank) return MLORA_ERR_LIMIT;
    a.rank[i] = ranks[i];
    rmax = ranks[i] > rmax ? ranks[i] : rmax;
  }
  a.n_adapters = n_adapters;
  a.Ci = (int32_t)C;
  ws_floats = plan_f32_outer(a, rmax, split);
  return MLORA_OK;
}

template <bool DIRECT, int OL>
static void launch_f32_outer(const F32OuterArgs &a, int rmax, unsigned items, hipStream_t stream) {
  if (f32_outer_bn(rmax) == 64) {
    using C = F32Cfg<1, 1, 4, 2, 1, true, true, DIRECT, 2>;
    static_assert(C::BM == kOuterC && C::BN == 64, "the plan's tile");
    hipLaunchKernelGGL((f32_outer_kernel<C, OL>), dim3(items), dim3(C::THREADS), 0, stream, a);
  } else {
    using C = F32Cfg<1, 1, 4, 4, 1, true, true, DIRECT, 2>;
    static_assert(C::BM == kOuterC && C::BN == 128, "the plan's tile");
    hipLaunchKernelGGL((f32_outer_kernel<C, OL>), dim3(items), dim3(C::THREADS), 0, stream, a);
  }
}

static int f32_outer_run(F32OuterArgs &a, int rmax, int64_t ws_floats, const void *p, int64_t ldp, int64_t M, int64_t C,
                         const void *h, int64_t ldh, void *const *out_ptrs, int out_layout, void *workspace,
                         hipStream_t stream) {
  int st;
  if (out_layout != 0 && out_layout != 1) return MLORA_ERR_INVALID;
  if (a.n_adapters > 0 && out_ptrs == nullptr) return MLORA_ERR_INVALID;
  bool direct = direct_ok(p, ldp, C) && direct_ok(h, ldh, 4);
  for (int i = 0; i < kMaxAdapters; ++i) {
    a.out[i] = i < a.n_adapters ? static_cast<float *>(out_ptrs[i]) : nullptr;
    if (a.rank[i] > 0 && C > 0 && (a.out[i] == nullptr || !aligned4(a.out[i]))) return MLORA_ERR_INVALID;
    direct = direct && a.rank[i] % 4 == 0;
  }
  if ((st = check_f32_matrix(p, ldp, M, C))) return st;
  if ((st = check_f32_matrix(h, ldh, M, rmax))) return st;
  if (C == 0 || rmax == 0) return MLORA_OK;
  const int32_t items = a.item_start[a.n_adapters];
  if (items < 0) return MLORA_ERR_LIMIT;
  a.P = static_cast<const float *>(p);
  a.ldp = ldp;
  a.H = static_cast<const float *>(h);
  a.ldh = ldh;
  a.ws = static_cast<float *>(workspace);
  if (direct) {
    if (out_layout == 0) launch_f32_outer<true, 0>(a, rmax, (unsigned)items, stream);
    else launch_f32_outer<true, 1>(a, rmax, (unsigned)items, stream);
  } else {
    if (out_layout == 0) launch_f32_outer<false, 0>(a, rmax, (unsigned)items, stream);
    else launch_f32_outer<false, 1>(a, rmax, (unsigned)items, stream);
  }
  if ((st = launch_status()) || ws_floats == 0) return st;
  const int64_t blocks = (C * rmax + 1023) / 1024;
  if (blocks > INT32_MAX) return MLORA_ERR_LIMIT;
  hipLaunchKernelGGL(f32_outer_reduce_kernel, dim3((unsigned)blocks, (unsigned)a.n_adapters), dim3(256), 0, stream, a);
  return launch_status();
}

}  // namespace mlora

using namespace mlora;

extern "C" int mlora_f32_shrink(const void *p, int64_t ldp, int64_t M, int64_t K, const void *const *op_ptrs,
                                int op_layout, const int32_t *ranks, const float *scales, int32_t n_adapters,
                                const int64_t *seg_offsets, const int32_t *adapter_ids, int32_t n_segments, void *h,
                                int64_t ldh, int64_t width, void *stream) {
  F32LinArgs a{};
  if (!f32_dims_ok(M, K, width)) return MLORA_ERR_LIMIT;
  int st = build_segtable(a.seg, M, seg_offsets, adapter_ids, n_segments, n_adapters);
  if (st) return st;
  // layout 0: Op_a [r, K] (contraction-contiguous); layout 1: Op_a [K, r] (natural)
  bool direct = direct_ok(p, ldp, K);
  if ((st = f32_adapters(a, op_ptrs, ranks, scales, n_adapters, op_layout == 0 ? K : 0, direct))) return st;
  if (op_layout != 0 && op_layout != 1) return MLORA_ERR_INVALID;
  const int rmax = f32_max_rank(a);
  if (width < rmax) return MLORA_ERR_INVALID;
  if ((st = check_f32_matrix(p, ldp, M, K))) return st;
  if ((st = check_f32_matrix(h, ldh, M, width))) return st;
  if (M == 0 || width == 0) return MLORA_OK;
  a.P = static_cast<const float *>(p);
  a.ldp = ldp;
  a.C = static_cast<float *>(h);
  a.ldc = ldh;
  a.M = (int32_t)M;
  a.Kc = (int32_t)K;
  a.Ncols = (int32_t)width;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (op_layout == 0) return direct ? dispatch_f32_shrink<false, true>(a, rmax, s) : dispatch_f32_shrink<false, false>(a, rmax, s);
  return direct ? dispatch_f32_shrink<true, true>(a, rmax, s) : dispatch_f32_shrink<true, false>(a, rmax, s);
}

extern "C" int mlora_f32_gemm_fwd(const void *x, int64_t ldx, int64_t M, int64_t K, const void *w, int64_t ldw,
                                  int64_t N, const void *bias, const void *h_rows, int64_t ldh,
                                  const void *const *b_ptrs, const int32_t *ranks, int32_t n_adapters,
                                  const int64_t *seg_offsets, const int32_t *adapter_ids, int32_t n_segments, void *y,
                                  int64_t ldy, void *stream) {
  F32LinArgs a{};
  if (!f32_dims_ok(M, K, N)) return MLORA_ERR_LIMIT;
  int st = build_segtable(a.seg, M, seg_offsets, adapter_ids, n_segments, n_adapters);
  if (st) return st;
  bool direct = direct_ok(x, ldx, K) && direct_ok(w, ldw, K);
  if ((st = f32_adapters(a, b_ptrs, ranks, nullptr, n_adapters, 0, direct))) return st;  // B_a [N, r]
  const int rmax = f32_max_rank(a);
  if ((st = check_f32_matrix(x, ldx, M, K))) return st;
  if ((st = check_f32_matrix(w, ldw, N, K))) return st;
  if ((st = check_f32_matrix(y, ldy, M, N))) return st;
  if (rmax > 0 && (st = check_f32_matrix(h_rows, ldh, M, rmax))) return st;
  if (bias != nullptr && !aligned4(bias)) return MLORA_ERR_UNSUPPORTED;
  if (M == 0 || N == 0) return MLORA_OK;
  if (rmax > 0) direct = direct && direct_ok(h_rows, ldh, 4);
  a.P = static_cast<const float *>(x);
  a.ldp = ldx;
  a.Q = static_cast<const float *>(w);
  a.ldq = ldw;
  a.E = rmax > 0 ? static_cast<const float *>(h_rows) : nullptr;
  a.lde = ldh;
  a.bias = static_cast<const float *>(bias);
  a.C = static_cast<float *>(y);
  a.ldc = ldy;
  a.M = (int32_t)M;
  a.Kc = (int32_t)K;
  a.Ncols = (int32_t)N;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return direct ? dispatch_f32_gemm<false, true>(a, s) : dispatch_f32_gemm<false, false>(a, s);
}

extern "C" int mlora_f32_gemm_dx(const void *dy, int64_t lddy, int64_t M, int64_t N, const void *w, int64_t ldw,
                                 int64_t K, const void *g_rows, int64_t ldg, const void *const *a_ptrs,
                                 const int32_t *ranks, int32_t n_adapters, const int64_t *seg_offsets,
                                 const int32_t *adapter_ids, int32_t n_segments, void *dx, int64_t lddx,
                                 void *stream) {
  F32LinArgs a{};
  if (!f32_dims_ok(M, N, K)) return MLORA_ERR_LIMIT;
  int st = build_segtable(a.seg, M, seg_offsets, adapter_ids, n_segments, n_adapters);
  if (st) return st;
  // W [N, K] and A_a [r, K] are natural operands: their rows are the contraction
  bool direct = direct_ok(dy, lddy, N) && direct_ok(w, ldw, K);
  if ((st = f32_adapters(a, a_ptrs, ranks, nullptr, n_adapters, K, direct))) return st;
  const int rmax = f32_max_rank(a);
  if ((st = check_f32_matrix(dy, lddy, M, N))) return st;
  if ((st = check_f32_matrix(w, ldw, N, K))) return st;
  if ((st = check_f32_matrix(dx, lddx, M, K))) return st;
  if (rmax > 0 && (st = check_f32_matrix(g_rows, ldg, M, rmax))) return st;
  if (M == 0 || K == 0) return MLORA_OK;
  if (rmax > 0) direct = direct && direct_ok(g_rows, ldg, 4);
  a.P = static_cast<const float *>(dy);
  a.ldp = lddy;
  a.Q = static_cast<const float *>(w);
  a.ldq = ldw;
  a.E = rmax > 0 ? static_cast<const float *>(g_rows) : nullptr;
  a.lde = ldg;
  a.bias = nullptr;
  a.C = static_cast<float *>(dx);
  a.ldc = lddx;
  a.M = (int32_t)M;
  a.Kc = (int32_t)N;
  a.Ncols = (int32_t)K;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return direct ? dispatch_f32_gemm<true, true>(a, s) : dispatch_f32_gemm<true, false>(a, s);
}

extern "C" int64_t mlora_f32_seg_outer_workspace_bytes(int64_t M, int64_t C, const int32_t *ranks, int32_t n_adapters,
                                                       const int64_t *seg_offsets, const int32_t *adapter_ids,
                                                       int32_t n_segments) {
  F32OuterArgs a{};
  int rmax = 0;
  int64_t ws = 0;
  const int st = f32_outer_setup(a, M, C, ranks, n_adapters, seg_offsets, adapter_ids, n_segments, true, rmax, ws);
  return st ? st : ws * (int64_t)sizeof(float);
}

extern "C" int mlora_f32_seg_outer_split(const void *p, int64_t ldp, int64_t M, int64_t C, const void *h, int64_t ldh,
                                         void *const *out_ptrs, int out_layout, const int32_t *ranks,
                                         int32_t n_adapters, const int64_t *seg_offsets, const int32_t *adapter_ids,
                                         int32_t n_segments, void *workspace, int64_t workspace_bytes, void *stream) {
  F32OuterArgs a{};
  int rmax = 0;
  int64_t ws = 0;
  const int st = f32_outer_setup(a, M, C, ranks, n_adapters, seg_offsets, adapter_ids, n_segments, true, rmax, ws);
  if (st) return st;
  if (ws > 0 && (workspace == nullptr || workspace_bytes < ws * (int64_t)sizeof(float))) return MLORA_ERR_WORKSPACE;
  if (ws > 0 && !aligned16(workspace)) return MLORA_ERR_UNSUPPORTED;
  return f32_outer_run(a, rmax, ws, p, ldp, M, C, h, ldh, out_ptrs, out_layout, workspace,
                       static_cast<hipStream_t>(stream));
}

extern "C" int mlora_f32_seg_outer(const void *p, int64_t ldp, int64_t M, int64_t C, const void *h, int64_t ldh,
                                   void *const *out_ptrs, int out_layout, const int32_t *ranks, int32_t n_adapters,
                                   const int64_t *seg_offsets, const int32_t *adapter_ids, int32_t n_segments,
                                   void *stream) {
  F32OuterArgs a{};
  int rmax = 0;
  int64_t ws = 0;
  const int st = f32_outer_setup(a, M, C, ranks, n_adapters, seg_offsets, adapter_ids, n_segments, false, rmax, ws);
  if (st) return st;
  return f32_outer_run(a, rmax, 0, p, ldp, M, C, h, ldh, out_ptrs, out_layout, nullptr,
                       static_cast<hipStream_t>(stream));
}
