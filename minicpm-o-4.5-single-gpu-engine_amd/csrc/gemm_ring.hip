// bf16 MFMA GEMM for calls whose 256-row tile grids would leave most CUs idle: streaming windows (the deferred GEMMs from
// one window's ~100 rows on), prompt setups, several streams at once, up to a few thousand rows.
//
// Small tiles (64x64, 128x64, 128x128) put a workgroup on every CU; what bounds them is the latency of a K stage, so the
// stages run through a ring of NS LDS buffers filled by global_load_lds, NS - 1 of them in flight, with one
// barrier per 64-K stage and the next stage's fragments read into registers while this stage's MFMAs run.  A stage then
// costs 0.15 us on a 64x64 tile (0.24 with two buffers and no fragment prefetch), 0.235 on 128x64, 0.34 on 128x128:
// about 65-95 bytes per ns and CU, near the LDS traffic of its copies and fragment reads.  Deeper rings (5, 6, 8 stages)
// measured the same, and waves that each ran their own K slices without barriers were slower (the closing
// reduction cost 1.5 us).  EPI_PART splits K over g.splits workgroups per tile as well; the row kernel that
// reads the sums next finishes the epilogue (Pend).
//
// Measured in graphs of back-to-back launches (us; the two-kernel split-K path or the 128x128 tile grid before -> this
// kernel, split sums included):
//   rows   qkv (3072x1024)  proj (1024x1024)  conv (1024x3072)  fc1 (2048x1024)  fc2 (1024x2048)
//    100     8.2 ->  7.1       5.2 ->  4.1       7.7 ->  5.4          -             6.4 ->  4.7
//    450    23.8 ->  9.5      18.2 ->  5.1      25.5 ->  7.6     20.2 ->  6.4      20.6 ->  6.4
//   1024    14.5 -> 12.3      21.7 ->  6.4      38.4 -> 11.0     14.6 ->  8.7      27.0 ->  9.1
//   2000        -             14.5 ->  8.7      32.5 -> 18.7     15.6 -> 13.8      24.5 -> 14.3
//   3000        -             14.8 -> 11.5      32.9 -> 26.1         -             25.4 -> 18.3
#include "common.h"
#include "t2w_internal.h"
#include "gemm_tile.h"

namespace t2w {

namespace {

// s_waitcnt vmcnt(N) for N known at compile time, and no LDS read of this wave outstanding; a compiler barrier
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

template <int BM, int BN, int WM, int WN, int NS, bool TAPS>
struct Ring {
  static constexpr int NW = WM * WN;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  static constexpr int APW = BM / 8 / NW, BPW = BN / 8 / NW;  // 1 KB load blocks (8 rows of 128 bytes) per wave and stage
  static constexpr int L = APW + BPW;
  static constexpr int STAGE = (BM + BN) * 8;  // uint4 per stage: A rows, then W rows
  static_assert(APW * NW * 8 == BM && BPW * NW * 8 == BN, "load blocks must divide over the waves");
  static_assert(WTM % 16 == 0 && WTN % 32 == 0, "wave tiles");
  static_assert(NS >= 3 && (NS - 2) * L < 64, "ring depth");

  uint32_t asrc[APW], bsrc[BPW];
  const GemmArgs& g;
  int lane, wave, wm, wn;

  __device__ __forceinline__ Ring(const GemmArgs& g_, int m0, int n0) : g(g_) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wm = wave / WN;
    wn = wave % WN;
    const int lrow = lane >> 3;
#pragma unroll
    for (int p = 0; p < APW; ++p) {
      const int trow = (wave + p * NW) * 8 + lrow;
      const int m = min(m0 + trow, g.M - 1);  // rows past M load row M - 1; their results are never stored
      asrc[p] = (uint32_t)(TAPS ? g.a_src[m] : m) * (uint32_t)(g.lda * 2) + ((lane & 7) ^ swz_key(trow)) * 16;
    }
#pragma unroll
    for (int p = 0; p < BPW; ++p) {
      const int trow = (wave + p * NW) * 8 + lrow;
      bsrc[p] = (uint32_t)min(n0 + trow, g.N - 1) * (uint32_t)(g.ldb * 2) + ((lane & 7) ^ swz_key(trow)) * 16;
    }
  }

  // Stage kt into the ring slot at LDS byte address `slot`.  The copies are inline assembly so that the compiler does
  // not count them: it would wait for every load in flight before the first fragment read of a loop, which is what
  // the ring is there to avoid; wait_vm and the barrier in stage() order them instead.  They have no output registers.
  __device__ __forceinline__ void dma(uint32_t lds, uint32_t off, const void* base) const {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
  }
  __device__ __forceinline__ void issue(uint32_t slot, int kt) const {
    const uint32_t koff = (uint32_t)kt * (BK * 2);  // taps: a row's frames follow each other, so K runs on across them
#pragma unroll
    for (int p = 0; p < BPW; ++p) dma(slot + BM * 128 + (wave + p * NW) * 1024, bsrc[p] + koff, g.B);
#pragma unroll
    for (int p = 0; p < APW; ++p) dma(slot + (wave + p * NW) * 1024, asrc[p] + koff, g.A);
  }

  typedef bf16x8 fragA_t[2][TM];
  typedef bf16x8 fragB_t[2][TN];
  __device__ __forceinline__ void frags(const uint4* s, fragA_t& af, fragB_t& bf) const {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int chunk = kk * 4 + (lane >> 4);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[kk][j] = as_bf16x8(s[BM * 8 + swz(wn * WTN + j * 16 + (lane & 15), chunk)]);
#pragma unroll
      for (int i = 0; i < TM; ++i) af[kk][i] = as_bf16x8(s[swz(wm * WTM + i * 16 + (lane & 15), chunk)]);
    }
  }
  __device__ __forceinline__ void mma(const fragA_t& af, const fragB_t& bf, f32x4 (&acc)[TM][TN]) const {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[kk][j], af[kk][i], acc[i][j], 0, 0, 0);
  }

  // Stage kt, whose fragments (ca, cb) are in registers: wait until stage kt + 1 has landed (AFTER stages behind it may
  // be in flight), meet the other waves (their copies of it have landed too, and everybody has read stage kt out of
  // its slot), refill that slot with stage kt + NS, read the next fragments while the MFMAs run.
  template <int AFTER, bool REFILL>
  __device__ __forceinline__ void stage(const uint4* next, uint32_t refill, int kt, const fragA_t& ca, const fragB_t& cb,
                                        fragA_t& na, fragB_t& nb, f32x4 (&acc)[TM][TN]) const {
    wait_vm<AFTER * L>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (REFILL) issue(refill, kt + NS);
    frags(next, na, nb);
    mma(ca, cb, acc);
    constexpr int NR = 2 * (TM + TN), NM = 2 * TM * TN;
#pragma unroll
    for (int x = 0; x < NM; ++x) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      const int r0 = x * NR / NM, r1 = (x + 1) * NR / NM;
      if (r1 - r0 == 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      else if (r1 - r0 == 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    asm volatile("" ::: "memory");
  }
  // stages kt .. k1 - 1, at most REM + 1 of them behind the one in registers
  template <int REM>
  __device__ __forceinline__ void tail(const uint4* ring, int slot, int kt, int k1, fragA_t& ca, fragB_t& cb, f32x4 (&acc)[TM][TN]) const {
    if constexpr (REM >= 0) {
      if (kt + 1 + REM < k1) {
        fragA_t na;
        fragB_t nb;
        slot = slot + 1 == NS ? 0 : slot + 1;
        stage<REM, false>(ring + slot * STAGE, 0, kt, ca, cb, na, nb, acc);
        tail<REM - 1>(ring, slot, kt + 1, k1, na, nb, acc);
      } else {
        tail<REM - 1>(ring, slot, kt, k1, ca, cb, acc);
      }
    } else {
      mma(ca, cb, acc);
    }
  }
};

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool TAPS>
__global__ void __launch_bounds__(64 * WM * WN) gemm_ring_kernel(GemmArgs g, int S, int colmajor) {
  typedef Ring<BM, BN, WM, WN, NS, TAPS> T;
  __shared__ uint4 ring[NS * T::STAGE];
  const int gm = (g.M + BM - 1) / BM, gn = (g.N + BN - 1) / BN;
  const int nblk = gm * gn * S, per = nblk / 8, full = per * 8;
  int b = blockIdx.x;
  if (b < full) b = (b % 8) * per + b / 8;
  int mb, nb;
  const int z = b / (gm * gn);
  b -= z * gm * gn;
  if (colmajor) { mb = b % gm; nb = b / gm; }
  else { mb = b / gn; nb = b % gn; }
  const int m0 = mb * BM, n0 = nb * BN;
  const int KT = g.K / BK, k0 = z * KT / S, k1 = (z + 1) * KT / S;

  T t(g, m0, n0);
  f32x4 acc[T::TM][T::TN];
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int j = 0; j < T::TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_ptr_t)ring;
  constexpr uint32_t SB = T::STAGE * 16;
#pragma unroll
  for (int i = 0; i < NS; ++i)
    if (k0 + i < k1) t.issue(base + i * SB, k0 + i);
  const int n = k1 - k0;
  if (n >= NS) wait_vm<(NS - 1) * T::L>();
  else wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  typename T::fragA_t a0, a1;
  typename T::fragB_t b0, b1;
  t.frags(ring, a0, b0);
  int slot = 0, kt = k0;
  auto step = [&](const typename T::fragA_t& ca, const typename T::fragB_t& cb, typename T::fragA_t& na, typename T::fragB_t& nb) {
    const int nx = slot + 1 == NS ? 0 : slot + 1;
    t.template stage<NS - 2, true>(ring + nx * T::STAGE, base + slot * SB, kt, ca, cb, na, nb, acc);
    slot = nx;
    ++kt;
  };
  // stages that refill a slot, two at a time (the two fragment sets keep fixed roles)
  for (; kt + NS + 1 < k1; ) {
    step(a0, b0, a1, b1);
    step(a1, b1, a0, b0);
  }
  if (kt + NS < k1) {
    step(a0, b0, a1, b1);
    t.template tail<NS - 2>(ring, slot, kt, k1, a1, b1, acc);
  } else {
    t.template tail<NS - 2>(ring, slot, kt, k1, a0, b0, acc);
  }
  // every load has landed (the last stage waited for all); once every wave has read its last fragments, the stage
  // buffers become epilogue slabs
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();
  constexpr int SLAB = 32 * T::WTN / 4;  // uint4 per wave slab
  static_assert(NS * T::STAGE >= T::NW * SLAB, "epilogue slabs do not fit");
  float4* st = (float4*)ring + t.wave * SLAB;
  if constexpr (EPI == EPI_PART) {
    GemmArgs h = g;
    h.C = (float*)g.C + (size_t)z * g.c_split;
    tile_store<EPI, 16, T::TM, T::TN, T::WTM, T::WTN>(h, acc, st, m0 + t.wm * T::WTM, n0 + t.wn * T::WTN, t.lane);
  } else {
    tile_store<EPI, 16, T::TM, T::TN, T::WTM, T::WTN>(g, acc, st, m0 + t.wm * T::WTM, n0 + t.wn * T::WTN, t.lane);
  }
}

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool TAPS>
hipError_t launch_ring(const GemmArgs& g, hipStream_t st) {
  const int S = EPI == EPI_PART ? g.splits : 1;
  const int gm = (g.M + BM - 1) / BM, gn = (g.N + BN - 1) / BN;
  // an XCD's tiles share W columns (column-major) or activation rows: the larger operand is the one that only one XCD
  // fetches
  const int colmajor = (long)g.M * (g.a_src ? g.lda : g.K) <= (long)g.N * g.K ? 1 : 0;
  hipLaunchKernelGGL((gemm_ring_kernel<BM, BN, WM, WN, NS, EPI, TAPS>), dim3(gm * gn * S), dim3(64 * WM * WN), 0, st, g, S, colmajor);
  return hipGetLastError();
}

// The qkv epilogue needs a whole head (64 columns) in one wave tile, so its wave grids differ.
template <int EPI, bool TAPS>
hipError_t ring_cfg(const GemmArgs& g, int cfg, hipStream_t st) {
  if constexpr (EPI == EPI_QKV) {
    switch (cfg) {
      case 0: return launch_ring<64, 64, 4, 1, 4, EPI, TAPS>(g, st);
      case 2: return launch_ring<128, 128, 4, 2, 3, EPI, TAPS>(g, st);
    }
  } else {
    switch (cfg) {
      case 0: return launch_ring<64, 64, 2, 2, 4, EPI, TAPS>(g, st);
      case 1: return launch_ring<128, 64, 4, 2, 4, EPI, TAPS>(g, st);
      case 2: return launch_ring<128, 128, 2, 4, 3, EPI, TAPS>(g, st);
    }
  }
  return hipErrorInvalidValue;
}

// Tile shapes with their fixed time, time per 64-K stage and most workgroups (in ns, one workgroup per CU; two 64x64
// workgroups share a CU without a second fixed part, and up to three rounds of them still beat the large tiles)
struct RingTile { int bm, bn, fixed, stage, most; };
constexpr RingTile RING[3] = {{64, 64, 3700, 165, 768}, {128, 64, 3800, 240, 256}, {128, 128, 5000, 340, 256}};

// ns of one call on RING[c] with K split S ways: rounds of 256 CUs, and for split sums their write and read by the row
// kernel (about 4.5 bytes per ns each way, most of it overlapped)
long ring_ns(int c, int M, int N, int K, int S) {
  const RingTile& t = RING[c];
  const long wgs = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * S;
  if (wgs > t.most) return -1;
  const long rounds = (wgs + 255) / 256;
  return t.fixed + rounds * ((K / 64 + S - 1) / S) * t.stage + (S > 1 ? (long)S * M * N * 4 / 4500 : 0);
}

}  // namespace

RingPlan ring_plan(int M, int N, int K, int max_splits, bool qkv) {
  RingPlan p{-1, 1};
  long best = -1;
  if (K % 64) return p;
  for (int c = 0; c < 3; ++c) {
    if (qkv && c == 1) continue;
    for (int S = 1; S <= max_splits && S <= K / 64; ++S) {
      const long ns = ring_ns(c, M, N, K, S);
      if (ns >= 0 && (best < 0 || ns < best)) best = ns, p.cfg = c, p.splits = S;
    }
  }
  return p;
}

bool gemm_ring_fits(const GemmArgs& g, int epi) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.w_scale || g.K % 64 || g.lda % 8 || g.ldb % 8) return false;
  if (((size_t)g.A | (size_t)g.B) & 15) return false;  // 16-byte copies
  const bool taps = g.a_src != nullptr;
  switch (epi) {
    case EPI_QKV: return !taps && g.qk.H % 64 == 0 && g.N == 3 * g.qk.H && !g.qk.rfreq;
    case EPI_PART: return g.splits >= 1 && g.splits <= 4 && g.splits <= g.K / 64 && g.ldc % 4 == 0 && ((size_t)g.C & 15) == 0 && g.c_split % 4 == 0;
    case EPI_F32: return g.ldc % 4 == 0 && ((size_t)g.C & 15) == 0;
    case EPI_GELU_BF16: case EPI_F16:
      if (taps) return false;
      [[fallthrough]];
    case EPI_BF16: case EPI_RESID_F16: return g.ldc % 8 == 0 && ((size_t)g.C & 15) == 0;
  }
  return false;
}

hipError_t gemm_ring(const GemmArgs& g, int epi, int cfg, hipStream_t st) {
  if (!gemm_ring_fits(g, epi)) return hipErrorInvalidValue;
  switch (epi * 2 + (g.a_src ? 1 : 0)) {
    case EPI_BF16 * 2: return ring_cfg<EPI_BF16, false>(g, cfg, st);
    case EPI_BF16 * 2 + 1: return ring_cfg<EPI_BF16, true>(g, cfg, st);
    case EPI_GELU_BF16 * 2: return ring_cfg<EPI_GELU_BF16, false>(g, cfg, st);
    case EPI_RESID_F16 * 2: return ring_cfg<EPI_RESID_F16, false>(g, cfg, st);
    case EPI_RESID_F16 * 2 + 1: return ring_cfg<EPI_RESID_F16, true>(g, cfg, st);
    case EPI_F16 * 2: return ring_cfg<EPI_F16, false>(g, cfg, st);
    case EPI_F32 * 2: return ring_cfg<EPI_F32, false>(g, cfg, st);
    case EPI_F32 * 2 + 1: return ring_cfg<EPI_F32, true>(g, cfg, st);
    case EPI_QKV * 2: return ring_cfg<EPI_QKV, false>(g, cfg, st);
    case EPI_PART * 2: return ring_cfg<EPI_PART, false>(g, cfg, st);
    case EPI_PART * 2 + 1: return ring_cfg<EPI_PART, true>(g, cfg, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace t2w
