// bf16 and fp8 MFMA GEMM for calls whose 256-row tile grids would leave most CUs idle: the K-split convs of a streaming
// window, several windows at once, prompt setups, batches of up to about 8,000 rows.
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
//   3600     27.5 -> 25.6     14.8 -> 11.9      32.9 -> 24.5     22.8 -> 20.1      25.4 -> 18.6
//   5000        -             19.7 -> 15.8      42.7 -> 33.6        -             30.4 -> 24.9
//   8000        -             22.0 -> 20.9      48.7 -> 44.1        -             35.1 -> 33.4
//
// 192x128 and 256x128 tiles (HALF) fill the chip once from ~4100 to ~8200 rows of N = 1024, where the 128x128 grid had
// just begun a second round.  fp8 (MX activations) runs on the same ring, 128 K values per stage, the activation scale
// dwords of a stage copied into its slot: solves of one window 35.2 -> 16.2 ms, two rows of 200-300 frames 36.2 -> 20.6,
// seven of 150-450 44.9 -> 40.3; bf16 batches of four rows of 250-400 frames 44.2 -> 37.1 and of nine 61.5 -> 56.0.
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

// HALF: the fragments of one 32-K step (fp8: 64) are in registers at a time and the barrier sits between the steps,
// for wave tiles whose whole-stage fragments would not fit next to their accumulators.
template <int BM, int BN, int WM, int WN, int NS, bool TAPS, bool FP8>
struct Ring {
  static constexpr int NW = WM * WN;
  static constexpr int MBE = FP8 ? 32 : 16;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / MBE, TN = WTN / MBE;
  static constexpr bool HALF = FP8 || TM * TN >= 12;
  static constexpr int APW = BM / 8 / NW, BPW = BN / 8 / NW;  // 1 KB load blocks (8 rows of 128 bytes) per wave and stage
  static constexpr int L = APW + BPW + (FP8 ? 1 : 0);
  static constexpr int SROWS = FP8 ? (BM + 63) / 64 : 0;            // 64-row blocks of activation scales
  static constexpr int STAGE = (BM + BN) * 8 + SROWS * 16;          // uint4 per stage: A rows, W rows, A's scale dwords
  static constexpr int ES = FP8 ? 1 : 2, BKE = BK * 2 / ES;         // bytes per element, K values per stage
  static_assert(APW * NW * 8 == BM && BPW * NW * 8 == BN, "load blocks must divide over the waves");
  static_assert(WTM % MBE == 0 && WTN % 32 == 0 && (!FP8 || WTM % 32 == 0), "wave tiles");
  static_assert(NS >= 3 && (NS - 1) * L < 64 && SROWS <= NW, "ring depth");
  typedef typename FragT<FP8>::type frag_t;
  typedef typename AccT<MBE>::type acc_t;

  uint32_t asrc[APW], bsrc[BPW], ssrc;
  const GemmArgs& g;
  int lane, wave, wm, wn;

  __device__ __forceinline__ Ring(const GemmArgs& g_, int m0, int n0) : g(g_) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wm = wave / WN;
    wn = wave % WN;
    const int lrow = lane >> 3;
    auto arow = [&](int trow) {
      const int m = min(m0 + trow, g.M - 1);  // rows past M load row M - 1; their results are never stored
      return (uint32_t)(TAPS ? g.a_src[m] : m);
    };
#pragma unroll
    for (int p = 0; p < APW; ++p) {
      const int trow = (wave + p * NW) * 8 + lrow;
      asrc[p] = arow(trow) * (uint32_t)(g.lda * ES) + ((lane & 7) ^ swz_key(trow)) * 16;
    }
#pragma unroll
    for (int p = 0; p < BPW; ++p) {
      const int trow = (wave + p * NW) * 8 + lrow;
      bsrc[p] = (uint32_t)min(n0 + trow, g.N - 1) * (uint32_t)(g.ldb * ES) + ((lane & 7) ^ swz_key(trow)) * 16;
    }
    // fp8: each wave copies 64 rows' scale dwords (waves beyond the tile's rows repeat a block, so that every wave has
    // the same number of copies in flight)
    ssrc = FP8 ? arow(min((wave % (SROWS ? SROWS : 1)) * 64 + lane, BM - 1)) * (uint32_t)g.a_sld : 0;
  }

  // Stage kt into the ring slot at LDS byte address `slot`.  The copies are inline assembly so that the compiler does
  // not count them: it would wait for every load in flight before the first fragment read of a loop, which is what
  // the ring is there to avoid; wait_vm and the barrier in stage() order them instead.  They have no output registers.
  __device__ __forceinline__ void dma(uint32_t lds, uint32_t off, const void* base) const {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
  }
  __device__ __forceinline__ void dma4(uint32_t lds, uint32_t off, const void* base) const {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
  }
  __device__ __forceinline__ void issue(uint32_t slot, int kt) const {
    const uint32_t koff = (uint32_t)kt * (BK * 2);  // taps: a row's frames follow each other, so K runs on across them
    if constexpr (FP8) dma4(slot + (BM + BN) * 128 + (wave % SROWS) * 256, ssrc + (uint32_t)kt * (BKE / 32), g.a_scale);
#pragma unroll
    for (int p = 0; p < BPW; ++p) dma(slot + BM * 128 + (wave + p * NW) * 1024, bsrc[p] + koff, g.B);
#pragma unroll
    for (int p = 0; p < APW; ++p) dma(slot + (wave + p * NW) * 1024, asrc[p] + koff, g.A);
  }

  // fragments of step kk of the stage in s; sc: fp8, the lane's activation scales (E8M0) of the step
  __device__ __forceinline__ void frag(const uint4* s, int kk, frag_t (&af)[TM], frag_t (&bf)[TN], int (&sc)[TM]) const {
    if constexpr (FP8) {
      const int c0 = kk * 4 + (lane >> 5);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = wn * WTN + j * 32 + (lane & 31);
        bf[j] = join8(s[BM * 8 + swz(r, c0)], s[BM * 8 + swz(r, c0 + 2)]);
      }
      const uint32_t* sw = (const uint32_t*)(s + (BM + BN) * 8);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = wm * WTM + i * 32 + (lane & 31);
        af[i] = join8(s[swz(r, c0)], s[swz(r, c0 + 2)]);
        sc[i] = (int)((sw[r] >> (8 * (kk * 2 + (lane >> 5)))) & 255u);
      }
    } else {
      const int chunk = kk * 4 + (lane >> 4);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = as_bf16x8(s[BM * 8 + swz(wn * WTN + j * 16 + (lane & 15), chunk)]);
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = as_bf16x8(s[swz(wm * WTM + i * 16 + (lane & 15), chunk)]);
    }
  }
  __device__ __forceinline__ void mma(const frag_t (&af)[TM], const frag_t (&bf)[TN], const int (&sc)[TM], acc_t (&acc)[TM][TN]) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (FP8) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[j], af[i], acc[i][j], 0, 0, 0, 127, 0, sc[i]);
        else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j], af[i], acc[i][j], 0, 0, 0);
      }
  }
  // NR LDS reads spread over NM MFMAs
  template <int NR, int NM>
  __device__ __forceinline__ void interleave() const {
#pragma unroll
    for (int x = 0; x < NM; ++x) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      constexpr int most = (NR + NM - 1) / NM;
      const int r = (x + 1) * NR / NM - x * NR / NM;
      if (r == most) __builtin_amdgcn_sched_group_barrier(0x100, most, 0);
      else if (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, most - 1, 0);
    }
  }
  template <int AFTER>
  __device__ __forceinline__ void meet() const {
    wait_vm<AFTER * L>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }

  // a stage's fragments: both steps, or (HALF) one at a time in turn
  struct Frags {
    frag_t a[2][TM], b[2][TN];
    int s[2][TM];
  };
  static constexpr int RPF = FP8 ? 2 : 1, NR = (TM + TN) * RPF + (FP8 ? TM : 0), NM = TM * TN;
  __device__ __forceinline__ void first(const uint4* s, Frags& f) const {
    frag(s, 0, f.a[0], f.b[0], f.s[0]);
    if (!HALF) frag(s, 1, f.a[1], f.b[1], f.s[1]);
  }

  // Stage kt, whose fragments (HALF: those of its first step) are in c: wait until stage kt + 1 has landed (AFTER
  // stages behind it may be in flight), meet the other waves (their copies of it have landed too, and everybody has
  // read stage kt out of its slot), refill that slot with stage kt + NS, read the next fragments while the MFMAs run.
  template <int AFTER, bool REFILL>
  __device__ __forceinline__ void stage(const uint4* cur, const uint4* next, uint32_t refill, int kt, Frags& c, Frags& n,
                                        acc_t (&acc)[TM][TN]) const {
    if constexpr (HALF) {
      frag(cur, 1, c.a[1], c.b[1], c.s[1]);
      mma(c.a[0], c.b[0], c.s[0], acc);
      interleave<NR, NM>();
      meet<AFTER>();
      if (REFILL) issue(refill, kt + NS);
      frag(next, 0, c.a[0], c.b[0], c.s[0]);
      mma(c.a[1], c.b[1], c.s[1], acc);
      interleave<NR, NM>();
    } else {
      meet<AFTER>();
      if (REFILL) issue(refill, kt + NS);
      first(next, n);
      mma(c.a[0], c.b[0], c.s[0], acc);
      mma(c.a[1], c.b[1], c.s[1], acc);
      interleave<2 * NR, 2 * NM>();
    }
    asm volatile("" ::: "memory");
  }
  __device__ __forceinline__ void last(const uint4* cur, Frags& c, acc_t (&acc)[TM][TN]) const {
    if (HALF) frag(cur, 1, c.a[1], c.b[1], c.s[1]);
    mma(c.a[0], c.b[0], c.s[0], acc);
    mma(c.a[1], c.b[1], c.s[1], acc);
  }
  // stages kt .. k1 - 1, at most REM + 1 of them behind the one in registers
  template <int REM>
  __device__ __forceinline__ void tail(const uint4* ring, int slot, int kt, int k1, Frags& c, acc_t (&acc)[TM][TN]) const {
    if constexpr (REM >= 0) {
      if (kt + 1 + REM < k1) {
        Frags n;
        const int nx = slot + 1 == NS ? 0 : slot + 1;
        stage<REM, false>(ring + slot * STAGE, ring + nx * STAGE, 0, kt, c, n, acc);
        tail<REM - 1>(ring, nx, kt + 1, k1, HALF ? c : n, acc);
      } else {
        tail<REM - 1>(ring, slot, kt, k1, c, acc);
      }
    } else {
      last(ring + slot * STAGE, c, acc);
    }
  }
};

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool TAPS, bool FP8>
__global__ void __launch_bounds__(64 * WM * WN) gemm_ring_kernel(GemmArgs g, int S, int colmajor) {
  typedef Ring<BM, BN, WM, WN, NS, TAPS, FP8> T;
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
  const int KT = g.K / T::BKE, k0 = z * KT / S, k1 = (z + 1) * KT / S;

  T t(g, m0, n0);
  typename T::acc_t acc[T::TM][T::TN];
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int j = 0; j < T::TN; ++j)
#pragma unroll
      for (int r = 0; r < (int)(sizeof(typename T::acc_t) / 4); ++r) acc[i][j][r] = 0.0f;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_ptr_t)ring;
  constexpr uint32_t SB = T::STAGE * 16;
#pragma unroll
  for (int i = 0; i < NS; ++i)
    if (k0 + i < k1) t.issue(base + i * SB, k0 + i);
  if (k1 - k0 >= NS) t.template meet<NS - 1>();
  else t.template meet<0>();
  typename T::Frags f0, f1;
  t.first(ring, f0);
  int slot = 0, kt = k0;
  auto step = [&](typename T::Frags& c, typename T::Frags& n) {
    const int nx = slot + 1 == NS ? 0 : slot + 1;
    t.template stage<NS - 2, true>(ring + slot * T::STAGE, ring + nx * T::STAGE, base + slot * SB, kt, c, n, acc);
    slot = nx;
    ++kt;
  };
  if constexpr (T::HALF) {
    while (kt + NS < k1) step(f0, f0);
    t.template tail<NS - 2>(ring, slot, kt, k1, f0, acc);
  } else {
    // stages that refill a slot, two at a time (the two fragment sets keep fixed roles)
    while (kt + NS + 1 < k1) {
      step(f0, f1);
      step(f1, f0);
    }
    if (kt + NS < k1) {
      step(f0, f1);
      t.template tail<NS - 2>(ring, slot, kt, k1, f1, acc);
    } else {
      t.template tail<NS - 2>(ring, slot, kt, k1, f0, acc);
    }
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
    tile_store<EPI, T::MBE, T::TM, T::TN, T::WTM, T::WTN>(h, acc, st, m0 + t.wm * T::WTM, n0 + t.wn * T::WTN, t.lane);
  } else {
    tile_store<EPI, T::MBE, T::TM, T::TN, T::WTM, T::WTN>(g, acc, st, m0 + t.wm * T::WTM, n0 + t.wn * T::WTN, t.lane);
  }
}

template <int BM, int BN, int WM, int WN, int NS, int EPI, bool TAPS, bool FP8 = false>
hipError_t launch_ring(const GemmArgs& g, hipStream_t st) {
  const int S = EPI == EPI_PART ? g.splits : 1;
  const int gm = (g.M + BM - 1) / BM, gn = (g.N + BN - 1) / BN;
  // an XCD's tiles share W columns (column-major) or activation rows: the larger operand is the one that only one XCD
  // fetches
  const int colmajor = (long)g.M * (g.a_src ? g.lda : g.K) <= (long)g.N * g.K ? 1 : 0;
  hipLaunchKernelGGL((gemm_ring_kernel<BM, BN, WM, WN, NS, EPI, TAPS, FP8>), dim3(gm * gn * S), dim3(64 * WM * WN), 0, st, g, S, colmajor);
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
  if constexpr (EPI != EPI_PART) {
    if (cfg == 3) return launch_ring<192, 128, 4, 2, 3, EPI, TAPS>(g, st);
    if (cfg == 4) return launch_ring<256, 128, 4, 2, 3, EPI, TAPS>(g, st);
  }
  return hipErrorInvalidValue;
}

template <int EPI, bool TAPS>
hipError_t ring_cfg8(const GemmArgs& g, int cfg, hipStream_t st) {
  if constexpr (EPI == EPI_QKV) {
    if (cfg == 0) return launch_ring<64, 64, 2, 1, 4, EPI, TAPS, true>(g, st);
  } else {
    switch (cfg) {
      case 0: return launch_ring<64, 64, 2, 2, 4, EPI, TAPS, true>(g, st);
      case 1: return launch_ring<128, 64, 4, 2, 4, EPI, TAPS, true>(g, st);
      case 3: return launch_ring<192, 128, 2, 4, 3, EPI, TAPS, true>(g, st);
    }
  }
  if (cfg == 2) return launch_ring<128, 128, 4, 2, 3, EPI, TAPS, true>(g, st);
  if (cfg == 4) return launch_ring<256, 128, 4, 2, 3, EPI, TAPS, true>(g, st);
  return hipErrorInvalidValue;
}

// Tile shapes with their fixed time, time per stage of 128-byte rows and most workgroups (in ns, one workgroup per CU;
// two 64x64 workgroups share a CU without a second fixed part, and up to three rounds of them still beat the large
// tiles; a second round of the others loses to the two-buffer grids)
struct RingTile { int bm, bn, fixed, stage, most; };
constexpr RingTile RING[5] = {{64, 64, 3700, 175, 768}, {128, 64, 3800, 240, 256}, {128, 128, 5000, 370, 256},
                              {192, 128, 6900, 540, 256}, {256, 128, 8600, 670, 256}};

// ns of one call on RING[c] with K of KT stages split S ways: rounds of 256 CUs, and for split sums their write and read
// by the row kernel (about 4.5 bytes per ns each way, most of it overlapped)
long ring_ns(int c, int M, int N, int KT, int S) {
  const RingTile& t = RING[c];
  const long wgs = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * S;
  if (wgs > t.most) return -1;
  const long rounds = (wgs + 255) / 256;
  return t.fixed + rounds * ((KT + S - 1) / S) * t.stage + (S > 1 ? (long)S * M * N * 4 / 4500 : 0);
}

}  // namespace

RingPlan ring_plan(int M, int N, int K, int max_splits, bool qkv, bool fp8) {
  RingPlan p{-1, 1};
  long best = -1;
  const int ke = fp8 ? 128 : 64;
  if (K % ke) return p;
  for (int c = 0; c < 5; ++c) {
    if (qkv && (c == 1 || (fp8 && c == 3) || N % RING[c].bn)) continue;
    for (int S = 1; S <= (c < 3 ? max_splits : 1) && S <= K / ke; ++S) {
      const long ns = ring_ns(c, M, N, K / ke, S);
      if (ns >= 0 && (best < 0 || ns < best)) best = ns, p.cfg = c, p.splits = S;
    }
  }
  return p;
}

bool gemm_ring_fits(const GemmArgs& g, int epi) {
  const bool taps = g.a_src != nullptr;
  if (g.M <= 0 || g.N <= 0 || g.K <= 0 || (((size_t)g.A | (size_t)g.B) & 15)) return false;  // 16-byte copies
  // both operands are addressed by 32-bit byte offsets (taps: frame rows up to M + 65536)
  const size_t es = g.w_scale ? 1 : 2;
  if (((size_t)g.M + 65536) * g.lda * es >= ((size_t)1 << 32) || (size_t)g.N * g.ldb * es >= ((size_t)1 << 32)) return false;
  if (g.w_scale) {
    // codes and scale dwords (4 blocks of 32 K values); taps: the scale rows run on across frames like the codes
    if (g.K % 128 || g.lda % 16 || g.ldb % 16 || g.a_sld % 4 || ((size_t)g.a_scale & 3) || (taps && g.a_sld * 32 != g.lda)) return false;
    if (epi == EPI_GELU_MX8) return !taps && g.c_scale && g.N % 32 == 0 && g.ldc % 4 == 0 && ((size_t)g.C & 3) == 0;
  } else {
    if (g.K % 64 || g.lda % 8 || g.ldb % 8) return false;
  }
  switch (epi) {
    case EPI_QKV: return !taps && g.qk.H % 64 == 0 && g.N == 3 * g.qk.H && !g.qk.rfreq;
    case EPI_PART:
      return !g.w_scale && g.splits >= 1 && g.splits <= 4 && g.splits <= g.K / 64 && g.ldc % 4 == 0 && ((size_t)g.C & 15) == 0 &&
             g.c_split % 4 == 0;
    case EPI_F32: return !g.w_scale && g.ldc % 4 == 0 && ((size_t)g.C & 15) == 0;
    case EPI_GELU_BF16: case EPI_F16:
      if (taps || g.w_scale) return false;
      [[fallthrough]];
    case EPI_BF16: case EPI_RESID_F16: return g.ldc % 8 == 0 && ((size_t)g.C & 15) == 0;
  }
  return false;
}

hipError_t gemm_ring(const GemmArgs& g, int epi, int cfg, hipStream_t st) {
  if (cfg < 0 || cfg >= 5 || !gemm_ring_fits(g, epi)) return hipErrorInvalidValue;
  // the qkv store has no column guard: columns past N would be written as one more head of v
  if (epi == EPI_QKV && g.N % RING[cfg].bn) return hipErrorInvalidValue;
  const int e = epi * 2 + (g.a_src ? 1 : 0);
  if (g.w_scale) {
    switch (e) {
      case EPI_BF16 * 2: return ring_cfg8<EPI_BF16, false>(g, cfg, st);
      case EPI_BF16 * 2 + 1: return ring_cfg8<EPI_BF16, true>(g, cfg, st);
      case EPI_RESID_F16 * 2: return ring_cfg8<EPI_RESID_F16, false>(g, cfg, st);
      case EPI_RESID_F16 * 2 + 1: return ring_cfg8<EPI_RESID_F16, true>(g, cfg, st);
      case EPI_GELU_MX8 * 2: return ring_cfg8<EPI_GELU_MX8, false>(g, cfg, st);
      case EPI_QKV * 2: return ring_cfg8<EPI_QKV, false>(g, cfg, st);
    }
    return hipErrorInvalidValue;
  }
  switch (e) {
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
