// Main loops of the bf16 GEMM whose two operands both go HBM/L2 -> LDS by
// buffer DMA: C[M,P] = A[M,Q] * B, B given either as [P][Q] rows (NN = false)
// or as [Q][P] rows (NN = true, read transposed by ds_read_b64_tr_b16).
// v_mfma_f32_16x16x32_bf16 with fp32 accumulation.
//
// What bounds it: at full load the card lowers its clock (a 4096^3 product
// takes 106 us on random operands and 78 us on zeros, the same instructions),
// so bytes moved per flop count as much as latency.  A 128x64 wave tile (256x256)
// reads 24 KiB of LDS per k-step of 1 MFLOP, the 64x64 one (256x128) 16 KiB
// per half of that;
// 16x16x32 ran 4-5% faster than 32x32x16 at full load (down-projection shape
// 2048 x 4096 x 14336: 186 against 194 us), and equally fast on zeros.
#pragma once
#include <type_traits>

#include "common.h"

namespace st {

// s_waitcnt for at most VM vector-memory and LGKM LDS/scalar operations in
// flight (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 7 = no wait,
// lgkmcnt in bits 11:8; VM = 63 / LGKM = 15 leave that counter alone)
template <int VM, int LGKM = 15>
__device__ __forceinline__ void wait_cnt() {
  static_assert(VM >= 0 && VM < 64 && LGKM >= 0 && LGKM < 16, "counter range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (LGKM << 8) | ((VM >> 4) << 14));
}
// Workgroup barrier without the fence of __syncthreads (which would also wait
// for every LDS DMA in flight): the caller first waits for exactly the
// operations other waves depend on.  The memory clobber keeps the compiler
// from moving memory accesses across it.
__device__ __forceinline__ void bar() { asm volatile("s_barrier" ::: "memory"); }

// Chunk swizzles (16-byte chunks; both are XORs, so a DMA lane applies the
// same one to its source address).  Rows of 64 contraction elements: the 16
// rows of a quarter-wave read hit distinct banks.  [k][BN] rows: the 8 rows
// of 32 bytes that a half-wave's transposing read takes hit distinct banks.
__device__ __forceinline__ int dma_kswz(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int dma_nswz(int n) { return 2 * ((n & 3) | ((n >> 1) & 4)); }

// B operand of a 16x16x32 MFMA from a [k][BN] tile: lane (column kc + lane%16,
// quarter g = lane/16) gets rows n0 + 8g .. +7.  The tile is read through a
// __restrict__ pointer: the caller has waited for the tile's DMAs and passed
// the barrier, and without it the compiler waits for every DMA in flight.
template <int BN>
__device__ __forceinline__ bf16x8 tr_operand16(const uint4* __restrict__ bs, int n0, int kc,
                                               int lane) {
  typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
  const int g = lane >> 4, i = lane & 15, col = kc + 4 * (i & 3);
  v4bf r[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int n = n0 + 8 * g + 4 * h + (i >> 2);
    const uint16_t* e =
        (const uint16_t*)(bs + n * (BN / 8) + ((col >> 3) ^ dma_nswz(n))) + (col & 7);
    r[h] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) v4bf*)e);
  }
  return __builtin_shufflevector(r[0], r[1], 0, 1, 2, 3, 4, 5, 6, 7);
}

// Instruction order of one phase: an LDS read after each of the first NR of
// NM MFMAs, so the next phase's fragments arrive under this phase's products
// (reads first, free scheduling and groups of four measured 2-6% slower).
template <int NR, int NM>
__device__ __forceinline__ void dma_order() {
#pragma unroll
  for (int i = 0; i < NM; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (i < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// one 1 KiB DMA: lane l's 16 bytes at byte offset voff (+ scalar soff) of rs go to dst[l]
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, uint4* dst, uint32_t voff,
                                      uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16,
                                           (int)voff, (int)soff, 0, 0);
}

struct DmaOperands {
  const uint16_t *A, *B;
  int64_t lda, ldb, a_bytes, b_bytes;
};

// 16-byte chunk (of the 8 of a k-step) that lane quarter g of slice sl takes.
// Natural order, or (PERM) the order of the register-operand 4-bit forward,
// whose 16-deep slices pair chunks s and 4 + s: the same sums in the same order.
template <bool PERM>
__device__ __forceinline__ int dma_chunk(int sl, int g) {
  return PERM ? 2 * sl + (g >> 1) + 4 * (g & 1) : 4 * sl + g;
}

// DMA side of a workgroup: each wave moves DA + DB instructions of 64 16-byte
// chunks per k-step of 64.  Lane offsets are fixed; the k-step moves the
// scalar offset.  Rows past the operand and contraction elements past Q start
// at kOOB and read as zero; whole k-steps carry no checks.  K-steps past the
// last are issued all the same (zeros), which keeps the wait counts static.
template <bool NN, int BM, int BN, int WAVES>
struct DmaTile {
  static constexpr int DA = BM * 8 / 64 / WAVES, DB = BN * 8 / 64 / WAVES;
  uint32_t va[DA], vb[DB], bstep;
  __amdgpu_buffer_rsrc_t rsA, rsB;
  int KF, KT, Q, wave, lane;

  __device__ __forceinline__ DmaTile(const DmaOperands& o, int m0, int M, int p0, int P, int Q_,
                                     int wave_, int lane_)
      : rsA(make_rsrc(o.A, o.a_bytes)), rsB(make_rsrc(o.B, o.b_bytes)), Q(Q_), wave(wave_),
        lane(lane_) {
    KT = (Q + 63) / 64;
    KF = Q / 64;
    bstep = NN ? (uint32_t)(64 * o.ldb * 2) : 128u;
#pragma unroll
    for (int q = 0; q < DA; ++q) {
      const int row = a_row(q), c = (lane & 7) ^ dma_kswz(row);
      va[q] = m0 + row < M ? (uint32_t)(((m0 + row) * o.lda + c * 8) * 2) : kOOB;
    }
#pragma unroll
    for (int q = 0; q < DB; ++q) {
      if constexpr (NN) {
        const int n = b_row(q), c = (lane % (BN / 8)) ^ dma_nswz(n);
        vb[q] = p0 + c * 8 < P ? (uint32_t)((n * o.ldb + p0 + c * 8) * 2) : kOOB;
      } else {
        const int row = b_row(q), c = (lane & 7) ^ dma_kswz(row);
        vb[q] = p0 + row < P ? (uint32_t)(((p0 + row) * o.ldb + c * 8) * 2) : kOOB;
      }
    }
  }
  // tile row that this lane's chunk of instruction q belongs to
  __device__ __forceinline__ int a_row(int q) const { return (wave * DA + q) * 8 + (lane >> 3); }
  __device__ __forceinline__ int b_row(int q) const {
    return NN ? ((wave * DB + q) * 64 + lane) / (BN / 8) : (wave * DB + q) * 8 + (lane >> 3);
  }
  // instructions [Q0, Q0 + QN) of operand A (B) of k-step kt
  template <int Q0 = 0, int QN = DA>
  __device__ __forceinline__ void a(int kt, uint4* slot) const {
    uint4* dst = slot + wave * DA * 64;
    const uint32_t soff = kt < KT ? (uint32_t)kt * 128u : 0u;
    if (kt < KF) {
#pragma unroll
      for (int q = Q0; q < Q0 + QN; ++q) dma16(rsA, dst + q * 64, va[q], soff);
    } else {
      const int rem = Q - kt * 64;
#pragma unroll
      for (int q = Q0; q < Q0 + QN; ++q) {
        const int k = ((lane & 7) ^ dma_kswz(a_row(q))) * 8;
        dma16(rsA, dst + q * 64, k < rem ? va[q] : kOOB, soff);
      }
    }
  }
  template <int Q0 = 0, int QN = DB>
  __device__ __forceinline__ void b(int kt, uint4* slot) const {
    uint4* dst = slot + wave * DB * 64;
    const uint32_t soff = kt < KT ? (uint32_t)kt * bstep : 0u;
    if (kt < KF) {
#pragma unroll
      for (int q = Q0; q < Q0 + QN; ++q) dma16(rsB, dst + q * 64, vb[q], soff);
    } else {
      const int rem = Q - kt * 64;
#pragma unroll
      for (int q = Q0; q < Q0 + QN; ++q) {
        const int k = NN ? b_row(q) : ((lane & 7) ^ dma_kswz(b_row(q))) * 8;
        dma16(rsB, dst + q * 64, k < rem ? vb[q] : kOOB, soff);
      }
    }
  }
};

// 256x256 tile, 8 waves (two per SIMD) of 128x64.  A k-step of 64 is four
// phases of 16 MFMAs: (slice 0, rows 0-63), (0, 64-127), (1, 0-63), (1,
// 64-127) of the wave's rows.  One barrier per k-step, before the last phase:
// every wave has then read the step's operands, so A(kt+2) and B(kt+3) may go
// into their slots (two A and three B slots of 32 KiB: all of the LDS; the
// weights come from farther away than the activations, and a third slot for
// B was worth 2-8% over two, a third one for A less).  Each phase issues two
// of the eight DMAs: all eight behind the barrier filled the address unit's
// queue and held the waves back (2048 x 4096 x 4096 on half the CUs 92 -> 80
// us, 2048 x 28672 x 4096 409 -> 393).
template <bool NN, bool PERM>
struct DmaLoop256 {
  static constexpr bool NN_B = NN;
  static_assert(!(NN && PERM), "PERM: [P][Q] weights only");
  static constexpr int BM = 256, BN = 256, WAVES = 8, NT = 512, WM = 128, WN = 64, WAVES_N = 4;
  static constexpr int FM = 8, FN = 4, SLOT = 2048, AST = 2, BST = 3;
  static constexpr int LDS16 = (AST + BST) * SLOT, MIN_WG_WAVES = 1;

  static __device__ __forceinline__ void run(const DmaOperands& o, uint4* lds, int m0, int M,
                                             int p0, int P, int Q, int wave, int lane,
                                             f32x4 (&acc)[FM][FN]) {
    const DmaTile<NN, BM, BN, WAVES> d(o, m0, M, p0, P, Q, wave, lane);
    uint4 *const As = lds, *const Bs = lds + AST * SLOT;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int lr = lane & 15, lh = lane >> 4, f = dma_kswz(lr);
    const int a_lane = (wm * WM + lr) * 8, b_lane = (wn * WN + lr) * 8;
    bf16x8 a0[4], a1[4], b0[4], b1[4];
    auto read_a = [&](const uint4* __restrict__ s, int sl, int half, bf16x8 (&a)[4]) {
      const uint4* p = s + a_lane + half * 64 * 8 + (dma_chunk<PERM>(sl, lh) ^ f);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = __builtin_bit_cast(bf16x8, p[i * 16 * 8]);
    };
    auto read_b = [&](const uint4* __restrict__ s, int sl, bf16x8 (&b)[4]) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (NN)
          b[j] = tr_operand16<BN>(s, sl * 32, wn * WN + j * 16, lane);
        else
          b[j] = __builtin_bit_cast(bf16x8, s[b_lane + (dma_chunk<PERM>(sl, lh) ^ f) + j * 16 * 8]);
      }
    };
    auto mfmas = [&](int half, const bf16x8 (&a)[4], const bf16x8 (&b)[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[half * 4 + i][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[half * 4 + i][j], 0, 0, 0);
    };
    constexpr int RB = NN ? 8 : 4;  // LDS reads of a slice's B fragments
    constexpr int DT = 4;           // DMAs per wave and slot
    static_assert(d.DA == DT && d.DB == DT, "wait counts below");
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.0f;

    // A0 B0 | half of A1, B1: all but the first pair may be in flight
    d.a(0, As);
    d.b(0, Bs);
    d.template a<0, 2>(1, As + SLOT);
    d.b(1, Bs + SLOT);
    wait_cnt<2 + DT>();
    bar();
    read_a(As, 0, 0, a0);
    read_b(Bs, 0, b0);
    int as = 0, bs = 0;
#pragma unroll 1
    for (int kt = 0; kt < d.KT; ++kt) {
      uint4 *const A = As + as * SLOT, *const B = Bs + bs * SLOT;
      as ^= 1;
      uint4* const A1 = As + as * SLOT;
      uint4* const B2 = Bs + (bs == 0 ? BST - 1 : bs - 1) * SLOT;  // of kt-1, and kt+2
      bs = bs == BST - 1 ? 0 : bs + 1;
      d.template a<2, 2>(kt + 1, A1);
      read_a(A, 0, 1, a1);
      read_b(B, 1, b1);
      mfmas(0, a0, b0);
      dma_order<4 + RB, 16>();
      d.template b<0, 2>(kt + 2, B2);
      read_a(A, 1, 0, a0);
      mfmas(1, a1, b0);
      dma_order<4, 16>();
      d.template b<2, 2>(kt + 2, B2);
      read_a(A, 1, 1, a1);
      mfmas(0, a0, b1);
      dma_order<4, 16>();
      // step kt+1 has landed (this step's B(kt+2) may be in flight) and this
      // wave's reads of step kt are done
      wait_cnt<DT, 0>();
      bar();
      d.template a<0, 2>(kt + 2, A);
      read_a(A1, 0, 0, a0);
      read_b(Bs + bs * SLOT, 0, b0);
      mfmas(1, a1, b1);
      dma_order<4 + RB, 16>();
    }
    wait_cnt<0, 0>();
    __syncthreads();
  }
};

// (64 WM) x (64 WN) tile of 64x64 wave tiles, ST slots of a whole k-step, one
// phase of 16 MFMAs per 32-deep slice, one barrier per k-step before its last
// phase.  <4, 2, 3>: 256x128, one workgroup per CU.  <2, 2, 2>: 128x128, two
// workgroups per CU, each with 64 KiB.  <2, 2, 4>: 128x128 alone on a CU with
// two more steps in flight.  With three slots or more B's DMAs go out in the
// first phase and A's in the second (3-5% faster than both behind the
// barrier); with two there is no step to spare and both follow the barrier.
template <bool NN, bool PERM, int WMS, int WNS, int ST>
struct DmaLoop64 {
  static constexpr bool NN_B = NN;
  static_assert(!(NN && PERM), "PERM: [P][Q] weights only");
  static constexpr int WM = 64, WN = 64, BM = WM * WMS, BN = WN * WNS, WAVES = WMS * WNS;
  static constexpr int NT = 64 * WAVES, WAVES_N = WNS, FM = 4, FN = 4;
  static constexpr int AS = BM * 8, BS = BN * 8, LDS16 = ST * (AS + BS);
  static constexpr int MIN_WG_WAVES = LDS16 * 16 <= 80 * 1024 ? 2 : 1;

  static __device__ __forceinline__ void run(const DmaOperands& o, uint4* lds, int m0, int M,
                                             int p0, int P, int Q, int wave, int lane,
                                             f32x4 (&acc)[FM][FN]) {
    const DmaTile<NN, BM, BN, WAVES> d(o, m0, M, p0, P, Q, wave, lane);
    constexpr int D = d.DA + d.DB;
    uint4 *const As = lds, *const Bs = lds + ST * AS;
    const int wm = wave / WNS, wn = wave % WNS;
    const int lr = lane & 15, lh = lane >> 4, f = dma_kswz(lr);
    const int a_lane = (wm * WM + lr) * 8, b_lane = (wn * WN + lr) * 8;
    bf16x8 a[2][4], b[2][4];
    auto read = [&](const uint4* __restrict__ sa, const uint4* __restrict__ sb, int sl,
                    bf16x8 (&x)[4], bf16x8 (&y)[4]) {
      const uint4* p = sa + a_lane + (dma_chunk<PERM>(sl, lh) ^ f);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = __builtin_bit_cast(bf16x8, p[i * 16 * 8]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (NN)
          y[j] = tr_operand16<BN>(sb, sl * 32, wn * WN + j * 16, lane);
        else
          y[j] = __builtin_bit_cast(bf16x8, sb[b_lane + (dma_chunk<PERM>(sl, lh) ^ f) + j * 16 * 8]);
      }
    };
    auto mfmas = [&](const bf16x8 (&x)[4], const bf16x8 (&y)[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i], y[j], acc[i][j], 0, 0, 0);
    };
    constexpr int NR = NN ? 12 : 8;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.0f;
    constexpr bool SPREAD = ST > 2;  // B(kt+ST-1) is issued in step kt's first phase
#pragma unroll
    for (int j = 0; j < ST; ++j) {
      d.a(j, As + j * AS);
      if (!SPREAD || j < ST - 1) d.b(j, Bs + j * BS);
    }
    wait_cnt<D*(ST - 1) - (SPREAD ? d.DB : 0)>();
    bar();
    read(As, Bs, 0, a[0], b[0]);
    int s = 0;
#pragma unroll 1
    for (int kt = 0; kt < d.KT; ++kt) {
      uint4 *const A = As + s * AS, *const B = Bs + s * BS;
      if constexpr (SPREAD) d.b(kt + ST - 1, Bs + (s == 0 ? ST - 1 : s - 1) * BS);
      s = s + 1 == ST ? 0 : s + 1;
      read(A, B, 1, a[1], b[1]);
      mfmas(a[0], b[0]);
      dma_order<NR, 16>();
      wait_cnt<D*(ST - 2), 0>();
      bar();
      d.a(kt + ST, A);
      if constexpr (!SPREAD) d.b(kt + ST, B);
      read(As + s * AS, Bs + s * BS, 0, a[0], b[0]);
      mfmas(a[1], b[1]);
      dma_order<NR, 16>();
    }
    wait_cnt<0, 0>();
    __syncthreads();
  }
};

}  // namespace st
