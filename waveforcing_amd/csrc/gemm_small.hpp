// GEMM for outputs that do not fill the GPU with the 128 x 256 / 256 x 256 tiles of gemm_w8a8.hip, and for the
// bf16 linears: y[m,n] = epilogue(sum_k a[m,k] * w[n,k]), int8, e4m3 or bf16 operands.
//
// What bounds it: with few tiles neither the matrix cores nor memory, but the time of one K step in a workgroup
// (barrier, fragment reads, a chain of MFMAs) times the steps, and below that the operand stream, (BM + BN) rows
// of K through the 64 B/clk vector-memory path of one CU.  So the tiles are small (more CUs share the stream), the
// smallest keep two kinds of work side by side, fragments are read a step ahead of their MFMAs, and the LDS ring keeps
// up to ST - 1 steps in flight.  Side by side: int8 splits K over groups of waves (int32 sums have the same bits in any
// order); bf16, whose fp32 sums do not, gives the DMAs to waves of their own.  Bytes move global -> LDS by DMA in
// the layout of gemm_w8a8.hip (1 KB blocks of 8 rows, K chunks swizzled by the row), and every fp32 sum takes the
// same MFMAs in the same K order as there and in the other bf16 kernels: the bits of an output do not depend on
// the tile, nor on the call's other rows.
//
// One K step (DN = 0): wait for the own DMAs of step kb, barrier (every wave's have landed and every wave is done with
// step kb - 1's stage), read step kb's fragments, DMA step kb + ST - 1 into that freed stage, then the MFMAs of
// step kb - 1.  DMAs past K read zeros into stages that nobody reads any more.  With DN loading waves these wait and
// DMA, the others read and multiply, and the barrier of a step joins both.
#pragma once

#include <type_traits>

#include "gemm_core.hpp"

namespace wf {
namespace gemm {

// BM x BN outputs per workgroup of KS groups of WM x WN waves, each wave (BM / WM) x (BN / WN) in 32 x 32 blocks;
// group g takes K steps g, g + KS, ... of U x 128 bytes through its own ring of ST LDS stages, and the groups' sums
// are added at the end (int8 only: KS > 1 changes the order of sums).  DN > 0: DN more waves issue all DMAs.
template <int BM_, int BN_, int WM_, int WN_, int ST_, int KS_ = 1, int U_ = 1, int DN_ = 0>
struct SmallTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, ST = ST_, KS = KS_, U = U_, DN = DN_;
  static constexpr int NW = WM * WN, THREADS = (KS * NW + DN) * 64;  // NW: waves of one group
  static constexpr int NL = DN > 0 ? DN : NW;                        // waves that load
  static constexpr int MI = BM / WM / 32, NI = BN / WN / 32;
  static constexpr int NBA = BM / 8 / NL, NBB = BN / 8 / NL, NDMA = NBA + NBB;
  static constexpr int CHUNK = (BM + BN) * BK, STAGE = U * CHUNK;
  static constexpr int WPITCH = BN / WN * 2 + 16;   // row pitch of a wave's 32-row output slab
  static constexpr int SLABS = MI > 1 ? 2 : 1;
  static_assert(MI >= 1 && NI >= 1 && MI * WM * 32 == BM && NI * WN * 32 == BN, "32 x 32 blocks");
  static_assert(NBA * 8 * NL == BM && NBB * 8 * NL == BN, "DMA blocks");
  static_assert(ST >= 3 && U * NDMA * (ST - 2) < 64, "outstanding DMAs");
  static constexpr int LDS = KS * ST * STAGE;
  static constexpr int ACC = MI * NI * 64 * 64;     // one wave's sums (bytes)
  static_assert(NW * SLABS * 32 * WPITCH <= LDS && LDS <= 160 * 1024, "LDS of one workgroup");
  static_assert(DN == 0 || KS == 1, "loading waves of their own serve one group");
  static_assert(KS == 1 || (KS - 1) * NW * ACC <= LDS, "the groups' sums fit the stages");
};

struct SmallArgs {
  const void* a;         // [M] rows of kb bytes, lda bytes apart
  const void* w;         // [N] rows of kb bytes
  const float* sx;       // int8: [M];  e4m3: [1]
  const float* sw;       // int8: [N];  e4m3: [1]
  const uint16_t* bias;  // [N] bf16 or null
  uint16_t* y;           // [M, N] bf16 (ldy)
  int M, N, kb, lda;
  int64_t ldy;
  int vec16;             // y and ldy allow 16-byte row stores
  int bias8;             // bias is 8-byte aligned
};

// ACT, on the bf16 result: 0 none, 1 SiLU, 2 GELU(tanh).
template <typename T, typename OP, int ACT>
__global__ __launch_bounds__(T::THREADS) void gemm_small_kernel(SmallArgs p) {
  constexpr int BM = T::BM, BN = T::BN, WN = T::WN, NW = T::NW, MI = T::MI, NI = T::NI, ST = T::ST;
  constexpr int STAGE = T::STAGE, NBA = T::NBA, NDMA = T::NDMA, WPITCH = T::WPITCH;
  constexpr bool kI8 = std::is_same<OP, OpI8>::value, kFp8 = std::is_same<OP, OpFp8>::value;
  constexpr int SUB = OP::SUB, PIECES = OP::PIECES;
  constexpr int CPS = BK / 16 / SUB;
  constexpr int KS = T::KS, U = T::U, DN = T::DN, NL = T::NL;
  __shared__ __attribute__((aligned(1024))) uint8_t lds_all[T::LDS];

  // Tiles in bands of GROUP_M tile rows swept column by column, a contiguous range of them per XCD.
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  const int n_tiles = tiles_m * tiles_n;
  const int per_xcd = (n_tiles + NUM_XCD - 1) / NUM_XCD;
  const int t = (blockIdx.x % NUM_XCD) * per_xcd + blockIdx.x / NUM_XCD;
  if (blockIdx.x / NUM_XCD >= per_xcd || t >= n_tiles) return;
  const int per_group = GROUP_M * tiles_n;
  const int first_m = (t / per_group) * GROUP_M;
  const int band = min(tiles_m - first_m, GROUP_M);
  const int m0 = (first_m + (t % per_group) % band) * BM;
  const int n0 = ((t % per_group) / band) * BN;

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = KS > 1 ? wave_all % NW : wave_all, ks = KS > 1 ? wave_all / NW : 0;
  const int lwave = DN > 0 ? wave_all - NW : wave;  // of the loading waves
  uint8_t* const lds = lds_all + ks * (ST * STAGE);
  const int wm = wave / WN, wn = wave % WN;
  const int l32 = lane & 31, half = lane >> 5;

  const __amdgpu_buffer_rsrc_t rsrc_a =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.a), 0, (p.M - 1) * p.lda + p.kb, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_w =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.w), 0, p.N * p.kb, kBufferRsrcWord3);

  // DMA block j of this wave: rows (j * NL + lwave) * 8 .. + 7 of A (j < NBA) or of W.
  int doff[NDMA], dcol[NDMA];
#pragma unroll
  for (int j = 0; j < NDMA; ++j) {
    const bool is_a = j < NBA;
    const int r = ((is_a ? j : j - NBA) * NL + lwave) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    dcol[j] = c * 16;
    doff[j] = is_a ? (m0 + r) * p.lda + c * 16 : (n0 + r) * p.kb + c * 16;
  }
  // The group's step kb (step KS kb + ks of the whole) into stage STG.
  auto dma_step = [&](int kb, int stage) {
    const int k0 = (KS * kb + ks) * (U * BK);
    auto issue = [&](auto WHOLE) {
      static_for<U * NDMA>([&](auto J) {
        constexpr int u = decltype(J)::value / NDMA, j = decltype(J)::value % NDMA;
        uint8_t* const dst = lds + stage * STAGE + u * T::CHUNK +
                             (j < NBA ? j * NL : BM / 8 + (j - NBA) * NL) * 1024 + lwave * 1024;
        const int k = k0 + u * BK;
        const int off = decltype(WHOLE)::value || dcol[j] < p.kb - k ? doff[j] + k : kOutOfRange;
        dma16(j < NBA ? rsrc_a : rsrc_w, dst, off);
      });
    };
    // a whole step within K needs no check per chunk (rows past M and N are past the buffers' ends)
    if (k0 + U * BK <= p.kb)
      issue(ic<1>{});
    else
      issue(ic<0>{});
  };

  const int nk = ((p.kb + BK - 1) / BK + KS * U - 1) / (KS * U);  // steps per group (a last one past K adds zeros)
  if constexpr (DN > 0) {
    if (wave_all >= NW) {
#pragma unroll
      for (int s = 0; s < ST - 1; ++s) dma_step(s, s);
      for (int kb = 0, stage = ST - 1; kb < nk; ++kb) {
        wait_counts<U * NDMA * (ST - 2), 15>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        dma_step(kb + ST - 1, stage);
        stage = stage + 1 == ST ? 0 : stage + 1;
      }
      wait_counts<0, 0>();
      __builtin_amdgcn_s_barrier();
      return;
    }
  }

  // Epilogue operands of the lane's outputs (block (j, i): row m = l32, columns 8 g + 4 half + 0..3 of block j),
  // loaded ahead of the operand stream.  N % 4 == 0: a group of 4 columns is inside N or not at all.
  float sxv[MI];
  float scale = 1.f;
  float4 swv[NI][4];
  uint2 bv[NI][4];
  if constexpr (kI8) {
#pragma unroll
    for (int i = 0; i < MI; ++i) sxv[i] = p.sx[min(m0 + (wm * MI + i) * 32 + l32, p.M - 1)];
  }
  if constexpr (kFp8) scale = p.sx[0] * p.sw[0];
  auto col = [&](int j, int g) { return min(n0 + (wn * NI + j) * 32 + 8 * g + 4 * half, p.N - 4); };
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bv[j][g] = make_uint2(0x80008000u, 0x80008000u);  // no bias: -0, which leaves every sum as it is
      if constexpr (kI8) swv[j][g] = *reinterpret_cast<const float4*>(p.sw + col(j, g));
    }
  if (p.bias != nullptr) {
    if (p.bias8) {
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) bv[j][g] = *reinterpret_cast<const uint2*>(p.bias + col(j, g));
    } else {
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const uint16_t* b = p.bias + col(j, g);
          bv[j][g] = make_uint2(b[0] | (static_cast<uint32_t>(b[1]) << 16), b[2] | (static_cast<uint32_t>(b[3]) << 16));
        }
    }
  }

  // Fragment pieces: sub-step s, lane half h, piece e is K chunk c = s*CPS + h*PIECES + e of the lane's row R,
  // at R*128 + 16*(c ^ ((R/2)%8)).
  const int x = (l32 >> 1) & 7;
  const int lane_a = (wm * MI * 32 + l32) * BK;
  const int lane_b = BM * BK + (wn * NI * 32 + l32) * BK;
  int koff[SUB][PIECES];
#pragma unroll
  for (int s = 0; s < SUB; ++s)
#pragma unroll
    for (int e = 0; e < PIECES; ++e) koff[s][e] = 16 * ((s * CPS + half * PIECES + e) ^ x);

  typename OP::acc_t acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = typename OP::acc_t{};

  if constexpr (DN == 0) static_for<ST - 1>([&](auto S) { dma_step(decltype(S)::value, decltype(S)::value); });
  // Fragments in two register sets: step kb's are read while the MFMAs of step kb - 1 run.  The stages and the
  // sets are compile-time (the loop is unrolled over both), so a step costs no address arithmetic but its DMAs'.
  v4i fa[2][U * SUB][MI][PIECES], fw[2][U * SUB][NI][PIECES];
  auto mma = [&](auto B) {
    constexpr int b = decltype(B)::value;
#pragma unroll
    for (int s = 0; s < U * SUB; ++s)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[j][i] = OP::mfma(fw[b][s][j], fa[b][s][i], acc[j][i]);
  };
  auto fetch = [&](auto B, auto STG, int kb) {
    constexpr int b = decltype(B)::value, stage = decltype(STG)::value;
    // own DMAs of step kb landed (those of the ST - 2 steps behind it may be in flight), own reads of the stage
    // before it done; the barrier makes both hold for every wave
    wait_counts<DN == 0 ? U * NDMA * (ST - 2) : 63, 0>();
    if constexpr (KS * NW + DN > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int s = 0; s < U * SUB; ++s) {
      const uint8_t* st = lds + stage * STAGE + s / SUB * T::CHUNK;
#pragma unroll
      for (int e = 0; e < PIECES; ++e) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          fa[b][s][i][e] = *reinterpret_cast<const v4i*>(st + i * 32 * BK + (lane_a + koff[s % SUB][e]));
#pragma unroll
        for (int j = 0; j < NI; ++j)
          fw[b][s][j][e] = *reinterpret_cast<const v4i*>(st + j * 32 * BK + (lane_b + koff[s % SUB][e]));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (DN == 0) dma_step(kb + ST - 1, (stage + ST - 1) % ST);
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(ic<0>{}, ic<0>{}, 0);
  constexpr int UNROLL = ST % 2 == 0 ? ST : 2 * ST;
  for (int kb = 1; kb < nk;) {
    static_for<UNROLL>([&](auto U) {
      constexpr int u = decltype(U)::value + 1;
      if (kb < nk) {
        fetch(ic<u & 1>{}, ic<u % ST>{}, kb);
        mma(ic<(u & 1) ^ 1>{});
        ++kb;
      }
    });
  }
  if (nk & 1)
    mma(ic<0>{});
  else
    mma(ic<1>{});
  // every DMA landed and every wave past its last LDS read before the stages are reused for the output staging
  wait_counts<0, 0>();
  if constexpr (KS * NW + DN > 1) __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  if constexpr (KS > 1) {
    // groups 1.. hand their sums to group 0 (16 bytes per lane and store), which adds them in group order and
    // finishes alone
    static_assert(kI8, "only int32 sums may be split");
    v4i* const sums = reinterpret_cast<v4i*>(lds_all);
    auto at = [&](int g, int j, int i, int q) { return (((((g - 1) * NW + wave) * NI + j) * MI + i) * 4 + q) * 64 + lane; };
    if (ks > 0) {
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            sums[at(ks, j, i, q)] =
                v4i{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
    }
    __syncthreads();
    if (ks == 0) {
#pragma unroll
      for (int g = 1; g < KS; ++g)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const v4i o = sums[at(g, j, i, q)];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[j][i][4 * q + e] += o[e];
            }
    }
    __syncthreads();  // the sums are read before group 0's slabs overwrite them
    if (ks > 0) return;
  }

  uint8_t* const wst = lds_all + wave * (T::SLABS * 32 * WPITCH);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    uint8_t* const slab = wst + (i & (T::SLABS - 1)) * 32 * WPITCH;
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int cw = j * 32 + 8 * g + 4 * half;
        const float b4[4] = {bf16_lo_to_f32(bv[j][g].x), bf16_hi_to_f32(bv[j][g].x), bf16_lo_to_f32(bv[j][g].y),
                             bf16_hi_to_f32(bv[j][g].y)};
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (kI8) {
            const float sw4[4] = {swv[j][g].x, swv[j][g].y, swv[j][g].z, swv[j][g].w};
            y[e] = __fmul_rn(__fmul_rn(static_cast<float>(acc[j][i][4 * g + e]), sxv[i]), sw4[e]);
          } else if constexpr (kFp8) {
            y[e] = __fmul_rn(acc[j][i][4 * g + e], scale);
          } else {
            y[e] = acc[j][i][4 * g + e];
          }
          y[e] = __fadd_rn(y[e], b4[e]);
          if constexpr (ACT != 0) {
            const float r = __uint_as_float(pack_bf16x2_hw(y[e], 0.f) << 16);
            y[e] = ACT == 1 ? silu(r) : gelu_tanh(r);
          }
        }
        *reinterpret_cast<uint2*>(slab + l32 * WPITCH + cw * 2) =
            make_uint2(pack_bf16x2_hw(y[0], y[1]), pack_bf16x2_hw(y[2], y[3]));
      }
    // the slab's rows are read back by other lanes of this wave: LDS executes a wave's accesses in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int LPR = NI * 4;        // lanes of 8 columns per output row
    constexpr int RPI = 64 / LPR;      // rows per store instruction
    const int ch = lane % LPR;
    const int gn = n0 + wn * NI * 32 + ch * 8;
#pragma unroll
    for (int it = 0; it < 32 / RPI; ++it) {
      const int rr = it * RPI + lane / LPR;
      const uint4 v = *reinterpret_cast<const uint4*>(slab + rr * WPITCH + ch * 16);
      const int gm = m0 + (wm * MI + i) * 32 + rr;
      if (gm < p.M && gn < p.N) {
        uint16_t* dst = p.y + static_cast<int64_t>(gm) * p.ldy + gn;
        if (p.vec16 && gn + 8 <= p.N) {
          *reinterpret_cast<uint4*>(dst) = v;
        } else {
          *reinterpret_cast<uint2*>(dst) = make_uint2(v.x, v.y);
          if (gn + 8 <= p.N) *reinterpret_cast<uint2*>(dst + 4) = make_uint2(v.z, v.w);
        }
      }
    }
  }
}

template <typename T, typename OP, int ACT>
void launch_small(const SmallArgs& p, hipStream_t stream) {
  const int64_t tiles = static_cast<int64_t>((p.M + T::BM - 1) / T::BM) * ((p.N + T::BN - 1) / T::BN);
  const dim3 grid(static_cast<uint32_t>((tiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD));
  hipLaunchKernelGGL((gemm_small_kernel<T, OP, ACT>), grid, dim3(T::THREADS), 0, stream, p);
}

// The tiles.  The time of the two small ones is the latency of a K step (about 350-450 cycles whatever its bytes).
// int8 runs groups of waves beside each other (KS).  bf16 has waves that only load, and two 128-byte chunks per step:
// 64 x 1536 -> 1536 4.9 us, 512 x 4096 -> 1536 14.3 us; the waves loading for themselves 6.3 and 16.8, a K split
// (another order of the sums) 5.7 and 14.8.  e4m3 keeps one group that loads for itself.
template <typename OP>
struct SmallTiles {
  static constexpr bool i8 = std::is_same<OP, OpI8>::value, bf16 = std::is_same<OP, OpBf16>::value;
  using T0 = typename std::conditional<
      i8, SmallTile<32, 64, 1, 2, 3, 4>,
      typename std::conditional<bf16, SmallTile<32, 64, 1, 2, 4, 1, 2, 4>, SmallTile<32, 64, 1, 2, 6>>::type>::type;
  using T1 = typename std::conditional<
      i8, SmallTile<64, 64, 2, 2, 4, 2>,
      typename std::conditional<bf16, SmallTile<64, 64, 2, 2, 4, 1, 2, 4>, SmallTile<64, 64, 2, 2, 4>>::type>::type;
  using T2 = SmallTile<64, 128, 2, 4, 3>;
  using T3 = SmallTile<128, 128, 2, 4, 4>;
};

// The tile of an M x N output with kb bytes of K, or -1 when `always` is false and the large tiles are the better
// ones: the smallest tile that covers the output in one round of workgroups (one per CU), because a round's time
// grows with the tile and a second round costs more than the next tile up.  us of 32 x 64, 64 x 64, 64 x 128, 128 x 128
// and 128 x 256 (M x N, K; where a rounds count is given, of more than one):
//   int8  300 x 1536, 1536: 5.2 5.5 6.0 8.5 10.6     300 x 1536, 8960: 13.7 14.9 22.4 30.5 40.1
//   e4m3  300 x 1536, 1536: 5.1 5.2 5.5 8.0 10.1     300 x 1536, 8960: 14.8 16.7 22.0 29.5 38.4
//   bf16  300 x 1536, 1536: 5.5 5.9 8.3 12.5         300 x 5120, 4096: 39 (3 rounds) 26.5 (2) 23.4 31.2
//   512 x 1536, 1536: int8 8.8 (2) 5.6 6.1, e4m3 5.9 (2) 5.3 5.6, bf16 9.4 (2) 6.2 8.4
// Past one round of 128 x 128 the 128 x 256 tile is ahead (1560 x 4608, K = 1536: int8 16.8 against 19.6, e4m3 16.0
// against 18.5).  A K of at most four steps is all launch, fill and stores: 64 x 128, two workgroups per CU
// (4680 x 1536, K = 64 bf16: 8.1 against 17 / 25 us for 64 x 64 / 32 x 64).
inline int pick_small(int M, int N, int kb, bool always) {
  if (g_tile_policy >= 2) return g_tile_policy - 2;
  const int64_t cus = device_cus();
  auto tiles = [&](int bm, int bn) { return static_cast<int64_t>((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (always && kb <= 4 * BK) return 2;
  if (tiles(32, 64) <= cus) return 0;
  if (tiles(64, 64) <= cus) return 1;
  if (tiles(64, 128) <= cus) return 2;
  if (always || tiles(128, 128) <= cus) return 3;
  return -1;
}

template <typename OP, int ACT>
void launch_small(int tile, const SmallArgs& p, hipStream_t stream) {
  using S = SmallTiles<OP>;
  switch (tile) {
    case 0: launch_small<typename S::T0, OP, ACT>(p, stream); break;
    case 1: launch_small<typename S::T1, OP, ACT>(p, stream); break;
    case 2: launch_small<typename S::T2, OP, ACT>(p, stream); break;
    default: launch_small<typename S::T3, OP, ACT>(p, stream); break;
  }
}

}  // namespace gemm
}  // namespace wf
