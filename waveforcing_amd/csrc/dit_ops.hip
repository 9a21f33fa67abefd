// The Wan DiT's layers around the quantized blocks, in bf16 as the reference
// runs them (its W8A8 swap replaces only the blocks' linears,
// wave_rt/runtime/fp8.py:93-137):
//
//  * a bf16 GEMM on the matrix cores for the patch embedding, the text and
//    time embeddings, the time projection and the output head
//    (naive_rt/rolling_forcing/wan/modules/causal_model.py:517-528,406-433):
//      y[m,n] = act_out( bf16( sum_k act_in(a[m,k]) * w[n,k] + bias[n] ) )
//    with fp32 accumulation; act_in = SiLU (the time projection's
//    nn.SiLU() before its Linear), act_out = SiLU or GELU(tanh), each
//    applied to a bf16 value and rounded to bf16 as torch's bf16 modules do;
//  * the patch gather of the Conv3d patch embedding (kernel = stride =
//    (1, 2, 2)): token (f, y, x) takes the 2 x 2 patch of every channel in
//    the weight's (c, kh, kw) order, so the embedding is that GEMM;
//  * unpatchify (causal_model.py:1080-1103: 'fhwpqrc->cfphqwr') fused with
//    the flow-matching x0 conversion of wan_wrapper.py:169-193,
//    x0 = xt - sigma * flow in float64, written in the (B, T, C, H, W)
//    layout the wavefront hands on (backend.py:456-490), converted to bf16
//    as torch converts float64 (through float32).
//
// The GEMM has three forms, chosen by size in wf_gemm_bf16: few rows (the W stream bounds it), LDS tiles
// (gemm_small.hpp) and the direct kernel for what the other two do not take.
#include <type_traits>

#include "gemm_core.hpp"
#include "gemm_small.hpp"
#include "wf_common.hpp"

namespace wf {
namespace {

using namespace gemm;

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf16_round(float x) { return __uint_as_float(pack_bf16x2_hw(x, 0.f) << 16); }

struct Bf16GemmArgs {
  const uint16_t* a;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* y;
  int64_t lda, ldy;
  int M, N, K;
  int act;      // 0 none, 1 SiLU, 2 GELU(tanh)
  int m_tiles;  // the few-row kernel's groups of rows
};

constexpr int kWaves = 4;
constexpr int kTileM = 64, kTileN = 128;

constexpr int kSkinnyWaves = 4;  // streaming waves of a workgroup; one more wave multiplies

// y for 8 NA rows of A and 16 NB rows of W, the few-row products of the time embedding.  The bound is the stream
// of W: K goes to the four streaming waves in pieces of 64 elements (whole 128-byte lines of every W row), which
// each of them brings into its own LDS ring of P pieces by DMA.  A piece of A is loaded, SiLU'd and handed over in
// LDS by the wave itself, 16 bytes per lane, so that the activation costs what the rows hold and not a 16-row tile.
// After each step of four pieces a barrier hands them to the fifth wave, which alone multiplies, in K order: one
// 16x16x32 MFMA adds in the order of the two 32x32x16 MFMAs of the other kernels, so a row has the same bits
// whichever kernel its call takes.  v_mfma_f32_16x16x32_bf16 takes 16 bytes of one row per lane (row l % 16, K
// elements 8 (l / 16) .. + 7); chunk c of row r lies at 16 (c ^ ((r / 2) % 8)).
template <bool SILU_IN, int NA, int NB>
__global__ __launch_bounds__((kSkinnyWaves + 1) * 64) void gemm_bf16_skinny_kernel(Bf16GemmArgs p) {
  constexpr int P = NB == 1 ? 4 : 3, S = kSkinnyWaves;
  constexpr int ROWS = 8 * NA, COLS = 16 * NB, MB = (NA + 1) / 2;
  constexpr int APIECE = ROWS * 128, WPIECE = COLS * 128;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S * P * WPIECE + 2 * S * APIECE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = static_cast<int>(blockIdx.x % static_cast<uint32_t>(p.m_tiles)) * ROWS;
  const int n0 = static_cast<int>(blockIdx.x / static_cast<uint32_t>(p.m_tiles)) * COLS;
  const int steps = ((p.K + 63) / 64 + S - 1) / S;  // the last pieces may be past K: zeros
  uint8_t* const abuf = lds + S * P * WPIECE;  // A's pieces of a step, two steps in turn

  if (wave < S) {
    const int rows = min(p.M - m0, ROWS), cols = min(p.N - n0, COLS);
    uint8_t* const ring = lds + wave * (P * WPIECE);
    // rows past M / N and chunks past K read zeros
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.a + static_cast<int64_t>(m0) * p.lda), 0,
        ((rows - 1) * static_cast<int>(p.lda) + p.K) * 2, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.w + static_cast<int64_t>(n0) * p.K), 0, cols * p.K * 2, kBufferRsrcWord3);
    // Lane l moves chunk l % 8 of row l / 8 (+ 8 i) of A, and of W the chunk that belongs at position l % 8 there.
    const int r8 = lane >> 3, c8 = lane & 7;
    u32x4 ar[P][NA];
    int aoff[NA], woff[2 * NB], wk[2 * NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) aoff[i] = ((r8 + 8 * i) * static_cast<int>(p.lda) + 8 * c8) * 2;
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i) {
      wk[i] = 8 * (c8 ^ (((r8 + 8 * i) >> 1) & 7));
      woff[i] = ((r8 + 8 * i) * p.K + wk[i]) * 2;
    }
    auto load = [&](auto SLOT, int step) {
      constexpr int s = decltype(SLOT)::value;
      const int k0 = 64 * (wave + S * step);
#pragma unroll
      for (int i = 0; i < NA; ++i)
        ar[s][i] =
            __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, k0 + 8 * c8 < p.K ? aoff[i] + 2 * k0 : kOutOfRange, 0, 0);
#pragma unroll
      for (int i = 0; i < 2 * NB; ++i)
        dma16(rsrc_w, ring + s * WPIECE + i * 1024, k0 + wk[i] < p.K ? woff[i] + 2 * k0 : kOutOfRange);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto hand_over = [&](auto SLOT, int step) {
      constexpr int s = decltype(SLOT)::value;
      uint8_t* const aw = abuf + (step & 1) * (S * APIECE) + wave * APIECE;
      // this piece's loads landed; those of the P - 2 pieces behind it may be in flight
      wait_counts<(P - 2) * (2 * NB + NA), 15>();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        u32x4 v = ar[s][i];
        if constexpr (SILU_IN) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = pack_bf16x2_hw(silu(bf16_lo_to_f32(v[e])), silu(bf16_hi_to_f32(v[e])));
        }
        const int r = r8 + 8 * i;
        *reinterpret_cast<u32x4*>(aw + r * 128 + 16 * (c8 ^ ((r >> 1) & 7))) = v;
      }
      wait_counts<63, 0>();
      if (step <= steps) __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    static_for<P - 1>([&](auto I) { load(I, decltype(I)::value); });
    // Whole rounds of the ring: with an exit inside, the compiler would wait at the top for loads that are to stay in
    // flight.  Steps past the last hand over nothing; the first of them waits until the last is read.
    for (int i = 0; i < steps; i += P) {
      static_for<P>([&](auto I) {
        constexpr int s = decltype(I)::value;
        hand_over(I, i + s);
        load(ic<(s + P - 1) % P>{}, i + s + P - 1);  // the slot of step i + s - 1, read before this step's barrier
      });
    }
    wait_counts<0, 0>();  // nothing of this wave is under way to LDS when it ends
    return;
  }

  const int r16 = lane & 15, kq = lane >> 4;
  auto at = [&](int r, int u) { return r * 128 + 16 * ((4 * u + kq) ^ ((r >> 1) & 7)); };
  // the lane's rows m0 + 16 i + l % 16, columns n0 + 16 j + 4 (l / 16) .. + 3 (N % 4 == 0: all inside N or none)
  const int m = m0 + r16, n = n0 + 4 * kq;
  float bias[NB][4];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) bias[j][e] = -0.f;  // no bias: -0, which leaves every sum as it is
  if (p.bias != nullptr) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[j][e] = bf16_bits_to_f32(p.bias[min(n + 16 * j, p.N - 4) + e]);
  }
  v4f acc[NB][MB] = {};
  for (int i = 0; i < steps; ++i) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint8_t* const wp = lds + (i % P) * WPIECE;
    const uint8_t* const ap = abuf + (i & 1) * (S * APIECE);
    v8bf av[S][2][MB], wv[S][2][NB];
#pragma unroll
    for (int w = 0; w < S; ++w)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          wv[w][u][j] = *reinterpret_cast<const v8bf*>(wp + w * (P * WPIECE) + at(16 * j + r16, u));
#pragma unroll
        for (int b = 0; b < MB; ++b)  // (NA = 1: rows 8.. are rows 0.. again, and not stored)
          av[w][u][b] = *reinterpret_cast<const v8bf*>(ap + w * APIECE + at((16 * b + r16) & (ROWS - 1), u));
      }
#pragma unroll
    for (int w = 0; w < S; ++w)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int b = 0; b < MB; ++b)
            acc[j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[w][u][j], av[w][u][b], acc[j][b], 0, 0, 0);
    // the step's fragments are in registers before the next barrier frees their slots
    wait_counts<63, 0>();
    asm volatile("" ::: "memory");
  }
  if (steps % P != 0) __builtin_amdgcn_s_barrier();  // of the first step past the last
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      if (m + 16 * b >= min(p.M, m0 + ROWS) || n + 16 * j >= p.N) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = bf16_round(__fadd_rn(acc[j][b][e], bias[j][e]));
        if (p.act == 1) v[e] = silu(v[e]);
        if (p.act == 2) v[e] = gelu_tanh(v[e]);
      }
      *reinterpret_cast<uint2*>(p.y + static_cast<int64_t>(m + 16 * b) * p.ldy + n + 16 * j) =
          make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
    }
}

template <bool SILU_IN>
__device__ inline v8bf load_frag(const uint16_t* row, int k, int K) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (k < K) v = *reinterpret_cast<const uint4*>(row + k);
  if constexpr (SILU_IN) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = pack_bf16x2_hw(silu(bf16_lo_to_f32(w[i])), silu(bf16_hi_to_f32(w[i])));
    v = make_uint4(o[0], o[1], o[2], o[3]);
  }
  return __builtin_bit_cast(v8bf, v);
}

// The general form: any size, 64-bit row addresses.  A workgroup of 4 waves owns a 64 x 128 output tile, each wave
// 32 rows x 64 columns as two v_mfma_f32_32x32x16_bf16 blocks whose fragments (16 contiguous bytes of one row of
// A and of W: lane l row l % 32, K elements 8 (l / 32) .. + 7) come straight from global memory, one K step
// ahead of the MFMAs.  A latency chain per K step; it serves what the kernels above do not take.
template <bool SILU_IN>
__global__ __launch_bounds__(kWaves * 64) void gemm_bf16_kernel(Bf16GemmArgs p) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int m0 = blockIdx.y * kTileM + (wave >> 1) * 32;
  const int n0 = blockIdx.x * kTileN + (wave & 1) * 64;
  // rows past M / N read a clamped row (their results are not stored)
  const uint16_t* arow = p.a + static_cast<int64_t>(min(m0 + l32, p.M - 1)) * p.lda;
  const uint16_t* wrow0 = p.w + static_cast<int64_t>(min(n0 + l32, p.N - 1)) * p.K;
  const uint16_t* wrow1 = p.w + static_cast<int64_t>(min(n0 + 32 + l32, p.N - 1)) * p.K;
  v16f acc0 = {}, acc1 = {};
  const int kh = 8 * half;
  v8bf a = load_frag<SILU_IN>(arow, kh, p.K);
  v8bf w0 = load_frag<false>(wrow0, kh, p.K);
  v8bf w1 = load_frag<false>(wrow1, kh, p.K);
  for (int k = 16; k < p.K + 16; k += 16) {
    // the next step's fragments load under this step's MFMAs (zeros past K)
    const v8bf an = load_frag<SILU_IN>(arow, k + kh, p.K);
    const v8bf w0n = load_frag<false>(wrow0, k + kh, p.K);
    const v8bf w1n = load_frag<false>(wrow1, k + kh, p.K);
    acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, a, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, a, acc1, 0, 0, 0);
    a = an;
    w0 = w0n;
    w1 = w1n;
  }
  // lane's row m0 + l32; register r of block j is column n0 + 32 j + 8 (r / 4) + 4 half + r % 4.  The
  // wave's 32 x 64 results go through its own LDS rows, so each row is stored as one 128-byte segment.
  constexpr int YP = 64 * 2 + 8;  // staged row pitch (bytes)
  __shared__ __attribute__((aligned(16))) uint8_t ys[kWaves * 32 * YP];
  uint8_t* yw = ys + wave * 32 * YP;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const v16f& acc = j == 0 ? acc0 : acc1;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n0 + 32 * j + 8 * g + 4 * half;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = acc[4 * g + e];
        if (p.bias && n < p.N) t = __fadd_rn(t, bf16_bits_to_f32(p.bias[n + e]));
        t = bf16_round(t);
        if (p.act == 1) t = silu(t);
        if (p.act == 2) t = gelu_tanh(t);
        v[e] = t;
      }
      *reinterpret_cast<uint2*>(yw + l32 * YP + 2 * (32 * j + 8 * g + 4 * half)) =
          make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * i + (lane >> 4);
    const int m = m0 + row, n = n0 + 4 * (lane & 15);
    const uint2 w = *reinterpret_cast<const uint2*>(yw + row * YP + 8 * (lane & 15));
    if (m < p.M && n < p.N) *reinterpret_cast<uint2*>(p.y + static_cast<int64_t>(m) * p.ldy + n) = w;
  }
}

// Patch gather: out[b][t][c * 4 + kh * 2 + kw] = x[b][c][f][2 y + kh][2 x + kw], token t = (f, y, x).
// One thread per (b, t, c): 4 values, one 8-byte store.
__global__ __launch_bounds__(256) void patchify_kernel(const uint16_t* __restrict__ x, int64_t B, int C, int F, int H,
                                                       int W, uint16_t* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int hp = H / 2, wp = W / 2;
  const int64_t tokens = static_cast<int64_t>(F) * hp * wp;
  if (i >= B * tokens * C) return;
  const int c = static_cast<int>(i % C);
  const int64_t bt = i / C;
  const int64_t t = bt % tokens;
  const int64_t b = bt / tokens;
  const int xw = static_cast<int>(t % wp), yh = static_cast<int>((t / wp) % hp), f = static_cast<int>(t / (wp * hp));
  const uint16_t* src = x + (((b * C + c) * F + f) * H + 2 * yh) * static_cast<int64_t>(W) + 2 * xw;
  const uint32_t top = *reinterpret_cast<const uint32_t*>(src);
  const uint32_t bot = *reinterpret_cast<const uint32_t*>(src + W);
  *reinterpret_cast<uint2*>(out + (b * tokens + t) * (4 * C) + 4 * c) = make_uint2(top, bot);
}

// float64 -> bf16 as torch converts it: to float32 (round to nearest even), then to bf16.
__device__ inline uint16_t f64_to_bf16_via_f32(double d) { return f32_to_bf16_rne(static_cast<float>(d)); }

// x0[b][f][c][y][x] = bf16(xt[b][c][f][y][x] - sigma * flow[b][c][f][y][x]) in float64, with flow the
// unpatchified head output: flow[b][c][f][2 y' + q][2 x' + r] = head[b][t(f, y', x')][(2 q + r) * C + c].
// One thread per (b, f, c, y, x pair): two outputs.
__global__ __launch_bounds__(256) void unpatchify_x0_kernel(const uint16_t* __restrict__ head,
                                                            const uint16_t* __restrict__ xt, int64_t B, int C, int F,
                                                            int H, int W, double sigma, uint16_t* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int wh = W / 2;
  const int64_t total = B * F * static_cast<int64_t>(C) * H * wh;
  if (i >= total) return;
  const int xp = static_cast<int>(i % wh);
  int64_t r = i / wh;
  const int yy = static_cast<int>(r % H);
  r /= H;
  const int c = static_cast<int>(r % C);
  r /= C;
  const int f = static_cast<int>(r % F);
  const int64_t b = r / F;
  const int hp = H / 2;
  const int64_t t = (static_cast<int64_t>(f) * hp + yy / 2) * wh + xp;
  const int q = yy & 1;
  const uint16_t* hrow = head + (b * (static_cast<int64_t>(F) * hp * wh) + t) * (4 * C);
  const uint16_t fl0 = hrow[(2 * q + 0) * C + c];
  const uint16_t fl1 = hrow[(2 * q + 1) * C + c];
  const uint32_t xv = *reinterpret_cast<const uint32_t*>(xt + (((b * C + c) * F + f) * H + yy) * static_cast<int64_t>(W) +
                                                         2 * xp);
  const double x0a = static_cast<double>(bf16_lo_to_f32(xv)) - sigma * static_cast<double>(bf16_bits_to_f32(fl0));
  const double x0b = static_cast<double>(bf16_hi_to_f32(xv)) - sigma * static_cast<double>(bf16_bits_to_f32(fl1));
  const uint32_t o = static_cast<uint32_t>(f64_to_bf16_via_f32(x0a)) |
                     (static_cast<uint32_t>(f64_to_bf16_via_f32(x0b)) << 16);
  *reinterpret_cast<uint32_t*>(out + (((b * F + f) * C + c) * H + yy) * static_cast<int64_t>(W) + 2 * xp) = o;
}

template <bool SILU_IN, int NA, int NB>
void launch_skinny(Bf16GemmArgs p, hipStream_t st) {
  p.m_tiles = (p.M + 8 * NA - 1) / (8 * NA);
  const int64_t blocks = static_cast<int64_t>(p.m_tiles) * ((p.N + 16 * NB - 1) / (16 * NB));
  hipLaunchKernelGGL((gemm_bf16_skinny_kernel<SILU_IN, NA, NB>), dim3(static_cast<uint32_t>(blocks)),
                     dim3((kSkinnyWaves + 1) * 64), 0, st, p);
}
template <bool SILU_IN, int NA>
void launch_skinny(bool wide, const Bf16GemmArgs& p, hipStream_t st) {
  wide ? launch_skinny<SILU_IN, NA, 2>(p, st) : launch_skinny<SILU_IN, NA, 1>(p, st);
}

template <bool SILU_IN>
void launch_direct(const Bf16GemmArgs& p, hipStream_t st) {
  const dim3 grid((p.N + kTileN - 1) / kTileN, (p.M + kTileM - 1) / kTileM);
  hipLaunchKernelGGL(gemm_bf16_kernel<SILU_IN>, grid, dim3(kWaves * 64), 0, st, p);
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace wf

extern "C" {

int wf_gemm_bf16(const void* a, int64_t m, int64_t k, int64_t lda, const void* w, int64_t n, const void* bias,
                 void* y, int64_t ldy, int32_t flags, void* stream) {
  static const char* fn = "wf_gemm_bf16";
  WF_REQUIRE(m >= 0 && n >= 0 && k > 0 && lda >= k && ldy >= n, WF_E_INVALID,
             "%s: bad sizes m=%lld n=%lld k=%lld lda=%lld ldy=%lld", fn, (long long)m, (long long)n, (long long)k,
             (long long)lda, (long long)ldy);
  if (m == 0 || n == 0) return WF_OK;
  WF_REQUIRE(a && w && y, WF_E_INVALID, "%s: null pointer", fn);
  WF_REQUIRE(m < (1 << 30) && n < (1 << 30) && k < (1 << 30), WF_E_SHAPE, "%s: size too large", fn);
  WF_REQUIRE(k % 8 == 0 && lda % 8 == 0 && n % 4 == 0 && ldy % 4 == 0, WF_E_SHAPE,
             "%s: k and lda must be multiples of 8, n and ldy of 4", fn);
  WF_REQUIRE(wf::a16(a) && wf::a16(w) && (reinterpret_cast<uintptr_t>(y) & 7u) == 0 &&
                 (reinterpret_cast<uintptr_t>(bias) & 1u) == 0,
             WF_E_ALIGN, "%s: a and w must be 16-byte, y 8-byte aligned", fn);
  const int act = (flags & WF_BF16_SILU_OUT) ? 1 : (flags & WF_BF16_GELU_OUT) ? 2 : 0;
  WF_REQUIRE((flags & ~(WF_BF16_SILU_IN | WF_BF16_SILU_OUT | WF_BF16_GELU_OUT)) == 0 &&
                 !((flags & WF_BF16_SILU_OUT) && (flags & WF_BF16_GELU_OUT)),
             WF_E_INVALID, "%s: bad flags 0x%x", fn, flags);
  hipStream_t st = wf::as_stream(stream);
  const bool silu_in = (flags & WF_BF16_SILU_IN) != 0;
  constexpr int64_t kSpan = (1ll << 31) - 16;  // buffer offsets are 32-bit
  wf::Bf16GemmArgs p{static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(w),
                     static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(y), lda, ldy,
                     static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), act, 0};
  // Few rows (the time embedding's 1-21 frames): the W stream's kernel; 3 x 1536 -> 9216 with SiLU 6.6 us against
  // 35.1 us for the direct kernel (28.3 MB of W), 3 x 5120 -> 30720 49.8 us (6.3 TB/s) against 148.  Without SiLU the
  // tiles take over at 17 rows (17 x 1536 -> 1536: 4.8 us); with it, which only this kernel and the direct one apply,
  // at 65.  Above 8 rows the SiLU that every workgroup repeats costs as much as the stream: where 32-column
  // workgroups still give each CU one they halve it (16 x 5120 -> 30720: 58 against 69 us; 16 x 4096 -> 1536, which
  // they would leave to 48 CUs, 9.5 against 6.4), and from 17 rows on take 32 rows at a time (21 x 1536 -> 9216:
  // 13.6 against 18.0 us).
  const int64_t skinny_max = silu_in ? 64 : 16;
  if (m <= skinny_max && wf::product_below({32, lda, 2}, kSpan) && wf::product_below({32, k, 2}, kSpan)) {
    const bool wide = (n + 31) / 32 >= wf::gemm::device_cus();
    if (silu_in && wide && m > 16)
      wf::launch_skinny<true, 4, 2>(p, st);
    else if (silu_in)
      m <= 8 ? wf::launch_skinny<true, 1, 1>(p, st) : wf::launch_skinny<true, 2>(wide, p, st);
    else
      m <= 8 ? wf::launch_skinny<false, 1, 1>(p, st) : wf::launch_skinny<false, 2>(wide, p, st);
    return wf::check_launch(fn);
  }
  // LDS-tiled: 512 x 4096 -> 1536 with GELU 14.3 us against 97 us, 4680 x 1536 -> 64 (head) 5.0 against 28.5 us,
  // 4680 x 64 -> 1536 (patch embedding) 8.1 against 13.3 us for the direct kernel.
  if (!silu_in && wf::product_below({m + 256, lda, 2}, kSpan) && wf::product_below({n + 256, k, 2}, kSpan)) {
    const wf::gemm::SmallArgs q{a, w, nullptr, nullptr, p.bias, p.y, p.M, p.N, 2 * p.K, static_cast<int>(2 * lda), ldy,
                                ldy % 8 == 0 && wf::a16(y), (reinterpret_cast<uintptr_t>(bias) & 7u) == 0};
    const int tile = wf::gemm::pick_small(p.M, p.N, q.kb, true);
    if (act == 0)
      wf::gemm::launch_small<wf::gemm::OpBf16, 0>(tile, q, st);
    else if (act == 1)
      wf::gemm::launch_small<wf::gemm::OpBf16, 1>(tile, q, st);
    else
      wf::gemm::launch_small<wf::gemm::OpBf16, 2>(tile, q, st);
    return wf::check_launch(fn);
  }
  silu_in ? wf::launch_direct<true>(p, st) : wf::launch_direct<false>(p, st);
  return wf::check_launch(fn);
}

int wf_patchify_bf16(const void* x, int64_t b, int32_t c, int32_t f, int32_t h, int32_t w, void* out, void* stream) {
  static const char* fn = "wf_patchify_bf16";
  WF_REQUIRE(b >= 0 && c > 0 && f > 0 && h > 0 && w > 0, WF_E_INVALID, "%s: bad sizes", fn);
  WF_REQUIRE(h % 2 == 0 && w % 2 == 0, WF_E_SHAPE, "%s: h=%d and w=%d must be even (2 x 2 patches)", fn, h, w);
  if (b == 0) return WF_OK;
  WF_REQUIRE(x && out, WF_E_INVALID, "%s: null pointer", fn);
  WF_REQUIRE((reinterpret_cast<uintptr_t>(x) & 3u) == 0 && (reinterpret_cast<uintptr_t>(out) & 7u) == 0, WF_E_ALIGN,
             "%s: x must be 4-byte and out 8-byte aligned", fn);
  // one thread per item: a launch holds fewer than 2^32 threads
  WF_REQUIRE(wf::product_below({b, f, h / 2, w / 2, c}, (1ll << 32) - 256), WF_E_SHAPE,
             "%s: b*f*(h/2)*(w/2)*c must stay below 2^32 - 256", fn);
  const int64_t items = b * static_cast<int64_t>(f) * (h / 2) * (w / 2) * c;
  hipLaunchKernelGGL(wf::patchify_kernel, dim3(static_cast<uint32_t>((items + 255) / 256)), dim3(256), 0,
                     wf::as_stream(stream), static_cast<const uint16_t*>(x), b, c, f, h, w,
                     static_cast<uint16_t*>(out));
  return wf::check_launch(fn);
}

int wf_unpatchify_flow_x0_bf16(const void* head, const void* xt, int64_t b, int32_t c, int32_t f, int32_t h,
                               int32_t w, double sigma, void* x0, void* stream) {
  static const char* fn = "wf_unpatchify_flow_x0_bf16";
  WF_REQUIRE(b >= 0 && c > 0 && f > 0 && h > 0 && w > 0, WF_E_INVALID, "%s: bad sizes", fn);
  WF_REQUIRE(h % 2 == 0 && w % 2 == 0, WF_E_SHAPE, "%s: h=%d and w=%d must be even (2 x 2 patches)", fn, h, w);
  if (b == 0) return WF_OK;
  WF_REQUIRE(head && xt && x0, WF_E_INVALID, "%s: null pointer", fn);
  WF_REQUIRE((reinterpret_cast<uintptr_t>(xt) & 3u) == 0 && (reinterpret_cast<uintptr_t>(x0) & 3u) == 0 &&
                 (reinterpret_cast<uintptr_t>(head) & 1u) == 0,
             WF_E_ALIGN, "%s: xt and x0 must be 4-byte aligned", fn);
  // one thread per item: a launch holds fewer than 2^32 threads
  WF_REQUIRE(wf::product_below({b, f, c, h, w / 2}, (1ll << 32) - 256), WF_E_SHAPE,
             "%s: b*f*c*h*(w/2) must stay below 2^32 - 256", fn);
  const int64_t items = b * static_cast<int64_t>(f) * c * h * (w / 2);
  hipLaunchKernelGGL(wf::unpatchify_x0_kernel, dim3(static_cast<uint32_t>((items + 255) / 256)), dim3(256), 0,
                     wf::as_stream(stream), static_cast<const uint16_t*>(head), static_cast<const uint16_t*>(xt), b, c,
                     f, h, w, sigma, static_cast<uint16_t*>(x0));
  return wf::check_launch(fn);
}

}  // extern "C"
