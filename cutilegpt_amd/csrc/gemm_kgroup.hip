// 16-bit GEMM for problems with few output tiles: C[M,N] = epilogue(A W^T + bias),
// K shared between the wave groups of a block.
//
// The projections back to the model width (N = d) give the tiled kernels about
// one tile a CU, or far fewer for short prompts, and a single four-wave tile
// leaves the CU waiting for its stage, its LDS reads and its barrier in turn.
// Here a block has KG groups of 2 x 2 waves.  Group i multiplies the k64 stages
// i, i + KG, ... of the block's tile from LDS buffers of its own, so every
// barrier interval moves KG stages and each SIMD has KG waves to switch
// between; the groups' sums are added through LDS at the end, each group
// finishing its share of the tile.
//
// Stages reach LDS by DMA (buffer_load ... lds), S - 1 stages ahead, in the
// layout of the pipeline kernels (gemm.hip): 128-byte rows, 16-byte chunk c of
// row r at chunk c ^ (r & 7).  The bias and, for the residual epilogue, the old
// C values of a group's share are loaded before the K loop.
#include "common.h"
#include "gemm_common.h"
#include "internal.h"

namespace cgpt {

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void load4(__amdgpu_buffer_rsrc_t r, uint32_t off, float* v, const float*) {
  const u32x4_t x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(x[i]);
}
__device__ __forceinline__ void load4(__amdgpu_buffer_rsrc_t r, uint32_t off, float* v, const bf16_t*) {
  const u32x2_t x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(i % 2 ? x[i / 2] & 0xffff0000u : x[i / 2] << 16);
}
__device__ __forceinline__ void load4(__amdgpu_buffer_rsrc_t r, uint32_t off, float* v, const f16_t*) {
  const u32x2_t x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = i % 2 ? f16_hi(x[i / 2]) : f16_lo(x[i / 2]);
}
#endif

// Requires K % 64 == 0, N % 4 == 0, rows of A, W and C that take 16-byte (a
// 16-bit C: 8-byte) accesses, and the operands and C within 2 GiB.
template <typename TIn, int BM, int BN, int WGM, int WGN, int KG, int S, int EPI, typename TOut>
__global__ __launch_bounds__(64 * WGM * WGN * KG) void gemm_kgroup_kernel(
    const TIn* __restrict__ A, const TIn* __restrict__ W, const void* __restrict__ bias,
    bool bias_half, TOut* __restrict__ C, int M, int N, int K, int lda, int ldw, int ldc, int tiles_m,
    int tiles_n) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = WGM * WGN;  // waves of a group
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "whole 16x16 tiles a wave");
  constexpr int ROWB = 128, STAGE = (BM + BN) * ROWB;
  // DMA instructions of a stage (8 rows each, A's then W's), dealt round-robin
  // to the group's waves: the first INS % NW waves have one more.
  constexpr int A_ALL = BM / 8, INS = (BM + BN) / 8, LPS = (INS + NW - 1) / NW, LMIN = INS / NW;
  static_assert(S >= 2 && S <= 5 && (S - 2) * LPS < 64, "stages");
  constexpr int TILES = TM * TN, OWN = (TILES + KG - 1) / KG;  // 16x16 tiles of a wave; a group's share
  constexpr int XCH = KG * (KG - 1) * OWN * NW * 1024;
  constexpr int SMEM = KG * S * STAGE > XCH ? KG * S * STAGE : XCH;
  static_assert(SMEM <= 160 * 1024, "LDS budget of one CU");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];

  const int lane = threadIdx.x & 63;
  const int bwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = KG > 1 ? bwave / NW : 0, wave = KG > 1 ? bwave % NW : bwave;
  const int wm0 = wave / WGN * WM, wn0 = wave % WGN * WN;
  const int frow = lane & 15, fgrp = lane >> 4;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // This lane's place in C, by tile of the wave: row, first column, byte offset
  // (past the resource where the row or the columns are outside C).
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
      C, 0, static_cast<int>(((M - 1) * static_cast<int64_t>(ldc) + N) * static_cast<int64_t>(sizeof(TOut))),
      kBufferRsrcWord3);
  auto c_off = [&](int t) -> uint32_t {
    const int m = m0 + wm0 + t / TN * 16 + frow, n = n0 + wn0 + t % TN * 16 + 4 * fgrp;
    return m < M && n < N ? static_cast<uint32_t>((static_cast<int64_t>(m) * ldc + n) * sizeof(TOut)) : 0x80000000u;
  };
  // The bias and old C values of the group's tiles grp * OWN ..
  float bv[OWN][4], cv[EPI == CGPT_EPI_BIAS_RESID ? OWN : 1][4];
  if constexpr (EPI != CGPT_EPI_NONE) {
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(bias), 0, N << (bias_half ? 1 : 2), kBufferRsrcWord3);
#pragma unroll
    for (int q = 0; q < OWN; ++q) {
      const int n = n0 + wn0 + (grp * OWN + q) % TN * 16 + 4 * fgrp;  // past N: reads zero
      if (bias_half)
        load4(rb, n * 2, bv[q], static_cast<const TIn*>(nullptr));
      else
        load4(rb, n * 4, bv[q], static_cast<const float*>(nullptr));
    }
  }
  if constexpr (EPI == CGPT_EPI_BIAS_RESID) {
#pragma unroll
    for (int q = 0; q < OWN; ++q) load4(rc, c_off(grp * OWN + q), cv[q], static_cast<const TOut*>(nullptr));
  }

  // DMA instruction j fills rows 8 j .. 8 j + 7 of the stage; rows past the
  // matrix are clamped to the last one.
  const u32x4_t ra = buffer_desc(A, static_cast<uint32_t>((M - 1) * static_cast<int64_t>(lda) + K) * 2);
  const u32x4_t rw = buffer_desc(W, static_cast<uint32_t>((N - 1) * static_cast<int64_t>(ldw) + K) * 2);
  const int lrow = lane >> 3, chunk = ((lane & 7) ^ lrow) << 4;
  uint32_t off[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const int j = i * NW + wave;
    off[i] = j < A_ALL ? static_cast<uint32_t>(min(m0 + j * 8 + lrow, M - 1)) * lda * 2 + chunk
                       : static_cast<uint32_t>(min(n0 + (j - A_ALL) * 8 + lrow, N - 1)) * ldw * 2 + chunk;
  }
  uint8_t* const gbase = smem + grp * S * STAGE;
  const int KT = K / 64;
  auto issue = [&](int it, int buf) {  // the group's stage it, if there is one
    const int kt = it * KG + grp;
    if (kt >= KT) return;
    uint8_t* p = gbase + buf * STAGE;
#pragma unroll
    for (int i = 0; i < LPS; ++i) {
      const int j = i * NW + wave;
      if (INS % NW == 0 || i < LMIN || j < INS) {
        if (j < A_ALL)
          dma_lds16(ra, lds_addr(p + j * 1024), off[i], kt * ROWB);
        else
          dma_lds16(rw, lds_addr(p + j * 1024), off[i], kt * ROWB);
      }
    }
  };
  // Waits until the group's stage it has landed (up to S - 2 later ones, as
  // many as there are, stay in flight) and this wave's LDS reads are done.
  auto wait_later = [&](auto n) {
    constexpr int L = decltype(n)::value;
    if (INS % NW == 0 || wave < INS % NW)
      wait_vmcnt<L * LPS>();
    else
      wait_vmcnt<L * LMIN>();
  };
  auto wait_stage = [&](int it) {
    const int last = (KT - 1 - grp) / KG;  // the group's last stage (KT > grp)
    const int later = min(last - it, S - 2);
    if constexpr (S >= 5) if (later >= 3) { wait_later(std::integral_constant<int, 3>{}); return; }
    if constexpr (S >= 4) if (later >= 2) { wait_later(std::integral_constant<int, 2>{}); return; }
    if constexpr (S >= 3) if (later >= 1) { wait_later(std::integral_constant<int, 1>{}); return; }
    wait_vmcnt<0>();
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int a_base = (wm0 + frow) * ROWB, w_base = BM * ROWB + (wn0 + frow) * ROWB;
  const int x0 = (fgrp ^ (frow & 7)) << 4, x1 = ((4 + fgrp) ^ (frow & 7)) << 4;

  const int iters = (KT + KG - 1) / KG;  // the same for every group (barriers)
#pragma unroll
  for (int it = 0; it < S - 1; ++it) issue(it, it);
  wait_stage(0);
  int cur = 0, nxt = S - 1;  // buffers of stages it and it + S - 1
  for (int it = 0; it < iters; ++it) {
    raw_barrier();
    issue(it + S - 1, nxt);
    if (it * KG + grp < KT) {
      const uint8_t* buf = gbase + cur * STAGE;
      u32x4_t a[2][TM], w[2][TN];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          a[s][i] = *reinterpret_cast<const u32x4_t*>(buf + a_base + i * 16 * ROWB + (s ? x1 : x0));
#pragma unroll
        for (int j = 0; j < TN; ++j)
          w[s][j] = *reinterpret_cast<const u32x4_t*>(buf + w_base + j * 16 * ROWB + (s ? x1 : x0));
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) Mfma<TIn>::run(w[s][j], a[s][i], acc[i][j]);
    }
    wait_stage(it + 1);
    cur = cur + 1 == S ? 0 : cur + 1;
    nxt = nxt + 1 == S ? 0 : nxt + 1;
  }

  // Every group hands the others its sums of their tiles and adds theirs to
  // its own, in group order.
  if constexpr (KG > 1) __syncthreads();
  f32x4_t* x = reinterpret_cast<f32x4_t*>(smem);
  const int tid = wave * 64 + lane;
  auto slot = [&](int owner, int src, int q) {  // src: the writer's place among the others
    return ((owner * (KG - 1) + src) * OWN + q) * (64 * NW) + tid;
  };
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int owner = t / OWN;
    if (owner != grp) x[slot(owner, grp - (grp > owner), t % OWN)] = acc[t / TN][t % TN];
  }
  if constexpr (KG > 1) __syncthreads();
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    if (t / OWN != grp) continue;
    f32x4_t sum = acc[t / TN][t % TN];
#pragma unroll
    for (int o = 0; o < KG - 1; ++o) sum += x[slot(t / OWN, o, t % OWN)];
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float z = sum[r];
      if (EPI != CGPT_EPI_NONE) z += bv[t % OWN][r];
      if (EPI == CGPT_EPI_BIAS_GELU) z = gelu_tanh(z);
      if constexpr (EPI == CGPT_EPI_BIAS_RESID) z += cv[t % OWN][r];
      v[r] = z;
    }
    const uint32_t off = c_off(t);
    if constexpr (sizeof(TOut) == 4)
      __builtin_amdgcn_raw_buffer_store_b128(
          u32x4_t{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])},
          rc, off, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{pack2<TOut>(v[0], v[1]), pack2<TOut>(v[2], v[3])}, rc, off,
                                            0, 0);
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <typename TIn, int BM, int BN, int WGM, int WGN, int KG, int S, int EPI, typename TOut>
static int launch_kgroup_tile(const void* a, const void* w, const void* bias, bool bias_half, void* c,
                              int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc, hipStream_t s) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_kgroup_kernel<TIn, BM, BN, WGM, WGN, KG, S, EPI, TOut>),
                     dim3(static_cast<unsigned>(tiles_m * tiles_n)), dim3(64 * WGM * WGN * KG), 0, s,
                     static_cast<const TIn*>(a), static_cast<const TIn*>(w), bias, bias_half,
                     static_cast<TOut*>(c), M, N, K, static_cast<int>(lda), static_cast<int>(ldw),
                     static_cast<int>(ldc), tiles_m, tiles_n);
  return hip_status(hipGetLastError());
}

template <typename TIn, int EPI, typename TOut>
static int launch_kgroup_epi(int tile, const void* a, const void* w, const void* bias, bool bias_half,
                             void* c, int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                             hipStream_t s) {
#define CGPT_KG_CASE(id, BM, BN, WGM, WGN, KG, S)                                                     \
  case id:                                                                                           \
    return launch_kgroup_tile<TIn, BM, BN, WGM, WGN, KG, S, EPI, TOut>(a, w, bias, bias_half, c, M, N, \
                                                                       K, lda, ldw, ldc, s);
  switch (tile) {
    CGPT_KG_CASE(0, 32, 32, 2, 2, 4, 3)
    CGPT_KG_CASE(1, 64, 32, 2, 2, 4, 3)
    CGPT_KG_CASE(2, 64, 64, 2, 2, 2, 3)
    CGPT_KG_CASE(3, 64, 96, 2, 2, 2, 3)
    CGPT_KG_CASE(4, 96, 96, 2, 2, 2, 3)
    CGPT_KG_CASE(5, 128, 96, 4, 2, 1, 3)
    CGPT_KG_CASE(6, 128, 128, 4, 2, 1, 4)
    CGPT_KG_CASE(7, 192, 96, 4, 2, 1, 4)
    default: return CGPT_EINVAL;
  }
#undef CGPT_KG_CASE
}

template <typename TIn, typename TOut>
static int launch_kgroup_out(int epi, int tile, const void* a, const void* w, const void* bias, bool bias_half,
                             void* c, int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                             hipStream_t s) {
#define CGPT_KG_EPI(E)                                                                                 \
  case E:                                                                                              \
    return launch_kgroup_epi<TIn, E, TOut>(tile, a, w, bias, bias_half, c, M, N, K, lda, ldw, ldc, s);
  switch (epi) {
    CGPT_KG_EPI(CGPT_EPI_NONE)
    CGPT_KG_EPI(CGPT_EPI_BIAS)
    CGPT_KG_EPI(CGPT_EPI_BIAS_GELU)
    CGPT_KG_EPI(CGPT_EPI_BIAS_RESID)
    default: return CGPT_EINVAL;
  }
#undef CGPT_KG_EPI
}

bool gemm_kgroup_ok(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int64_t ldc, const void* c,
                    bool out16) {
  const int64_t lim = int64_t{1} << 31, es = out16 ? 2 : 4;
  return K % 64 == 0 && N % 4 == 0 && ldc % 4 == 0 && reinterpret_cast<uintptr_t>(c) % (4 * es) == 0 &&
         M * lda * 2 < lim && N * ldw * 2 < lim && M * ldc * es < lim;
}

int launch_gemm_kgroup(bool f16, int epilogue, int tile, const void* a, const void* w, const void* bias,
                       bool bias_half, void* c, bool out16, int M, int N, int K, int64_t lda, int64_t ldw,
                       int64_t ldc, hipStream_t s) {
  if (f16)
    return out16 ? launch_kgroup_out<f16_t, f16_t>(epilogue, tile, a, w, bias, bias_half, c, M, N, K, lda, ldw, ldc, s)
                 : launch_kgroup_out<f16_t, float>(epilogue, tile, a, w, bias, bias_half, c, M, N, K, lda, ldw, ldc, s);
  return out16 ? launch_kgroup_out<bf16_t, bf16_t>(epilogue, tile, a, w, bias, bias_half, c, M, N, K, lda, ldw, ldc, s)
               : launch_kgroup_out<bf16_t, float>(epilogue, tile, a, w, bias, bias_half, c, M, N, K, lda, ldw, ldc, s);
}

}  // namespace cgpt
