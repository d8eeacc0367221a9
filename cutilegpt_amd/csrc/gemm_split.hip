// fp32 GEMM on the bf16 matrix cores: C[M,N] = epilogue(A[M,K] W[N,K]^T + bias).
//
// The fp32 MFMA runs at 1/16 of the bf16 rate.  Each fp32 operand is split
// exactly into three bf16 values, x = h + m + l (h = bf16(x), m = bf16(x - h),
// l = x - h - m, round to nearest; 8 + 8 + 8 significant bits), and the product
// is the six bf16 products whose size is at least 2^-18 of h h:
//     h h + (h m + m h) + (h l + l h + m m),
// all accumulated in fp32 by the MFMA.  The dropped m l, l m and l l are below
// 2^-26 of the product, a quarter of fp32's own rounding of it, and one MFMA
// adds 16 products at a time where the fp32 one adds 4: the error against
// float64 is below the fp32 MFMA's (K = 768: 4.3e-7 against 5.0e-7 of the
// result's norm, K = 6400: 1.27e-6 against 1.43e-6).  The small tiles, which add
// the small terms up apart, leave a third of that: 50 rows through a 768-wide
// MLP 1.7e-7 (the skinny kernel 4.1e-7), 48 x 50257 x 768 8.8e-8 (1.8e-7).
//
// Both operands are split at 2^23 times their size (split.h), so that no part of
// a small value is subnormal, and the sums are scaled back by 2^-46.  A block
// whose sums are not all finite computes its tile again with the fp32 MFMA
// straight from global memory: infinities, NaN, values of 2^105 and more, and
// sums of 2^82 and more (those that overflow fp32 among them).
#include "common.h"
#include "gemm_common.h"
#include "internal.h"
#include "split.h"

namespace cgpt {

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void mfma32(const u32x4_t& a, const u32x4_t& b, f32x16_t& c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                              __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
#endif

// A block of KG groups of WGM x WGN wavefronts owns a BM x BN tile; group i
// takes the k16 stages i, i + KG, ... with LDS buffers of its own, and the
// groups' sums are added through LDS at the end (problems with fewer tiles
// than the chip has room for get their waves from K).
//
// Stages are double-buffered in LDS.  While a stage is multiplied, the fp32
// values of the group's next one, loaded a whole step before, are split by the
// threads that hold them (each element once a block) and written to the other
// buffer, and the loads of the one after go out.  An operand's stage is
// [plane][k half][row] 16-byte chunks (8 k of one row); each run of rows is
// followed by 64 bytes so that the 8-byte writes of the runs fall in different
// banks, and a fragment read takes 32 consecutive chunks of both halves.
template <int BM, int BN, int WGM, int WGN, int KG, int PD, int EPI, typename TOut>
__global__ __launch_bounds__(64 * WGM * WGN * KG, BM * BN == 128 * 128 && KG == 1 ? 3 : 2) void gemm_split_kernel(
    const float* __restrict__ A, const float* __restrict__ W, const void* __restrict__ bias,
    bool bias_bf16, TOut* __restrict__ C, int M, int N, int K, int lda, int ldw, int64_t ldc,
    int tiles_m, int tiles_n, bool vec_store) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = WGM * WGN, NT = 64 * NW;  // one group's waves and threads
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "32x32 MFMA tiles");
  // Waves of one 32x32 product have the registers to keep the five smaller
  // products' sums (2^-8 of h h) apart: one rounding of the large sum a stage,
  // not six, and two chains of MFMAs, not one.
  constexpr bool kLow = TM * TN == 1;
  constexpr int BK = 16, QPR = BK / 4;  // 16-byte fp32 chunks a row and stage
  constexpr int A_LD = BM * QPR / NT, W_LD = BN * QPR / NT;
  static_assert(BM * QPR % NT == 0 && BN * QPR % NT == 0, "tile/thread mismatch");
  constexpr int A_RUN = BM * 16 + 64, W_RUN = BN * 16 + 64;
  constexpr int A_PLANE = 2 * A_RUN, W_PLANE = 2 * W_RUN;
  constexpr int STAGE = 3 * (A_PLANE + W_PLANE);
  constexpr int QUADS = TM * TN * 4;      // 4-register quads of a wave's accumulators
  constexpr int OWN = QUADS > KG ? QUADS / KG : 1;  // quads a group finishes (the first QUADS groups, if fewer)
  static_assert(QUADS % KG == 0 || KG > QUADS, "groups share the tile's quads evenly");
  constexpr int XCH = KG > 1 ? QUADS * (KG - 1) * NW * 1024 : 0;
  constexpr int SMEM = 2 * STAGE * KG > XCH ? 2 * STAGE * KG : XCH;
  static_assert(SMEM <= 160 * 1024, "LDS budget of one CU");
  __shared__ __attribute__((aligned(16))) uint8_t smem[SMEM];

  const int lane = threadIdx.x & 63;
  const int bwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = KG > 1 ? bwave / NW : 0, wave = KG > 1 ? bwave % NW : bwave;
  const int tid = wave * 64 + lane;
  const int wm0 = (wave / WGN) * WM, wn0 = (wave % WGN) * WN;
  const int r32 = lane & 31, g = lane >> 5;

  int tile_m, tile_n;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const uint8_t* ab = reinterpret_cast<const uint8_t*>(A + static_cast<int64_t>(m0) * lda);
  const uint8_t* wb = reinterpret_cast<const uint8_t*>(W + static_cast<int64_t>(n0) * ldw);

  // Byte offsets of this thread's rows in the tile, unsigned: the host keeps a
  // tile's rows within 4 GiB (256 rows less than 2^22 floats apart); rows past the matrix are clamped to the last one
  // (loaded, never stored).
  uint32_t ao[A_LD], wo[W_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i)
    ao[i] = static_cast<uint32_t>(min((tid + i * NT) / QPR, M - 1 - m0) * lda) * 4;
#pragma unroll
  for (int i = 0; i < W_LD; ++i)
    wo[i] = static_cast<uint32_t>(min((tid + i * NT) / QPR, N - 1 - n0) * ldw) * 4;
  const int kq = tid % QPR;
  u32x4_t ra[PD][A_LD], rw[PD][W_LD];
  // k past K is loaded from the row's last chunk and zeroed before the split.
  auto koff = [&](int kt) { return static_cast<uint32_t>(min(kt * BK + kq * 4, K - 4)) * 4; };
  auto load_a = [&](int d, int i, uint32_t ko) {
    ra[d][i] = *reinterpret_cast<const u32x4_t*>(ab + (ao[i] + ko));
  };
  auto load_w = [&](int d, int i, uint32_t ko) {
    rw[d][i] = *reinterpret_cast<const u32x4_t*>(wb + (wo[i] + ko));
  };
  auto put = [&](uint8_t* base, int run, int plane, int row, const u32x4_t& v) {
    u32x2_t h, m, l;
    split3(v, kSplitUp, h, m, l);
    uint8_t* p = base + (kq >> 1) * run + row * 16 + (kq & 1) * 8;
    *reinterpret_cast<u32x2_t*>(p) = h;
    *reinterpret_cast<u32x2_t*>(p + plane) = m;
    *reinterpret_cast<u32x2_t*>(p + 2 * plane) = l;
  };
  uint8_t* const gbase = smem + grp * 2 * STAGE;
  // Chunk c (A's, then W's) of stage kt from register set d into buffer `buf`,
  // its register reloaded with the stage at `ko`.  `whole`: the stage is known
  // to end within K.
  constexpr int NCH = A_LD + W_LD;
  auto put_chunk = [&](int c, int d, int kt, int buf, uint32_t ko, bool whole) {
    const bool live = whole || kt * BK + kq * 4 < K;
    uint8_t* sa = gbase + buf * STAGE;
    if (c < A_LD) {
      if (!whole) ra[d][c] = live ? ra[d][c] : u32x4_t{0, 0, 0, 0};
      put(sa, A_RUN, A_PLANE, (tid + c * NT) / QPR, ra[d][c]);
      load_a(d, c, ko);
    } else {
      const int w = c - A_LD;
      if (!whole) rw[d][w] = live ? rw[d][w] : u32x4_t{0, 0, 0, 0};
      put(sa + 3 * A_PLANE, W_RUN, W_PLANE, (tid + w * NT) / QPR, rw[d][w]);
      load_w(d, w, ko);
    }
  };
  // A group of one wave shares its buffers with no other wave.
  auto stage_sync = [&]() {
    wait_lgkm0();
    if constexpr (NW > 1) raw_barrier(); else asm volatile("" ::: "memory");
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  f32x16_t low;
#pragma unroll
  for (int r = 0; r < 16; ++r) low[r] = 0.f;

  const int KT = (K + BK - 1) / BK;
  const int iters = (KT + KG - 1) / KG;  // the same for every group: a stage past K is zero
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    const uint32_t ko = koff(grp + d * KG);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) load_a(d, i, ko);
#pragma unroll
    for (int i = 0; i < W_LD; ++i) load_w(d, i, ko);
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c) put_chunk(c, 0, grp, 0, koff(grp + PD * KG), false);
  stage_sync();
  // One step: multiply stage it (buffer it & 1) and put stage it + 1 (register
  // set d) into the other buffer.
  auto step = [&](int it, int buf, int d, bool whole) {
    const uint8_t* sa = gbase + buf * STAGE + g * A_RUN + (wm0 + r32) * 16;
    const uint8_t* sw = gbase + buf * STAGE + 3 * A_PLANE + g * W_RUN + (wn0 + r32) * 16;
    u32x4_t af[3][TM], wf[3][TN];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[p][i] = *reinterpret_cast<const u32x4_t*>(sa + p * A_PLANE + i * 512);
#pragma unroll
      for (int j = 0; j < TN; ++j) wf[p][j] = *reinterpret_cast<const u32x4_t*>(sw + p * W_PLANE + j * 512);
    }
    // The next stage's chunks go between the MFMAs, one MFMA and its share of
    // the splitting at a time, so that the vector unit works while the matrix
    // core does (16384 x 3072 x 768 450 -> 406 us, 4096 x 768 x 3072 127 -> 121,
    // against the whole split before the first MFMA, which also spilled).
    constexpr int NMF = 6 * TM * TN;
    const int kt = (it + 1) * KG + grp;
    const uint32_t ko = koff((it + 1 + PD) * KG + grp);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      put_chunk(c, d, kt, buf ^ 1, ko, whole);
#pragma unroll
      for (int x = c * NMF / NCH; x < (c + 1) * NMF / NCH; ++x)
        mfma32(wf[kSplitA[x / (TM * TN)]][x % TN], af[kSplitB[x / (TM * TN)]][x / TN % TM],
               kLow && x > 0 ? low : acc[x / TN % TM][x % TN]);
#pragma unroll
      for (int x = c * NMF / NCH; x < (c + 1) * NMF / NCH; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                              // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (32 * NCH + NMF - 1) / NMF, 0);  // VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stage_sync();
  };
  if constexpr (PD == 1) {
    // Steps whose next stage is whole for every group, then the others (the
    // stage after the last one is zero and never read).
    const int n_whole = K / BK / KG - 1;
    int it = 0;
    for (; it < n_whole; ++it) step(it, it & 1, 0, true);
    for (; it < iters; ++it) step(it, it & 1, 0, false);
  } else {
    static_assert(PD == 1 || PD % 2 == 0, "buffer parity of the unrolled steps");
    // Stages past K are zero: up to PD - 1 more of them, and the loop needs no exits.
    for (int it = 0; it < iters; it += PD)
#pragma unroll
      for (int u = 0; u < PD; ++u) step(it + u, u & 1, (u + 1) % PD, false);
  }
  if constexpr (kLow) acc[0][0] += low;
  if constexpr (NW == 1 && KG > 1) __syncthreads();

  // Each group adds the others' sums of its quads (in group order).
  if constexpr (KG > 1) {
    f32x4_t* x = reinterpret_cast<f32x4_t*>(smem);
    auto slot = [&](int owner, int src, int quad) {  // src: the writer's place among the others
      return ((owner * (KG - 1) + src) * OWN + quad) * NT + tid;
    };
#pragma unroll
    for (int q = 0; q < QUADS; ++q) {
      const int owner = q / OWN;
      if (owner != grp) {
        const f32x16_t& t = acc[q / 4 / TN][q / 4 % TN];
        const int e = 4 * (q % 4);
        x[slot(owner, grp - (grp > owner), q % OWN)] = f32x4_t{t[e], t[e + 1], t[e + 2], t[e + 3]};
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QUADS; ++q) {
      if (q / OWN == grp) {
        f32x16_t& t = acc[q / 4 / TN][q / 4 % TN];
        const int e = 4 * (q % 4);
#pragma unroll
        for (int o = 0; o < KG - 1; ++o) {
          const f32x4_t v = x[slot(q / OWN, o, q % OWN)];
#pragma unroll
          for (int r = 0; r < 4; ++r) t[e + r] += v[r];
        }
      }
    }
  }

  // x * 0 is NaN exactly for infinities and NaN.
  float chk = 0.f;
#pragma unroll
  for (int q = 0; q < QUADS; ++q)
    if (q / OWN == grp)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        chk = __builtin_fmaf(acc[q / 4 / TN][q / 4 % TN][4 * (q % 4) + r], 0.f, chk);
  float down = kSplitDown * kSplitDown;
  if (__syncthreads_or(chk != chk)) {
    down = 1.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        // Lane l supplies row l % 32 of both operands, and of every 2 KV k the KV
        // from KV (l / 32) on (any one order of k serves).  Four k a load, one
        // where the accumulators leave no registers for it (one -> four, a NaN in
        // every tile: 4096 x 3072 x 768 1088 -> 400 us, 87 rows of it 177 -> 57).
        constexpr int KV = TM * TN > 4 ? 1 : 4;
        const float* pa = A + static_cast<int64_t>(min(m0 + wm0 + i * 32 + r32, M - 1)) * lda;
        const float* pw = W + static_cast<int64_t>(min(n0 + wn0 + j * 32 + r32, N - 1)) * ldw;
        f32x16_t t;
#pragma unroll
        for (int r = 0; r < 16; ++r) t[r] = 0.f;
        for (int k0 = 0; k0 < K; k0 += 2 * KV) {
          const int k = k0 + KV * g, at = min(k, K - KV);
          float va[KV], vw[KV];
#pragma unroll
          for (int e = 0; e < KV; ++e) va[e] = pa[at + e], vw[e] = pw[at + e];
#pragma unroll
          for (int e = 0; e < KV; ++e)
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(k < K ? vw[e] : 0.f, k < K ? va[e] : 0.f, t, 0, 0, 0);
        }
        acc[i][j] = t;
      }
  }

  // Lane (g, r32) holds C[m = r32][n = 8 q + 4 g + r] in element 4 q + r.
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    if (q / OWN != grp) continue;
    const int i = q / 4 / TN, j = q / 4 % TN, e = 4 * (q % 4);
    const int m = m0 + wm0 + i * 32 + r32;
    const int n = n0 + wn0 + j * 32 + 2 * e + 4 * g;
    if (m >= M || n >= N) continue;
    TOut* out = C + static_cast<int64_t>(m) * ldc + n;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float t = acc[i][j][e + r] * down;
      if (EPI != CGPT_EPI_NONE && n + r < N)
        t += bias_bf16 ? bf16_to_f32(static_cast<const bf16_t*>(bias)[n + r])
                       : static_cast<const float*>(bias)[n + r];
      if (EPI == CGPT_EPI_BIAS_GELU) t = gelu_tanh(t);
      if (EPI == CGPT_EPI_BIAS_RESID && n + r < N) t += Elem<TOut>::load(out + r);
      v[r] = t;
    }
    if (vec_store && n + 3 < N) {
      store4_out(out, v);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) Elem<TOut>::store(out + r, v[r]);
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <int BM, int BN, int WGM, int WGN, int KG, int PD, int EPI, typename TOut>
static int launch_split_tile(const float* a, const float* w, const void* bias, bool bias_bf16, TOut* c,
                             int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                             bool vec_store, hipStream_t s) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int64_t tiles = static_cast<int64_t>(tiles_m) * tiles_n;
  if (tiles > 0x7fffffff) return CGPT_ESHAPE;
  hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WGM, WGN, KG, PD, EPI, TOut>),
                     dim3(static_cast<unsigned>(tiles)), dim3(64 * WGM * WGN * KG), 0, s, a, w, bias,
                     bias_bf16, c, M, N, K, static_cast<int>(lda), static_cast<int>(ldw), ldc,
                     tiles_m, tiles_n, vec_store);
  return hip_status(hipGetLastError());
}

// Tiles, by id: {rows, columns, K groups}.
enum SplitTile { k256x256, k128x128, k128x128k2, k128x64k2, k64x64k4, k32x32k4, k32x32k8 };

template <int EPI, typename TOut>
static int launch_split_epi(int tile, const void* a, const void* w, const void* bias, bool bias_bf16,
                            void* c, int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                            bool vec_store, hipStream_t s) {
#define CGPT_SPLIT_CASE(id, BM, BN, WGM, WGN, KG, PD)                                               \
  case id:                                                                                          \
    return launch_split_tile<BM, BN, WGM, WGN, KG, PD, EPI, TOut>(                                   \
        static_cast<const float*>(a), static_cast<const float*>(w), bias, bias_bf16,                 \
        static_cast<TOut*>(c), M, N, K, lda, ldw, ldc, vec_store, s);
  switch (tile) {
    CGPT_SPLIT_CASE(k256x256, 256, 256, 2, 4, 1, 1)
    CGPT_SPLIT_CASE(k128x128, 128, 128, 2, 2, 1, 1)
    CGPT_SPLIT_CASE(k128x128k2, 128, 128, 2, 2, 2, 1)
    CGPT_SPLIT_CASE(k128x64k2, 128, 64, 2, 2, 2, 1)
    CGPT_SPLIT_CASE(k64x64k4, 64, 64, 2, 2, 4, 2)
    CGPT_SPLIT_CASE(k32x32k4, 32, 32, 1, 1, 4, 4)
    CGPT_SPLIT_CASE(k32x32k8, 32, 32, 1, 1, 8, 2)
    default: return CGPT_EINVAL;
  }
#undef CGPT_SPLIT_CASE
}

// The tile of a problem, from a sweep of 15 tiles over 19 shapes (us a launch,
// replayed from a graph; the fp32-MFMA kernel this replaces first):
//  * 256x256 (8 waves, one block a CU; half the LDS reads a product of the
//    others) when it fills three quarters of its rounds over the CUs and its
//    rows take 16-byte stores: 16384 x 3072 x 768 655 -> 382 (128x128 425); its
//    epilogue overlaps nothing, so scalar stores go to the smaller tiles:
//    1000 x 50257 x 768 732 -> 509 with 128x128 (256x256 566);
//  * 128x128, three blocks a CU, from 2.5 of them a CU: 4096 x 3072 x 768
//    201 -> 123; of one row of tiles and K up to 256 from one a CU: 100 x 50257 x
//    128 30.2 (128x64 34.5), 70 x 50304 x 256 26.0 (32.8), x 384 the same;
//  * fewer, and long K: 128x128 with two K groups, 4096 x 768 x 3072 173 -> 123
//    (one group 156), 1500 x 1600 x 6400 351 -> 220 (128x64 239);
//  * 128x64 with two K groups: 4096 x 2304 x 768 138 -> 96, 4096 x 768 x 768
//    48 -> 38 (128x128 with two 39), 520 x 3072 x 768 37 -> 24,
//    and whenever 64x64 tiles, one block a CU, would need a second round:
//    1500 x 768 x 768 24.2 (64x64 29.8), 7000 x 192 x 192 11.8 (16.9);
//  * 64x64 with four K groups from 5/8 of a tile a CU: 200 x 3072 x 768
//    24 -> 15 (128x64 21, 32x32 18), and when 32x32 tiles, two blocks a CU, would
//    need a second round: 1500 x 384 x 768 16.0 (32x32 20.3), x 128 7.5 (11.4);
//    up to K = 128 when they are more than one a CU: 900 x 384 x 96 7.0 (7.8);
//  * 32x32, a wave a K group: eight groups while that is one round of blocks,
//    87 x 768 x 3072 77 -> 20 (64x64 38), 87 x 2304 x 768 23 -> 8.8; four
//    beyond (two blocks a CU), 65 x 3072 x 768 22 -> 12.2 (eight: 15); of
//    64 rows or fewer those beyond are one row of tiles, 64 x 4800 x 1600 26.9
//    with 64x64 (32x32 29.2), 64 x 50304 x 768 73 (32x32 90, 128x128 78).
static int split_tile(int M, int N, int K, bool vec_store) {
  const int64_t cus = num_cus();
  auto tiles = [&](int bm, int bn) {
    return static_cast<int64_t>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  };
  if (M <= 64) return tiles(32, 32) <= cus ? k32x32k8 : M <= 32 ? k32x32k4 : k64x64k4;
  const int64_t t256 = tiles(256, 256), rounds = (t256 + cus - 1) / cus;
  if (t256 >= cus && vec_store && 4 * t256 >= 3 * rounds * cus) return k256x256;
  const int64_t t128 = tiles(128, 128);
  if (2 * t128 >= 5 * cus || (M <= 128 && t128 > cus && K <= 256)) return k128x128;
  if (2 * t128 >= cus && K >= 1536) return k128x128k2;
  const int64_t t64 = tiles(64, 64), t32 = tiles(32, 32);
  if (8 * tiles(128, 64) >= 6 * cus || t64 > cus) return k128x64k2;
  if (8 * t64 >= 5 * cus || t32 > (K <= 128 ? 1 : 2) * cus) return k64x64k4;
  return t32 <= cus ? k32x32k8 : k32x32k4;
}

bool gemm_split_ok(int64_t lda, int64_t ldw) { return lda < (1 << 22) && ldw < (1 << 22); }

int launch_gemm_split(int epilogue, int tile, const void* a, const void* w, const void* bias,
                      bool bias_bf16, void* c, bool out_bf16, int M, int N, int K, int64_t lda,
                      int64_t ldw, int64_t ldc, bool vec_store, hipStream_t s) {
  const int t = tile == 0 ? k128x128 : tile == 1 ? k64x64k4 : split_tile(M, N, K, vec_store);
#define CGPT_SPLIT_EPI(E)                                                                          \
  case E:                                                                                          \
    return out_bf16 ? launch_split_epi<E, bf16_t>(t, a, w, bias, bias_bf16, c, M, N, K, lda, ldw,   \
                                                  ldc, vec_store, s)                               \
                    : launch_split_epi<E, float>(t, a, w, bias, bias_bf16, c, M, N, K, lda, ldw,    \
                                                 ldc, vec_store, s);
  switch (epilogue) {
    CGPT_SPLIT_EPI(CGPT_EPI_NONE)
    CGPT_SPLIT_EPI(CGPT_EPI_BIAS)
    CGPT_SPLIT_EPI(CGPT_EPI_BIAS_GELU)
    CGPT_SPLIT_EPI(CGPT_EPI_BIAS_RESID)
    default: return CGPT_EINVAL;
  }
#undef CGPT_SPLIT_EPI
}

}  // namespace cgpt
