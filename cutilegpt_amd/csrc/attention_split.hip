// Causal flash attention for fp32 inputs of head_dim 64 on the bf16 matrix
// cores: Q, K, V and the probabilities as three bf16 parts each (split.h), six
// MFMAs in place of an fp32 product whose MFMA runs at 1/16 of the rate.
//
// The work split and the formulation are attn_fwd_dma_kernel's (attention.hip):
// four waves a block, 16 queries a sub-tile, 64-key blocks, S^T = K Q^T so that
// a lane owns one query, O^T = V^T P^T with P from the S^T registers and V^T
// through the transposing LDS read, the running maximum moved only when a
// row's grows by more than 2^8.  K and V come through registers: the thread
// that loads four values splits them and writes each part to its own row-major
// plane, the planes of one key block filling 48 KiB (three blocks a CU hide the
// two barriers around a refill).
//
// K, V and P are split at 2^23 times their size (split.h: no part of a small
// value is subnormal), Q at 2^-23, so that the scores keep their size and
// overflow where fp32's do; the sums of P V are scaled back with the normaliser.
// A block whose sums are not all finite (infinities or NaN in the inputs, values
// of K and V of 2^105 and more) or whose Q has a value below 2^-80, whose scaled
// parts bf16 cannot hold, computes its rows again with the fp32 MFMA.
#include "common.h"
#include "internal.h"
#include "split.h"

namespace cgpt {

constexpr int kAsThreads = 256;
[[maybe_unused]] constexpr int kAsBKV = 64, kAsHD = 64;  // keys a block, head_dim

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void mfma_bf16(const u32x4_t& a, const u32x4_t& b, f32x4_t& c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                              __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// One wave's 16 queries with fp32 products, keys 16 at a time straight from
// global memory.  q, k, v: the (batch, head)'s rows; lane l's query qi, its
// last visible key lim; kv_end: keys the 16 queries need.
__device__ __forceinline__ void attn_rows_fp32(const float* q, const float* k, const float* v, int64_t k_st,
                                            int64_t v_st, int Tk, int kv_end, int lim, float scale_log2,
                                            int lane, f32x4_t* o, float* l_out) {
  const int g = lane >> 4, frow = lane & 15;
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
  for (int dt = 0; dt < kAsHD / 16; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int kv0 = 0; kv0 < kv_end; kv0 += 16) {
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
    const float* krow = k + static_cast<int64_t>(min(kv0 + frow, Tk - 1)) * k_st;
#pragma unroll
    for (int c = 0; c < kAsHD / 16; ++c)
      Mfma<float>::run(*reinterpret_cast<const u32x4_t*>(krow + 16 * c + 4 * g),
                       *reinterpret_cast<const u32x4_t*>(q + 16 * c + 4 * g), s);
    float mloc = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (kv0 + 4 * g + r > lim) s[r] = -INFINITY;
      mloc = fmaxf(mloc, s[r]);
    }
    const float m_new = fmaxf(m_run, column_max(mloc) * scale_log2);
    const float alpha = m_new == m_run ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    const float neg_m = m_run == -INFINITY ? 0.f : -m_run;  // only masked keys so far: p is 0
    l_run *= alpha;
    u32x4_t p;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale_log2, neg_m));
      p[r] = __float_as_uint(e);
      l_run += e;
    }
#pragma unroll
    for (int dt = 0; dt < kAsHD / 16; ++dt) {
      u32x4_t vf;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        vf[j] = __float_as_uint(v[static_cast<int64_t>(min(kv0 + 4 * g + j, Tk - 1)) * v_st + dt * 16 + frow]);
      f32x4_t t = o[dt];
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] *= alpha;
      Mfma<float>::run(vf, p, t);
      o[dt] = t;
    }
  }
  *l_out = l_run;
}
#endif

template <int QT>
__global__ __launch_bounds__(kAsThreads, QT == 1 ? 3 : 2) void attn_fwd_split_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    float* __restrict__ O, int H, int Tq, int Tk, int64_t q_sb, int64_t q_sh, int64_t q_st,
    int64_t k_sb, int64_t k_sh, int64_t k_st, int64_t v_sb, int64_t v_sh, int64_t v_st,
    int64_t o_sb, int64_t o_sh, int64_t o_st, float scale_log2, int causal, int n_bh) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int HD = kAsHD, BKV = kAsBKV, BQ = 4 * 16 * QT;
  constexpr int KROW = HD * 2;           // bytes of a plane's row
  constexpr int PLANE = BKV * KROW;
  constexpr int CPR = HD / 4;            // 16-byte fp32 chunks a row
  constexpr int LD = BKV * CPR / kAsThreads;
  constexpr int NKS = HD / 32, ND = HD / 16;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[6 * PLANE];
  uint8_t* const sk = smem;
  uint8_t* const sv = smem + 3 * PLANE;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, frow = lane & 15;
  const int n_qblk = (Tq + BQ - 1) / BQ;
  const int qb = n_qblk - 1 - static_cast<int>(blockIdx.x) / n_bh;  // heavy blocks first
  const int bh = static_cast<int>(blockIdx.x) % n_bh;
  const int b = bh / H, h = bh % H;
  const int q0 = qb * BQ;
  const int off = Tk - Tq;
  const float* Qb = Q + b * q_sb + h * q_sh;
  const float* Kb = K + b * k_sb + h * k_sh;
  const float* Vb = V + b * v_sb + h * v_sh;

  const int last_q = min(q0 + BQ, Tq) - 1 + off;
  const int kv_end = causal ? min(last_q + 1, Tk) : Tk;
  const int n_kv = (kv_end + BKV - 1) / BKV;
  const int wave_q0 = q0 + wave * 16 * QT;
  const int wave_last = min(wave_q0 + 16 * QT, Tq) - 1 + off;
  const bool wave_live = wave_q0 < Tq;

  // Thread (row tid / CPR, chunk tid % CPR) of every 16 rows.
  const int lrow = tid / CPR, lchunk = tid % CPR;
  u32x4_t rk[LD], rv[LD];
  auto gload = [&](int j) {
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int64_t key = min(j * BKV + lrow + i * (kAsThreads / CPR), Tk - 1);
      rk[i] = *reinterpret_cast<const u32x4_t*>(Kb + key * k_st + lchunk * 4);
      rv[i] = *reinterpret_cast<const u32x4_t*>(Vb + key * v_st + lchunk * 4);
    }
  };
  // 16-byte chunk c of a plane's row r sits at chunk c ^ (r & 7).
  auto swrite = [&]() {
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      const int row = lrow + i * (kAsThreads / CPR);
      const int at = row * KROW + (((lchunk >> 1) ^ (row & 7)) << 4) + (lchunk & 1) * 8;
      u32x2_t hh, mm, ll;
      split3(rk[i], kSplitUp, hh, mm, ll);
      *reinterpret_cast<u32x2_t*>(sk + at) = hh;
      *reinterpret_cast<u32x2_t*>(sk + PLANE + at) = mm;
      *reinterpret_cast<u32x2_t*>(sk + 2 * PLANE + at) = ll;
      split3(rv[i], kSplitUp, hh, mm, ll);
      *reinterpret_cast<u32x2_t*>(sv + at) = hh;
      *reinterpret_cast<u32x2_t*>(sv + PLANE + at) = mm;
      *reinterpret_cast<u32x2_t*>(sv + 2 * PLANE + at) = ll;
    }
  };

  gload(0);
  // Q's parts stay in registers for the whole key loop (rows past Tq: zero).
  u32x4_t qf[3][QT][NKS];
  bool odd = false;  // what the split does not hold was met
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int qi = q0 + wave * 16 * QT + qt * 16 + frow;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const float* p = Qb + static_cast<int64_t>(min(qi, Tq - 1)) * q_st + 32 * ks + 8 * g;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        u32x4_t v = *reinterpret_cast<const u32x4_t*>(p + 4 * x);
        if (qi >= Tq) v = u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; ++e) odd = odd || (v[e] << 1) - 1 < ((127u - 80) << 24) - 1;  // 0 < |v| < 2^-80
        u32x2_t hh, mm, ll;
        split3(v, kSplitDown, hh, mm, ll);
        qf[0][qt][ks][2 * x] = hh[0], qf[0][qt][ks][2 * x + 1] = hh[1];
        qf[1][qt][ks][2 * x] = mm[0], qf[1][qt][ks][2 * x + 1] = mm[1];
        qf[2][qt][ks][2 * x] = ll[0], qf[2][qt][ks][2 * x + 1] = ll[1];
      }
    }
  }

  f32x4_t o_acc[QT][ND];
  float nm[QT], l_run[QT];  // minus the running maximum (+inf: none yet), normaliser
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    nm[qt] = INFINITY;
    l_run[qt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) o_acc[qt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // V^T read: lane (g, k) of a 16-lane group points at row 4g + k/4 (plus the
  // slab's base key) and d = dt*16 + 4 (k % 4).
  const int tr_row = 4 * g + (frow >> 2), tr_byte = 8 * (frow & 3);
  auto vt_read = [&](const uint8_t* p0, int row, int dt) -> u32x2_t {
    const int byte = dt * 32 + tr_byte;
    const uint8_t* p = p0 + row * KROW + ((((byte >> 4) ^ (row & 7))) << 4) + (byte & 15);
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)((__attribute__((address_space(3))) uint8_t*)(p)));
    return __builtin_bit_cast(u32x2_t, r);
  };

  for (int j = 0; j < n_kv; ++j) {
    wait_lgkm0();
    raw_barrier();  // every wave's reads of the previous block have landed
    swrite();
    if (j + 1 < n_kv) gload(j + 1);
    wait_lgkm0();
    raw_barrier();
    const int kv0 = j * BKV;
    if (!wave_live || (causal && kv0 > wave_last)) continue;
    f32x4_t s[QT][4];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) s[qt][kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < 4; k0 += 2) {  // two key tiles at a time
      u32x4_t kf[3][NKS][2];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int kt = 0; kt < 2; ++kt) {
            const int key = (k0 + kt) * 16 + frow;
            kf[p][ks][kt] = *reinterpret_cast<const u32x4_t*>(sk + p * PLANE + key * KROW +
                                                              (((4 * ks + g) ^ (key & 7)) << 4));
          }
      // The small products of all of head_dim first: the running sum is then
      // rounded at its full size only by the last ones.
#pragma unroll
      for (int t = 5; t >= 0; --t)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
              mfma_bf16(kf[kSplitA[t]][ks][kt], qf[kSplitB[t]][qt][ks], s[qt][k0 + kt]);
    }
    constexpr float kLazyLog2 = 8.0f;
    if ((causal && kv0 + BKV - 1 > wave_q0 + off) || kv0 + BKV > Tk) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const int qpos = wave_q0 + qt * 16 + frow + off;
        const int lim = (causal ? min(qpos, Tk - 1) : Tk - 1) - kv0 - 4 * g;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[qt][kt][r] = (kt * 16 + r > lim) ? -INFINITY : s[qt][kt][r];
      }
    }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float mloc = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, s[qt][kt][r]);
      const float mblk = column_max(mloc) * scale_log2;
      const float m_old = -nm[qt];
      const bool grow = mblk > m_old + kLazyLog2;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m_new = grow ? mblk : m_old;
        const float alpha = grow ? __builtin_amdgcn_exp2f(m_old - m_new) : 1.0f;
        nm[qt] = -m_new;
        l_run[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o_acc[qt][dt][r] *= alpha;
      }
      float lsum = 0.f;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][kt][r], scale_log2, nm[qt]));
          s[qt][kt][r] = p;
          lsum += p;
        }
      l_run[qt] += lsum;
    }
    // O^T += V^T P^T, k-slab c = keys 32c .. 32c + 31.  A slab's sum is built
    // from zero and added once, so that O is rounded once a slab.
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u32x4_t pf[3][QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          u32x2_t hh, mm, ll;
          split3(__builtin_bit_cast(u32x4_t, s[qt][2 * c + x]), kSplitUp, hh, mm, ll);
          pf[0][qt][2 * x] = hh[0], pf[0][qt][2 * x + 1] = hh[1];
          pf[1][qt][2 * x] = mm[0], pf[1][qt][2 * x + 1] = mm[1];
          pf[2][qt][2 * x] = ll[0], pf[2][qt][2 * x + 1] = ll[1];
        }
#pragma unroll
      for (int d0 = 0; d0 < ND; d0 += 2) {
        u32x4_t vf[3][2];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int dt = 0; dt < 2; ++dt) {
            const u32x2_t lo = vt_read(sv + p * PLANE, 32 * c + tr_row, d0 + dt);
            const u32x2_t hi = vt_read(sv + p * PLANE, 32 * c + 16 + tr_row, d0 + dt);
            vf[p][dt] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
          }
        f32x4_t sum[QT][2];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int dt = 0; dt < 2; ++dt) sum[qt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 5; t >= 0; --t)
#pragma unroll
          for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
              mfma_bf16(vf[kSplitA[t]][dt], pf[kSplitB[t]][qt], sum[qt][dt]);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o_acc[qt][d0 + dt][r] += sum[qt][dt][r];
      }
    }
  }

  float chk = 0.f;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    chk = __builtin_fmaf(l_run[qt], 0.f, chk);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) chk = __builtin_fmaf(o_acc[qt][dt][r], 0.f, chk);
  }
  const bool redo = __syncthreads_or(odd || chk != chk) != 0;
  if (!wave_live) return;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int qi = wave_q0 + qt * 16 + frow;
    if (redo) {
      const int qpos = qi + off;
      f32x4_t o[ND];
      const int keys = causal ? min(kv_end, wave_q0 + qt * 16 + 16 + off) : kv_end;
      attn_rows_fp32(Qb + static_cast<int64_t>(min(qi, Tq - 1)) * q_st, Kb, Vb, k_st, v_st, Tk, keys,
                     causal ? min(qpos, Tk - 1) : Tk - 1, scale_log2, lane, o, &l_run[qt]);
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) o_acc[qt][dt] = o[dt];
    }
    const float l = column_sum(l_run[qt]);
    if (qi >= Tq) continue;
    const float inv = (l > 0.f ? 1.0f / l : 0.f) * (redo ? 1.0f : kSplitDown * kSplitDown);
    float* orow = O + b * o_sb + h * o_sh + qi * o_st;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = o_acc[qt][dt][r] * inv;
      store_vec(orow + dt * 16 + 4 * g, v);
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

int launch_attention_split(const float* q, const float* k, const float* v, float* o, int B, int H,
                           int Tq, int Tk, const int64_t* st, float scale, int causal, int queries,
                           hipStream_t s) {
  const int n_bh = B * H;
  const int64_t blocks = static_cast<int64_t>(n_bh) * ((Tq + queries - 1) / queries);
  if (blocks > 0x7fffffff) return CGPT_ESHAPE;
  const float scale_log2 = scale * 1.4426950408889634f;
#define CGPT_AS_LAUNCH(QT)                                                                           \
  hipLaunchKernelGGL((attn_fwd_split_kernel<QT>), dim3(static_cast<unsigned>(blocks)),               \
                     dim3(kAsThreads), 0, s, q, k, v, o, H, Tq, Tk, st[0], st[1], st[2], st[3], st[4], \
                     st[5], st[6], st[7], st[8], st[9], st[10], st[11], scale_log2, causal, n_bh)
  if (queries == 64)
    CGPT_AS_LAUNCH(1);
  else
    CGPT_AS_LAUNCH(2);
#undef CGPT_AS_LAUNCH
  return hip_status(hipGetLastError());
}

}  // namespace cgpt
