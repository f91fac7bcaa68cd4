// Small GEMMs on the fp32 MFMA: 32 x 32 output tiles, the contraction split
// over the waves of a workgroup.  Included by gemm.hip (inside no namespace).
//
// What bounds a small product is not its arithmetic: 256 x 128 over K = 64
// (a projection of the training demo) ran as two 128 x 128 workgroups walking
// k in steps of load, split, barrier and MFMA, behind a launch of its own that
// reduced the operands' maxima.  Here a tile is 32 x 32, every wave of the
// workgroup takes its own range of k straight from global memory into
// v_mfma_f32_32x32x2_f32 (the operands are fp32: no exponents, so no maxima to
// wait for, and no LDS stage or barrier before the sums), and the waves' sums
// meet in LDS once, added in wave order.  The maxima that a caller's buffers
// are to hold are taken from the fragments of the first tile column and row as
// they pass.  The fp32 products are exact (the split form keeps 22 bits), the
// sums are fp32 as there; an MFMA of this kind rounds after every two terms
// (the fp16 one after sixteen), so chunks of 32 k are summed apart and then
// added up: the error against fp64 stays below the split form's at every K.
//
// Fragments: 8 k per step, lane l holding k = 4 (l / 32) + e, e = 0 .. 3, of row
// (column) l % 32; MFMA e takes element e, so the order of k inside a step is
// e, 4 + e for both operands.  A k-contiguous operand's step is one float4 per
// lane (VEC; else four loads), the others' four loads of 32 consecutive floats.
// Four steps are in flight while the four before them multiply.
#pragma once

namespace {

constexpr int kSmallTile = 32;
constexpr int kSmallJobs = 16;
constexpr int kSmallWaves = 8;
constexpr int kSmallSteps = 4;  // steps of 8 k per batch of loads

struct SJob {
  const float* A;
  const float* B;
  float* C;
  const float* resid;
  float* O;    // SwiGLU output (the fused form)
  float* xpa;  // maxima to fill, or null
  float* xpb;
  int M, N, K, lda, ldb, beta;  // fused SwiGLU: N = H, C row stride 2 H
  int tile0;
};
struct STable {
  int count, tiles;
  float* partial;  // K pieces, [z][M][N]; null: one piece
  RopeEpi rope;    // cols 0: none
  SJob job[kSmallJobs];
};
static_assert(sizeof(STable) <= 4096, "the job table travels as a kernel argument (4 KB at most)");

// One step's four elements: k = k0 .. k0 + 3 of row i (element (i, k) at
// p[i ld + k], KC) or column i (at p[k ld + i]); zeros from kend on.
template <bool KC, bool VEC, bool CHECKED>
__device__ __forceinline__ void small_load(const float* __restrict__ p, int ld, int i, int k0, int kend,
                                           float (&x)[4]) {
  if constexpr (KC && VEC) {
    if (!CHECKED || k0 < kend) {
      const float4 v = *reinterpret_cast<const float4*>(p + (size_t)i * ld + k0);
      x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
      x[0] = x[1] = x[2] = x[3] = 0.f;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      x[e] = !CHECKED || k0 + e < kend ? (KC ? p[(size_t)i * ld + k0 + e] : p[(size_t)(k0 + e) * ld + i]) : 0.f;
  }
}

__device__ __forceinline__ float max4(float m, const float (&x)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) m = fmaxf(m, finite_abs(x[e]));
  return m;
}

// x, with inf as the NaN that its split form is in the other kernels.
__device__ __forceinline__ float inf_to_nan(float x) { return fmaf(x, 0.f, x); }

// blockIdx.x: tile of the table's jobs; blockIdx.y: K piece; wave w of the
// workgroup's W: k in [(y W + w) kc, + kc).  Dynamic LDS: (SW ? 2 : 1) * W * 4 KB.
template <bool AK, bool BKc, bool VEC, bool SW>
__global__ void __launch_bounds__(64 * kSmallWaves) gemm_small_kernel(STable t) {
  extern __shared__ float sm[];
  __shared__ float wmax[2][kSmallWaves];
  int q = 0;
  while (q + 1 < t.count && (int)blockIdx.x >= t.job[q + 1].tile0) ++q;
  const SJob& jb = t.job[q];
  const int M = jb.M, N = jb.N, K = jb.K, lda = jb.lda, ldb = jb.ldb;
  const int tile = blockIdx.x - jb.tile0, nTm = (M + 31) / 32, nTn = (N + 31) / 32;
  const int mt = tile / nTn, nt = tile - mt * nTn;
  const int W = blockDim.x >> 6, S = gridDim.y;
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kc = ((K + W * S - 1) / (W * S) + 7) & ~7;
  const int kbeg = min(K, ((int)blockIdx.y * W + wave) * kc), kend = min(K, kbeg + kc);
  // rows and columns past the edge repeat the last one: their sums are not stored
  const int ia = min(mt * 32 + (lane & 31), M - 1), ib = min(nt * 32 + (lane & 31), N - 1);
  const bool fill_a = jb.xpa && nt == 0, fill_b = jb.xpb && mt == 0;
  float ma = 0.f, mb = 0.f;
  f32x16 sum, sum2, acc, acc2;  // sums of whole chunks; the chunk's
#pragma unroll
  for (int i = 0; i < 16; ++i) sum[i] = 0.f;
  if constexpr (SW) sum2 = sum;

  float a[2][kSmallSteps][4], b[2][kSmallSteps][4], u[SW ? 2 : 1][kSmallSteps][4];
  auto load = [&](auto checked, auto stage, int k) {
    constexpr bool CH = decltype(checked)::value;
    constexpr int st = decltype(stage)::value;
#pragma unroll
    for (int s = 0; s < kSmallSteps; ++s) {
      const int k0 = k + 8 * s + 4 * half;
      small_load<AK, VEC, CH>(jb.A, lda, ia, k0, kend, a[st][s]);
      small_load<BKc, VEC, CH>(jb.B, ldb, ib, k0, kend, b[st][s]);
      if constexpr (SW) small_load<BKc, VEC, CH>(jb.B + (size_t)N * ldb, ldb, ib, k0, kend, u[st][s]);
    }
  };
  auto mma = [&](auto stage, int k) {
    constexpr int st = decltype(stage)::value;
#pragma unroll
    for (int s = 0; s < kSmallSteps; ++s) {
      if (k + 8 * s < kend) {
      if (fill_a) ma = max4(ma, a[st][s]);
      if (fill_b) {
        mb = max4(mb, b[st][s]);
        if constexpr (SW) mb = max4(mb, u[st][s]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float av = inf_to_nan(a[st][s][e]);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, inf_to_nan(b[st][s][e]), acc, 0, 0, 0);
        if constexpr (SW) acc2 = __builtin_amdgcn_mfma_f32_32x32x2f32(av, inf_to_nan(u[st][s][e]), acc2, 0, 0, 0);
      }
      }
    }
  };
  constexpr int kBatch = 8 * kSmallSteps;
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  auto fetch = [&](auto stage, int k) {
    if (k + kBatch <= kend)
      load(std::false_type(), stage, k);
    else if (k < kend)
      load(std::true_type(), stage, k);
  };
  fetch(C0(), kbeg);
  for (int k = kbeg; k < kend; k += 2 * kBatch) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if constexpr (SW) acc2 = acc;
    fetch(C1(), k + kBatch);
    mma(C0(), k);
    sum += acc;
    if constexpr (SW) sum2 += acc2;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if constexpr (SW) acc2 = acc;
    fetch(C0(), k + 2 * kBatch);
    mma(C1(), k + kBatch);
    sum += acc;
    if constexpr (SW) sum2 += acc2;
  }

  // the waves' sums, in wave order
  float* mine = sm + (size_t)wave * 1024;
#pragma unroll
  for (int r = 0; r < 16; ++r) mine[r * 64 + lane] = sum[r];
  if constexpr (SW) {
#pragma unroll
    for (int r = 0; r < 16; ++r) mine[(size_t)W * 1024 + r * 64 + lane] = sum2[r];
  }
  if (fill_a || fill_b) {
    ma = fg_wave_max(ma);
    mb = fg_wave_max(mb);
    if (lane == 0) {
      wmax[0][wave] = ma;
      wmax[1][wave] = mb;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (fill_a) {
      for (int w = 0; w < W; ++w) ma = fmaxf(ma, wmax[0][w]);
      jb.xpa[mt * S + blockIdx.y] = ma;
    }
    if (fill_b) {
      for (int w = 0; w < W; ++w) mb = fmaxf(mb, wmax[1][w]);
      jb.xpb[nt * S + blockIdx.y] = mb;
    }
  }
  if (tile == 0 && blockIdx.y == 0) {  // the parts that no workgroup writes
    if (jb.xpa)
      for (int i = nTm * S + threadIdx.x; i < kXpParts; i += blockDim.x) jb.xpa[i] = 0.f;
    if (jb.xpb)
      for (int i = nTn * S + threadIdx.x; i < kXpParts; i += blockDim.x) jb.xpb[i] = 0.f;
  }
  for (int o = threadIdx.x; o < 1024; o += blockDim.x) {
    const int r = o >> 6, l = o & 63;
    const int row = mt * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), col = nt * 32 + (l & 31);
    float s = sm[o];
    for (int w = 1; w < W; ++w) s += sm[w * 1024 + o];
    if constexpr (SW) {
      float s2 = sm[W * 1024 + o];
      for (int w = 1; w < W; ++w) s2 += sm[(W + w) * 1024 + o];
      if (row < M && col < N) {
        float* c = jb.C + (size_t)row * 2 * N;
        c[col] = s;
        c[N + col] = s2;
        jb.O[(size_t)row * N + col] = fg::swiglu_fwd1(s, s2);
      }
      continue;
    }
    if (t.rope.cols) {  // column pairs (even, odd) are neighbouring lanes
      const float other = __shfl_xor(s, 1);
      if (row < M && col < t.rope.cols) {
        const int pos = t.rope.pos0 + (t.rope.posStride > 0 ? row % t.rope.posStride : row);
        const size_t at = (size_t)pos * (t.rope.dH >> 1) + (col % t.rope.dH) / 2;
        const bool odd = col & 1;
        float x = odd ? other : s, y = odd ? s : other;
        rope_turn(x, y, t.rope.c[at], t.rope.s[at]);
        s = odd ? y : x;
      }
    }
    if (row >= M || col >= N) continue;
    const size_t e = (size_t)row * N + col;
    if (t.partial) {
      t.partial[(size_t)blockIdx.y * M * N + e] = s;
      continue;
    }
    if (jb.beta) s = jb.C[e] + s;
    if (jb.resid) s = jb.resid[e] + s;
    jb.C[e] = s;
  }
}

// When it pays, and with how many waves per tile and K pieces.  The lines come
// from a sweep of 45 shapes (each with its maxima, forward / input / weight
// gradient, us, other kernels -> these):
//   64^3               14.5 / 13.2 / 10.9 -> 6.3 / 6.3 / 6.1
//   256 x 64 x 128      9.4 / 20.5 / 21.2 -> 6.3 / 6.7 / 6.6   (M x K x N)
//   512^3              19.0 / 19.7 / 18.7 -> 11.4 / 15.0 / 8.7
//   1024 x 512 x 500   45.6 / 45.6 / 26.0 -> 16.0 / 14.1 / 12.7 (ragged)
//   512 x 512 x 1024   20.0 / 20.9 / 20.1 -> 16.0 / 14.0 / 12.8
//   1024^3             25.5 / 25.7 / 23.8 -> 43.6 / 39.2 / 37.9
// The fp32 MFMA's rate ends it at 2^28 products; at twice that where 64 rows
// or columns leave half of the other kernels' 128-row tiles empty (8192 x 1024
// over 64 as an input gradient 41 -> 25); earlier over a short K, where the
// loads of 32 x 32 tiles weigh more (4096 x 256 over 256 16.8 -> 17.8), and
// where 32-wide stores of a large output are the whole launch (2048 x 2048 over
// 32: 9.5 -> 13.9).
//
// Waves: as many as leave each 8 k, up to eight (more share the SIMDs' one MFMA
// pipe and halve the registers).  K pieces: a workgroup's CU takes 8 cycles per
// k, so few tiles over a long K (>= 1536: 5 us) are cut into pieces of 768 and
// more (their sum is a second launch of 3 us).
struct SmallPlan {
  int waves = 0;  // 0: not this kernel
  int splits = 1;
};
constexpr int64_t kSmallMax = (int64_t)1 << 28;  // M N K
inline int64_t small_tiles(int M, int N) { return (int64_t)((M + 31) / 32) * ((N + 31) / 32); }
inline int small_waves(int64_t tiles, int K) {
  int W = 1;
  while (W < kSmallWaves && tiles * W < 2048 && K / (2 * W) >= 8) W *= 2;
  return W;
}
inline SmallPlan plan_small(int M, int N, int K, int force_splits) {
  SmallPlan p;
  const int64_t T = small_tiles(M, N);
  const int64_t work = (int64_t)M * N * K;
  if (K <= 128   ? work >= kSmallMax / 2
      : K <= 256 ? work > kSmallMax / 4 * 3
                 : work > (M <= 64 || N <= 64 ? 2 : 1) * kSmallMax)
    return p;
  if (T > (K < 64 ? 1024 : 4096)) return p;
  const int W = small_waves(T, K);
  int S = force_splits ? force_splits : 1;
  if (!force_splits && K >= 1536)
    while (S < 16 && T * S < 256 && K / S >= 768) S *= 2;
  if ((int64_t)((M + 31) / 32) * S > kXpParts || (int64_t)((N + 31) / 32) * S > kXpParts) return p;
  p.waves = W;
  p.splits = S;
  return p;
}
inline bool small_vec(bool ak, bool bk, const float* A, const float* B, int K, int lda, int ldb) {
  return (!ak || (K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % 16 == 0)) &&
         (!bk || (K % 4 == 0 && ldb % 4 == 0 && (uintptr_t)B % 16 == 0));
}

template <bool AK, bool BKc, bool SW = false>
int launch_small(const STable& t, const SmallPlan& p, bool vec) {
  const dim3 grid((unsigned)t.tiles, (unsigned)p.splits), block(64 * p.waves);
  const size_t lds = (size_t)p.waves * 4096 * (SW ? 2 : 1);
  if (vec)
    FG_LAUNCH((gemm_small_kernel<AK, BKc, true, SW>), grid, block, lds, t);
  else
    FG_LAUNCH((gemm_small_kernel<AK, BKc, false, SW>), grid, block, lds, t);
  return FG_OK;
}
// A table of one GEMM; the maxima that xp's buffers lack are filled.
inline STable small_table(float* C, const float* A, const float* B, int M, int N, int K, int lda, int ldb, int beta,
                          const float* resid, const XpArgs& xp) {
  STable t;
  t.count = 1;
  t.tiles = (int)small_tiles(M, N);
  t.partial = nullptr;
  t.rope = RopeEpi{nullptr, nullptr, 0, 0, 0, 0};
  t.job[0] = SJob{A,     B, C, resid, nullptr, xp.have & 1 ? nullptr : xp.a, xp.have & 2 ? nullptr : xp.b, M, N, K, lda,
                  ldb, beta ? 1 : 0, 0};
  return t;
}

}  // namespace
