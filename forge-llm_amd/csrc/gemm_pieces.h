// GEMM on operands split ahead of time (included by gemm.hip, inside its
// anonymous namespace).
//
// The kernels of gemm.hip split every operand element into its fp16 pieces
// while staging it to LDS, once per workgroup that reads it: five VALU
// instructions per MFMA, and a register round trip for every tile, which held
// the widest of them at 53% MFMA busy (8192 x 4096 over K = 768: 175 us, 296
// fp32 TFLOP/s).  For outputs large enough to pay for it, the operands are
// split once instead:
//
//   * split_pieces_kernel reads each fp32 operand (either orientation) and
//     writes its pieces in the order the MFMA fragments take them:
//       [block of 32 rows][chunk of 16 k][hi | lo][lane 0..63][8 fp16]
//     lane l of a fragment holds row l % 32, k = 8 (l / 32) .. +7.  Rows and
//     k past the operand are zero pieces, so the GEMM needs no bounds checks
//     on its loads, whatever the sizes and strides of the fp32 operands.  8 B
//     per element: 5.0 - 5.3 TB/s, what a large copy reaches.
//   * pieces_tile copies the fragments of its tile straight into LDS
//     (global_load_lds, 1 KB per wave instruction, S - 1 chunks ahead) and
//     reads each back as one conflict-free ds_read_b128 per lane; its main
//     loop holds nothing but those reads, the MFMAs and one barrier per chunk.
//     The fragments of chunk c + 1 are read while chunk c multiplies.
//
// Every output element gets the same three products per 16-k chunk, in the
// same order, as in the other kernels.
//
// Measured in place (us, the GEMM alone, before -> after, then its split):
// 4096 x 28672 over K = 4096 with the SwiGLU epilogue 2536 -> 2159, 209; the
// four weight gradients of a 4096-wide layer over 4096 tokens 5345 -> 4541,
// 440; 8192 x 32000 over 768 1220 -> 1078, 40.  4096 x 28672 reaches 470 fp32
// TFLOP/s (1410 on the fp16 pipes, what a large library product reaches in
// fp16): the clock the card holds under a dense MFMA stream bounds it.  With
// short K or few columns the split costs what the GEMM gains (8192 x 4096
// over 768: 184 -> 152 + 17 and a launch), and plan_pieces leaves those.

struct SplitJob {
  const float* src;
  char* dst;
  const float* parts;  // the operand's partial maxima
  int rows, k, ld;     // the operand as rows x k
  int nkc, rbs;        // chunks of 16 k; blocks of 32 rows (padded to whole tiles)
  int kc;              // 1: element (r, k) at src[r*ld + k]; 0: at src[k*ld + r]
  int swh;             // > 0: row r of the operand is row swiglu_row(r, swh) of src
  int unit0;           // units of the jobs before this one
};
constexpr int kSplitJobs = 32;
struct SplitTable {
  int count, units;
  SplitJob job[kSplitJobs];
};
static_assert(sizeof(SplitTable) <= 4096, "the split table travels as a kernel argument (4 KB at most)");
constexpr int kSplitNC = 4;  // chunks per unit: a wave loads 32 rows x 64 k (256 B of each row) at once

inline int split_units(const SplitJob& j) { return (j.nkc + kSplitNC - 1) / kSplitNC * j.rbs; }

// One unit: a block of 32 rows x kSplitNC chunks, by one wave.  All loads of
// the unit are in flight before the first split.  Consecutive waves take
// consecutive k (kc) or consecutive row blocks (otherwise): the direction in
// which the source is contiguous.
__device__ __forceinline__ void split_unit(const SplitJob& j, int u, int e) {
  const int lane = threadIdx.x & 63;
  const int units_k = (j.nkc + kSplitNC - 1) / kSplitNC;
  int rb, c0;
  if (j.kc) {
    rb = u / units_k;
    c0 = (u - rb * units_k) * kSplitNC;
  } else {
    const int q = u / j.rbs;
    rb = u - q * j.rbs;
    c0 = q * kSplitNC;
  }
  int r = rb * 32 + (lane & 31);
  const bool in = r < j.rows;
  if (j.swh > 0 && in) r = swiglu_row(r, j.swh);
  float f[kSplitNC][8];
#pragma unroll
  for (int c = 0; c < kSplitNC; ++c) {
    const int k = (c0 + c) * 16 + (lane >> 5) * 8;
    if (j.kc && in && k + 8 <= j.k) {  // 16-byte loads at any element (rows of odd length)
      __builtin_memcpy(f[c], j.src + (size_t)r * j.ld + k, 16);
      __builtin_memcpy(f[c] + 4, j.src + (size_t)r * j.ld + k + 4, 16);
    } else if (j.kc) {
#pragma unroll
      for (int q = 0; q < 8; ++q) f[c][q] = in && k + q < j.k ? j.src[(size_t)r * j.ld + k + q] : 0.f;
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) f[c][q] = in && k + q < j.k ? j.src[(size_t)(k + q) * j.ld + r] : 0.f;
    }
  }
  char* d = j.dst + ((size_t)rb * j.nkc + c0) * 2048 + lane * 16;
#pragma unroll
  for (int c = 0; c < kSplitNC; ++c) {
    if (c0 + c >= j.nkc) break;
    u32x4 h, l;
    split8h(f[c], e, h, l);
    *reinterpret_cast<u32x4*>(d + c * 2048) = h;
    *reinterpret_cast<u32x4*>(d + c * 2048 + 1024) = l;
  }
}

__global__ void __launch_bounds__(256) split_pieces_kernel(SplitTable t) {
  const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int j = 0, have = -1, e = 0;
  for (int u = wave; u < t.units; u += gridDim.x * 4) {
    while (j + 1 < t.count && u >= t.job[j + 1].unit0) ++j;
    if (j != have) e = xp_exponent(t.job[have = j].parts);
    split_unit(t.job[j], u - t.job[j].unit0, e);
  }
}

// 16 bytes per lane from each src[i] + voff straight into LDS at `lds` + 1024 i +
// 16 * lane (lds wave-uniform).  The instructions have no register result; their
// arrival is waited for explicitly (wait_lds_loads).  m0, which holds the LDS
// address, cannot be named as clobbered (the compiler reserves it), so it is
// given back; once per four or six loads that costs nothing (4096 x 28672 over K
// = 4096 2362 us without, 2362 with, 2388 when every load gives it back).
__device__ __forceinline__ void loads_to_lds(uint32_t lds, const char* const (&src)[4], uint32_t voff) {
  uint32_t m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %5\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %6\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(m0)
      : "s"(lds), "v"(voff), "s"(src[0]), "s"(src[1]), "s"(src[2]), "s"(src[3])
      : "memory", "scc");
}
__device__ __forceinline__ void loads_to_lds(uint32_t lds, const char* const (&src)[6], uint32_t voff) {
  uint32_t m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %5\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %6\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %7\n\t"
      "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %8\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(m0)
      : "s"(lds), "v"(voff), "s"(src[0]), "s"(src[1]), "s"(src[2]), "s"(src[3]), "s"(src[4]), "s"(src[5])
      : "memory", "scc");
}
// All but this wave's N newest loads to LDS have arrived and its LDS reads are
// done; then every wave's (barrier).
template <int N>
__device__ __forceinline__ void wait_lds_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Workgroup of WM x 2 waves, wave tile 64 x 32 NB: output tile 64 WM x 64 NB.
// S stages of one chunk each.  The fragments of a chunk go to registers one
// chunk ahead of their MFMAs, so a stage is free again one barrier after it
// was read, and the copies run up to S chunks ahead.
template <int WM, int NB, int S>
struct PieceTile {
  static constexpr int TM = 64 * WM, TN = 64 * NB, threads = 128 * WM;
  static constexpr int blocks = 2 * WM + 2 * NB;            // 32-row blocks of A and B per chunk
  static constexpr int stage = blocks * 2048;               // bytes per chunk
  static constexpr int loads = 2 * blocks / (2 * WM);       // 1 KB copies per wave per chunk
  static_assert(2 * blocks % (2 * WM) == 0, "the waves share a chunk evenly");
  static constexpr int lds = S * stage;
};

// acc = the tile's products over chunks [c0, c0 + nk) of the pieces A and B
// (row blocks of nkc chunks), nk >= 1.
template <int WM, int NB, int S>
__device__ __forceinline__ void pieces_tile(char* lds, const char* __restrict__ A, const char* __restrict__ B,
                                            int nkc, int tm, int tn, int c0, int nk, f32x16 (&acc)[2][NB]) {
  using T = PieceTile<WM, NB, S>;
  constexpr int L = T::loads;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * L * 1024;
  const char* src[L];  // the wave's share of a chunk: L runs of 1 KB
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int u = wave * L + i, rb = u >> 1;
    const char* blk = rb < 2 * WM ? A + (size_t)(tm * 2 * WM + rb) * nkc * 2048
                                  : B + (size_t)(tn * 2 * NB + rb - 2 * WM) * nkc * 2048;
    src[i] = blk + (u & 1) * 1024 + (size_t)c0 * 2048;
  }
  uint32_t vo = lane * 16;
  int ws = 0, rs = 0;  // stage of the next copy / read
  auto issue = [&]() {
    loads_to_lds(l0 + ws * T::stage, src, vo);
    vo += 2048;
    ws = ws == S - 1 ? 0 : ws + 1;
  };
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
  f16x8 ah[2][2], al[2][2], bh[2][NB], bl[2][NB];
  auto read = [&](int p) {
    const char* st = lds + rs * T::stage + lane * 16;
    const char* sa = st + wm * 2 * 2048;
    const char* sb = st + (2 * WM + wn * NB) * 2048;
#pragma unroll
    for (int r = 0; r < 2; ++r) al[p][r] = *reinterpret_cast<const f16x8*>(sa + r * 2048 + 1024);
#pragma unroll
    for (int r = 0; r < NB; ++r) bh[p][r] = *reinterpret_cast<const f16x8*>(sb + r * 2048);
#pragma unroll
    for (int r = 0; r < 2; ++r) ah[p][r] = *reinterpret_cast<const f16x8*>(sa + r * 2048);
#pragma unroll
    for (int r = 0; r < NB; ++r) bl[p][r] = *reinterpret_cast<const f16x8*>(sb + r * 2048 + 1024);
    rs = rs == S - 1 ? 0 : rs + 1;
  };
#define FG_P1(X, Y, p)                                                               \
  _Pragma("unroll") for (int a = 0; a < 2; ++a) _Pragma("unroll") for (int b = 0; b < NB; ++b) \
      acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(X[p][a], Y[p][b], acc[a][b], 0, 0, 0);
#define FG_P3(p) FG_P1(al, bh, p) FG_P1(ah, bl, p) FG_P1(ah, bh, p)
  // steady state: one fragment read of chunk c + 1 after each of the first MFMAs
#define FG_P_STEP(p)                                                                 \
  {                                                                                  \
    wait_lds_loads<(S - 2) * L>();                                                   \
    issue();                                                                         \
    read(1 - p);                                                                     \
    FG_P3(p)                                                                         \
    _Pragma("unroll") for (int q = 0; q < 4 + 2 * NB; ++q) {                         \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                             \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                             \
    }                                                                                \
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * NB - 4, 0);                      \
  }
  // the last chunks: nothing left to load, or less than the steady wait counts on
#define FG_P_LAST(p)                                                                 \
  {                                                                                  \
    if (c + 1 < nk) {                                                                \
      wait_lds_loads<0>();                                                           \
      if (c + S < nk) issue();                                                       \
      read(1 - p);                                                                   \
    }                                                                                \
    FG_P3(p)                                                                         \
    ++c;                                                                             \
  }
  for (int i = 0; i < (nk < S ? nk : S); ++i) issue();
  if (nk >= S)
    wait_lds_loads<(S - 1) * L>();
  else
    wait_lds_loads<0>();
  read(0);
  int c = 0;
  for (; c + 1 + S < nk; c += 2) {
    FG_P_STEP(0)
    FG_P_STEP(1)
  }
  while (c < nk) {
    FG_P_LAST(0)
    if (c >= nk) break;
    FG_P_LAST(1)
  }
#undef FG_P_LAST
#undef FG_P_STEP
#undef FG_P3
#undef FG_P1
}

// Tile-rows per group of the grouped-M order: 1024 output rows (4 x 256
// against 8 x 256: 8192 x 4096 over K = 768 146 -> 132 us).
template <int WM>
__device__ __forceinline__ void piece_origin(int pid, int nTm, int nTn, int& tm, int& tn) {
  constexpr int G = 16 / WM;
  const int in_group = G * nTn;
  const int group = pid / in_group;
  const int first = group * G;
  const int gs = min(nTm - first, G);
  tm = first + (pid % in_group) % gs;
  tn = (pid % in_group) / gs;
}

template <int WM, int NB, int S, bool CHECKED>
__global__ void __launch_bounds__(128 * WM, 2)
    gemm_pieces_kernel(float* __restrict__ C, const char* __restrict__ A, const char* __restrict__ B, int M, int N,
                       int nkc, int ksplit, int beta, float* __restrict__ partial, const float* __restrict__ resid,
                       const float* __restrict__ xpa, const float* __restrict__ xpb) {
  using T = PieceTile<WM, NB, S>;
  __shared__ __attribute__((aligned(1024))) char lds[T::lds];
  const int nTm = (M + T::TM - 1) / T::TM, nTn = (N + T::TN - 1) / T::TN;
  int tm, tn;
  piece_origin<WM>(remap_xcd(blockIdx.x, nTm * nTn), nTm, nTn, tm, tn);
  const int c0 = blockIdx.y * ksplit;
  f32x16 acc[2][NB];
  pieces_tile<WM, NB, S>(lds, A, B, nkc, tm, tn, c0, min(nkc - c0, ksplit), acc);
  const int wave = threadIdx.x >> 6;
  store_acc<2, NB, CHECKED>(partial ? partial + (size_t)blockIdx.y * M * N : C, partial ? nullptr : resid, acc, M, N,
                            tm * T::TM + (wave >> 1) * 64, tn * T::TN + (wave & 1) * 32 * NB, partial ? 0 : beta,
                            -(xp_exponent(xpa) + xp_exponent(xpb)));
}

// The fused gate/up projection on pieces: B's rows split in swiglu_row order,
// so accumulator blocks 2p and 2p + 1 of a lane hold G and U of one hidden
// unit (M % TM == 0, H % 128 == 0).
template <int WM, int S>
__global__ void __launch_bounds__(128 * WM, 2)
    gemm_pieces_swiglu_kernel(float* __restrict__ O, float* __restrict__ GU, const char* __restrict__ A,
                              const char* __restrict__ B, int M, int H, int nkc, const float* __restrict__ xpa,
                              const float* __restrict__ xpb) {
  using T = PieceTile<WM, 4, S>;
  __shared__ __attribute__((aligned(1024))) char lds[T::lds];
  const int nTm = M / T::TM, nTn = 2 * H / T::TN;
  int tm, tn;
  piece_origin<WM>(remap_xcd(blockIdx.x, nTm * nTn), nTm, nTn, tm, tn);
  f32x16 acc[2][4];
  pieces_tile<WM, 4, S>(lds, A, B, nkc, tm, tn, 0, nkc, acc);
  const int esc = -(xp_exponent(xpa) + xp_exponent(xpb));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      const int j = tn * 128 + wn * 64 + pr * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int i = tm * T::TM + wm * 64 + a * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const float g = __builtin_amdgcn_ldexpf(acc[a][2 * pr][v], esc);
        const float u = __builtin_amdgcn_ldexpf(acc[a][2 * pr + 1][v], esc);
        GU[(size_t)i * 2 * H + j] = g;
        GU[(size_t)i * 2 * H + H + j] = u;
        O[(size_t)i * H + j] = fg::swiglu_fwd1(g, u);
      }
    }
}

// Several weight gradients in one launch (see GTable): job pieces per table
// entry, one K split for all jobs (gridDim.y), its partial sums job after job
// in `slab` ([job][split][M x N], each job's from a 16-byte boundary on).  Unlike
// gemm_pieces_kernel it spills (140 registers, 468 - 484 B a lane: the zero
// accumulators of an empty piece and the job's fields meet in the epilogue); the
// main loop is clean, the epilogue stores at 2.1 TB/s, and 4096-wide layers reach
// 403 TFLOP/s where the plain kernel reaches 449 - 470.
struct PJob {
  float* C;
  const char* A;
  const char* B;
  const float* xpa;
  const float* xpb;
  int64_t slab0;
  int M, N, nkc, beta, tile0;
};
constexpr int kPieceJobs = 48;
struct PTable {
  int count, tiles, splits;
  float* slab;
  PJob job[kPieceJobs];
};
static_assert(sizeof(PTable) <= 4096, "the job table travels as a kernel argument (4 KB at most)");

template <int WM, int NB, int S>
__global__ void __launch_bounds__(128 * WM, 2) gemm_pieces_grouped(PTable t) {
  using T = PieceTile<WM, NB, S>;
  __shared__ __attribute__((aligned(1024))) char lds[T::lds];
  const int g = remap_xcd(blockIdx.x, t.tiles);
  int j = 0;
  while (j + 1 < t.count && g >= t.job[j + 1].tile0) ++j;
  const PJob& jb = t.job[j];
  int tm, tn;
  piece_origin<WM>(g - jb.tile0, (jb.M + T::TM - 1) / T::TM, (jb.N + T::TN - 1) / T::TN, tm, tn);
  const int per = (jb.nkc + t.splits - 1) / t.splits, c0 = blockIdx.y * per, nk = min(jb.nkc - c0, per);
  const int wave = threadIdx.x >> 6;
  const int i0 = tm * T::TM + (wave >> 1) * 64, j0 = tn * T::TN + (wave & 1) * 32 * NB;
  f32x16 acc[2][NB];
  if (nk > 0) {
    pieces_tile<WM, NB, S>(lds, jb.A, jb.B, jb.nkc, tm, tn, c0, nk, acc);
  } else {  // a short job under the common split
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
  }
  const int esc = -(xp_exponent(jb.xpa) + xp_exponent(jb.xpb));
  float* out = t.splits > 1 ? t.slab + jb.slab0 + (int64_t)blockIdx.y * jb.M * jb.N : jb.C;
  store_acc<2, NB, true>(out, nullptr, acc, jb.M, jb.N, i0, j0, t.splits > 1 ? 0 : jb.beta, esc);
}
