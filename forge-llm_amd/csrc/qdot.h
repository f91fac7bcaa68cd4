// Row dot products of half and quantized weight matrices for the matvecs (the
// QuantLinear forward and the decode step): y = W x with W rows of GGML blocks
// (qformat.h) and x in LDS.
//
// A row is a list of units, one per lane and step: 32 elements of a K-quant
// block (Q4_K, Q5_K, Q6_K: a run of 16 low and 16 high nibbles, so two
// sub-blocks with a scale each), 16 of a Q8_0 block, 8 halves.  A unit's
// quants are one 16-byte load per plane, at whatever alignment the block size
// leaves.  A wave takes R rows at a time: their loads of a step are issued
// together and a step ahead of their use, the unit's x values and their sums
// are formed once for all of them.
//
// x sits in LDS in the order the lanes read it: granules of four values,
// [64 units][granule of the unit][unit], so that every read is one
// conflict-free ds_read_b128 (in element order a K-quant unit's lanes are 64 B
// apart, a four-way conflict, which bounded one row per wave at 2.6 TB/s).
//
// Arithmetic as the element-order dots of qformat.h: integer-times-x products
// in fp32 over the same runs (16 for Q4_K and Q5_K, 4 for Q6_K and Q8_0, 8 for
// F16), everything across runs, block scales and rows in fp64.  A block scale
// times a 6- or 8-bit sub-block scale is exact in fp32 (11 + 8 bits), so one
// conversion takes it to fp64.
#pragma once

#include "qformat.h"

namespace fgq {

// Elements per unit; 0: the type has no unit form (qrows_dot serves it).
__host__ __device__ constexpr int unit_elems(int t) {
  return t == kQ4_K || t == kQ5_K || t == kQ6_K ? 32 : t == kQ8_0 ? 16 : t == kF16 ? 8 : 0;
}
__host__ __device__ constexpr bool has_units(int t) { return unit_elems(t) > 0; }
// Place of x[i] (i a multiple of 4: a granule) in the LDS copy of x for rows
// of U units.
template <int QT>
__device__ __forceinline__ int x_place(int i, int U) {
  constexpr int G = unit_elems(QT) / 4;
  int u, v;
  if constexpr (QT == kQ4_K || QT == kQ5_K) {
    u = (i >> 8) * 8 + ((i >> 6) & 3) * 2 + ((i >> 4) & 1);
    v = ((i >> 5) & 1) * 4 + ((i >> 2) & 3);
  } else if constexpr (QT == kQ6_K) {
    u = (i >> 8) * 8 + ((i >> 7) & 1) * 4 + ((i >> 5) & 1) * 2 + ((i >> 4) & 1);
    v = ((i >> 6) & 1) * 4 + ((i >> 2) & 3);
  } else if constexpr (QT == kQ8_0) {
    u = i >> 4;
    v = (i >> 2) & 3;
  } else {
    u = i >> 3;
    v = (i >> 2) & 1;
  }
  const int u0 = u & ~63, n = U - u0 < 64 ? U - u0 : 64;
  return 4 * (u0 * G + v * n + (u - u0));
}

// Loads at any alignment (blocks of 34 and 210 bytes are 2-byte aligned): one
// instruction.  Reading the words around the block and shifting them into
// place measured slower (Q6_K, 128256 x 4096: 122 against 160 us).
template <typename T>
__device__ __forceinline__ T ld_any(const uint8_t* p) {
  T v;
  __builtin_memcpy(&v, p, sizeof(T));
  return v;
}

// A unit's bytes in registers.
template <int QT>
struct Unit;
template <>
struct Unit<kQ4_K> {
  uint4 hd, q;
};
template <>
struct Unit<kQ5_K> {
  uint4 hd, q, qh;
};
template <>
struct Unit<kQ6_K> {
  uint4 q, qh;
  uint2 sc;
  uint32_t d;
};
template <>
struct Unit<kQ8_0> {
  uint4 q;
  uint32_t d;
};
template <>
struct Unit<kF16> {
  uint4 q;
};

template <int QT>
__device__ __forceinline__ void unit_load(Unit<QT>& f, const uint8_t* row, int u) {
  if constexpr (QT == kQ4_K || QT == kQ5_K) {
    constexpr int BB = block_bytes(QT);
    const uint8_t* B = row + BB * (u >> 3);
    f.hd = *reinterpret_cast<const uint4*>(B);
    f.q = *reinterpret_cast<const uint4*>(B + (BB - 128) + 16 * (u & 7));
    if constexpr (QT == kQ5_K) f.qh = *reinterpret_cast<const uint4*>(B + 16 + 16 * (u & 1));
  } else if constexpr (QT == kQ6_K) {
    const uint8_t* B = row + 210 * (u >> 3);
    const int s = u & 7;
    f.q = ld_any<uint4>(B + 16 * s);  // [half][low / high 32][16]: s = 4 h + 2 a + l / 16
    f.qh = ld_any<uint4>(B + 128 + 32 * (s >> 2) + 16 * (s & 1));
    f.sc = ld_any<uint2>(B + 192 + 8 * (s >> 2));
    f.d = ld16(B + 208);
  } else if constexpr (QT == kQ8_0) {
    const uint8_t* B = row + 34 * (u >> 1);
    f.q = ld_any<uint4>(B + 2 + 16 * (u & 1));
    f.d = ld16(B);
  } else {
    f.q = *reinterpret_cast<const uint4*>(row + 16 * u);
  }
}

// The unit's x values and what its rows share of them.
template <int QT>
struct UnitX {
  float x[unit_elems(QT)];
  double s0, s1;  // sums over the two runs (K-quants), over all (Q8_0)
};
template <int QT>
__device__ __forceinline__ void unit_x(UnitX<QT>& X, const float* xs, int u, int U) {
  constexpr int E = unit_elems(QT), G = E / 4;
  const int u0 = u & ~63, n = U - u0 < 64 ? U - u0 : 64;
  const float4* p = reinterpret_cast<const float4*>(xs) + u0 * G + (u - u0);
#pragma unroll
  for (int v = 0; v < G; ++v) {
    const float4 a = p[v * n];
    X.x[4 * v] = a.x;
    X.x[4 * v + 1] = a.y;
    X.x[4 * v + 2] = a.z;
    X.x[4 * v + 3] = a.w;
  }
  if constexpr (QT == kQ4_K || QT == kQ5_K) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      a += X.x[i];
      b += X.x[16 + i];
    }
    X.s0 = a;
    X.s1 = b;
  } else if constexpr (QT == kQ6_K || QT == kQ8_0) {
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int v = 0; v < G; ++v)
      s[v >> 2] += (double)((X.x[4 * v] + X.x[4 * v + 1]) + (X.x[4 * v + 2] + X.x[4 * v + 3]));
    X.s0 = s[0];
    X.s1 = s[1];
  }
}

// The four bytes of w as they are: without this the compiler sees through the
// masks that made them and extracts each nibble before converting it, an
// instruction more per element (v_cvt_f32_ubyte1..3 take bytes in place).
__device__ __forceinline__ uint32_t as_bytes(uint32_t w) {
  asm("" : "+v"(w));
  return w;
}

// Four bytes of w times x, one fp32 run.
__device__ __forceinline__ float dot4(uint32_t w, const float* x) {
  float f[4];
  w = as_bytes(w);
  bytes_f32(w, f);
  float t = f[0] * x[0];
  t = fmaf(f[1], x[1], t);
  t = fmaf(f[2], x[2], t);
  return fmaf(f[3], x[3], t);
}

template <int QT>
__device__ __forceinline__ void unit_dot(double& acc, const Unit<QT>& f, const UnitX<QT>& X, int u) {
  if constexpr (QT == kQ4_K || QT == kQ5_K) {
    const int c = (u & 7) >> 1, sh = (c & 1) * 16;
    // sub-blocks 2c and 2c + 1: two 6-bit scales and mins at once (getScaleMinK4)
    const uint32_t A = f.hd.y >> sh, B = f.hd.z >> sh, C = f.hd.w >> sh;
    const uint32_t sc = c < 2 ? A & 0x3F3Fu : (C & 0x0F0Fu) | ((A >> 2) & 0x3030u);
    const uint32_t mn = c < 2 ? B & 0x3F3Fu : ((C >> 4) & 0x0F0Fu) | ((B >> 2) & 0x3030u);
    const float d = h2f(f.hd.x & 0xffffu), dm = h2f(f.hd.x >> 16);
    const uint32_t qw[4] = {f.q.x, f.q.y, f.q.z, f.q.w};
    float al = 0.f, ah = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      uint32_t lo = qw[v] & 0x0F0F0F0Fu, hi = (qw[v] >> 4) & 0x0F0F0F0Fu;
      if constexpr (QT == kQ5_K) {  // the fifth bit: bit 2c (low) / 2c + 1 (high)
        const uint32_t h = v == 0 ? f.qh.x : v == 1 ? f.qh.y : v == 2 ? f.qh.z : f.qh.w;
        const uint32_t hs = h >> (2 * c);
        lo |= (hs & 0x01010101u) << 4;
        hi |= ((hs >> 1) & 0x01010101u) << 4;
      }
      float fl[4], fh[4];
      bytes_f32(as_bytes(lo), fl);
      bytes_f32(as_bytes(hi), fh);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        al = fmaf(fl[i], X.x[4 * v + i], al);
        ah = fmaf(fh[i], X.x[16 + 4 * v + i], ah);
      }
    }
    acc = fma((double)(d * (float)(sc & 0xffu)), (double)al, acc);
    acc = fma(-(double)(dm * (float)(mn & 0xffu)), X.s0, acc);
    acc = fma((double)(d * (float)(sc >> 8)), (double)ah, acc);
    acc = fma(-(double)(dm * (float)(mn >> 8)), X.s1, acc);
  } else if constexpr (QT == kQ6_K) {
    const int s = u & 7, a2 = s & 2, by = 8 * ((s & 1) + a2);  // group a = a2 / 2 and a + 2, scale byte l / 16 + 2 a
    const uint32_t qw[4] = {f.q.x, f.q.y, f.q.z, f.q.w};
    const uint32_t hw[4] = {f.qh.x, f.qh.y, f.qh.z, f.qh.w};
    double al = -32.0 * X.s0, ah = -32.0 * X.s1;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint32_t h = hw[v] >> a2;
      al += (double)dot4((qw[v] & 0x0F0F0F0Fu) | ((h & 0x03030303u) << 4), X.x + 4 * v);
      ah += (double)dot4(((qw[v] >> 4) & 0x0F0F0F0Fu) | (h & 0x30303030u), X.x + 16 + 4 * v);
    }
    const float d = h2f(f.d);
    acc = fma((double)(d * (float)(int8_t)(f.sc.x >> by)), al, acc);
    acc = fma((double)(d * (float)(int8_t)(f.sc.y >> by)), ah, acc);
  } else if constexpr (QT == kQ8_0) {
    // int8 q = (q ^ 0x80) - 128: unsigned bytes convert at full rate
    const uint32_t qw[4] = {f.q.x, f.q.y, f.q.z, f.q.w};
    double a = -128.0 * (X.s0 + X.s1);
#pragma unroll
    for (int v = 0; v < 4; ++v) a += (double)dot4(qw[v] ^ 0x80808080u, X.x + 4 * v);
    acc = fma((double)h2f(f.d), a, acc);
  } else {
    const uint32_t hw[4] = {f.q.x, f.q.y, f.q.z, f.q.w};
    float a = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) a = fmaf(h2f((hw[i >> 1] >> (16 * (i & 1))) & 0xffffu), X.x[i], a);
    acc += (double)a;
  }
}

// R rows of one wave over its part of the units: steps part, part + P, ... of
// 64 units.  `start` issues the loads of the first step (before x is there),
// `finish` sums: acc[r] is this lane's share of row r.
template <int QT, int R>
struct UnitRows {
  const uint8_t* row[R];
  Unit<QT> f[R];
  __device__ __forceinline__ void start(int U, int part) {
    const int u = part * 64 + (threadIdx.x & 63);
    if (u < U) {
#pragma unroll
      for (int r = 0; r < R; ++r) unit_load<QT>(f[r], row[r], u);
    }
  }
  __device__ __forceinline__ void finish(double (&acc)[R], const float* xs, int U, int part, int P) {
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0;
    for (int u = part * 64 + (threadIdx.x & 63); u < U;) {
      const int un = u + 64 * P;
      Unit<QT> n[R];
      if (un < U) {
#pragma unroll
        for (int r = 0; r < R; ++r) unit_load<QT>(n[r], row[r], un);
      }
      UnitX<QT> X;
      unit_x<QT>(X, xs, u, U);
#pragma unroll
      for (int r = 0; r < R; ++r) unit_dot<QT>(acc[r], f[r], X, u);
#pragma unroll
      for (int r = 0; r < R; ++r) f[r] = n[r];
      u = un;
    }
  }
};

// Workgroups of kUnitWaves waves: P waves share the units of a row group (P a
// power of two, at most one step each), kUnitWaves / P groups at a time.
constexpr int kUnitWaves = 4, kUnitThreads = 64 * kUnitWaves;
inline int unit_parts(int U) {
  int P = 1;
  while (P < kUnitWaves && 64 * P < U) P <<= 1;
  return P;
}
// The share of its lanes that P waves use over the steps of a row of U units.
inline double unit_fill(int U) {
  const int step = 64 * unit_parts(U);
  return (double)U / ((U + step - 1) / step * step);
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov_d(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
// Sum over each row of 16 lanes (rotations within the row), in every lane.
__device__ __forceinline__ double row16_sum(double v) {
  v += dpp_mov_d<0x128>(v);  // row_ror:8
  v += dpp_mov_d<0x124>(v);
  v += dpp_mov_d<0x122>(v);
  v += dpp_mov_d<0x121>(v);
  return v;
}
__device__ __forceinline__ double lane_d(double v, int l) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
// acc[r] = its sum over the wave, in every lane.  Four rows: two exchanges
// leave each quarter of the wave one row to sum over its 16 lanes.
template <int R>
__device__ __forceinline__ void wave_rows_sum(double (&acc)[R]) {
  if constexpr (R == 4) {
    const int lane = threadIdx.x & 63;
    const bool up = lane & 32, odd = lane & 16;
    const double s0 = __shfl_xor(up ? acc[0] : acc[2], 32, 64), s1 = __shfl_xor(up ? acc[1] : acc[3], 32, 64);
    const double a = (up ? acc[2] : acc[0]) + s0, b = (up ? acc[3] : acc[1]) + s1;
    double c = (odd ? b : a) + __shfl_xor(odd ? a : b, 16, 64);
    c = row16_sum(c);
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = lane_d(c, 16 * r);
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double c = row16_sum(acc[r]);
      acc[r] = (lane_d(c, 0) + lane_d(c, 16)) + (lane_d(c, 32) + lane_d(c, 48));
    }
  }
}

// Sums acc over the wave and the P waves of the group; the result is valid in
// lane 0 of part 0.  Every wave of the workgroup calls it (barriers for P > 1).
template <int R>
__device__ __forceinline__ void unit_reduce(double (&acc)[R], double (*red)[R], int P) {
  const int wave = threadIdx.x >> 6;
  wave_rows_sum<R>(acc);
  if (P == 1) return;
  __syncthreads();  // the previous group's sums have been read
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) red[wave][r] = acc[r];
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0 && (wave & (P - 1)) == 0) {
    for (int p = 1; p < P; ++p) {
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] += red[wave + p][r];
    }
  }
}

}  // namespace fgq
