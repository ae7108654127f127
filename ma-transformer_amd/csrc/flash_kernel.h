// flash_kernel.h -- banded attention, forward and backward, for head_dims 8 to
// 128 (a multiple of 8) on 16x16x32 MFMA: windows [i-left, i+right] of any
// dilation, dense and causal rows (bands as wide as the sequence).
//
// float32 is computed on the bf16 matrix cores.  x = x0 + x1 + x2 with x0, x1,
// x2 the successive bf16 roundings of what is left (24 bits in all, float32's
// exponent range), and a product takes the six partial products whose bf16
// planes p, p' have p + p' <= 2, smallest first; the three left out come to
// 2^-24 of it at most (x1 reaches 2^-8 of x, x2 2^-17), 2^-27.5 rms over uniform
// mantissas.  Six 16x16x32 MFMAs take 6/16 of the time of the sixteen 16x16x4 fp32
// MFMAs they replace, and 64-term dot products came out closer to 64-bit ones
// (relative error 4.6e-8 against 1.44e-7 on normal data; 7.7e-8 against 1.24e-7 on
// data spread over e^(+-9)): each MFMA rounds once per 32 terms instead of once per
// term.
//
// 16-bit inputs multiply exactly (one plane).  Probabilities and dS are float32
// and enter their products in planes too, so that nothing but the stored
// results is rounded to 16 bits: bf16 as the three planes above (all 24 bits),
// f16 as a value and its remainder (22 bits) times a power of two that puts the
// largest just below f16's maximum, as f16 has no bits below 2^-24 (FlScale).
// A sum then keeps the bits of weights down to 2^-26 of its largest, below a
// float32 sum's own rounding.  head_dim 64 is the exception: P and dS are one
// 16-bit plane there, as on the kernels that share its calls.
//
// Operand layouts (lane = 16 g + c).  Row operand: lane (c, g) holds row c at
// head_dim 32 j + 8 g .. +7 for each j (one 16-byte LDS read, or registers).
// rows . rows^T of 16 x 16 lands with lane (c, g) holding column c of rows
// 4 g .. 4 g + 3, which is the B operand of the products with the other
// matrix's transpose; that transpose is read from the LDS rows by the
// transpose read (tr_read), two 16-row sub-tiles per MFMA.  A lane ends with
// head_dim 32 h + 8 g .. +7 of its column for each h.
//
// LDS rows are 64 ND + 32 bytes (ND = ceil(head_dim / 32)): the 32-byte pad
// keeps a transpose read's four rows on disjoint banks.  Columns from head_dim
// to 32 ND read as zero and are not stored.
#pragma once

#include "device_common.h"

namespace ma_dev {

struct FlArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* dout;
  void* o;          // forward: O; backward: dQ
  void* dk;
  void* dv;
  const void* fo;   // backward from saved statistics: the forward's O
  float* lse;       // forward: optional statistics out; backward from saved statistics: in ([B*N*H])
  float* stats;     // backward: {lse2, delta} per row, [B*N*H][2]
  int64_t N;
  int32_t H, D, left, right, dil;
  int32_t tiles;      // tiles of the longest residue class
  int32_t desc;       // 1: the last tile first (causal rows: longest first)
  int32_t globals;    // forward, GL kernels: keys 0..globals-1 (at most 16) join every row's window
  uint32_t tok_bytes; // bytes between consecutive rows of a residue class
  float scale, scale_log2;
};

// Element type of the MFMA operands and the number of planes of an input.
template <typename T>
struct FlElt {
  using E = T;
  static constexpr int NP = 1;
  // planes of a probability or dS operand
  static constexpr int NPB = __is_same(T, __bf16) ? 3 : 2;
};
template <>
struct FlElt<float> {
  using E = __bf16;
  static constexpr int NP = 3;
  static constexpr int NPB = 3;
};

// Powers of two on f16's two-plane operands; other operands take none.
template <typename T, int NPB>
struct FlScale {
  static constexpr bool kOn = __is_same(T, _Float16) && NPB == 2;
  static constexpr float kFwd = kOn ? 7.0f : 0.0f;   // forward weights: up to 2^kSlack, so up to 2^15
  static constexpr float kProb = kOn ? 15.0f : 0.0f; // normalised probabilities: up to 1
  // exponents' offsets of a weight (mu: the row's maximum) and of a probability
  static __device__ __forceinline__ float fwd(float mu) { return kOn ? kFwd - mu : -mu; }
  static __device__ __forceinline__ float prob(float lse2) { return kOn ? kProb - lse2 : -lse2; }
  // the exponent that takes values up to x to [2^(top - 1), 2^top)
  static __device__ __forceinline__ int exponent(float x, int top) {
    return min(top - __builtin_amdgcn_frexp_expf(x), 100);
  }
};

template <typename E>
__device__ __forceinline__ float fl_lo(uint32_t w) {
  if constexpr (__is_same(E, __bf16))
    return __uint_as_float(w << 16);
  else
    return static_cast<float>(__builtin_bit_cast(E, (uint16_t)(w & 0xffffu)));
}
template <typename E>
__device__ __forceinline__ float fl_hi(uint32_t w) {
  if constexpr (__is_same(E, __bf16))
    return __uint_as_float(w & 0xffff0000u);
  else
    return static_cast<float>(__builtin_bit_cast(E, (uint16_t)(w >> 16)));
}

// Planes of two values: w[p] holds plane p of both.
template <typename E, int NPL>
__device__ __forceinline__ void fl_split2(float x, float y, uint32_t (&w)[NPL]) {
#pragma unroll
  for (int p = 0; p < NPL; ++p) {
    w[p] = Mma<E>::pack2(x, y);
    if (p + 1 < NPL) {
      x -= fl_lo<E>(w[p]);
      y -= fl_hi<E>(w[p]);
    }
  }
}

// The three bf16 planes of 8 floats.  A value that rounds to a bf16 infinity
// (above 3.39e38, or an infinity itself) is clamped to bf16's largest in its
// first planes, so that its planes still add up to it.
__device__ __forceinline__ void fl_split8(const uint4& a, const uint4& b, uint4 (&o)[3]) {
  float x[8] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w)};
  constexpr float kBig = 3.3895313892515355e38f;  // bf16's largest finite value
  const float mx = fmaxf(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))),
                         fmaxf(fmaxf(fabsf(x[4]), fabsf(x[5])), fmaxf(fabsf(x[6]), fabsf(x[7]))));
  uint32_t w[3][4];
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(mx > kBig) == 0, 1)) {  // NaNs pass: fmaxf skips them
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t t[3];
      fl_split2<__bf16, 3>(x[2 * i], x[2 * i + 1], t);
      w[0][i] = t[0];
      w[1][i] = t[1];
      w[2][i] = t[2];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y = x[2 * i], z = x[2 * i + 1];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const float cy = p < 2 && fabsf(y) > kBig ? copysignf(kBig, y) : y;
        const float cz = p < 2 && fabsf(z) > kBig ? copysignf(kBig, z) : z;
        w[p][i] = Mma<__bf16>::pack2(cy, cz);
        y -= fl_lo<__bf16>(w[p][i]);
        z -= fl_hi<__bf16>(w[p][i]);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) o[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

// ---------------------------------------------------------------- operands

template <int ND>
constexpr int fl_rs() {
  return 64 * ND + 32;  // bytes per LDS row of one plane
}

// A register row operand: row c at head_dim 32 j + 8 g .. +7, per plane.
template <typename T, int ND>
struct FlFrag {
  static constexpr int NP = FlElt<T>::NP;
  uint4 r[NP][ND];
  // `row`: byte offset of the row (kOob or past the range: zeros)
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t row, int D, int g) {
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const int d = 32 * j + 8 * g;
      const uint32_t off = d < D ? row + (uint32_t)(d * sizeof(T)) : kOob;
      if constexpr (NP == 1) {
        r[0][j] = bload16(rs, off);
      } else {
        const uint4 a = bload16(rs, off), b = bload16(rs, off + 16);
        uint4 s[3];
        fl_split8(a, b, s);
#pragma unroll
        for (int p = 0; p < 3; ++p) r[p][j] = s[p];
      }
    }
  }
};

// R rows of one matrix on their way to LDS: 8-element units, a thread's unit i
// is number tid + threads * i in row order.
template <typename T, int ND, int R, int NW>
struct FlStage {
  static constexpr int kUnits = R * 4 * ND, kThr = 64 * NW;
  static constexpr int NU = (kUnits + kThr - 1) / kThr;
  static constexpr bool kEven = kUnits % kThr == 0;
  static constexpr int NP = FlElt<T>::NP;
  static constexpr int RS = fl_rs<ND>();
  static constexpr int kPlane = R * RS, kMat = NP * kPlane;
  uint4 r[NU][sizeof(T) == 4 ? 2 : 1];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int row0, int tid, uint32_t tb, int D) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + kThr * i, row = u / (4 * ND), col = u % (4 * ND);
      const bool ok = (kEven || u < kUnits) && 8 * col < D;
      const uint32_t off = ok ? (uint32_t)(row0 + row) * tb + (uint32_t)(8 * col * sizeof(T)) : kOob;
      r[i][0] = bload16(rs, off);
      if constexpr (sizeof(T) == 4) r[i][1] = bload16(rs, off + 16);
    }
  }
  __device__ __forceinline__ void store(uint8_t* m, int tid) const {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + kThr * i, row = u / (4 * ND), col = u % (4 * ND);
      if (!kEven && u >= kUnits) continue;
      uint8_t* p = m + row * RS + 16 * col;
      if constexpr (sizeof(T) == 2) {
        *reinterpret_cast<uint4*>(p) = r[i][0];
      } else {
        uint4 s[3];
        fl_split8(r[i][0], r[i][1], s);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint4*>(p + q * kPlane) = s[q];
      }
    }
  }
};

// z[n] = 16 LDS rows (at p, the lane's address in plane 0) . frags[n]^T.
template <typename T, int ND, int PL, int NF>
__device__ __forceinline__ void fl_rowdot(const uint8_t* p, const FlFrag<T, ND> (&f)[NF], f32x4 (&z)[NF]) {
  using E = typename FlElt<T>::E;
#pragma unroll
  for (int n = 0; n < NF; ++n) z[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (FlElt<T>::NP == 1) {
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const uint4 a = *reinterpret_cast<const uint4*>(p + 64 * j);
#pragma unroll
      for (int n = 0; n < NF; ++n) z[n] = Mma<E>::x32(a, f[n].r[0][j], z[n]);
    }
  } else {
    // LDS planes 2, 1, 0 against register planes with p + p' <= 2, smallest first
#pragma unroll
    for (int s = 2; s >= 0; --s)
#pragma unroll
      for (int pa = s; pa >= 0; --pa)
#pragma unroll
        for (int j = 0; j < ND; ++j) {
          const uint4 a = *reinterpret_cast<const uint4*>(p + pa * PL + 64 * j);
#pragma unroll
          for (int n = 0; n < NF; ++n) z[n] = Mma<E>::x32(a, f[n].r[s - pa][j], z[n]);
        }
  }
}

// B operand planes of two sub-tiles' values (4 per lane each).
template <typename T, int NPB = FlElt<T>::NPB>
struct FlB {
  uint4 b[NPB];
  __device__ __forceinline__ void set(const float (&p0)[4], const float (&p1)[4]) {
    using E = typename FlElt<T>::E;
    uint32_t w[4][NPB];
    fl_split2<E, NPB>(p0[0], p0[1], w[0]);
    fl_split2<E, NPB>(p0[2], p0[3], w[1]);
    fl_split2<E, NPB>(p1[0], p1[1], w[2]);
    fl_split2<E, NPB>(p1[2], p1[3], w[3]);
#pragma unroll
    for (int p = 0; p < NPB; ++p) b[p] = make_uint4(w[0][p], w[1][p], w[2][p], w[3][p]);
  }
};

// acc[n] += M^T B[n]^T over two 16-row sub-tiles of M: m0, m1 the lane's
// transpose-read addresses (fl_tr_lane) in their plane 0.
template <int ND>
__device__ __forceinline__ uint32_t fl_tr_lane(int c, int g) {
  return (uint32_t)((4 * g + (c >> 2)) * fl_rs<ND>() + 16 * (c & 3));
}
// LOCAL (float32): the six products of a pair of sub-tiles are summed from zero
// and added to acc once, so that acc is rounded once per 32 rows instead of six
// times.  The forward up to head_dim 64 takes it: relative error at head_dim 64 of
// [i-300, i+300] 3.9e-7 -> 1.7e-7 and of windows over all of 4096 earlier rows
// 3.9e-7 -> 1.6e-7 (fp32 FMA kernels before: 2.7e-7 both), for 0 to 4 % of the time.
// Where the kernels before were further off already it is left out: above head_dim
// 64 (4.0e-7 against 5.9e-7) and for the long dense rows of two query groups (8 heads
// of 16384 rows 1243 us, with it 1302).
template <typename T, int ND, int PL, int NF, int NPB = FlElt<T>::NPB, bool LOCAL = false>
__device__ __forceinline__ void fl_trmul(const uint8_t* m0, const uint8_t* m1, const FlB<T, NPB> (&b)[NF],
                                         f32x4 (&acc)[NF][2 * ND]) {
  using E = typename FlElt<T>::E;
#pragma unroll
  for (int dt = 0; dt < 2 * ND; ++dt) {
    const int o = 64 * (dt >> 1) + 8 * (dt & 1);
    if constexpr (FlElt<T>::NP == 1) {
      const uint2 a0 = tr_read(m0 + o), a1 = tr_read(m1 + o);
      const uint4 a = make_uint4(a0.x, a0.y, a1.x, a1.y);
#pragma unroll
      for (int n = 0; n < NF; ++n) {
#pragma unroll
        for (int p = NPB - 1; p >= 0; --p) acc[n][dt] = Mma<E>::x32(a, b[n].b[p], acc[n][dt]);  // remainders first
      }
    } else {
      uint4 a[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const uint2 a0 = tr_read(m0 + p * PL + o), a1 = tr_read(m1 + p * PL + o);
        a[p] = make_uint4(a0.x, a0.y, a1.x, a1.y);
      }
      f32x4 t[NF];
#pragma unroll
      for (int n = 0; n < NF; ++n) t[n] = LOCAL ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[n][dt];
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int pa = s; pa >= 0; --pa)
#pragma unroll
          for (int n = 0; n < NF; ++n) t[n] = Mma<E>::x32(a[pa], b[n].b[s - pa], t[n]);
#pragma unroll
      for (int n = 0; n < NF; ++n) acc[n][dt] = LOCAL ? acc[n][dt] + t[n] : t[n];
    }
  }
}

// A finished row: acc * s at head_dim 32 h + 8 g .. +7.
template <typename T, int ND>
__device__ __forceinline__ void fl_store(const f32x4 (&acc)[2 * ND], float s, __amdgpu_buffer_rsrc_t rs,
                                         uint32_t row, int D, int g) {
#pragma unroll
  for (int h = 0; h < ND; ++h) {
    const int d = 32 * h + 8 * g;
    const uint32_t off = d < D ? row + (uint32_t)(d * sizeof(T)) : kOob;
    const f32x4 x = acc[2 * h] * s, y = acc[2 * h + 1] * s;
    if constexpr (sizeof(T) == 4) {
      bstore16(rs, off, __builtin_bit_cast(uint4, x));
      bstore16(rs, off + 16, __builtin_bit_cast(uint4, y));
    } else {
      bstore16(rs, off, make_uint4(Mma<T>::pack2(x[0], x[1]), Mma<T>::pack2(x[2], x[3]), Mma<T>::pack2(y[0], y[1]),
                                   Mma<T>::pack2(y[2], y[3])));
    }
  }
}

// Whether any of the lane's sums is an infinity or NaN (0 * x is NaN then).
template <int ND>
__device__ __forceinline__ bool fl_bad(const f32x4 (&acc)[2 * ND]) {
  float t = 0.0f;
#pragma unroll
  for (int i = 0; i < 2 * ND; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) t = fmaf(acc[i][r], 0.0f, t);
  return t != 0.0f;  // true for NaN
}

// The (batch, head, residue class) stream and tile of a workgroup.
struct FlPos {
  int tile, rho, h, b, Nr;
  int64_t base;  // elements of the stream's first row
  uint32_t nrec;
};
__device__ __forceinline__ FlPos fl_pos(const FlArgs& a, int elt) {
  FlPos p;
  int lin = xcd_row_order(blockIdx.x, gridDim.x);
  p.tile = lin % a.tiles;
  if (a.desc) p.tile = a.tiles - 1 - p.tile;
  lin /= a.tiles;
  p.rho = lin % a.dil;
  lin /= a.dil;
  p.h = lin % a.H;
  p.b = lin / a.H;
  p.Nr = (int)((a.N - p.rho + a.dil - 1) / a.dil);
  p.base = (((int64_t)p.b * a.N + p.rho) * a.H + p.h) * a.D;
  p.nrec = p.Nr > 0 ? (uint32_t)(p.Nr - 1) * a.tok_bytes + (uint32_t)(a.D * elt) : 0u;
  return p;
}

// Rows of a workgroup of NW waves with W rows each: wave w has first .. first +
// W - 1 (first = Nr: none), the workgroup lo .. hi.  PAIR: the first half of
// the waves on tile p, the second half on tile T - 1 - p.
struct FlRows {
  int first, lo, hi;
};
template <int W, int NW, bool PAIR>
__device__ __forceinline__ bool fl_rows(const FlPos& ps, int wv, FlRows& r) {
  if constexpr (PAIR) {
    constexpr int HT = W * NW / 2;
    const int last = (ps.Nr + HT - 1) / HT - 1 - ps.tile;
    if (ps.tile > last) return false;
    const bool second = wv >= NW / 2;
    r.first = (second ? last : ps.tile) * HT + W * (wv % (NW / 2));
    if (second && last == ps.tile) r.first = ps.Nr;  // the middle tile of an odd count: one half is enough
    r.lo = ps.tile * HT;
    r.hi = last * HT + HT - 1;
    return true;
  } else {
    r.lo = ps.tile * (W * NW);
    r.hi = r.lo + W * NW - 1;
    r.first = r.lo + W * wv;
    return r.lo < ps.Nr;
  }
}

// ---------------------------------------------------------------- rows redone
//
// The weight of a masked pair is 0, but 0 times an infinity or NaN in its row
// of V (K, Q, dO) is NaN and reaches sums that do not hold that pair; likewise
// an infinity times an operand's negative remainder plane.  A group of 16 rows
// with such sums is computed again in float32 over each row's own set: lane
// (c, g) holds row c at head_dim 32 h + 8 g .. +7 for each h, as the sums do,
// and walks the group's keys (queries).  Rows that are NaN throughout in either
// computation keep their sums: those whose statistics are NaN, and keys of such
// queries (fl_dkv_nan).
//
// Bound by the VALU's products (two of head_dim 64 for a pair of the forward, four
// for the backward's dK and dV), after the clean call's own time.  Causal, 8 heads
// of 8192 rows, clean call / every row redone (an infinite first V row; infinite
// output gradients): float32 at head_dim 64 0.51 / 5.9 and 1.5 / 5.9 ms, f16 at
// head_dim 128 0.27 / 6.0 and 1.1 / 7.5 ms.  One row and key at a time took 14 to
// 46 ms for 2048 rows; 16 rows at once take 0.6 to 1.8.
template <typename T, int ND>
struct FlRow {
  float x[8 * ND];
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t row, int D, int g) {
#pragma unroll
    for (int h = 0; h < ND; ++h) {
      const int d = 32 * h + 8 * g;
      const uint32_t off = d < D ? row + (uint32_t)(d * sizeof(T)) : kOob;
      const uint4 a = bload16(rs, off);
      const uint32_t w[4] = {a.x, a.y, a.z, a.w};
      if constexpr (sizeof(T) == 4) {
        const uint4 b = bload16(rs, off + 16);
        const uint32_t y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[8 * h + i] = __uint_as_float(w[i]);
          x[8 * h + 4 + i] = __uint_as_float(y[i]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[8 * h + 2 * i] = fl_lo<T>(w[i]);
          x[8 * h + 2 * i + 1] = fl_hi<T>(w[i]);
        }
      }
    }
  }
  __device__ __forceinline__ float dot(const FlRow& o) const {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) s = fmaf(x[i], o.x[i], s);
    return col_sum(s);
  }
  __device__ __forceinline__ void add(float f, const FlRow& o) {
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) x[i] = fmaf(f, o.x[i], x[i]);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) x[i] = 0.0f;
  }
  __device__ __forceinline__ void scale(float f) {
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) x[i] *= f;
  }
  // as a product's accumulator, for fl_store
  __device__ __forceinline__ void sums(f32x4 (&acc)[2 * ND]) const {
#pragma unroll
    for (int i = 0; i < 2 * ND; ++i) acc[i] = f32x4{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
  }
};

// ---------------------------------------------------------------- forward
//
// One workgroup (NW waves) per 16 NQ NW queries of one stream; a wave holds
// NQ groups of 16 queries, so that every K and V operand it reads from LDS
// feeds NQ MFMAs.  Key blocks of KB rows go through LDS (one buffer, refilled
// between two barriers from loads issued a block earlier), softmax online in registers, rescaled only
// when a row's maximum rose.  The running maximum is kept times scale log2(e),
// rounded: a row whose maximum stayed is rescaled by 2^0 exactly (a difference
// formed from the raw maximum inside one fma would leave that product's
// rounding error, once per key block).  16-key sub-tiles outside every window of the
// wave are skipped.
//
// Rows of the group r0 .. r0 + 15 (lane's own: r0 + c) over their own keys:
// unnormalised sums and the weights' total.
template <typename T, int ND, bool GL>
__device__ __forceinline__ void fl_fwd_rows(const FlArgs& a, const FlPos& ps, __amdgpu_buffer_rsrc_t Qr,
                                            __amdgpu_buffer_rsrc_t Kr, __amdgpu_buffer_rsrc_t Vr, int r0, int c, int g,
                                            f32x4 (&sums)[2 * ND], float& l) {
  constexpr int U = ND == 1 ? 4 : ND == 2 ? 2 : 1;
  const uint32_t tb = a.tok_bytes;
  const int i = r0 + c, lo = max(0, r0 - a.left), hi = min(ps.Nr, r0 + 16 + a.right);
  const int ng = GL ? min(a.globals, lo) : 0;
  FlRow<T, ND> q, acc;
  q.load(Qr, (uint32_t)i * tb, a.D, g);
  acc.zero();
  float m = -INFINITY;
  l = 0.0f;
  for (int e = 0; e < ng + hi - lo; e += U) {
    FlRow<T, ND> k[U], v[U];
    float s[U], mn = m;
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = e + u < ng ? e + u : lo + e + u - ng;  // past hi: in range of the buffer or zeros, and masked
      k[u].load(Kr, (uint32_t)j * tb, a.D, g);
      v[u].load(Vr, (uint32_t)j * tb, a.D, g);
      in[u] = j < hi && j <= i + a.right && (j >= i - a.left || (GL && j < a.globals));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u] = q.dot(k[u]) * a.scale_log2;
      s[u] = in[u] ? s[u] : -INFINITY;
      mn = fmaxf(mn, s[u]);
    }
    const float mu = mn == -INFINITY ? 0.0f : mn, corr = __builtin_amdgcn_exp2f(m - mu);
    l *= corr;
    acc.scale(corr);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - mu);
      l += p;
      if (in[u]) acc.add(p, v[u]);
    }
    m = mn;
  }
  acc.sums(sums);
}

constexpr float kSlack = 8.0f;

// GL (Longformer windows; one residue class): after the window's
// blocks one more holds the global keys, of which a row takes those before its
// window.  Rows below `globals` are not written: they attend every key and
// another kernel splits them.
template <typename T, int ND, int NQ, int NW, int KB, int NPB, int OCC, bool GL>
__global__ __launch_bounds__(64 * NW, OCC) void flash_fwd_kernel(FlArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using St = FlStage<T, ND, KB, NW>;
  using Sc = FlScale<T, NPB>;
  constexpr int RS = St::RS, PL = St::kPlane, MAT = St::kMat;
  constexpr int NU = KB / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const FlPos ps = fl_pos(a, sizeof(T));
  const int Nr = ps.Nr, L = a.left, R = a.right, D = a.D;
  const int q0 = ps.tile * (16 * NQ * NW);
  if (q0 >= Nr) return;  // uniform per workgroup, before any barrier
  const uint32_t tb = a.tok_bytes;
  const __amdgpu_buffer_rsrc_t Qr = make_rsrc(static_cast<const T*>(a.q) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Kr = make_rsrc(static_cast<const T*>(a.k) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Vr = make_rsrc(static_cast<const T*>(a.v) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Or = make_rsrc(static_cast<T*>(a.o) + ps.base, ps.nrec);

  const int qa = q0 + 16 * NQ * wv;  // the wave's first query
  const int k0 = max(0, q0 - L) & ~15;
  const int kend = min(Nr, q0 + 16 * NQ * NW + R);
  const int nwin = (kend - k0 + KB - 1) / KB;
  const int nb = nwin + (GL && q0 + 16 * NQ * NW - 1 > L ? 1 : 0);

  St ks, vs;
  ks.load(Kr, k0, tid, tb, D);
  vs.load(Vr, k0, tid, tb, D);
  FlFrag<T, ND> qf[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) qf[n].load(Qr, (uint32_t)(qa + 16 * n + c) * tb, D, g);
  const uint32_t kl = (uint32_t)(c * RS + 16 * g), vl = (uint32_t)MAT + fl_tr_lane<ND>(c, g);

  float m_run[NQ], l_run[NQ];
  f32x4 acc[NQ][2 * ND];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m_run[n] = -INFINITY;
    l_run[n] = 0.0f;
#pragma unroll
    for (int d = 0; d < 2 * ND; ++d) acc[n][d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const float sl2 = a.scale_log2;
  ks.store(lds, tid);
  vs.store(lds + MAT, tid);
  __syncthreads();

  for (int e = 0; e < nb; ++e) {
    if (e + 1 < nb) {
      const int next = GL && e + 1 == nwin ? 0 : k0 + (e + 1) * KB;
      ks.load(Kr, next, tid, tb, D);
      vs.load(Vr, next, tid, tb, D);
    }
    __builtin_amdgcn_sched_barrier(0);
    const bool glob = GL && e == nwin;
    const int key0 = glob ? 0 : k0 + e * KB;
    // sub-tiles [u0, u1] of the block meet some window of the wave
    const int u0 = glob ? 0 : max(0, (qa - L - key0) >> 4);
    const int u1 = qa >= Nr ? -1
                   : glob   ? (qa + 16 * NQ - 1 > L ? 0 : -1)
                            : min(NU - 1, (min(qa + 16 * NQ - 1 + R, Nr - 1) - key0) >> 4);
    if (u0 <= u1) {  // wave-uniform
      f32x4 sc[NU][NQ];
      float mx[NQ], mu[NQ];
#pragma unroll
      for (int n = 0; n < NQ; ++n) mx[n] = -INFINITY;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if (u >= u0 && u <= u1) {
          fl_rowdot<T, ND, PL, NQ>(lds + u * 16 * RS + kl, qf, sc[u]);
          const int key = key0 + 16 * u;
#pragma unroll
          for (int n = 0; n < NQ; ++n) {
            const int rel = key - (qa + 16 * n);  // key - query offsets span rel -+ 15
            if (GL && glob) {
              const int x = rel + 4 * g - c;
#pragma unroll
              for (int r = 0; r < 4; ++r)
                sc[u][n][r] = x + r < -L && 4 * g + r < a.globals ? sc[u][n][r] : -INFINITY;
            } else if (rel - 15 < -L || rel + 15 > R || key + 15 >= Nr) {
              const int x = rel + 4 * g - c, hi = min(R, Nr - 1 - (qa + 16 * n) - c);
#pragma unroll
              for (int r = 0; r < 4; ++r) sc[u][n][r] = x + r >= -L && x + r <= hi ? sc[u][n][r] : -INFINITY;
            }
          }
        } else {
#pragma unroll
          for (int n = 0; n < NQ; ++n) sc[u][n] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        }
      }
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int n = 0; n < NQ; ++n)
          mx[n] = fmaxf(mx[n], fmaxf(fmaxf(sc[u][n][0], sc[u][n][1]), fmaxf(sc[u][n][2], sc[u][n][3])));
      bool rose = false;
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        // a maximum up to 2^kSlack times the running one (in weights) keeps it;
        // weights rounded to 16 bits follow every rise, which leaves the
        // largest of them exact (relative error of bf16 rows against float64
        // with the slack 2.27e-3, without 2.13e-3)
        constexpr float slack = NPB == 1 ? 0.0f : kSlack;
        mx[n] = col_max(mx[n]) * sl2;
        const bool up = !(mx[n] <= m_run[n] + slack);
        mx[n] = up ? fmaxf(m_run[n], mx[n]) : m_run[n];
        mu[n] = mx[n] == -INFINITY ? 0.0f : mx[n];
        rose = rose || up;
      }
      if (__builtin_amdgcn_ballot_w64(rose) != 0) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          const float corr = __builtin_amdgcn_exp2f(m_run[n] - mu[n]);  // 0 on a row's first block, 1 without a rise
          l_run[n] *= corr;
#pragma unroll
          for (int d = 0; d < 2 * ND; ++d) acc[n][d] *= corr;
          m_run[n] = mx[n];
        }
      }
#pragma unroll
      for (int u = 0; u < NU; u += 2) {
        if (u + 1 < u0 || u > u1) continue;  // wave-uniform
        FlB<T, NPB> pb[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          float p0[4], p1[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p0[r] = __builtin_amdgcn_exp2f(fmaf(sc[u][n][r], sl2, Sc::fwd(mu[n])));
            p1[r] = __builtin_amdgcn_exp2f(fmaf(sc[u + 1][n][r], sl2, Sc::fwd(mu[n])));
            l_run[n] += p0[r] + p1[r];
          }
          pb[n].set(p0, p1);
        }
        fl_trmul<T, ND, PL, NQ, NPB, ND <= 2 && NQ == 1>(lds + u * 16 * RS + vl, lds + (u + 1) * 16 * RS + vl, pb, acc);
      }
    }
    if (e + 1 < nb) {
      __syncthreads();
      ks.store(lds, tid);
      vs.store(lds + MAT, tid);
      __syncthreads();
    }
  }

  if (qa >= Nr) return;  // no barrier below
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const float l_tot = col_sum(l_run[n]);
    const float inv = l_tot != 0.0f ? 1.0f / l_tot : 0.0f;
    const int i = qa + 16 * n + c;
    const bool mine = !(GL && i < a.globals);
    const uint64_t bad = __builtin_amdgcn_ballot_w64(i < Nr && mine && fl_bad<ND>(acc[n]) && l_tot < INFINITY);
    const bool own_bad = (bad >> c & 0x0001000100010001ull) != 0;  // in some lane of the row
    fl_store<T, ND>(acc[n], inv, Or, own_bad || !mine ? kOob : (uint32_t)i * tb, D, g);
    if (a.lse && g == 0 && i < Nr)
      a.lse[((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h] =
          l_tot > 0.0f ? m_run[n] + (__log2f(l_tot) - Sc::kFwd) : 0.0f;
    if (__builtin_expect(bad != 0, 0)) {
      float l;
      fl_fwd_rows<T, ND, GL>(a, ps, Qr, Kr, Vr, qa + 16 * n, c, g, acc[n], l);
      fl_store<T, ND>(acc[n], l != 0.0f ? 1.0f / l : 0.0f, Or, own_bad ? (uint32_t)i * tb : kOob, D, g);
    }
  }
}

// ---------------------------------------------------------------- forward, paired tiles
//
// Causal (and other one-sided, sequence-wide) rows on few tiles: a launch lasts
// as long as its longest row of blocks.  The first half of the waves takes tile
// p, the second half tile T - 1 - p, so that every workgroup has the same
// number of (wave, block) products and each SIMD holds a wave of either tile;
// both walk the key blocks from 0 and share them.  The long tile's wave is
// alone on its SIMD for most of them, so a block's two halves overlap: while
// block e's scores turn into probabilities (VALU), the products of block e + 1
// with the queries run on the matrix cores.  K is therefore one block ahead of
// V in LDS (one buffer each, refilled between two barriers from loads issued a
// block earlier).  float32, head_dim 64, 8 heads of 4096 rows: 138 us, against
// 170-190 us unpaired and 214 us on the fp32 matrix cores.
//
// NPB: planes of a probability.
__device__ __forceinline__ float fl_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }

template <typename T, int ND, int NQ, int NW, int KB, int NPB>
__global__ __launch_bounds__(64 * NW, 2) void flash_pair_fwd_kernel(FlArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using St = FlStage<T, ND, KB, NW>;
  using Sc = FlScale<T, NPB>;
  constexpr int RS = St::RS, PL = St::kPlane, MAT = St::kMat;
  constexpr int NU = KB / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const FlPos ps = fl_pos(a, sizeof(T));
  const int Nr = ps.Nr, L = a.left, R = a.right, D = a.D;
  FlRows rows;
  if (!fl_rows<16 * NQ, NW, true>(ps, wv, rows)) return;  // uniform per workgroup, before any barrier
  const int qa = rows.first, qmin = rows.lo, qmax = rows.hi;
  const uint32_t tb = a.tok_bytes;
  const __amdgpu_buffer_rsrc_t Qr = make_rsrc(static_cast<const T*>(a.q) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Kr = make_rsrc(static_cast<const T*>(a.k) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Vr = make_rsrc(static_cast<const T*>(a.v) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Or = make_rsrc(static_cast<T*>(a.o) + ps.base, ps.nrec);
  const int k0 = max(0, qmin - L) & ~15;
  const int kend = min(Nr, qmax + R + 1);
  const int nb = (kend - k0 + KB - 1) / KB;

  St ks, vs;
  ks.load(Kr, k0, tid, tb, D);
  FlFrag<T, ND> qf[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) qf[n].load(Qr, (uint32_t)(qa + 16 * n + c) * tb, D, g);
  const uint32_t kl = (uint32_t)(c * RS + 16 * g), vl = (uint32_t)MAT + fl_tr_lane<ND>(c, g);
  float m_run[NQ], l_run[NQ];
  f32x4 acc[NQ][2 * ND];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m_run[n] = -INFINITY;
    l_run[n] = 0.0f;
#pragma unroll
    for (int d = 0; d < 2 * ND; ++d) acc[n][d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const float sl2 = a.scale_log2;

  // block e holds a pair of the wave's band / only pairs of it
  auto live = [&](int e) {
    const int key0 = k0 + e * KB;
    return e < nb && qa < Nr && key0 + KB - 1 >= qa - L && key0 <= min(qa + 16 * NQ - 1 + R, Nr - 1);
  };
  auto full = [&](int e) {
    const int key0 = k0 + e * KB;
    return e < nb && qa < Nr && key0 >= qa + 16 * NQ - 1 - L && key0 + KB - 1 <= min(qa + R, Nr - 1);
  };
  auto products = [&](f32x4 (&sc)[NU][NQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; ++u) fl_rowdot<T, ND, PL, NQ>(lds + u * 16 * RS + kl, qf, sc[u]);
  };
  auto masks = [&](int e, f32x4 (&sc)[NU][NQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int i = qa + 16 * n + c, x = k0 + e * KB + 4 * g - i;  // key - query of element 0
      const int hi = min(R, Nr - 1 - i);
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = x + 16 * u + r;
          sc[u][n][r] = d >= -L && d <= hi ? sc[u][n][r] : -INFINITY;
        }
    }
  };
  // the online softmax of a block's scores: a row's maximum moves only when
  // some score's weight would pass 2^kSlack times the largest so far
  auto weights = [&](f32x4 (&sc)[NU][NQ], float (&mu)[NQ]) __attribute__((always_inline)) {
    bool rose = false;
    float mn[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      float mx = fl_max(fl_max(sc[0][n][0], sc[0][n][1]), fl_max(sc[0][n][2], sc[0][n][3]));
#pragma unroll
      for (int u = 1; u < NU; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fl_max(mx, sc[u][n][r]);
      mx = col_max(mx) * sl2;
      const bool up = !(mx <= m_run[n] + kSlack);
      mn[n] = up ? fmaxf(m_run[n], mx) : m_run[n];
      mu[n] = mn[n] == -INFINITY ? 0.0f : mn[n];
      rose = rose || up;
    }
    if (__builtin_amdgcn_ballot_w64(rose) != 0) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        const float corr = __builtin_amdgcn_exp2f(m_run[n] - mu[n]);  // 0 on a row's first block, 1 without a rise
        l_run[n] *= corr;
#pragma unroll
        for (int d = 0; d < 2 * ND; ++d) acc[n][d] *= corr;
        m_run[n] = mn[n];
      }
    }
  };
  auto apply = [&](f32x4 (&sc)[NU][NQ], const float (&mu)[NQ], FlB<T, NPB> (&pb)[NU / 2][NQ])
                   __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; u += 2)
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        float p0[4], p1[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p0[r] = __builtin_amdgcn_exp2f(fmaf(sc[u][n][r], sl2, Sc::fwd(mu[n])));
          p1[r] = __builtin_amdgcn_exp2f(fmaf(sc[u + 1][n][r], sl2, Sc::fwd(mu[n])));
          l_run[n] += p0[r] + p1[r];
        }
        pb[u / 2][n].set(p0, p1);
      }
  };
  auto values = [&](const FlB<T, NPB> (&pb)[NU / 2][NQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; u += 2)
      fl_trmul<T, ND, PL, NQ, NPB, ND <= 2>(lds + u * 16 * RS + vl, lds + (u + 1) * 16 * RS + vl, pb[u / 2], acc);
  };

  f32x4 sa[NU][NQ], sb[NU][NQ];
  ks.store(lds, tid);
  __syncthreads();
  ks.load(Kr, k0 + KB, tid, tb, D);
  vs.load(Vr, k0, tid, tb, D);
  if (live(0)) {
    products(sa);
    masks(0, sa);
  }
  __syncthreads();
  ks.store(lds, tid);
  vs.store(lds + MAT, tid);
  __syncthreads();

  auto step = [&](int e, f32x4 (&cur)[NU][NQ], f32x4 (&nxt)[NU][NQ]) __attribute__((always_inline)) {
    ks.load(Kr, k0 + (e + 2) * KB, tid, tb, D);
    vs.load(Vr, k0 + (e + 1) * KB, tid, tb, D);
    __builtin_amdgcn_sched_barrier(0);
    const bool lv = live(e);
    if (lv && full(e + 1)) {  // wave-uniform
      float mu[NQ];
      FlB<T, NPB> pb[NU / 2][NQ];
      weights(cur, mu);
      products(nxt);
      apply(cur, mu, pb);
      values(pb);
    } else {
      if (lv) {
        float mu[NQ];
        FlB<T, NPB> pb[NU / 2][NQ];
        weights(cur, mu);
        apply(cur, mu, pb);
        values(pb);
      }
      if (live(e + 1)) {
        products(nxt);
        masks(e + 1, nxt);
      }
    }
    if (e + 1 < nb) {
      __syncthreads();
      ks.store(lds, tid);
      vs.store(lds + MAT, tid);
      __syncthreads();
    }
  };
  for (int e = 0; e < nb; e += 2) {
    step(e, sa, sb);
    if (e + 1 >= nb) break;
    step(e + 1, sb, sa);
  }

  if (qa >= Nr) return;  // no barrier below
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const float l_tot = col_sum(l_run[n]);
    const float inv = l_tot != 0.0f ? 1.0f / l_tot : 0.0f;
    const int i = qa + 16 * n + c;
    const uint64_t bad = __builtin_amdgcn_ballot_w64(i < Nr && fl_bad<ND>(acc[n]) && l_tot < INFINITY);
    const bool own_bad = (bad >> c & 0x0001000100010001ull) != 0;
    fl_store<T, ND>(acc[n], inv, Or, own_bad ? kOob : (uint32_t)i * tb, D, g);
    if (a.lse && g == 0 && i < Nr)
      a.lse[((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h] =
          l_tot > 0.0f ? m_run[n] + (__log2f(l_tot) - Sc::kFwd) : 0.0f;
    if (__builtin_expect(bad != 0, 0)) {
      float l;
      fl_fwd_rows<T, ND, false>(a, ps, Qr, Kr, Vr, qa + 16 * n, c, g, acc[n], l);
      fl_store<T, ND>(acc[n], l != 0.0f ? 1.0f / l : 0.0f, Or, own_bad ? (uint32_t)i * tb : kOob, D, g);
    }
  }
}

// ---------------------------------------------------------------- backward
//
// Two launches: dQ (and each row's statistics) by query tiles, then dK and dV
// by key tiles.  With p_ij = 2^(s_ij sl2 - lse2_i), dp_ij = dO_i . V_j,
// delta_i = sum_j p_ij dp_ij and ds_ij = p_ij (dp_ij - delta_i):
// dQ_i = scale sum_j ds_ij K_j, dK_j = scale sum_i ds_ij Q_i,
// dV_j = sum_i p_ij dO_i.  Each output row has one writer.
//
// Sums of dQ's rows r0 .. r0 + 15 over their own keys: p = 2^(s - mu) inv,
// with the row's delta dlt.
template <typename T, int ND>
__device__ __forceinline__ void fl_dq_rows(const FlArgs& a, const FlPos& ps, __amdgpu_buffer_rsrc_t Qr,
                                           __amdgpu_buffer_rsrc_t Gr, __amdgpu_buffer_rsrc_t Kr,
                                           __amdgpu_buffer_rsrc_t Vr, int r0, int c, int g, float mu, float inv,
                                           float dlt, f32x4 (&sums)[2 * ND]) {
  constexpr int U = ND == 1 ? 2 : 1;
  const uint32_t tb = a.tok_bytes;
  const int i = r0 + c, lo = max(0, r0 - a.left), hi = min(ps.Nr, r0 + 16 + a.right);
  FlRow<T, ND> q, go, acc;
  q.load(Qr, (uint32_t)i * tb, a.D, g);
  go.load(Gr, (uint32_t)i * tb, a.D, g);
  acc.zero();
  for (int e = lo; e < hi; e += U) {
    FlRow<T, ND> k[U], v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      k[u].load(Kr, (uint32_t)(e + u) * tb, a.D, g);
      v[u].load(Vr, (uint32_t)(e + u) * tb, a.D, g);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float s = q.dot(k[u]), dp = go.dot(v[u]);
      const float ds = __builtin_amdgcn_exp2f(fmaf(s, a.scale_log2, -mu)) * inv * (dp - dlt);
      if (e + u < hi && e + u >= i - a.left && e + u <= i + a.right) acc.add(ds, k[u]);
    }
  }
  acc.sums(sums);
}

// Sums of dK's and dV's rows r0 .. r0 + 15 over their own queries.
template <typename T, int ND>
__device__ __forceinline__ void fl_dkv_rows(const FlArgs& a, const FlPos& ps, __amdgpu_buffer_rsrc_t Qr,
                                            __amdgpu_buffer_rsrc_t Gr, __amdgpu_buffer_rsrc_t Kr,
                                            __amdgpu_buffer_rsrc_t Vr, int r0, int c, int g, f32x4 (&sk)[2 * ND],
                                            f32x4 (&sv)[2 * ND]) {
  constexpr int U = ND == 1 ? 2 : 1;
  const uint32_t tb = a.tok_bytes;
  const int j = r0 + c, lo = max(0, r0 - a.right), hi = min(ps.Nr, r0 + 16 + a.left);
  FlRow<T, ND> k, v, dk, dv;
  k.load(Kr, (uint32_t)j * tb, a.D, g);
  v.load(Vr, (uint32_t)j * tb, a.D, g);
  dk.zero();
  dv.zero();
  for (int e = lo; e < hi; e += U) {
    FlRow<T, ND> q[U], go[U];
    f32x2 st[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      q[u].load(Qr, (uint32_t)(e + u) * tb, a.D, g);
      go[u].load(Gr, (uint32_t)(e + u) * tb, a.D, g);
      const int64_t row = ((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * min(e + u, hi - 1)) * a.H + ps.h;
      st[u] = *reinterpret_cast<const f32x2*>(a.stats + 2 * row);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float s = k.dot(q[u]), dp = v.dot(go[u]);
      const float p = __builtin_amdgcn_exp2f(fmaf(s, a.scale_log2, -st[u][0]));
      if (e + u < hi && e + u >= j - a.right && e + u <= j + a.left) {
        dv.add(p, go[u]);
        dk.add(p * (dp - st[u][1]), q[u]);
      }
    }
  }
  dk.sums(sk);
  dv.sums(sv);
}

// Whether the sums of dK and dV stand for the keys r0 .. r0 + 15: each has, in
// its query set, a query whose statistics are NaN, or whose delta and whole dO
// row are (dK and dV all NaN in either computation), or whose delta is NaN where
// dV's sums are finite (v_ok; dK all NaN).
template <typename T, int ND>
__device__ __forceinline__ bool fl_dkv_nan(const FlArgs& a, const FlPos& ps, __amdgpu_buffer_rsrc_t Gr, int r0,
                                           int lane, bool v_ok) {
  bool nan_l = false;
  int w = -1;
  for (int i = max(0, r0 + 15 - a.right) + lane; i <= min(ps.Nr - 1, r0 + a.left); i += 64) {
    const int64_t row = ((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h;
    const f32x2 st = *reinterpret_cast<const f32x2*>(a.stats + 2 * row);
    nan_l = nan_l || st[0] != st[0];
    w = st[1] != st[1] ? i : w;
  }
  if (__builtin_amdgcn_ballot_w64(nan_l) != 0) return true;
  const uint64_t found = __builtin_amdgcn_ballot_w64(w >= 0);
  if (found == 0 || v_ok) return found != 0;
  FlRow<T, ND> go;
  go.load(Gr, (uint32_t)__shfl(w, __builtin_ctzll(found), 64) * a.tok_bytes, a.D, lane >> 4);
  bool all = true;
#pragma unroll
  for (int i = 0; i < 8 * ND; ++i)
    all = all && (go.x[i] != go.x[i] || 32 * (i >> 3) + 8 * (lane >> 4) >= a.D);
  return __builtin_amdgcn_ballot_w64(!all) == 0;
}

template <bool B>
struct FlBool {
  static constexpr bool value = B;
};

// dQ of 16 NQ NW queries.  Pass 1 over the key blocks: the online softmax's
// maximum, sum and sum of e dp.  Pass 2, backwards over the same blocks (the
// last one is still in LDS): p, ds, dQ^T += K^T ds^T.  SAVED: the forward's
// statistics are read and delta = dO . O, so only the second pass runs.  PAIR:
// fl_rows; NPB: planes of a dS (and probability) operand.
template <typename T, int ND, int NQ, int NW, int KB, int NPB, int OCC, bool SAVED, bool FAST, bool PAIR>
__global__ __launch_bounds__(64 * NW, OCC) void flash_dq_kernel(FlArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using St = FlStage<T, ND, KB, NW>;
  using Sc = FlScale<T, NPB>;
  constexpr int RS = St::RS, PL = St::kPlane, MAT = St::kMat;
  constexpr int NU = KB / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const FlPos ps = fl_pos(a, sizeof(T));
  const int Nr = ps.Nr, L = a.left, R = a.right, D = a.D;
  FlRows rows;
  if (!fl_rows<16 * NQ, NW, PAIR>(ps, wv, rows)) return;  // uniform per workgroup, before any barrier
  const uint32_t tb = a.tok_bytes;
  const __amdgpu_buffer_rsrc_t Qr = make_rsrc(static_cast<const T*>(a.q) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Gr = make_rsrc(static_cast<const T*>(a.dout) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Kr = make_rsrc(static_cast<const T*>(a.k) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Vr = make_rsrc(static_cast<const T*>(a.v) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Or = make_rsrc(static_cast<T*>(a.o) + ps.base, ps.nrec);

  const int qa = rows.first;
  const int k0 = max(0, rows.lo - L) & ~15;
  const int kend = min(Nr, rows.hi + 1 + R);
  const int nb = (kend - k0 + KB - 1) / KB;
  const int steps = SAVED ? nb : 2 * nb;
  auto block_at = [&](int e) { return !SAVED && e < nb ? e : steps - 1 - e; };

  St ks, vs;
  ks.load(Kr, k0 + block_at(0) * KB, tid, tb, D);
  vs.load(Vr, k0 + block_at(0) * KB, tid, tb, D);
  FlFrag<T, ND> qf[NQ], gf[NQ];
  float m[NQ], l[NQ], dl[NQ];  // pass 1: maximum, sum, sum of e dp; then mu, 1/sum, delta
  float top[NQ];  // f16: pass 1: largest |dp|; then the power of two on the row's dS, which is below 2 top
  const float sl2 = a.scale_log2;
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const uint32_t row = (uint32_t)(qa + 16 * n + c) * tb;
    qf[n].load(Qr, row, D, g);
    gf[n].load(Gr, row, D, g);
    m[n] = -INFINITY;
    l[n] = dl[n] = top[n] = 0.0f;
    if constexpr (SAVED) {
      const __amdgpu_buffer_rsrc_t Fr = make_rsrc(static_cast<const T*>(a.fo) + ps.base, ps.nrec);
      FlFrag<T, ND> of;
      of.load(Fr, row, D, g);
      using E = typename FlElt<T>::E;
      float d = 0.0f;
#pragma unroll
      for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float x0 = 0.0f, x1 = 0.0f, y0 = 0.0f, y1 = 0.0f;  // planes add up exactly, smallest first
#pragma unroll
          for (int p = FlElt<T>::NP - 1; p >= 0; --p) {
            const uint32_t gw = reinterpret_cast<const uint32_t*>(&gf[n].r[p][j])[w];
            const uint32_t ow = reinterpret_cast<const uint32_t*>(&of.r[p][j])[w];
            x0 += fl_lo<E>(gw);
            x1 += fl_hi<E>(gw);
            y0 += fl_lo<E>(ow);
            y1 += fl_hi<E>(ow);
          }
          d = fmaf(x0, y0, d);
          d = fmaf(x1, y1, d);
        }
      dl[n] = col_sum(d);
      const int i = qa + 16 * n + c;
      m[n] = i < Nr ? a.lse[((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h] : 0.0f;
      l[n] = 1.0f;
    }
  }
  const uint32_t rl = (uint32_t)(c * RS + 16 * g), tl = fl_tr_lane<ND>(c, g);
  f32x4 acc[NQ][2 * ND];
#pragma unroll
  for (int n = 0; n < NQ; ++n)
#pragma unroll
    for (int d = 0; d < 2 * ND; ++d) acc[n][d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  ks.store(lds, tid);
  vs.store(lds + MAT, tid);
  __syncthreads();

  // S and dP of sub-tile u of the block at key0, pairs outside the band
  // masked (their V row may hold anything: dP 0)
  auto scores = [&](auto full, int u, int key0, f32x4 (&sc)[NQ], f32x4 (&dp)[NQ]) __attribute__((always_inline)) {
    fl_rowdot<T, ND, PL, NQ>(lds + u * 16 * RS + rl, qf, sc);
    fl_rowdot<T, ND, PL, NQ>(lds + MAT + u * 16 * RS + rl, gf, dp);
    if constexpr (decltype(full)::value) return;
    const int key = key0 + 16 * u;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int rel = key - (qa + 16 * n);
      if (rel - 15 < -L || rel + 15 > R || key + 15 >= Nr) {
        const int x = rel + 4 * g - c, hi = min(R, Nr - 1 - (qa + 16 * n) - c);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = x + r >= -L && x + r <= hi;
          sc[n][r] = in ? sc[n][r] : -INFINITY;
          dp[n][r] = in ? dp[n][r] : 0.0f;
        }
      }
    }
  };

  for (int e = 0; e < steps; ++e) {
    const bool turn = !SAVED && e == nb - 1;  // the next step works on the same block
    const bool more = e + 1 < steps && !turn;
    if (more) {
      ks.load(Kr, k0 + block_at(e + 1) * KB, tid, tb, D);
      vs.load(Vr, k0 + block_at(e + 1) * KB, tid, tb, D);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int key0 = k0 + block_at(e) * KB;
    const int u0 = max(0, (qa - L - key0) >> 4);
    const int u1 = qa < Nr ? min(NU - 1, (min(qa + 16 * NQ - 1 + R, Nr - 1) - key0) >> 4) : -1;
    if (!SAVED && e < nb) {
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if (u < u0 || u > u1) continue;  // wave-uniform
        f32x4 sc[NQ], dp[NQ];
        scores(FlBool<false>{}, u, key0, sc, dp);
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          const float mn =
              fmaxf(m[n], col_max(fmaxf(fmaxf(sc[n][0], sc[n][1]), fmaxf(sc[n][2], sc[n][3]))) * sl2);
          const float mu = mn == -INFINITY ? 0.0f : mn;
          const float corr = __builtin_amdgcn_exp2f(m[n] - mu);  // 1 without a rise
          l[n] *= corr;
          dl[n] *= corr;
          m[n] = mn;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float p = __builtin_amdgcn_exp2f(fmaf(sc[n][r], sl2, -mu));
            l[n] += p;
            dl[n] = fmaf(p, dp[n][r], dl[n]);
            if constexpr (Sc::kOn) top[n] = fmaxf(top[n], fabsf(dp[n][r]));
          }
        }
      }
      if (e == nb - 1) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
          const float lt = col_sum(l[n]), dt = col_sum(dl[n]);
          const float mu = m[n] == -INFINITY ? 0.0f : m[n];
          l[n] = lt != 0.0f ? 1.0f / lt : 0.0f;
          dl[n] = dt * l[n];
          const int i = qa + 16 * n + c;
          if (g == 0 && i < Nr) {
            const int64_t row = ((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h;
            *reinterpret_cast<f32x2*>(a.stats + 2 * row) = f32x2{lt != 0.0f ? mu + __log2f(lt) : 0.0f, dl[n]};
          }
          m[n] = mu;
          if constexpr (Sc::kOn) {
            top[n] = __builtin_amdgcn_ldexpf(1.0f, Sc::exponent(col_max(top[n]), 14));
            l[n] *= top[n];
          }
        }
      }
    } else {
      auto pass2 = [&](auto full) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full)::value;
#pragma unroll
        for (int u = 0; u < NU; u += 2) {
          if (!FULL && (u + 1 < u0 || u > u1)) continue;  // wave-uniform
          f32x4 sc[2][NQ], dp[2][NQ];
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            if (FULL || (u + w >= u0 && u + w <= u1)) {
              scores(full, u + w, key0, sc[w], dp[w]);
            } else {
#pragma unroll
              for (int n = 0; n < NQ; ++n) {
                sc[w][n] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                dp[w][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
              }
            }
          }
          FlB<T, NPB> db[NQ];
#pragma unroll
          for (int n = 0; n < NQ; ++n) {
            float ds[2][4];
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(fmaf(sc[w][n][r], sl2, -m[n]));
                ds[w][r] = (SAVED ? p : p * l[n]) * (dp[w][n][r] - dl[n]);
              }
            db[n].set(ds[0], ds[1]);
          }
          fl_trmul<T, ND, PL, NQ, NPB>(lds + u * 16 * RS + tl, lds + (u + 1) * 16 * RS + tl, db, acc);
        }
      };
      // FAST: blocks wholly inside the band as straight-line code
      if (FAST && key0 >= qa + 16 * NQ - 1 - L && key0 + KB - 1 <= min(qa + R, Nr - 1) && qa < Nr)
        pass2(FlBool<true>{});
      else
        pass2(FlBool<false>{});
    }
    if (more) {
      __syncthreads();
      ks.store(lds, tid);
      vs.store(lds + MAT, tid);
      __syncthreads();
    }
  }

  if (qa >= Nr) return;  // no barrier below
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const int i = qa + 16 * n + c;
    if constexpr (SAVED) {  // the dK, dV kernel reads {lse2, delta}
      if (g == 0 && i < Nr) {
        const int64_t row = ((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h;
        *reinterpret_cast<f32x2*>(a.stats + 2 * row) = f32x2{m[n], dl[n]};
      }
    }
    float f = a.scale;
    if constexpr (Sc::kOn) {
      f /= top[n];
      l[n] /= top[n];
    }
    const uint64_t bad = __builtin_amdgcn_ballot_w64(i < Nr && fl_bad<ND>(acc[n]) && l[n] == l[n] && dl[n] == dl[n]);
    const bool own_bad = (bad >> c & 0x0001000100010001ull) != 0;  // in some lane of the row
    fl_store<T, ND>(acc[n], f, Or, own_bad ? kOob : (uint32_t)i * tb, D, g);
    if (__builtin_expect(bad != 0, 0)) {
      fl_dq_rows<T, ND>(a, ps, Qr, Gr, Kr, Vr, qa + 16 * n, c, g, m[n], l[n], dl[n], acc[n]);
      fl_store<T, ND>(acc[n], a.scale, Or, own_bad ? (uint32_t)i * tb : kOob, D, g);
    }
  }
}

// dK, dV of 16 NK NW keys: a wave holds NK groups of 16 keys' K and V rows as
// register operands; blocks of QB query rows (Q, dO and their statistics) go
// through LDS, and every operand read from them feeds NK MFMAs.  S and dP land
// with lane (c, g) holding queries 4 g .. 4 g + 3 of key c.
template <typename T, int ND, int NK, int NW, int QB, int NPB, int OCC, bool FAST, bool PAIR>
__global__ __launch_bounds__(64 * NW, OCC) void flash_dkv_kernel(FlArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using St = FlStage<T, ND, QB, NW>;
  using Sc = FlScale<T, NPB>;
  constexpr int RS = St::RS, PL = St::kPlane, MAT = St::kMat;
  constexpr int NU = QB / 16;
  float* lst = reinterpret_cast<float*>(lds + 2 * MAT);  // QB lse2, then QB delta
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const FlPos ps = fl_pos(a, sizeof(T));
  const int Nr = ps.Nr, L = a.left, R = a.right, D = a.D;
  FlRows rows;
  if (!fl_rows<16 * NK, NW, PAIR>(ps, wv, rows)) return;  // uniform per workgroup, before any barrier
  const uint32_t tb = a.tok_bytes;
  const __amdgpu_buffer_rsrc_t Qr = make_rsrc(static_cast<const T*>(a.q) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Gr = make_rsrc(static_cast<const T*>(a.dout) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Kr = make_rsrc(static_cast<const T*>(a.k) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t Vr = make_rsrc(static_cast<const T*>(a.v) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t dKr = make_rsrc(static_cast<T*>(a.dk) + ps.base, ps.nrec);
  const __amdgpu_buffer_rsrc_t dVr = make_rsrc(static_cast<T*>(a.dv) + ps.base, ps.nrec);

  const int ja = rows.first;  // the wave's first key
  const int i0 = max(0, rows.lo - R) & ~15;
  const int iend = min(Nr, rows.hi + 1 + L);
  const int nb = (iend - i0 + QB - 1) / QB;

  St qs, gs;
  f32x2 st;
  auto load_stats = [&](int r0) {  // threads 0 .. QB-1; rows past the end get p = 0
    const int i = r0 + tid;
    st = f32x2{INFINITY, 0.0f};
    if (tid < QB && i < Nr)
      st = *reinterpret_cast<const f32x2*>(a.stats +
                                           2 * (((int64_t)ps.b * a.N + ps.rho + (int64_t)a.dil * i) * a.H + ps.h));
  };
  auto store_stats = [&]() {
    if (tid < QB) {
      lst[tid] = st[0];
      lst[QB + tid] = st[1];
    }
  };
  qs.load(Qr, i0, tid, tb, D);
  gs.load(Gr, i0, tid, tb, D);
  load_stats(i0);
  FlFrag<T, ND> kf[NK], vf[NK];
#pragma unroll
  for (int n = 0; n < NK; ++n) {
    kf[n].load(Kr, (uint32_t)(ja + 16 * n + c) * tb, D, g);
    vf[n].load(Vr, (uint32_t)(ja + 16 * n + c) * tb, D, g);
  }
  const uint32_t rl = (uint32_t)(c * RS + 16 * g), tl = fl_tr_lane<ND>(c, g);
  const float sl2 = a.scale_log2;
  f32x4 ak[NK][2 * ND], av[NK][2 * ND];
  float sk[NK];  // f16: the power of two on the key's dS, lowered (and ak with it) when one would pass 2^15
#pragma unroll
  for (int n = 0; n < NK; ++n) sk[n] = 0x1p100f;
#pragma unroll
  for (int n = 0; n < NK; ++n)
#pragma unroll
    for (int d = 0; d < 2 * ND; ++d) ak[n][d] = av[n][d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  qs.store(lds, tid);
  gs.store(lds + MAT, tid);
  store_stats();
  __syncthreads();

  for (int e = 0; e < nb; ++e) {
    const bool more = e + 1 < nb;
    if (more) {
      qs.load(Qr, i0 + (e + 1) * QB, tid, tb, D);
      gs.load(Gr, i0 + (e + 1) * QB, tid, tb, D);
      load_stats(i0 + (e + 1) * QB);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int r0 = i0 + e * QB;
    // query sub-tiles [u0, u1] see some key of the wave: i in [ja - R, ja + 16 NK - 1 + L]
    const int u0 = max(0, (ja - R - r0) >> 4);
    const int u1 = ja < Nr ? min(NU - 1, (min(ja + 16 * NK - 1 + L, Nr - 1) - r0) >> 4) : -1;
    auto block = [&](auto full) __attribute__((always_inline)) {
      constexpr bool FULL = decltype(full)::value;
#pragma unroll
      for (int u = 0; u < NU; u += 2) {
        if (!FULL && (u + 1 < u0 || u > u1)) continue;  // wave-uniform
        float p[NK][2][4], ds[NK][2][4];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          if (FULL || (u + w >= u0 && u + w <= u1)) {
            f32x4 sc[NK], dp[NK];
            fl_rowdot<T, ND, PL, NK>(lds + (u + w) * 16 * RS + rl, kf, sc);
            fl_rowdot<T, ND, PL, NK>(lds + MAT + (u + w) * 16 * RS + rl, vf, dp);
            const int qb = r0 + 16 * (u + w);
            const f32x4 ls = *reinterpret_cast<const f32x4*>(lst + 16 * (u + w) + 4 * g);
            const f32x4 dt = *reinterpret_cast<const f32x4*>(lst + QB + 16 * (u + w) + 4 * g);
#pragma unroll
            for (int n = 0; n < NK; ++n) {
              if constexpr (!FULL) {
                const int rel = ja + 16 * n - qb;  // key - query offsets span rel -+ 15
                if (rel - 15 < -L || rel + 15 > R) {
                  const int x = rel + c - 4 * g;  // key - query of element 0
#pragma unroll
                  for (int r = 0; r < 4; ++r) {
                    const bool in = x - r >= -L && x - r <= R;
                    sc[n][r] = in ? sc[n][r] : -INFINITY;
                    dp[n][r] = in ? dp[n][r] : dt[r];
                  }
                }
              }
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                p[n][w][r] = __builtin_amdgcn_exp2f(fmaf(sc[n][r], sl2, Sc::prob(ls[r])));
                ds[n][w][r] = p[n][w][r] * (dp[n][r] - dt[r]);
              }
            }
          } else {
#pragma unroll
            for (int n = 0; n < NK; ++n)
#pragma unroll
              for (int r = 0; r < 4; ++r) p[n][w][r] = ds[n][w][r] = 0.0f;
          }
        }
        FlB<T, NPB> b[NK];
#pragma unroll
        for (int n = 0; n < NK; ++n) b[n].set(p[n][0], p[n][1]);
        fl_trmul<T, ND, PL, NK, NPB>(lds + MAT + u * 16 * RS + tl, lds + MAT + (u + 1) * 16 * RS + tl, b, av);
        if constexpr (Sc::kOn) {
          float mx[NK];
          bool over = false;
#pragma unroll
          for (int n = 0; n < NK; ++n) {
            mx[n] = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[n] = fmaxf(mx[n], fmaxf(fabsf(ds[n][0][r]), fabsf(ds[n][1][r])));
            over = over || mx[n] * sk[n] > 0x1p15f;
          }
          if (__builtin_amdgcn_ballot_w64(over) != 0) {
#pragma unroll
            for (int n = 0; n < NK; ++n) {
              mx[n] = col_max(mx[n]);
              const float s = mx[n] * sk[n] > 0x1p15f ? __builtin_amdgcn_ldexpf(1.0f, Sc::exponent(mx[n], 12)) : sk[n];
              const float f = s / sk[n];
#pragma unroll
              for (int d = 0; d < 2 * ND; ++d) ak[n][d] *= f;
              sk[n] = s;
            }
          }
#pragma unroll
          for (int n = 0; n < NK; ++n)
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
              for (int r = 0; r < 4; ++r) ds[n][w][r] *= sk[n];
        }
#pragma unroll
        for (int n = 0; n < NK; ++n) b[n].set(ds[n][0], ds[n][1]);
        fl_trmul<T, ND, PL, NK, NPB>(lds + u * 16 * RS + tl, lds + (u + 1) * 16 * RS + tl, b, ak);
      }
    };
    // FAST: blocks whose every pair is in the band as straight-line code (rows
    // past the end have lse2 = infinity)
    if (FAST && ja < Nr && r0 >= ja + 16 * NK - 1 - R && r0 + QB - 1 <= ja + L)
      block(FlBool<true>{});
    else
      block(FlBool<false>{});
    if (more) {
      __syncthreads();
      qs.store(lds, tid);
      gs.store(lds + MAT, tid);
      store_stats();
      __syncthreads();
    }
  }

  if (ja >= Nr) return;  // no barrier below
  // the lane's numbers again: held over the loop they would spill at head_dims above 64
  const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), ec = el & 15, eg = el >> 4;
#pragma unroll
  for (int n = 0; n < NK; ++n) {
    const int j = ja + 16 * n + ec;
    const uint64_t bad_v = __builtin_amdgcn_ballot_w64(j < Nr && fl_bad<ND>(av[n]));
    uint64_t bad = bad_v | __builtin_amdgcn_ballot_w64(j < Nr && fl_bad<ND>(ak[n]));
    if (__builtin_expect(bad != 0, 0) && fl_dkv_nan<T, ND>(a, ps, Gr, ja + 16 * n, el, bad_v == 0)) bad = 0;
    const bool own_bad = (bad >> ec & 0x0001000100010001ull) != 0;  // in some lane of the row
    const uint32_t row = (uint32_t)j * tb;
    constexpr float kUp = Sc::kOn ? 0x1p-15f : 1.0f;  // 2^-kProb
    fl_store<T, ND>(ak[n], Sc::kOn ? a.scale * kUp / sk[n] : a.scale, dKr, own_bad ? kOob : row, D, eg);
    fl_store<T, ND>(av[n], kUp, dVr, own_bad ? kOob : row, D, eg);
    if (__builtin_expect(bad != 0, 0)) {
      fl_dkv_rows<T, ND>(a, ps, Qr, Gr, Kr, Vr, ja + 16 * n, ec, eg, ak[n], av[n]);
      fl_store<T, ND>(ak[n], a.scale, dKr, own_bad ? row : kOob, D, eg);
      fl_store<T, ND>(av[n], 1.0f, dVr, own_bad ? row : kOob, D, eg);
    }
  }
}

}  // namespace ma_dev
