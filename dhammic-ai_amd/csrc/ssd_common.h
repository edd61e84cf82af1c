// Device-side building blocks shared by the SSD kernels (gfx950, wave64).
//
// MFMA tiling: one wave computes a 32x32 fp32 tile with
//   bf16: v_mfma_f32_32x32x16_bf16  (K = 16 per instruction)
//   fp32: 8 x v_mfma_f32_32x32x2_f32 (K = 16 per group of eight)
// Operand fragments: lane l supplies A[l%32][k0 + (l/32)*8 + t] and
// B[k0 + (l/32)*8 + t][l%32] for t = 0..7, i.e. eight consecutive k per lane,
// so every operand is kept k-contiguous in LDS (or global) and read as one
// 16-byte vector (bf16) or two (fp32). For fp32 the eight values of a lane are
// spread over eight K=2 instructions; A and B use the same spreading, so the
// sum over k is unchanged.
// Accumulator layout (both variants): lane l, register v holds
//   row 8*(v/4) + 4*(l/32) + v%4, column l%32.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

#define SSD_WAVE 64
// Rows of the token axis per block tile inside a chunk.
#define SSD_BLK 64
#define SSD_LO (-20.0f)
#define SSD_HI (20.0f)
// Largest exponent (nats) of either factor of the factorised decay
// exp(cs_l - cs_s) = exp(cs_l - c_j) * exp(c_j - cs_s) inside a 64-token block j, whose reference c_j
// is the midpoint of the block's cumsum range: blocks that drop by at most 2 SSD_FACT_RANGE take it
// (every factor then within e^{+-64}, inside fp32 and bf16 with room for the values it scales).
#define SSD_FACT_RANGE (64.0f)
// Largest rise of the in-chunk cumsum from one position to the next that the factorised-decay guard
// treats as non-increasing. The cumsum is a parallel scan whose lanes round their prefixes along
// different paths, so a flat stretch (positions past a packed sequence's end, a = 0) can rise by an
// ulp; the factorisation itself is exact for any cumsum, and a total rise below 256 x this bound
// leaves every factor within e^0.26 and no clamp at +20 binding.
#define SSD_FACT_RISE (1e-3f)

// exp(clamp(v, -20, 20)): every decay exponent of the reference path
// (r2/dhammic-ai/src/kernels/ssd_scan.py:53-54, :116, :212).
__device__ __forceinline__ float exp_clamp(float v) {
  return __expf(fminf(fmaxf(v, SSD_LO), SSD_HI));
}
// Strict pass mask of the clamp backward (ssd_scan.py:192, :230).
__device__ __forceinline__ float clamp_pass(float v) {
  return (v > SSD_LO && v < SSD_HI) ? 1.0f : 0.0f;
}

template <typename T> __device__ __forceinline__ float to_f(T v);
template <> __device__ __forceinline__ float to_f<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f<bf16>(bf16 v) { return (float)v; }

template <typename T> __device__ __forceinline__ T from_f(float v);
template <> __device__ __forceinline__ float from_f<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f<bf16>(float v) { return (bf16)v; }

template <typename T> struct Frag;
template <> struct Frag<bf16> { bf16x8 v; };
template <> struct Frag<float> { float v[8]; };

// Eight consecutive elements at p (16-byte aligned for bf16, 32-byte for fp32 in LDS).
__device__ __forceinline__ Frag<bf16> ld_frag(const bf16* p) {
  Frag<bf16> f;
  f.v = *reinterpret_cast<const bf16x8*>(p);
  return f;
}
__device__ __forceinline__ Frag<float> ld_frag(const float* p) {
  Frag<float> f;
  floatx4 a = *reinterpret_cast<const floatx4*>(p);
  floatx4 b = *reinterpret_cast<const floatx4*>(p + 4);
  f.v[0] = a[0]; f.v[1] = a[1]; f.v[2] = a[2]; f.v[3] = a[3];
  f.v[4] = b[0]; f.v[5] = b[1]; f.v[6] = b[2]; f.v[7] = b[3];
  return f;
}

// Eight consecutive fp32 values (global, 16-byte aligned) converted to T.
template <typename T> __device__ __forceinline__ Frag<T> ld_frag_f32(const float* p);
template <> __device__ __forceinline__ Frag<float> ld_frag_f32<float>(const float* p) {
  return ld_frag(p);
}
template <> __device__ __forceinline__ Frag<bf16> ld_frag_f32<bf16>(const float* p) {
  floatx4 a = *reinterpret_cast<const floatx4*>(p);
  floatx4 b = *reinterpret_cast<const floatx4*>(p + 4);
  Frag<bf16> f;
  f.v[0] = (bf16)a[0]; f.v[1] = (bf16)a[1]; f.v[2] = (bf16)a[2]; f.v[3] = (bf16)a[3];
  f.v[4] = (bf16)b[0]; f.v[5] = (bf16)b[1]; f.v[6] = (bf16)b[2]; f.v[7] = (bf16)b[3];
  return f;
}

__device__ __forceinline__ void mma(floatx16& acc, const Frag<bf16>& a, const Frag<bf16>& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma(floatx16& acc, const Frag<float>& a, const Frag<float>& b) {
#pragma unroll
  for (int t = 0; t < 8; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[t], b.v[t], acc, 0, 0, 0);
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
// Row (0..31) of accumulator register v for this lane; the column is lane % 32.
__device__ __forceinline__ int acc_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

__device__ __forceinline__ void zero(floatx16& a) {
#pragma unroll
  for (int v = 0; v < 16; ++v) a[v] = 0.0f;
}

// acc(32x32) += A[32 x K] * B[K x 32] with A(i, k) = a[i*lda + k] and
// B(k, j) = b[j*ldb + k] (both k-contiguous), K a multiple of 16.
template <typename T>
__device__ __forceinline__ void mma_tile(floatx16& acc, const T* a, int lda, const T* b, int ldb, int K) {
  const int lane = lane_id();
  const T* ap = a + (lane & 31) * lda + (lane >> 5) * 8;
  const T* bp = b + (lane & 31) * ldb + (lane >> 5) * 8;
  for (int k0 = 0; k0 < K; k0 += 16) {
    Frag<T> fa = ld_frag(ap + k0);
    Frag<T> fb = ld_frag(bp + k0);
    mma(acc, fa, fb);
  }
}

// ---------------------------------------------------------------------------
// Accumulator tile reused as an MFMA A operand (no LDS round trip).
// A 32x32 fp32 tile X in accumulator layout (lane: column b = lane%32; rows
// a = 8r + 4*(lane/32) + q in register 4r + q) serves as A'[i = b][k = a],
// i.e. A' = X^T. K-step kk (0 or 1) covers rows a = 16kk .. 16kk+15 of X,
// registers 8kk .. 8kk+7; their row order is a = 16kk + 8*(t/4) + 4*(lane/32)
// + t%4 for t = 0..7, so the B operand is read in the same permuted order.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <typename T> __device__ __forceinline__ Frag<T> frag_from_acc(const floatx16& x, int kk);
template <> __device__ __forceinline__ Frag<bf16> frag_from_acc<bf16>(const floatx16& x, int kk) {
  Frag<bf16> f;
#pragma unroll
  for (int t = 0; t < 8; ++t) f.v[t] = (bf16)x[8 * kk + t];
  return f;
}
template <> __device__ __forceinline__ Frag<float> frag_from_acc<float>(const floatx16& x, int kk) {
  Frag<float> f;
#pragma unroll
  for (int t = 0; t < 8; ++t) f.v[t] = x[8 * kk + t];
  return f;
}

// B'[a][j] for the permuted rows a of step kk, from row j of a [j][a] tile (a contiguous).
__device__ __forceinline__ Frag<bf16> ld_frag_perm(const bf16* row, int kk) {
  const int off = 16 * kk + 4 * (lane_id() >> 5);
  const bf16x4 lo = *reinterpret_cast<const bf16x4*>(row + off);
  const bf16x4 hi = *reinterpret_cast<const bf16x4*>(row + off + 8);
  Frag<bf16> f;
  f.v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return f;
}
__device__ __forceinline__ Frag<float> ld_frag_perm(const float* row, int kk) {
  const int off = 16 * kk + 4 * (lane_id() >> 5);
  const floatx4 lo = *reinterpret_cast<const floatx4*>(row + off);
  const floatx4 hi = *reinterpret_cast<const floatx4*>(row + off + 8);
  Frag<float> f;
  f.v[0] = lo[0]; f.v[1] = lo[1]; f.v[2] = lo[2]; f.v[3] = lo[3];
  f.v[4] = hi[0]; f.v[5] = hi[1]; f.v[6] = hi[2]; f.v[7] = hi[3];
  return f;
}

// out(32x32) += X^T B' with X a 32x32 accumulator tile and B'[a][j] = src[j*ld + a].
template <typename T>
__device__ __forceinline__ void mma_xt(floatx16& out, const floatx16& X, const T* src, int ld) {
  const T* row = src + (lane_id() & 31) * ld;
  mma(out, frag_from_acc<T>(X, 0), ld_frag_perm(row, 0));
  mma(out, frag_from_acc<T>(X, 1), ld_frag_perm(row, 1));
}

// Compile-time K version of mma_tile (fully unrolled; lda / ldb are usually
// compile-time too, so the LDS offsets become immediates).
template <typename T, int K>
__device__ __forceinline__ void mma_k(floatx16& acc, const T* a, int lda, const T* b, int ldb) {
  const int lane = lane_id();
  const T* ap = a + (lane & 31) * lda + (lane >> 5) * 8;
  const T* bp = b + (lane & 31) * ldb + (lane >> 5) * 8;
#pragma unroll
  for (int k = 0; k < K / 16; ++k) mma(acc, ld_frag(ap + 16 * k), ld_frag(bp + 16 * k));
}

// The two A fragments of an accumulator tile (see frag_from_acc), converted once.
template <typename T> struct AccFrags { Frag<T> f[2]; };
template <typename T>
__device__ __forceinline__ AccFrags<T> acc_frags(const floatx16& x) {
  AccFrags<T> a;
  a.f[0] = frag_from_acc<T>(x, 0);
  a.f[1] = frag_from_acc<T>(x, 1);
  return a;
}
// out(32x32) += X^T B' with X given by its converted fragments, B'[a][j] = src[j*ld + a].
template <typename T>
__device__ __forceinline__ void mma_xt_f(floatx16& out, const AccFrags<T>& X, const T* src, int ld) {
  const T* row = src + (lane_id() & 31) * ld;
  mma(out, X.f[0], ld_frag_perm(row, 0));
  mma(out, X.f[1], ld_frag_perm(row, 1));
}

// The 16 per-register row values base[row(v)] of this lane (rows 8r + 4*(lane/32) + q),
// read as four 16-byte LDS loads (base 16-byte aligned).
__device__ __forceinline__ void rows16(const float* base, float (&o)[16]) {
  const float* p = base + 4 * (lane_id() >> 5);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const floatx4 v = *reinterpret_cast<const floatx4*>(p + 8 * r);
    o[4 * r + 0] = v[0]; o[4 * r + 1] = v[1]; o[4 * r + 2] = v[2]; o[4 * r + 3] = v[3];
  }
}

// One MFMA operand fragment (8 consecutive features k .. k+7 of row `row`)
// read straight from a row-major global tensor, zero outside the row range /
// feature width. vec_ok: 16-byte loads are aligned (see stage_nat).
template <typename T>
__device__ __forceinline__ Frag<T> frag_global(const T* __restrict__ src, int64_t ld, int64_t col0, int64_t row,
                                               bool row_ok, int k, int width, bool vec_ok) {
  Frag<T> f;
  const T* g = src + row * ld + col0 + k;
  if (vec_ok && row_ok && k + 8 <= width) {
    if constexpr (sizeof(T) == 2) {
      f.v = *reinterpret_cast<const bf16x8*>(g);
    } else {
      const floatx4 a = *reinterpret_cast<const floatx4*>(g);
      const floatx4 b = *reinterpret_cast<const floatx4*>(g + 4);
      f.v[0] = a[0]; f.v[1] = a[1]; f.v[2] = a[2]; f.v[3] = a[3];
      f.v[4] = b[0]; f.v[5] = b[1]; f.v[6] = b[2]; f.v[7] = b[3];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) f.v[e] = (row_ok && k + e < width) ? g[e] : from_f<T>(0.0f);
  }
  return f;
}

// Sum over the 32 columns of each row: after the call every lane holds, for
// each of its 16 registers, the full row sum (lanes of one 32-lane half agree).
__device__ __forceinline__ float row_reduce32(float v) {
  v += __shfl_xor(v, 1, 64);
  v += __shfl_xor(v, 2, 64);
  v += __shfl_xor(v, 4, 64);
  v += __shfl_xor(v, 8, 64);
  v += __shfl_xor(v, 16, 64);
  return v;
}

// Round x up to a multiple of m.
__host__ __device__ __forceinline__ int round_up(int x, int m) { return (x + m - 1) / m * m; }

// LDS row pitch (elements) for a k-contiguous tile of width w: +16 bytes so
// consecutive rows start in different banks.
template <typename T> __host__ __device__ constexpr int lds_pitch(int w) { return w + 16 / (int)sizeof(T); }

// ---------------------------------------------------------------------------
// Global -> LDS staging of a 64-row block of a row-major (rows, features)
// tensor: rows row0 + [r0, r0 + 64) (valid below `len`), features
// [col0, col0 + width) of a row of `ld` elements, zero-filled up to `wpad`.
// `vec_ok` (uniform) says 16-byte loads are aligned (width, ld, col0 multiples
// of 16/sizeof(T) and a 16-byte aligned base); otherwise scalar loads.
// ---------------------------------------------------------------------------
template <typename T> struct Vec16;
template <> struct Vec16<bf16> { typedef bf16x8 type; static constexpr int n = 8; };
template <> struct Vec16<float> { typedef floatx4 type; static constexpr int n = 4; };

// natural layout: out[r][k] (pitch elements per row)
template <typename T>
__device__ __forceinline__ void stage_nat(T* __restrict__ out, int pitch, const T* __restrict__ src, int64_t ld,
                                          int64_t col0, int64_t row0, int r0, int len, int width, int wpad,
                                          bool vec_ok) {
  constexpr int V = Vec16<T>::n;
  typedef typename Vec16<T>::type VT;
  const int per_row = wpad / V;
  const int total = SSD_BLK * per_row;
  for (int id = threadIdx.x; id < total; id += blockDim.x) {
    const int r = id / per_row, k = (id - r * per_row) * V;
    const bool rv = r0 + r < len;
    const T* g = src + (row0 + r0 + r) * ld + col0 + k;
    VT v;
    if (vec_ok) {
      if (rv && k < width) v = *reinterpret_cast<const VT*>(g);
      else for (int e = 0; e < V; ++e) v[e] = from_f<T>(0.0f);
    } else {
      for (int e = 0; e < V; ++e) v[e] = (rv && k + e < width) ? g[e] : from_f<T>(0.0f);
    }
    *reinterpret_cast<VT*>(out + r * pitch + k) = v;
  }
}

// transposed layout: out[k][r]; lanes of a wave take consecutive rows so the
// 2-byte LDS stores of one feature land in consecutive banks.
template <typename T>
__device__ __forceinline__ void stage_tr(T* __restrict__ out, int pitch, const T* __restrict__ src, int64_t ld,
                                         int64_t col0, int64_t row0, int r0, int len, int width, int wpad,
                                         bool vec_ok) {
  constexpr int V = Vec16<T>::n;
  typedef typename Vec16<T>::type VT;
  const int total = SSD_BLK * (wpad / V);
  for (int id = threadIdx.x; id < total; id += blockDim.x) {
    const int r = id & (SSD_BLK - 1), k = (id >> 6) * V;
    const bool rv = r0 + r < len;
    const T* g = src + (row0 + r0 + r) * ld + col0 + k;
    VT v;
    if (vec_ok) {
      if (rv && k < width) v = *reinterpret_cast<const VT*>(g);
      else for (int e = 0; e < V; ++e) v[e] = from_f<T>(0.0f);
    } else {
      for (int e = 0; e < V; ++e) v[e] = (rv && k + e < width) ? g[e] : from_f<T>(0.0f);
    }
    for (int e = 0; e < V; ++e) out[(k + e) * pitch + r] = v[e];
  }
}

// transposed layout with every row scaled by scale[r] (fp32) before rounding.
template <typename T>
__device__ __forceinline__ void stage_tr_scaled(T* __restrict__ out, int pitch, const T* __restrict__ src,
                                                int64_t ld, int64_t col0, int64_t row0, int r0, int len, int width,
                                                int wpad, bool vec_ok, const float* __restrict__ scale) {
  constexpr int V = Vec16<T>::n;
  typedef typename Vec16<T>::type VT;
  const int total = SSD_BLK * (wpad / V);
  for (int id = threadIdx.x; id < total; id += blockDim.x) {
    const int r = id & (SSD_BLK - 1), k = (id >> 6) * V;
    const bool rv = r0 + r < len;
    const T* g = src + (row0 + r0 + r) * ld + col0 + k;
    VT v;
    if (vec_ok) {
      if (rv && k < width) v = *reinterpret_cast<const VT*>(g);
      else for (int e = 0; e < V; ++e) v[e] = from_f<T>(0.0f);
    } else {
      for (int e = 0; e < V; ++e) v[e] = (rv && k + e < width) ? g[e] : from_f<T>(0.0f);
    }
    const float sc = rv ? scale[r] : 0.0f;
    for (int e = 0; e < V; ++e) out[(k + e) * pitch + r] = from_f<T>(to_f(v[e]) * sc);
  }
}

// ---------------------------------------------------------------------------
// Register-staged tiles: a 64-row x wpad (<= 128) block is loaded by the 256
// threads of a block into registers first (all loads in flight together), then
// written to LDS in natural and/or transposed layout. Element (r, k) of the
// tile belongs to vector id = r + 64 * (k / V) (TR mapping: the 64 lanes of a
// wave hold 64 consecutive rows, so transposed 2-byte stores hit consecutive
// banks) or id = r * (wpad / V) + k / V (row-major mapping: a wave reads whole
// rows, fully coalesced). Thread t owns ids t, t + 256, ...
// ---------------------------------------------------------------------------
template <typename T, int MAXW = 128> struct TileRegs {
  static constexpr int V = Vec16<T>::n;
  static constexpr int MAXQ = SSD_BLK * MAXW / V / 256;  // vectors per thread for wpad = MAXW
  typename Vec16<T>::type v[MAXQ];
};

template <typename T, bool TRMAP, int MAXW>
__device__ __forceinline__ void tile_load(TileRegs<T, MAXW>& t, const T* __restrict__ src, int64_t ld, int64_t col0,
                                          int64_t row0, int r0, int len, int width, int wpad, bool vec_ok) {
  constexpr int V = Vec16<T>::n;
  const int per_row = wpad / V, total = SSD_BLK * per_row;
#pragma unroll
  for (int q = 0; q < TileRegs<T, MAXW>::MAXQ; ++q) {
    const int id = threadIdx.x + q * 256;
    if (id < total) {
      const int r = TRMAP ? (id & (SSD_BLK - 1)) : id / per_row;
      const int k = TRMAP ? (id >> 6) * V : (id - r * per_row) * V;
      const bool rv = r0 + r < len;
      const T* g = src + (row0 + r0 + r) * ld + col0 + k;
      if (vec_ok) {
        if (rv && k < width) t.v[q] = *reinterpret_cast<const typename Vec16<T>::type*>(g);
        else for (int e = 0; e < V; ++e) t.v[q][e] = from_f<T>(0.0f);
      } else {
        for (int e = 0; e < V; ++e) t.v[q][e] = (rv && k + e < width) ? g[e] : from_f<T>(0.0f);
      }
    }
  }
}

template <typename T, bool TRMAP, int MAXW>
__device__ __forceinline__ void tile_store_nat(const TileRegs<T, MAXW>& t, T* __restrict__ out, int pitch, int wpad) {
  constexpr int V = Vec16<T>::n;
  const int per_row = wpad / V, total = SSD_BLK * per_row;
#pragma unroll
  for (int q = 0; q < TileRegs<T, MAXW>::MAXQ; ++q) {
    const int id = threadIdx.x + q * 256;
    if (id < total) {
      const int r = TRMAP ? (id & (SSD_BLK - 1)) : id / per_row;
      const int k = TRMAP ? (id >> 6) * V : (id - r * per_row) * V;
      *reinterpret_cast<typename Vec16<T>::type*>(out + r * pitch + k) = t.v[q];
    }
  }
}

// transposed: out[k][r]; rows scaled by scale[r] when scale != nullptr
template <typename T, int MAXW>
__device__ __forceinline__ void tile_store_tr(const TileRegs<T, MAXW>& t, T* __restrict__ out, int pitch, int wpad,
                                              const float* __restrict__ scale = nullptr) {
  constexpr int V = Vec16<T>::n;
  const int total = SSD_BLK * (wpad / V);
#pragma unroll
  for (int q = 0; q < TileRegs<T, MAXW>::MAXQ; ++q) {
    const int id = threadIdx.x + q * 256;
    if (id < total) {
      const int r = id & (SSD_BLK - 1), k = (id >> 6) * V;
      if (scale) {
        const float sc = scale[r];
        for (int e = 0; e < V; ++e) out[(k + e) * pitch + r] = from_f<T>(to_f(t.v[q][e]) * sc);
      } else {
        for (int e = 0; e < V; ++e) out[(k + e) * pitch + r] = t.v[q][e];
      }
    }
  }
}

// One entry of the chunk table: chunk k of sequence `seq` covers rows
// [row0, row0 + len) of the packed token axis; `first` marks k == 0.
// The chunk states' bf16 rounding residual hin - bf16(hin), kept as OCP fp8 e4m3 of
// SSD_LO_SCALE times the residual (clamped to the format's +-448): |residual| <= 2^-8 |hin|,
// so states up to 448 / 8 in magnitude keep the residual to about 2^-4 of itself (hi + lo to
// about 2^-12), and the residual of a larger state saturates to a partial correction.
#define SSD_LO_SCALE 2048.0f
#define SSD_LO_MAX 448.0f

// Byte offset, within one (chunk, head) tile of hin_lo, of the 8 residuals (n, p .. p + 7)
// (p % 8 == 0): the tile is stored in the row kernel's MFMA A-fragment order, fragment
// (32-wide n tile, 16-deep p step) after fragment, 64 lanes of 8 values each (lane = 32 (p / 8 % 2)
// + n % 32), so one fragment is a contiguous 512 bytes.
__host__ __device__ __forceinline__ int64_t hin_lo_off(int Ppad, int n, int p) {
  const int frag = (n >> 5) * (Ppad >> 4) + (p >> 4);
  return ((int64_t)frag * 64 + 32 * ((p >> 3) & 1) + (n & 31)) * 8;
}

typedef short ssd_short2 __attribute__((ext_vector_type(2)));
typedef __bf16 ssd_bf16x2 __attribute__((ext_vector_type(2)));
// Four scaled residuals of v0..v3 (fp32 states) as four e4m3 bytes (v0 in the low byte). The
// conversion divides by its scale operand (the decode, cvt_scalef32_pk_bf16_fp8, multiplies by it)
// and overflows to NaN, so the residual is clamped to the format's range first.
__device__ __forceinline__ unsigned lo_pack4(float v0, float v1, float v2, float v3) {
  constexpr float lim = SSD_LO_MAX / SSD_LO_SCALE;
  auto r = [](float v) { return fminf(fmaxf(v - (float)(bf16)v, -lim), lim); };
  constexpr float sc = 1.0f / SSD_LO_SCALE;
  ssd_short2 w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(ssd_short2{0, 0}, r(v0), r(v1), sc, false);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(w, r(v2), r(v3), sc, true);
  return __builtin_bit_cast(unsigned, w);
}
// Eight such bytes as a bf16 MFMA operand.
__device__ __forceinline__ bf16x8 lo_frag(uint2 u) {
  bf16x8 f;
  constexpr float sc = 1.0f / SSD_LO_SCALE;
  const ssd_bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.x, sc, false);
  const ssd_bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.x, sc, true);
  const ssd_bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.y, sc, false);
  const ssd_bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u.y, sc, true);
  f[0] = a[0]; f[1] = a[1]; f[2] = b[0]; f[3] = b[1]; f[4] = c[0]; f[5] = c[1]; f[6] = d[0]; f[7] = d[1];
  return f;
}

struct ChunkInfo {
  int32_t row0;
  int32_t len;
  int32_t seq;
  int32_t idx_in_seq;
};
