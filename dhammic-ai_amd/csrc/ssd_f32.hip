// fp32 kernels of the chunked SSD scan (gfx950): the chunk scan of the forward and the per-chunk work of
// the backward (r2/dhammic-ai/src/kernels/ssd_scan.py:330-533), with v_mfma_f32_32x32x2_f32 and exact
// per-element decays.
//
// The fp32 matrix rate (154 TFLOP/s measured, a sixteenth of bf16's) is what these shapes are bound by, so
// the products are arranged to be done once: S = C B^T per (chunk, group) in 32 x 32 tiles (k_f32_cb) that
// every head of the group reads, dS = dM L summed over a slice's heads and multiplied with B and C once per
// group (k_f32_row), where a kernel per (chunk, head) would redo both for each head. At B=2 L=2048 H=24
// P=64 N=128 chunk 256 that is 32 of 96 MFLOP per (chunk, head).
//
// Tiles. A 32 x 32 tile T in accumulator layout (lane: column c = lane % 32; register v: row
// acc_row(v, lane)) is, register by register, the A operand T^T of v_mfma_f32_32x32x2: lane half h of step v
// supplies k = acc_row(v, lane), so its B operand is row acc_row(v, lane) of a row-major tile, one 4-byte
// LDS read with the lanes along the columns (no bank conflicts, no transposed copy). S and dS are kept in
// memory as [tile][4 register quads][lane][4], whole 1 KB rows of lanes per access, in the orientation the
// reader needs:
//   F: lane = output token l, registers over source tokens s   (S of the scan: M x)
//   R: lane = s, registers over l                              (S of the backward, dS: M^T dy, dS^T C)
// Tile (lt, st), st <= lt, of a unit (chunk, group) is number lt (lt + 1) / 2 + st.
#include <algorithm>

#include "ssd_launch.h"
#include "ssd_stage.h"
#include "ssd_tile.h"

namespace {

__host__ __device__ constexpr int nsub_of(int nl) { return nl * (nl + 1) / 2; }
__device__ __forceinline__ int sub_of(int lt, int st) { return lt * (lt + 1) / 2 + st; }

__device__ __forceinline__ void mfma32(floatx16& acc, float a, float b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
}

__device__ __forceinline__ floatx16 ld_tile(const float* __restrict__ t, int lane) {
  floatx16 f;
  const float* p = t + lane * 4;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const floatx4 v = *reinterpret_cast<const floatx4*>(p + 256 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * q + e] = v[e];
  }
  return f;
}
__device__ __forceinline__ void st_tile(float* __restrict__ t, int lane, const floatx16& f) {
  float* p = t + lane * 4;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<floatx4*>(p + 256 * q) = floatx4{f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]};
}

// Sum in pairs: the rounding of four additions, not of sixteen (the decay gradient is a difference of such sums).
__device__ __forceinline__ float sum16(const float (&a)[16]) {
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = a[2 * i] + a[2 * i + 1];
#pragma unroll
  for (int w = 4; w > 0; w >>= 1)
#pragma unroll
    for (int i = 0; i < w; ++i) s[i] = s[2 * i] + s[2 * i + 1];
  return s[0];
}

// Rows [0, nrows) (valid below len) x [0, W) columns (valid below width) of a row-major tensor into LDS
// (pitch floats per row), zeros elsewhere. Masked buffer loads, eight pieces per thread in flight; ssd_stage.h has
// the addresses.
template <int W, bool VEC>
__device__ __forceinline__ void stage_rows_v(float* __restrict__ out, int pitch, const float* __restrict__ src,
                                             int64_t ld, int nrows, int len, int width) {
  constexpr int CPR = W / 4, NB = 8;
  static_assert(64 % CPR == 0, "a wave holds whole rows");
  const int total = nrows * CPR, nthr = blockDim.x;
  for (int id0 = threadIdx.x; id0 < total; id0 += NB * nthr) {
    floatx4 v[NB];
    const int w0 = __builtin_amdgcn_readfirstlane(id0);
    const int k = stage_col(id0, CPR), off = stage_off(id0, w0, CPR, ld);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int id = id0 + q * nthr;
      const bool ok = id < total && stage_row(id, CPR) < len;
      const __amdgpu_buffer_rsrc_t rs = buf_rsrc(src + stage_base(w0, q, nthr, CPR) * ld);
      if constexpr (VEC) {
        v[q] = __builtin_bit_cast(
            floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, ok && k < width ? off * 4 : SSD_BUF_SIZE, 0, 0));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q][e] = buf_ldf(rs, (off + e) * 4, ok && k + e < width);
      }
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int id = id0 + q * nthr;
      if (id < total) *reinterpret_cast<floatx4*>(out + stage_row(id, CPR) * pitch + k) = v[q];
    }
  }
}
// `vec` (uniform): 16-byte loads are valid. The branch stays outside the loads (around each of them it made
// every load wait for the one before).
template <int W>
__device__ __forceinline__ void stage_rows(float* __restrict__ out, int pitch, const float* __restrict__ src,
                                           int64_t ld, int nrows, int len, int width, bool vec) {
  if (vec) stage_rows_v<W, true>(out, pitch, src, ld, nrows, len, width);
  else stage_rows_v<W, false>(out, pitch, src, ld, nrows, len, width);
}

// Operand pieces f[i] = columns 16 (i0 + i) + 8 hh .. + 7 of the row at element offset `off` from the resource's
// base, zeros outside the row mask and the width; masked buffer loads, all in flight (branch as above).
template <int M>
__device__ __forceinline__ void row_frags(Frag<float> (&f)[M], __amdgpu_buffer_rsrc_t r, int off, bool ok, int k0,
                                          int width, bool vec) {
  if (vec) {
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int k = k0 + 16 * i + 4 * q;
        const floatx4 v = __builtin_bit_cast(
            floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, ok && k < width ? (off + k) * 4 : SSD_BUF_SIZE, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) f[i].v[4 * q + e] = v[e];
      }
  } else {
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) f[i].v[e] = buf_ldf(r, (off + k0 + 16 * i + e) * 4, ok && k0 + 16 * i + e < width);
  }
}

// cs, dt (1 without) and, with s_D, D of one (chunk, head) into LDS: every load issued before the first wait.
__device__ __forceinline__ void stage_scalars(const SsdDims& d, const ChunkInfo& ci, const float* __restrict__ cs,
                                              const float* __restrict__ dt, const float* __restrict__ Dv,
                                              const float* __restrict__ Dtok, int h, float* s_cs, float* s_dt,
                                              float* s_D) {
  const __amdgpu_buffer_rsrc_t rc = buf_rsrc(cs), rt = buf_rsrc(d.has_dt ? dt + (int64_t)ci.row0 * d.H : cs);
  const bool tok = d.trapz != 0;
  const __amdgpu_buffer_rsrc_t rD = buf_rsrc(tok ? Dtok + (int64_t)ci.row0 * d.H : (d.has_D ? Dv : cs));
  for (int l = threadIdx.x; l < d.Qpad; l += blockDim.x) {
    const bool in = l < ci.len;
    const float c = buf_ldf(rc, l * 4, true);
    const float t = buf_ldf(rt, (l * d.H + h) * 4, d.has_dt && in);
    const float D = s_D ? buf_ldf(rD, ((tok ? l * d.H : 0) + h) * 4, tok ? in : d.has_D) : 0.0f;
    s_cs[l] = c;
    s_dt[l] = (d.has_dt && in) ? t : 1.0f;
    if (s_D) s_D[l] = D;
  }
}

struct F32Args {
  const ChunkInfo* chunks;
  const float* cs;    // [MC][H][Qpad]
  const float* x;
  const float* dt;
  const float* Bm;
  const float* Cm;
  const float* Dv;
  const float* Dtok;  // trapezoidal mode: D per token
  const float* hin;   // [MC][H][Ppad][Npad]
  const float* dst;   // [MC][H][Ppad][Npad], gradient leaving each chunk
  const float* dy;
  float* cb;          // S tiles of the units of this launch
  int unit0;          // first unit (chunk * G + group) of this launch; cb and the dS tiles count from it
};

}  // namespace

// S tiles of one orientation, one wave per tile: K = N from global (each row piece is read by the tiles of
// its row or column only, out of L1 / L2). 36 tiles x 64 MFMA per unit at chunk 256, N = 128.
template <int NT, bool FWD>
__global__ void __launch_bounds__(256) k_f32_cb(SsdDims d, F32Args a) {
  const int nl = d.Qpad / 32, nsub = nsub_of(nl), nb = (nsub + 3) / 4;
  const int u = blockIdx.x / nb;
  const int sub = (blockIdx.x % nb) * 4 + (threadIdx.x >> 6);
  if (sub >= nsub) return;
  const int unit = a.unit0 + u, c = unit / d.G, g = unit % d.G;
  const ChunkInfo ci = a.chunks[c];
  int lt = 0;
  while ((lt + 1) * (lt + 2) / 2 <= sub) ++lt;
  const int st = sub - lt * (lt + 1) / 2;
  if (32 * lt >= ci.len) return;
  const int lane = lane_id(), hh = lane >> 5, l32 = lane & 31;
  const int64_t brow = (int64_t)d.G * d.N;
  const int lr = 32 * lt + l32, sr = 32 * st + l32;
  floatx16 acc;
  zero(acc);
  const __amdgpu_buffer_rsrc_t rc = buf_rsrc(a.Cm + (int64_t)(ci.row0 + 32 * lt) * brow + (int64_t)g * d.N);
  const __amdgpu_buffer_rsrc_t rb = buf_rsrc(a.Bm + (int64_t)(ci.row0 + 32 * st) * brow + (int64_t)g * d.N);
  Frag<float> fc[2 * NT], fb[2 * NT];  // every operand in flight at once
  row_frags(fc, rc, l32 * (int)brow, lr < ci.len, 8 * hh, d.N, d.vec_bc);
  row_frags(fb, rb, l32 * (int)brow, sr < ci.len, 8 * hh, d.N, d.vec_bc);
#pragma unroll
  for (int k = 0; k < 2 * NT; ++k) {
    if (FWD) mma(acc, fb[k], fc[k]);  // rows s, columns l
    else mma(acc, fc[k], fb[k]);      // rows l, columns s
  }
  st_tile(a.cb + ((int64_t)u * nsub + sub) * 1024, lane, acc);
}

// ---------------------------------------------------------------------------
// Forward chunk scan, Y = M x + exp(cs) C h_in^T (+ D x): block (unit, head, 32 PT columns of P); wave w has
// the row tiles w and nl - 1 - w, whose 32 x 32 source tiles number nl + 1 together, so the waves of a block
// are even. x sits in LDS (70 KB at chunk 256, PT = 2: two blocks per CU); M is built in registers from the S tile
// (ready one tile ahead) and is the A operand as it is. In small batches (launch_f32_scan) a wave has one row tile
// and PT = 1; the two waves of a SIMD then share nl + 1 source tiles.
// ---------------------------------------------------------------------------
template <int PT, int NT, bool SELF>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_f32_scan(SsdDims d, F32Args a, float* __restrict__ y, int nph) {
  constexpr int PP = 32 * PT, XP = PP + 4;
  extern __shared__ __align__(16) unsigned char smem[];
  const int Qpad = d.Qpad, nl = Qpad / 32, nsub = nsub_of(nl);
  const int ph = blockIdx.x % nph, hk = blockIdx.x / nph % d.hpg, u = blockIdx.x / nph / d.hpg;
  const int unit = a.unit0 + u, c = unit / d.G, g = unit % d.G, h = g * d.hpg + hk;
  const ChunkInfo ci = a.chunks[c];
  if (ci.len == 0) return;
  const int p0 = ph * PP, pw = min(d.P - p0, PP);
  float* s_cs = reinterpret_cast<float*>(smem);  // [Qpad]
  float* s_dt = s_cs + Qpad;                     // [Qpad]
  float* xs = s_dt + Qpad;                       // [Qpad][XP]
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const float* csc = a.cs + ((int64_t)c * d.H + h) * Qpad;
  const int lane = lane_id(), hh = lane >> 5, l32 = lane & 31, w = threadIdx.x >> 6;
  const int nlv = (ci.len + 31) / 32;
  // tiles ta < tb; with a wave for every tile (two waves of a SIMD: 4 apart) the first alone
  const bool single = (int)blockDim.x == 64 * nl;
  const int ta = single && w >= 4 ? nl + 3 - w : w, tb = nl - 1 - w;
  const bool two = !single && tb < nlv;
  const int la = 32 * ta + l32, lb = 32 * tb + l32;
  const float Dh = d.has_D ? a.Dv[h] : 0.0f;
  // The operands of the state term's first 16 columns (SELF: of all, and C's again for S, whose first B rows come with
  // them) in flight through the staging
  constexpr int KC = SELF ? 2 * NT : 1;
  const float* hrow = a.hin + (((int64_t)c * d.H + h) * d.Ppad + p0 + l32) * d.Npad + 8 * hh;
  const __amdgpu_buffer_rsrc_t ra = buf_rsrc(a.Cm + (int64_t)(ci.row0 + 32 * ta) * brow + (int64_t)g * d.N);
  const __amdgpu_buffer_rsrc_t rb = buf_rsrc(a.Cm + (int64_t)(ci.row0 + (two ? 32 * tb : 0)) * brow + (int64_t)g * d.N);
  Frag<float> ca[KC], cb[KC], fh[KC][PT], fb[KC];
  auto load = [&](int k) {
    row_frags(ca, ra, l32 * (int)brow, la < ci.len, k + 8 * hh, d.N, d.vec_bc);
    row_frags(cb, rb, l32 * (int)brow, two && lb < ci.len, k + 8 * hh, d.N, d.vec_bc);
#pragma unroll
    for (int i = 0; i < KC; ++i)
#pragma unroll
      for (int t = 0; t < PT; ++t) fh[i][t] = ld_frag(hrow + (int64_t)(32 * t) * d.Npad + k + 16 * i);
  };
  auto load_B = [&](int st) {
    const __amdgpu_buffer_rsrc_t r = buf_rsrc(a.Bm + (int64_t)(ci.row0 + 32 * st) * brow + (int64_t)g * d.N);
    row_frags(fb, r, l32 * (int)brow, 32 * st + l32 < ci.len, 8 * hh, d.N, d.vec_bc);
  };
  load(0);
  if constexpr (SELF) load_B(0);
  stage_scalars(d, ci, csc, a.dt, nullptr, nullptr, h, s_cs, s_dt, nullptr);
  stage_rows<PP>(xs, XP, a.x + (int64_t)ci.row0 * xrow + (int64_t)h * d.P + p0, xrow, Qpad, ci.len, pw, d.vec_x);
  __syncthreads();
  if (ta >= nlv) return;
  floatx16 acc[2][PT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int t = 0; t < PT; ++t) zero(acc[q][t]);
  if constexpr (SELF) {
#pragma unroll
    for (int k = 0; k < KC; ++k)
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        mma(acc[0][t], ca[k], fh[k][t]);
        if (two) mma(acc[1][t], cb[k], fh[k][t]);
      }
  } else {
    // operands of the next 16 columns in flight while these are multiplied
#pragma unroll
    for (int k = 0; k < 32 * NT; k += 16) {
      const Frag<float> ca0 = ca[0], cb0 = cb[0];
      Frag<float> fh0[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) fh0[t] = fh[0][t];
      if (k + 16 < 32 * NT) load(k + 16);
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        mma(acc[0][t], ca0, fh0[t]);
        if (two) mma(acc[1][t], cb0, fh0[t]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float rc[16];
    rows16(s_cs + 32 * (q ? tb : ta), rc);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float e = exp_clamp(rc[v]);
#pragma unroll
      for (int t = 0; t < PT; ++t) acc[q][t][v] *= e;
    }
  }
  const float* cbu = a.cb + (int64_t)u * nsub * 1024;
  const float cs_a = s_cs[la], cs_b = s_cs[lb];
  const int strict = d.trapz ? 1 : 0;  // trapezoidal mode: strictly causal
  const int last = two ? tb : ta;
  // S of the next source tile, ahead of its use: from memory, or (SELF) multiplied here, the B rows of the tile after
  // it in flight
  floatx16 Sa, Sb;
  auto load_S = [&](int st, floatx16& A, floatx16& Bt) {
    if constexpr (SELF) {
      zero(A);
      zero(Bt);
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        if (st <= ta) mma(A, fb[k], ca[k]);
        if (two) mma(Bt, fb[k], cb[k]);
      }
      if (st < last) load_B(st + 1);
    } else {
      if (st <= ta) A = ld_tile(cbu + (int64_t)sub_of(ta, st) * 1024, lane);
      if (two) Bt = ld_tile(cbu + (int64_t)sub_of(tb, st) * 1024, lane);
    }
  };
  load_S(0, Sa, Sb);
  for (int st = 0; st <= last; ++st) {
    floatx16 Na, Nb;
    if (!SELF && st < last) load_S(st + 1, Na, Nb);
    float css[16], dts[16];
    rows16(s_cs + 32 * st, css);
    rows16(s_dt + 32 * st, dts);
    float xv[PT][16];
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) xv[t][v] = xs[(32 * st + acc_row(v, lane)) * XP + 32 * t + l32];
    if (two) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float m = Sb[v] * exp_clamp(cs_b - css[v]) * dts[v];
        Sb[v] = (st < tb || acc_row(v, lane) + strict <= l32) ? m : 0.0f;
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int t = 0; t < PT; ++t) mfma32(acc[1][t], Sb[v], xv[t][v]);
    }
    if (st <= ta) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float m = Sa[v] * exp_clamp(cs_a - css[v]) * dts[v];
        Sa[v] = (st < ta || acc_row(v, lane) + strict <= l32) ? m : 0.0f;
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int t = 0; t < PT; ++t) mfma32(acc[0][t], Sa[v], xv[t][v]);
    }
    if constexpr (SELF) {
      if (st < last) load_S(st + 1, Sa, Sb);
    } else {
      Sa = Na;
      Sb = Nb;
    }
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    if (q == 1 && !two) continue;
    const int l0 = 32 * (q ? tb : ta);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int l = l0 + acc_row(v, lane);
      if (l >= ci.len) continue;
      const float Dl = d.trapz ? a.Dtok[(int64_t)(ci.row0 + l) * d.H + h] : Dh;
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        const int p = 32 * t + l32;
        if (p >= pw) continue;
        float yv = acc[q][t][v];
        if (d.has_D || d.trapz) yv += Dl * xs[l * XP + p];
        y[(int64_t)(ci.row0 + l) * xrow + (int64_t)h * d.P + p0 + p] = yv;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Chunk states (fp32), out[c][h][p][n] = sum_l U[l][p] coef_l V[l][n] as k_chunk_state: both operands are
// row-major with the contraction along the rows, so every MFMA operand is one coalesced 4-byte load per lane
// and nothing goes through LDS but the coefficients. One wave per 32 x 32 tile of the state.
// ---------------------------------------------------------------------------
// STEP: tokens a step.
template <int MODE, int STEP>
__global__ void __launch_bounds__(512) k_f32_state(SsdDims d, F32Args a, const float* __restrict__ U,
                                                   const float* __restrict__ V, float* __restrict__ out) {
  constexpr int NL = STEP / 2;  // loads per lane and operand
  __shared__ float coef[256];
  const int c = blockIdx.x, h = blockIdx.y, g = h / d.hpg;
  const ChunkInfo ci = a.chunks[c];
  if (ci.len == 0) return;
  const int lane = lane_id(), hh = lane >> 5, l32 = lane & 31, w = threadIdx.x >> 6;  // one wave per tile
  const int ntn = d.Npad / 32, pt = w / ntn, n0 = w % ntn * 32, p = 32 * pt + l32, n = n0 + l32;
  const int64_t urow = (int64_t)d.H * d.P, vrow = (int64_t)d.G * d.N;
  // a step's operands one step ahead; masked buffer loads (no branches) from bases at the step's first row
  float uv[NL], vv[NL];
  auto load = [&](int l0) {
    const __amdgpu_buffer_rsrc_t ru = buf_rsrc(U + (int64_t)(ci.row0 + l0) * urow + (int64_t)h * d.P);
    const __amdgpu_buffer_rsrc_t rv = buf_rsrc(V + (int64_t)(ci.row0 + l0) * vrow + (int64_t)g * d.N);
#pragma unroll
    for (int t = 0; t < NL; ++t) {
      const int l = 2 * t + hh;
      const bool ok = l0 + l < ci.len;
      uv[t] = buf_ldf(ru, (l * (int)urow + p) * 4, ok && p < d.P);
      vv[t] = buf_ldf(rv, (l * (int)vrow + n) * 4, ok && n < d.N);
    }
  };
  load(0);
  const float* csc = a.cs + ((int64_t)c * d.H + h) * d.Qpad;
  const float cs_last = csc[d.Qpad - 1];
  for (int l = threadIdx.x; l < d.Qpad; l += blockDim.x) {
    float v = 0.0f;
    if (l < ci.len) {
      if (MODE == 0)
        v = exp_clamp(cs_last - csc[l]) * (d.has_dt ? a.dt[(int64_t)(ci.row0 + l) * d.H + h] : 1.0f);
      else
        v = exp_clamp(csc[l]);
    }
    coef[l] = v;
  }
  __syncthreads();
  floatx16 acc;
  zero(acc);
  for (int l0 = 0; l0 < ci.len; l0 += STEP) {
    float ua[NL], va[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
      ua[t] = uv[t];
      va[t] = vv[t] * coef[l0 + 2 * t + hh];  // (0 past the chunk; Qpad is a multiple of 64)
    }
    if (l0 + STEP < ci.len) load(l0 + STEP);
#pragma unroll
    for (int t = 0; t < NL; ++t) mfma32(acc, ua[t], va[t]);
  }
  float* o = out + ((int64_t)c * d.H + h) * d.Ppad * d.Npad;
#pragma unroll
  for (int v = 0; v < 16; ++v) o[(int64_t)(32 * pt + acc_row(v, lane)) * d.Npad + n] = acc[v];
}

// ---------------------------------------------------------------------------
// Backward, column side: block (unit, head slice), wave st has the source tokens of tile st and walks the
// output tiles lt >= st; the dy rows of a head sit in LDS for all waves. Per tile: P = dy x^T, G, M and
// dS in registers (layout R), dX += M^T dy with M as the A operand, dS to memory (added over the slice's
// heads). At 192 tokens and more a unit is two blocks, tiles {0, 1, nl - 2, nl - 1} and the others (18 of the
// 36 tiles each at chunk 256): with the dy rows 80 KB of LDS, so two blocks per CU, one staging while the other
// computes. Per head: dx, the sums of G over either index, E, x.dX and the D partial.
// ---------------------------------------------------------------------------
template <int PT, int NT, bool SELF>
__global__ void __launch_bounds__(256, 2) k_f32_col(SsdDims d, SsdBufs bf, F32Args a, float* __restrict__ dx, int hslice,
                                                 int nslices, float* __restrict__ dS, int64_t slice_stride) {
  constexpr int PP = 32 * PT, YP = PP + 4;
  extern __shared__ __align__(16) unsigned char smem[];
  const int Qpad = d.Qpad, nl = Qpad / 32, nsub = nsub_of(nl);
  const int nhalf = nl >= 6 ? 2 : 1, half = blockIdx.x % nhalf;
  const int slc = blockIdx.x / nhalf % nslices, u = blockIdx.x / nhalf / nslices;
  const int unit = a.unit0 + u, c = unit / d.G, g = unit % d.G;
  const ChunkInfo ci = a.chunks[c];
  if (ci.len == 0) return;
  const int h_lo = g * d.hpg + slc * hslice, h_hi = min(h_lo + hslice, (g + 1) * d.hpg);
  float* s_cs = reinterpret_cast<float*>(smem);  // [Qpad]
  float* s_dt = s_cs + Qpad;                     // [Qpad]
  float* s_D = s_dt + Qpad;                      // [Qpad] D at each token
  float* s_dD = s_D + Qpad;                      // [16]
  float* rowp = s_dD + 16;                       // [nl][Qpad]
  float* dys = rowp + nl * Qpad;                 // [Qpad][YP]
  int lane = lane_id(), hh = lane >> 5, l32 = lane & 31;
  // (per-lane offsets are recomputed from an opaque lane id where a phase starts: held across the head loop
  // they spill)
  auto relane = [&]() {
    lane = opaque_lane();
    hh = lane >> 5;
    l32 = lane & 31;
  };
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int st = nhalf == 1 ? w : (half ? 2 + w : (w < 2 ? w : nl - 4 + w));
  const int nlv = (ci.len + 31) / 32;
  const int nw = half ? nl - 4 : (int)(blockDim.x >> 6);  // waves with a tile
  const bool live = w < nw && st < nlv;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const int strict = d.trapz ? 1 : 0;
  const float* cbu = a.cb + (int64_t)u * nsub * 1024;
  float* dSu = dS + (int64_t)slc * slice_stride + (int64_t)u * nsub * 1024;
  for (int h = h_lo; h < h_hi; ++h) {
    __syncthreads();  // the previous head's LDS reads are done
    relane();
    const int s_me = 32 * st + l32;
    const float* csc = a.cs + ((int64_t)c * d.H + h) * Qpad;
    const int64_t xo = (int64_t)ci.row0 * xrow + (int64_t)h * d.P;
    // x rows of this wave's tile (base at its first row, so that offsets stay below 2 GiB)
    const int st_row = live ? 32 * st : 0;
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.x + xo + (int64_t)st_row * xrow);
    constexpr bool HOLD = PT <= 2;  // x operand held over the tiles (P = 128: re-read per tile)
    Frag<float> xf[HOLD ? PP / 16 : 1];
    if (HOLD) row_frags(xf, rx, l32 * (int)xrow, live && s_me < ci.len, 8 * hh, d.P, d.vec_x);
    stage_scalars(d, ci, csc, a.dt, a.Dv, a.Dtok, h, s_cs, s_dt, s_D);
    stage_rows<PP>(dys, YP, a.dy + xo, xrow, Qpad, ci.len, d.P, d.vec_x);
    __syncthreads();
    const int64_t hq = ((int64_t)c * d.H + h) * Qpad;
    if (live) {
      floatx16 dX[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) zero(dX[t]);
      const float cs_s = s_cs[s_me], dt_s = s_dt[s_me];
      float gcol = 0.0f;
      floatx16 S;
      // (AHEAD: the C rows of the tile after the next are in flight; with PT = 4 they would spill)
      constexpr bool AHEAD = SELF && PT <= 2;
      Frag<float> bs[SELF ? 2 * NT : 1], fc[SELF ? 2 * NT : 1];
      auto load_C = [&](int lt) {
        row_frags(fc, buf_rsrc(a.Cm + (int64_t)(ci.row0 + 32 * lt) * brow + (int64_t)g * d.N), l32 * (int)brow,
                  32 * lt + l32 < ci.len, 8 * hh, d.N, d.vec_bc);
      };
      if constexpr (SELF)
        row_frags(bs, buf_rsrc(a.Bm + (int64_t)(ci.row0 + st_row) * brow + (int64_t)g * d.N), l32 * (int)brow,
                  s_me < ci.len, 8 * hh, d.N, d.vec_bc);
      if constexpr (AHEAD) load_C(st);
      auto load_S = [&](int lt, floatx16& o) {
        if constexpr (SELF) {
          if constexpr (!AHEAD) load_C(lt);
          zero(o);
#pragma unroll
          for (int k = 0; k < 2 * NT; ++k) mma(o, fc[k], bs[k]);
          if (AHEAD && lt + 1 < nlv) load_C(lt + 1);
        } else {
          o = ld_tile(cbu + (int64_t)sub_of(lt, st) * 1024, lane);
        }
      };
      load_S(st, S);
      for (int lt = st; lt < nlv; ++lt) {
        floatx16 nS;
        const int64_t so = (int64_t)sub_of(lt, st) * 1024;
        if (!AHEAD && lt + 1 < nlv) load_S(lt + 1, nS);
        Frag<float> yf[PP / 16];
#pragma unroll
        for (int k = 0; k < PP / 16; ++k) yf[k] = ld_frag(dys + (32 * lt + l32) * YP + 16 * k + 8 * hh);
        floatx16 P;
        zero(P);
        int xoff = l32 * (int)xrow;
        asm volatile("" : "+v"(xoff));
#pragma unroll
        for (int k = 0; k < PP / 16; ++k) {
          Frag<float> xr[1];
          if (!HOLD) row_frags(xr, rx, xoff, s_me < ci.len, 16 * k + 8 * hh, d.P, d.vec_x);
          mma(P, yf[k], HOLD ? xf[HOLD ? k : 0] : xr[0]);
        }
        float csl[16], G[16];
        rows16(s_cs + 32 * lt, csl);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const bool ok = lt > st || l32 + strict <= acc_row(v, lane);
          const float dd = csl[v] - cs_s;
          const float L = ok ? exp_clamp(dd) : 0.0f;
          const float m = S[v] * L, dm = P[v] * dt_s;
          G[v] = dm * m * clamp_pass(dd);
          S[v] = m;
          P[v] = dm * L;
        }
        // (rows past the chunk's length have dy = 0; their S tile rows are zero as well)
        gcol += sum16(G);
        const float rs = half_reduce16(G, lane);
        if (!(lane & 1)) rowp[st * Qpad + 32 * lt + acc_row((l32 >> 1) & 15, lane)] = rs;
        if (h > h_lo) {
          const floatx16 old = ld_tile(dSu + so, lane);
#pragma unroll
          for (int v = 0; v < 16; ++v) P[v] += old[v];
        }
        st_tile(dSu + so, lane, P);
        __builtin_amdgcn_sched_barrier(0);  // (its LDS operands are not read ahead of the tile's own work)
        float yv[2][16];
        auto ldy = [&](int t) {
#pragma unroll
          for (int v = 0; v < 16; ++v) yv[t & 1][v] = dys[(32 * lt + acc_row(v, lane)) * YP + 32 * t + l32];
        };
        ldy(0);
#pragma unroll
        for (int t = 0; t < PT; ++t) {
          if (t + 1 < PT) ldy(t + 1);
#pragma unroll
          for (int v = 0; v < 16; ++v) mfma32(dX[t], S[v], yv[t & 1][v]);
        }
        if constexpr (AHEAD) {
          if (lt + 1 < nlv) load_S(lt + 1, S);
        } else {
          S = nS;
        }
      }
      gcol = add_xor32(gcol);
      if (hh == 0 && s_me < ci.len) bf.colG[hq + s_me] = gcol;
      __builtin_amdgcn_sched_barrier(0);
      relane();
      // state term B_s dst^T (K = N)
      floatx16 tmp[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) zero(tmp[t]);
      const float* dsth = a.dst + ((int64_t)c * d.H + h) * PP * d.Npad;
      const __amdgpu_buffer_rsrc_t rb = buf_rsrc(a.Bm + (int64_t)(ci.row0 + st_row) * brow + (int64_t)g * d.N);
      Frag<float> fb[1], fd[PT];
      auto load = [&](int k) {
        row_frags(fb, rb, l32 * (int)brow, s_me < ci.len, k + 8 * hh, d.N, d.vec_bc);
#pragma unroll
        for (int t = 0; t < PT; ++t) fd[t] = ld_frag(dsth + (int64_t)(32 * t + l32) * d.Npad + k + 8 * hh);
      };
      load(0);
#pragma unroll
      for (int k = 0; k < 32 * NT; k += 16) {
        const Frag<float> fb0 = fb[0];
        Frag<float> fd0[PT];
#pragma unroll
        for (int t = 0; t < PT; ++t) fd0[t] = fd[t];
        if (k + 16 < 32 * NT) load(k + 16);
#pragma unroll
        for (int t = 0; t < PT; ++t) mma(tmp[t], fb0, fd0[t]);
        __builtin_amdgcn_sched_barrier(0);
      }
      relane();
      const float cs_last = s_cs[Qpad - 1];
      float e[16], xs[16], dpart = 0.0f, d4 = 0.0f;  // (d4: of four rows)
      const __amdgpu_buffer_rsrc_t rdx = buf_rsrc(dx + xo + (int64_t)st_row * xrow);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int sl = acc_row(v, lane), s = 32 * st + sl;
        const bool in = s < ci.len;
        const float dl = cs_last - s_cs[s];
        const float ws = in ? exp_clamp(dl) : 0.0f, dts = s_dt[s];
        const float Dl = s_D[s];
        float ev = 0.0f, xv = 0.0f;
#pragma unroll
        for (int t = 0; t < PT; ++t) {
          const int p = 32 * t + l32;
          const bool ok = in && p < d.P;
          const int o = (sl * (int)xrow + p) * 4;
          const float xx = buf_ldf(rx, o, ok), yy = dys[s * YP + p];
          const float tx = tmp[t][v] * ws, dXv = dX[t][v] + tx;
          ev += xx * tx;
          xv += xx * dXv;
          d4 += xx * yy;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dts * dXv + Dl * yy), rdx, ok ? o : SSD_BUF_SIZE, 0, 0);
        }
        e[v] = ev * dts * clamp_pass(dl);
        xs[v] = xv;
        if ((v & 3) == 3) {
          dpart += d4;
          d4 = 0.0f;
          __builtin_amdgcn_sched_barrier(0);  // four rows' x loads in flight at a time
        }
      }
      const float er = half_reduce16(e, lane), xr = half_reduce16(xs, lane);
      const int s = 32 * st + acc_row((l32 >> 1) & 15, lane);
      if (!(lane & 1) && s < ci.len) {
        bf.eterm[hq + s] = er;
        bf.xdx[hq + s] = xr;
      }
      dpart = wave_sum(dpart);
      if (lane == 0) s_dD[st] = dpart;
    } else if (lane == 0 && w < nw) {
      s_dD[st] = 0.0f;
    }
    __syncthreads();
    // the second half's tiles start at token 64, where the finish kernel starts to add its partial
    float* rowG = bf.rowG + (int64_t)half * d.max_chunks * d.H * Qpad + hq;
    for (int l = 64 * half + threadIdx.x; l < ci.len; l += blockDim.x) {
      float r = 0.0f;
      for (int q = 0; q < nw; ++q) {
        const int sq = nhalf == 1 ? q : (half ? 2 + q : (q < 2 ? q : nl - 4 + q));
        if (sq <= l / 32) r += rowp[sq * Qpad + l];
      }
      rowG[l] = r;
    }
    if (lane == 0 && w < nw && !(st & 1))
      bf.dD_part[((int64_t)c * d.H + h) * (Qpad / 64) + st / 2] = s_dD[st] + s_dD[st + 1];
  }
}

// dS of a batch of units summed over the head slices, into slice 0.
__global__ void __launch_bounds__(256) k_f32_ds(SsdDims d, const ChunkInfo* __restrict__ chunks, int unit0,
                                                float* __restrict__ dS, int64_t slice_stride, int nslices) {
  const int nl = d.Qpad / 32, nsub = nsub_of(nl), nb = (nsub + 3) / 4;
  const int u = blockIdx.x / nb, w = threadIdx.x >> 6, lane = lane_id();
  const int sub = (blockIdx.x % nb) * 4 + w;
  int lt = 0;
  while ((lt + 1) * (lt + 2) / 2 <= sub) ++lt;
  if (sub >= nsub || 32 * lt >= chunks[(unit0 + u) / d.G].len) return;
  float* o = dS + ((int64_t)u * nsub + sub) * 1024;
  floatx16 f = ld_tile(o, lane);
  for (int k = 1; k < nslices; ++k) {
    const floatx16 q = ld_tile(o + k * slice_stride, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) f[v] += q[v];
  }
  st_tile(o, lane, f);
}

// ---------------------------------------------------------------------------
// Backward, row side: dC (role 0) and dB (role 1). Block (unit, role, four row tiles, slice), wave = one
// 32-row tile over 64 columns of N (all 128 in one wave took 256 registers and spilled: 150 us against
// 61 at B=2 L=2048 H=24 P=64 N=128). Slices 0 .. nhs - 1 take the state terms of their heads
// (dC += exp(cs) dy h_in, whose product with C is the decay gradient's Y_off term; dB += w dt x dst), with the
// head's state in LDS; the tile term (dS B, dS^T C) is one more slice, or the same block's when there is one
// head slice.
// ---------------------------------------------------------------------------
template <int PT, int NT>
__global__ void __launch_bounds__(NT > 2 ? 512 : 256, NT > 2 ? 2 : 1)
k_f32_row(SsdDims d, SsdBufs bf, F32Args a, const float* __restrict__ dS, float* __restrict__ dB, float* __restrict__ dC,
          int hslice, int nhs, int nsl) {
  constexpr int PP = 32 * PT, NP = 32 * NT;
  constexpr int NH = NT > 2 ? 2 : 1, TN = NT / NH, THR = 256 * NH;  // column halves, n tiles per wave
  extern __shared__ __align__(16) unsigned char smem[];
  float* hs = reinterpret_cast<float*>(smem);  // [PP][NP]
  float* s_off = hs + PP * NP;                 // [NH][128] the head's Y_off sums
  const int Qpad = d.Qpad, nl = Qpad / 32, nsub = nsub_of(nl), nbq = (nl + 3) / 4;
  int b = blockIdx.x;
  const int slc = b % nsl;
  b /= nsl;
  const int bq = b % nbq;
  b /= nbq;
  const int role = b & 1, u = b >> 1, unit = a.unit0 + u, c = unit / d.G, g = unit % d.G;
  const ChunkInfo ci = a.chunks[c];
  if (128 * bq >= ci.len) return;
  const int lane = lane_id(), hh = lane >> 5, l32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rw = w & 3, n0 = 32 * TN * (w >> 2);
  const int rt = 4 * bq + rw;
  const int nlv = (ci.len + 31) / 32;
  const bool live = rt < nlv;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const int r_me = 32 * rt + l32;
  const bool r_ok = live && r_me < ci.len;
  const int rt_row = live ? 32 * rt : 0;
  floatx16 acc[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) zero(acc[t]);
  const int h_lo = g * d.hpg + slc * hslice, h_hi = slc < nhs ? min(h_lo + hslice, (g + 1) * d.hpg) : h_lo;
  const __amdgpu_buffer_rsrc_t rc = buf_rsrc(a.Cm + (int64_t)(ci.row0 + rt_row) * brow + (int64_t)g * d.N);
  auto flush = [&](int h) {  // head h's dcs_off, after a barrier
    const int l = 128 * bq + threadIdx.x;
    if (role || threadIdx.x >= 128 || l >= ci.len) return;
    float o = s_off[threadIdx.x];
    if (NH > 1) o += s_off[128 + threadIdx.x];
    const int64_t q = ((int64_t)c * d.H + h) * Qpad + l;
    bf.dcs_off[q] = o * clamp_pass(a.cs[q]);
  };
  for (int h = h_lo; h < h_hi; ++h) {
    const int64_t ch = (int64_t)c * d.H + h;
    const float* src = (role ? a.dst : a.hin) + ch * PP * d.Npad;
    constexpr int NV = PP * NP / 4 / THR;  // 16-byte pieces per thread
    floatx4 pc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) pc[q] = *reinterpret_cast<const floatx4*>(src + 4 * (threadIdx.x + THR * q));
    const __amdgpu_buffer_rsrc_t rr =
        buf_rsrc((role ? a.x : a.dy) + (int64_t)(ci.row0 + rt_row) * xrow + (int64_t)h * d.P);
    Frag<float> fr[PP / 16];
    row_frags(fr, rr, l32 * (int)xrow, r_ok, 8 * hh, d.P, d.vec_x);
    const __amdgpu_buffer_rsrc_t rcs = buf_rsrc(a.cs + ch * Qpad);
    const __amdgpu_buffer_rsrc_t rdt = buf_rsrc(d.has_dt ? a.dt + (int64_t)(ci.row0 + rt_row) * d.H + h : a.cs);
    const float cs_r = buf_ldf(rcs, r_me * 4, r_ok), cs_last = buf_ldf(rcs, (Qpad - 1) * 4, true);
    const float dt_r = buf_ldf(rdt, l32 * d.H * 4, r_ok && d.has_dt);
    __syncthreads();  // the previous head's reads are done, its Y_off sums are written
    if (h > h_lo) flush(h - 1);
#pragma unroll
    for (int q = 0; q < NV; ++q) *reinterpret_cast<floatx4*>(hs + 4 * (threadIdx.x + THR * q)) = pc[q];
    float f = 0.0f;
    if (r_ok) f = role ? exp_clamp(cs_last - cs_r) * (d.has_dt ? dt_r : 1.0f) : exp_clamp(cs_r);
#pragma unroll
    for (int k = 0; k < PP / 16; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) fr[k].v[e] *= f;
    __syncthreads();
    if (role) {
#pragma unroll
      for (int k = 0; k < PP / 16; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int t = 0; t < TN; ++t)
            mfma32(acc[t], fr[k].v[e], hs[(16 * k + 8 * hh + e) * NP + n0 + 32 * t + l32]);
    } else {
      float off[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) off[v] = 0.0f;
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const int n = n0 + 32 * t + l32;
        float cv[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int ll = acc_row(v, lane);
          cv[v] = buf_ldf(rc, (ll * (int)brow + n) * 4, live && 32 * rt + ll < ci.len && n < d.N);
        }
        floatx16 tmp;
        zero(tmp);
#pragma unroll
        for (int k = 0; k < PP / 16; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            mfma32(tmp, fr[k].v[e], hs[(16 * k + 8 * hh + e) * NP + n0 + 32 * t + l32]);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          off[v] += tmp[v] * cv[v];
          acc[t][v] += tmp[v];
        }
      }
      const float o = half_reduce16(off, lane);
      if (!(lane & 1)) s_off[128 * (w >> 2) + 32 * rw + acc_row((l32 >> 1) & 15, lane)] = o;
    }
  }
  if (h_hi > h_lo) {
    __syncthreads();
    flush(h_hi - 1);
  }
  if (!live) return;
  if (slc == nsl - 1) {  // the tile term
    const float* T = dS + (int64_t)u * nsub * 1024;
    const float* M = role ? a.Cm : a.Bm;
    const int q0 = role ? rt : 0, q1 = role ? nlv - 1 : rt;
    floatx16 A;
    float m[TN][16];
    auto load = [&](int q) {
      if (role) {
        A = ld_tile(T + (int64_t)sub_of(q, rt) * 1024, lane);
      } else {  // the other orientation: lane = row l of the tile, register = s (sixteen 16-byte runs per access)
        const float* t = T + (int64_t)sub_of(rt, q) * 1024 + (l32 >> 3) * 256 + (l32 & 4) * 32 + (l32 & 3);
#pragma unroll
        for (int v = 0; v < 16; ++v) A[v] = t[4 * acc_row(v, lane)];
      }
      const __amdgpu_buffer_rsrc_t rm = buf_rsrc(M + (int64_t)(ci.row0 + 32 * q) * brow + (int64_t)g * d.N);
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = acc_row(v, lane), n = n0 + 32 * t + l32;
          m[t][v] = buf_ldf(rm, (r * (int)brow + n) * 4, 32 * q + r < ci.len && n < d.N);
        }
    };
    load(q0);
    for (int q = q0; q <= q1; ++q) {
      const floatx16 A0 = A;
      float m0[TN][16];
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) m0[t][v] = m[t][v];
      if (q < q1) load(q + 1);
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int t = 0; t < TN; ++t) mfma32(acc[t], A0[v], m0[t][v]);
    }
  }
  float* out = nsl == 1 ? (role ? dB : dC) : (role ? bf.dB_part : bf.dC_part) + (int64_t)slc * d.R * brow;
  const __amdgpu_buffer_rsrc_t ro = buf_rsrc(out + (int64_t)(ci.row0 + rt_row) * brow + (int64_t)g * d.N);
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const int n = n0 + 32 * t + l32;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = acc_row(v, lane);
      const bool ok = 32 * rt + r < ci.len && n < d.N;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[t][v]), ro, ok ? (r * (int)brow + n) * 4 : SSD_BUF_SIZE, 0, 0);
    }
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static F32Args f32_args(const SsdBufs& b, const SsdIn& in, const void* dy) {
  F32Args a;
  a.chunks = b.chunks;
  a.cs = b.cs;
  a.x = static_cast<const float*>(in.x);
  a.dt = in.dt;
  a.Bm = static_cast<const float*>(in.B);
  a.Cm = static_cast<const float*>(in.C);
  a.Dv = in.D;
  a.Dtok = b.Dtok;
  a.hin = static_cast<const float*>(b.hin);
  a.dst = b.dst;
  a.dy = static_cast<const float*>(dy);
  a.cb = b.f32_cb;
  a.unit0 = 0;
  return a;
}

// LDS of the kernels, for PT (and NT) tiles of 32 columns
static size_t lds_f32_scan(const SsdDims& d, int pt) {
  return sizeof(float) * ((size_t)2 * d.Qpad + (size_t)d.Qpad * (32 * pt + 4));
}
static size_t lds_f32_col(const SsdDims& d, int pt) {
  return sizeof(float) * ((size_t)3 * d.Qpad + 16 + (size_t)(d.Qpad / 32) * d.Qpad + (size_t)d.Qpad * (32 * pt + 4));
}
static size_t lds_f32_row(int pt, int nt) { return sizeof(float) * (1024 * pt * nt + 256); }

// Widths of 32, 64 and 128 columns in any pairing but 128 x 128 (the switches below, and one wave per state tile
// in k_f32_state).
bool f32_supported(const SsdDims& d, size_t max_lds) {
  const int pt = d.Ppad / 32, nt = d.Npad / 32;
  return pt * nt <= 8 && d.Qpad <= 256 && lds_f32_scan(d, pt < 2 ? pt : 2) <= max_lds && lds_f32_col(d, pt) <= max_lds &&
         lds_f32_row(pt, nt) <= max_lds;
}

size_t f32_unit_floats(const SsdDims& d) { return (size_t)nsub_of(d.Qpad / 32) * 1024; }

template <int NT, bool FWD>
static void cb_launch(const SsdDims& d, const F32Args& a, int units, hipStream_t s) {
  const int nb = (nsub_of(d.Qpad / 32) + 3) / 4;
  hipLaunchKernelGGL((k_f32_cb<NT, FWD>), dim3((unsigned)units * nb), dim3(256), 0, s, d, a);
}

// One head per group and N <= 32: the scan and the column kernel multiply S themselves (16 MFMA a tile; no other
// head would read the tiles, and a launch and their way through memory are saved).
bool f32_self(const SsdDims& d) { return d.hpg == 1 && d.Npad == 32; }

// `few`: a wave per tile.
template <int PT, int NT>
static hipError_t f32_scan_t(const SsdDims& d, const SsdBufs& b, F32Args a, float* y, bool few, hipStream_t s) {
  const int64_t units = (int64_t)d.max_chunks * d.G;
  const int nph = (d.P + 32 * PT - 1) / (32 * PT), nl = d.Qpad / 32;
  const size_t lds = lds_f32_scan(d, PT);
  const dim3 thr(64 * (few ? nl : (nl + 1) / 2));
  const bool self = f32_self(d);
  auto k = self ? k_f32_scan<PT, NT, NT == 1> : k_f32_scan<PT, NT, false>;
  ensure_lds(k, lds);
  for (int64_t u0 = 0; u0 < units; u0 += b.f32_batch) {
    const int n = (int)std::min<int64_t>(b.f32_batch, units - u0);
    a.unit0 = (int)u0;
    if (!self) cb_launch<NT, true>(d, a, n, s);
    hipLaunchKernelGGL(k, dim3((unsigned)n * d.hpg * nph), thr, lds, s, d, a, y, nph);
  }
  return hipGetLastError();
}

hipError_t launch_f32_scan(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  const F32Args a = f32_args(b, in, nullptr);
  float* yo = static_cast<float*>(y);
  // A wave per tile over 32 columns of P where those waves, two per SIMD, fit the chip at once: the scan is then one
  // wave's chain of products, half as long. Forward alone, two tiles of 64 columns / one of 32, us: 32 chunks of 64
  // tokens, 4 heads of 64 columns 50 / 37; 8 chunks of 64, 24 heads of 96 47 / 36; 128 chunk-heads of 256 tokens (2048
  // waves) 66 / 55; 512 of them 96 / 146.
  const bool few = (int64_t)d.max_chunks * d.H * ((d.P + 31) / 32) * (d.Qpad / 32) <= 2048;
  switch ((d.P > 32 && !few ? 20 : 10) + d.Npad / 32) {
    case 11: return f32_scan_t<1, 1>(d, b, a, yo, few, s);
    case 12: return f32_scan_t<1, 2>(d, b, a, yo, few, s);
    case 14: return f32_scan_t<1, 4>(d, b, a, yo, few, s);
    case 21: return f32_scan_t<2, 1>(d, b, a, yo, few, s);
    case 22: return f32_scan_t<2, 2>(d, b, a, yo, few, s);
    default: return f32_scan_t<2, 4>(d, b, a, yo, few, s);
  }
}

hipError_t launch_f32_state(int mode, const SsdDims& d, const SsdBufs& b, const void* U, const void* V, const float* dt,
                            float* out, hipStream_t s) {
  SsdIn in{};
  in.dt = dt;
  const F32Args a = f32_args(b, in, nullptr);
  const dim3 grid(d.max_chunks, d.H);
  const float *u = static_cast<const float*>(U), *v = static_cast<const float*>(V);
  const dim3 thr(64 * (d.Ppad / 32) * (d.Npad / 32));  // (at most 8 tiles: not 128 x 128)
  // Up to two waves per SIMD wait for their loads, so they take twice as many at once (48 states of 32 x 16 over 256
  // tokens 13.7 -> 12.1 us); more hide each other's, and short chunks would multiply padding (1536 states of 64 x 128
  // over one token: 6 us dearer with steps of 32).
  const bool few = (int64_t)d.max_chunks * d.H * (thr.x / 64) <= 2048 && d.Qpad > 64;
  auto k = mode == 0 ? (few ? k_f32_state<0, 32> : k_f32_state<0, 16>) : (few ? k_f32_state<1, 32> : k_f32_state<1, 16>);
  hipLaunchKernelGGL(k, grid, thr, 0, s, d, a, u, v, out);
  return hipGetLastError();
}

// Units [u0, u0 + n): the column kernel (after the S tiles), or the row kernel (after the dS sums).
template <int PT, int NT>
static hipError_t f32_bwd_t(const SsdDims& d, const SsdBufs& b, F32Args a, float* dx, float* dB, float* dC, int u0,
                            int n, bool row, hipStream_t s) {
  const int nl = d.Qpad / 32;
  const int64_t ss = (int64_t)b.f32_batch * f32_unit_floats(d);
  a.unit0 = u0;
  if (!row) {
    const size_t lds = lds_f32_col(d, PT);
    const int nhalf = nl >= 6 ? 2 : 1;
    const dim3 grid((unsigned)n * b.nslices * nhalf), thr(64 * min(nl, 4));
    if (f32_self(d)) {
      ensure_lds(k_f32_col<PT, NT, NT == 1>, lds);
      hipLaunchKernelGGL((k_f32_col<PT, NT, NT == 1>), grid, thr, lds, s, d, b, a, dx, b.hslice, b.nslices, b.f32_dS, ss);
    } else {
      ensure_lds(k_f32_col<PT, NT, false>, lds);
      cb_launch<NT, false>(d, a, n, s);
      hipLaunchKernelGGL((k_f32_col<PT, NT, false>), grid, thr, lds, s, d, b, a, dx, b.hslice, b.nslices, b.f32_dS, ss);
    }
  } else {
    if (b.nslices > 1)
      hipLaunchKernelGGL(k_f32_ds, dim3((unsigned)n * ((nsub_of(nl) + 3) / 4)), dim3(256), 0, s, d, b.chunks, u0,
                         b.f32_dS, ss, b.nslices);
    const size_t lds = lds_f32_row(PT, NT);
    hipLaunchKernelGGL((k_f32_row<PT, NT>), dim3((unsigned)n * 2 * ((nl + 3) / 4) * b.f32_rsl), dim3(NT > 2 ? 512 : 256), lds, s, d, b,
                       a, b.f32_dS, dB, dC, b.f32_rhs, b.f32_rsl > 1 ? b.f32_rsl - 1 : 1, b.f32_rsl);
  }
  return hipGetLastError();
}

static hipError_t f32_bwd(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, void* dB,
                          void* dC, int u0, int n, bool row, hipStream_t s) {
  const F32Args a = f32_args(b, in, dy);
  float *px = static_cast<float*>(dx), *pb = static_cast<float*>(dB), *pc = static_cast<float*>(dC);
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return f32_bwd_t<1, 1>(d, b, a, px, pb, pc, u0, n, row, s);
    case 12: return f32_bwd_t<1, 2>(d, b, a, px, pb, pc, u0, n, row, s);
    case 14: return f32_bwd_t<1, 4>(d, b, a, px, pb, pc, u0, n, row, s);
    case 21: return f32_bwd_t<2, 1>(d, b, a, px, pb, pc, u0, n, row, s);
    case 22: return f32_bwd_t<2, 2>(d, b, a, px, pb, pc, u0, n, row, s);
    case 24: return f32_bwd_t<2, 4>(d, b, a, px, pb, pc, u0, n, row, s);
    case 41: return f32_bwd_t<4, 1>(d, b, a, px, pb, pc, u0, n, row, s);
    case 42: return f32_bwd_t<4, 2>(d, b, a, px, pb, pc, u0, n, row, s);
    default: return hipErrorInvalidValue;  // (f32_supported)
  }
}

hipError_t launch_f32_col(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, int u0, int n,
                          hipStream_t s) {
  return f32_bwd(d, b, in, dy, dx, nullptr, nullptr, u0, n, false, s);
}
hipError_t launch_f32_row(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC, int u0,
                          int n, hipStream_t s) {
  return f32_bwd(d, b, in, dy, nullptr, dB, dC, u0, n, true, s);
}
