// Backward of the chunked SSD scan for B and C per head (one head per group), bf16, gfx950: the per-chunk work
// FusedSSDScan.backward (r2/dhammic-ai/src/kernels/ssd_scan.py:467-533) gets by re-running the forward under
// autograd, in one kernel. Notation of ssd_bwd_impl.h.
//
// With a group of many heads, S = C B^T and dS serve all of them and the column / row split pays (ssd_bwd_fact.hip,
// ssd_bwd_gemm.hip). With one head nothing is shared: the column blocks of a chunk each read dy, C and dst again and
// the dS tiles go to memory and come back twice, 1.1 MB per (chunk, head) at chunk 256, P = 64, N = 128 against the
// 0.4 MB of its inputs and outputs. Here a block owns a whole (chunk, head): every input is read once (B and dy a
// second time, out of L2) and dS stays in registers.
//
// Wave st owns the source tokens of 32-token tile st (waves w and w + 4 share a SIMD and take tiles st and
// nl - 1 - st, so that each SIMD has nl + 1 of the tiles (lt, st), st <= lt):
//   1a  per tile: S = C_l B_s^T, P = dy_l x_s^T (MFMA, lane = s, registers over l); L exactly, per element;
//       G = M dM in fp32 from fp32 S and the exact products P (its row and column sums cancel in the decay
//       gradient); M rounded to bf16 is the operand of dX^T += dy^T M in place, dS is kept in bf16
//   1b  dX's state term, dx, E, x.dX, the D partial; dB^T = w dt dst^T x^T + C^T dS
//   1c  with the tile's tokens as rows l: dC^T's state term exp(cs) h_in^T dy^T (+ its fp8 residual) and with it
//       the decay gradient's Y_off term
//   2   dS through LDS (over C, dy and the states), B rows beside it: dC^T += B^T dS^T
// Decays are exact (exp and both clamps per element; 36 tiles x 16 exps per lane and head hide beside the MFMAs),
// so no (chunk, head) needs the factorised kernels' fixup.
//
// At B=4 L=4096 H=32 P=64 N=128 chunk 256 (2048 blocks, one per CU), against the column and row kernels: the reference
// scan (MODE 0) 274 us / 342 + 323, its whole backward 317 / 725 (chunk 64: 483 / 788, chunk 256 with N = 16: 187 / 459;
// 64 tokens of 4 heads: 91 / 96); the trapezoidal scan with the gamma path's decay gradient (MODE 3) 338 us / 357 + 372.
// A block's 0.37 MB take 150 us of that at the copy rate; the rest is the block's own chain load -> tiles -> dS exchange
// with 8 waves and no second block beside it (LDS 150 KB, 256 VGPRs): waves wait 47% of their cycles, the MFMA pipes run
// 14%. With NT = 4 the 256 VGPRs do not quite do: 4 and 6 spill in MODE 0 and 1 (PT = 2), 12 and 21 in MODE 3
// (PT = 1 and 2) where the B rows of phase 2 are loaded late (LATE), 84 and 122 where they are in flight through 1c.
#include "ssd_launch.h"
#include "ssd_tile.h"

struct BwdHeadArgs {
  const ChunkInfo* chunks;
  const float* cs;     // [MC][H][Qpad]
  const bf16* hin;     // [MC][H][Ppad][Npad]
  const uint8_t* hin_lo;
  const bf16* hdec;    // MODE 3: the gamma path's states, for the decay term, and their residual
  const uint8_t* hdec_lo;
  const bf16* dst;     // [MC][H][Ppad][Npad], gradient leaving each chunk
  const bf16* x;
  const float* dt;
  const bf16* Bm;
  const bf16* Cm;
  const float* Dv;
  const float* Dtok;   // trapezoidal mode: D per token, and gamma per token
  const float* gam;
  const bf16* dy;
  bf16* dx;
  bf16* dB;
  bf16* dC;
  float* rowG;
  float* colG;
  float* eterm;
  float* xdx;
  float* dcs_off;
  float* dD_part;      // [MC][H][Qpad/64]
  float* xdy;          // trapezoidal mode
};

namespace {

// LDS: phase 1 C, dy, dst, h_in rows, per-token scalars, partial row sums of G; phase 2 the dS tiles and B rows.
template <int PT, int NT>
struct HeadLds {
  static constexpr int PP = 32 * PT, NP = 32 * NT, TS = 32 * tpitch<32>();
  int nl;
  __host__ __device__ int rows() const { return 32 * nl; }
  __host__ __device__ int dy() const { return rows() * tpitch<NP>(); }          // bf16 offsets
  __host__ __device__ int dst() const { return dy() + rows() * tpitch<PP>(); }
  __host__ __device__ int hin() const { return dst() + PP * tpitch<NP>(); }
  __host__ __device__ int scal() const { return hin() + PP * tpitch<NP>(); }
  __host__ __device__ int brows() const { return nl * (nl + 1) / 2 * TS; }      // phase 2
  __host__ __device__ size_t bytes() const {
    const size_t p1 = 2 * (size_t)scal() + 4 * ((size_t)(4 + nl) * rows() + 16);
    const size_t p2 = 2 * ((size_t)brows() + (size_t)rows() * tpitch<NP>());
    return p1 > p2 ? p1 : p2;
  }
};

// The chunk's rows (as many as the block has threads / 2) x W columns: with W / 16 pieces per thread whatever the
// block size, loaded in straight-line masked loads (zeros past nrows and width) and stored to a padded tile later.
template <int W>
struct HeadRows {
  static constexpr int CPR = W / 8, PER = W / 16;
  bf16x8 v[PER];
  __device__ __forceinline__ void load(const bf16* __restrict__ g, int64_t ld, int nrows, int width) {
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(g);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int id = threadIdx.x + q * blockDim.x, r = id / CPR, k = (id % CPR) * 8;
      v[q] = buf_ld16(rs, (int)(((int64_t)r * ld + k) * 2), r < nrows && k < width);
    }
  }
  __device__ __forceinline__ void store(bf16* __restrict__ t) const {
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int id = threadIdx.x + q * blockDim.x, r = id / CPR, k = (id % CPR) * 8;
      *reinterpret_cast<bf16x8*>(t + toff<W>(r, k)) = v[q];
    }
  }
};
// A state tile [PP][NP]: the pieces of a 512-thread block in registers, the rest (smaller blocks) straight through.
template <int PP, int NP>
struct HeadState {
  static constexpr int CPR = NP / 8, TOT = PP * CPR, PER = (TOT + 511) / 512;
  bf16x8 v[PER];
  __device__ __forceinline__ void load(const bf16* __restrict__ g) {
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(g);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int id = threadIdx.x + q * blockDim.x;
      v[q] = buf_ld16(rs, id * 16, id < TOT);
    }
  }
  __device__ __forceinline__ void store(bf16* __restrict__ t, const bf16* __restrict__ g) const {
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int id = threadIdx.x + q * blockDim.x;
      if (id < TOT) *reinterpret_cast<bf16x8*>(t + toff<NP>(id / CPR, (id % CPR) * 8)) = v[q];
    }
    for (int id = threadIdx.x + PER * blockDim.x; id < TOT; id += blockDim.x)
      *reinterpret_cast<bf16x8*>(t + toff<NP>(id / CPR, (id % CPR) * 8)) =
          *reinterpret_cast<const bf16x8*>(g + (int64_t)id * 8);
  }
};

}  // namespace

// MODE: 0 plain, 1 trapezoidal (strictly causal, D per token; the diagonal of dS is gamma x.dy), 3 the same with
// the gamma path's decay gradient (G and E weighted by gamma, the Y_off term over its states).
// LATE: phase 2's B rows are loaded after 1c, not in flight through it.
template <int PT, int NT, int MODE, bool LATE>
__global__ void __launch_bounds__(512, 2) k_bwd_head(SsdDims d, BwdHeadArgs a) {
  constexpr int PP = 32 * PT, NP = 32 * NT, PPI = tpitch<PP>(), NPI = tpitch<NP>(), TPI = tpitch<32>();
  constexpr bool TZ = MODE != 0;
  extern __shared__ __align__(16) unsigned char smem[];
  const int Qpad = d.Qpad, nl = Qpad / 32;
  // (heads fastest: the resident blocks read the columns of many heads at once)
  const int c = blockIdx.x / d.H, h = blockIdx.x % d.H;
  const ChunkInfo ci = a.chunks[c];
  if (ci.len == 0) return;
  const int nlv = (ci.len + 31) >> 5;
  const HeadLds<PT, NT> L{nl};
  bf16* base = reinterpret_cast<bf16*>(smem);
  bf16* Ct = base;               // [rows][NP] C
  bf16* dyt = base + L.dy();     // [rows][PP] dy
  bf16* dstT = base + L.dst();   // [PP][NP]
  bf16* hinT = base + L.hin();   // [PP][NP]
  float* s_cs = reinterpret_cast<float*>(base + L.scal());  // cs log2 e, dt, gamma, D at each token
  float *s_dt = s_cs + Qpad, *s_gm = s_dt + Qpad, *s_D = s_gm + Qpad;
  float* rowp = s_D + Qpad;      // [nl][Qpad]
  float* s_dD = rowp + nl * Qpad;
  int lane = lane_id(), hh = lane >> 5, l32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int st = w < 4 ? w : nl + 3 - w;
  const bool live = st < nlv;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const int64_t hq = ((int64_t)c * d.H + h) * Qpad;
  const bf16* xg = a.x + (int64_t)ci.row0 * xrow + (int64_t)h * d.P;
  const bf16* yg = a.dy + (int64_t)ci.row0 * xrow + (int64_t)h * d.P;
  const bf16* Bg = a.Bm + (int64_t)ci.row0 * brow + (int64_t)h * d.N;
  const bf16* Cg = a.Cm + (int64_t)ci.row0 * brow + (int64_t)h * d.N;
  const int64_t so = ((int64_t)c * d.H + h) * PP * NP;
  auto relane = [&]() {  // (per-lane offsets are recomputed per phase instead of living across all of them)
    lane = opaque_lane();
    hh = lane >> 5;
    l32 = lane & 31;
  };

  // ---- every input in flight: C, dy and the states for LDS, B and x of the tile's tokens as operands (lane =
  // token, 8 consecutive columns), the per-token scalars ----
  HeadRows<NP> rC;
  HeadRows<PP> rY;
  HeadState<PP, NP> rS, rH;
  rC.load(Cg, brow, ci.len, d.N);
  rY.load(yg, xrow, ci.len, d.P);
  rS.load(a.dst + so);
  rH.load(a.hin + so);
  bf16x8 bfr[2 * NT], xfr[2 * PT];
  {
    const int r = 32 * st + l32;
    const bool ok = live && r < ci.len;
    const __amdgpu_buffer_rsrc_t rb = buf_rsrc(Bg), rx = buf_rsrc(xg);
#pragma unroll
    for (int k = 0; k < 2 * NT; ++k)
      bfr[k] = buf_ld16(rb, (int)((r * brow + 16 * k + 8 * hh) * 2), ok && 16 * k + 8 * hh < d.N);
#pragma unroll
    for (int k = 0; k < 2 * PT; ++k)
      xfr[k] = buf_ld16(rx, (int)((r * xrow + 16 * k + 8 * hh) * 2), ok && 16 * k + 8 * hh < d.P);
  }
  {
    const __amdgpu_buffer_rsrc_t rc = buf_rsrc(a.cs + hq), rt = buf_rsrc(d.has_dt ? a.dt + (int64_t)ci.row0 * d.H : a.cs);
    const __amdgpu_buffer_rsrc_t rg = buf_rsrc(TZ ? a.gam + (int64_t)ci.row0 * d.H : a.cs);
    const __amdgpu_buffer_rsrc_t rD = buf_rsrc(TZ ? a.Dtok + (int64_t)ci.row0 * d.H : (d.has_D ? a.Dv : a.cs));
    const int l = threadIdx.x;  // (blockDim = 2 Qpad)
    if (l < Qpad) {
      const bool in = l < ci.len;
      const float c0 = buf_ldf(rc, l * 4, true), t0 = buf_ldf(rt, (l * d.H + h) * 4, d.has_dt && in);
      const float g0 = buf_ldf(rg, (l * d.H + h) * 4, TZ && in);
      const float D0 = buf_ldf(rD, ((TZ ? l * d.H : 0) + h) * 4, TZ ? in : d.has_D != 0);
      s_cs[l] = c0 * SSD_LOG2E;
      s_dt[l] = (d.has_dt && in) ? t0 : 1.0f;
      s_gm[l] = g0;
      s_D[l] = D0;
    }
  }
  rC.store(Ct);
  rY.store(dyt);
  rS.store(dstT, a.dst + so);
  rH.store(hinT, a.hin + so);
  __syncthreads();

  // ---- 1a ----
  floatx16 dX[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) zero(dX[p]);
  bf16x8 dS16[8][2];
  const int s_me = 32 * st + l32;
  if (live) {
    const float cs_s = s_cs[s_me], dt_s = s_dt[s_me], gm_s = s_gm[s_me];
    float gcol = 0.0f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int lt = st + t;
      if (lt < nlv) {
        floatx16 S, P;
        zero(S);
        zero(P);
        const bf16* cr = Ct + (32 * lt) * NPI;
        const bf16* yr = dyt + (32 * lt) * PPI;
#pragma unroll
        for (int k = 0; k < 2 * NT; ++k) mfma(S, tld8<NP>(cr, l32, 16 * k + 8 * hh), bfr[k]);
#pragma unroll
        for (int k = 0; k < 2 * PT; ++k) mfma(P, tld8<PP>(yr, l32, 16 * k + 8 * hh), xfr[k]);
        float csl[16], G[16];
        rows16(s_cs + 32 * lt, csl);
        float xd = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const bool ok = t > 0 || l32 + (TZ ? 1 : 0) <= acc_row(v, lane);
          const float dd = csl[v] - cs_s;
          const float Lv = ok ? exp2_fast(clamp_med3(dd, -SSD_T2, SSD_T2)) : 0.0f;
          const float m = S[v] * Lv, pl = P[v] * Lv;
          const float g = m * P[v] * (MODE == 3 ? gm_s : dt_s);
          G[v] = fabsf(dd) < SSD_T2 ? g : 0.0f;
          gcol += G[v];
          S[v] = m;
          float ds = pl * dt_s;
          if (TZ && t == 0 && acc_row(v, lane) == l32) {  // the diagonal: D's gamma (C . B) part
            xd = P[v];
            ds = gm_s * P[v];
          }
          P[v] = ds;
        }
        if (TZ && t == 0) {
          xd = add_xor32(xd);
          if (hh == 0 && s_me < ci.len) a.xdy[hq + s_me] = xd;
        }
        const bf16x8 m0 = acc_frag(S, 0), m1 = acc_frag(S, 1);
        dS16[t][0] = acc_frag(P, 0);
        dS16[t][1] = acc_frag(P, 1);
        const float rs = half_reduce16(G, lane);
        if (!(lane & 1)) rowp[st * Qpad + 32 * lt + acc_row((l32 >> 1) & 15, lane)] = rs;
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          mfma(dX[p], ttr_perm<PP>(yr, 0, 0, 32 * p, lane), m0);
          mfma(dX[p], ttr_perm<PP>(yr, 0, 1, 32 * p, lane), m1);
        }
      }
    }
    gcol = add_xor32(gcol);
    if (hh == 0 && s_me < ci.len) a.colG[hq + s_me] = gcol;
  }
  __syncthreads();  // row sums complete; every wave past the dy rows of the others
  for (int l = threadIdx.x; l < ci.len; l += blockDim.x) {
    float r = 0.0f;
    for (int q = 0; q <= l >> 5; ++q) r += rowp[q * Qpad + l];
    a.rowG[hq + l] = r;
  }

  // The wave's own 32 dy rows: read by this wave alone from here on, then the staging tile of its outputs.
  bf16* own = dyt + 32 * st * PPI;
  // 32 rows x PP columns of `own` to rows 32 st .. of a row-major tensor at g (column 0 of the pass), cols < width
  auto store_own = [&](bf16* g, int64_t ld, int width) {
    constexpr int CPR = PP / 8;
#pragma unroll
    for (int q = 0; q < 32 * CPR / 64; ++q) {
      const int id = lane + 64 * q, r = id / CPR, k = (id % CPR) * 8;
      if (32 * st + r < ci.len && k < width)
        *reinterpret_cast<bf16x8*>(g + (int64_t)(32 * st + r) * ld + k) = tld8<PP>(own, r, k);
    }
  };

  // ---- 1b ----
  bf16x8 yfr[2 * PT];
  uint2 lf[NT][2 * PT];  // residual of the decay term's states (1c), in flight through dB
  const uint8_t* lo = MODE == 3 ? a.hdec_lo : a.hin_lo;
  floatx16 acc[NT];
  if (MODE == 3) rS.load(a.hdec + so);
  if (live) {
    relane();
    const int s = 32 * st + l32;
    floatx16 dXs[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
      zero(dXs[p]);
#pragma unroll
      for (int k = 0; k < 2 * NT; ++k) mfma(dXs[p], tld8<NP>(dstT, 32 * p + l32, 16 * k + 8 * hh), bfr[k]);
    }
    const float dw = s_cs[Qpad - 1] - s_cs[s], dts = s_dt[s], Dl = s_D[s];
    const float ws = s < ci.len ? exp2_fast(clamp_med3(dw, -SSD_T2, SSD_T2)) : 0.0f;
    const float pw = fabsf(dw) < SSD_T2 ? 1.0f : 0.0f;
    float esum = 0.0f, xsum = 0.0f, dsum = 0.0f;
#pragma unroll
    for (int k = 0; k < 2 * PT; ++k) {
      // x at the accumulator's rows p: quads 16 k + 4 hh and 16 k + 8 + 4 hh of this lane's token, by trading
      // halves with the lane that holds the token's other eight columns
      const u32x4 u = __builtin_bit_cast(u32x4, xfr[k]);
      const auto r0 = __builtin_amdgcn_permlane32_swap(u[0], u[2], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(u[1], u[3], false, false);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bf16x2 xa = __builtin_bit_cast(bf16x2, (unsigned)r0[q]), xb = __builtin_bit_cast(bf16x2, (unsigned)r1[q]);
        const float xv[4] = {(float)xa[0], (float)xa[1], (float)xb[0], (float)xb[1]};
        const int p = k >> 1, r = 2 * (k & 1) + q, p0 = 32 * p + 8 * r + 4 * hh;
        const bf16x4 yv = tld4<PP>(own, l32, p0);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float yf = (float)yv[e], ds = ws * dXs[p][4 * r + e], dXv = dX[p][4 * r + e] + ds;
          esum = fmaf(xv[e], ds, esum);
          xsum = fmaf(xv[e], dXv, xsum);
          dsum = fmaf(xv[e], yf, dsum);
          o[e] = (bf16)fmaf(dts, dXv, Dl * yf);
        }
        *reinterpret_cast<bf16x4*>(own + toff<PP>(l32, p0)) = o;
      }
    }
    esum = add_xor32(esum);
    xsum = add_xor32(xsum);
    dsum = wave_sum(dsum);
    if (hh == 0 && s < ci.len) {
      a.eterm[hq + s] = esum * (MODE == 3 ? s_gm[s] : dts) * pw;
      a.xdx[hq + s] = xsum;
    }
    if (lane == 0) s_dD[st] = dsum;
    store_own(a.dx + (int64_t)ci.row0 * xrow + (int64_t)h * d.P, xrow, d.P);
    // dy rows of the tile's tokens again (1c's operand), in flight through dB
    {
      const __amdgpu_buffer_rsrc_t ry = buf_rsrc(yg);
#pragma unroll
      for (int k = 0; k < 2 * PT; ++k)
        yfr[k] = buf_ld16(ry, (int)((s * xrow + 16 * k + 8 * hh) * 2), s < ci.len && 16 * k + 8 * hh < d.P);
    }
    if (lo) {
      const __amdgpu_buffer_rsrc_t rl = buf_rsrc(lo + so);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int k = 0; k < 2 * PT; ++k)
          lf[n][k] = __builtin_bit_cast(
              uint2, __builtin_amdgcn_raw_buffer_load_b64(rl, (int)hin_lo_off(PP, 32 * n, 16 * k) + lane * 8, 0, 0));
    }
    relane();
    const float f = ws * dts;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      zero(acc[n]);
#pragma unroll
      for (int k = 0; k < 2 * PT; ++k) mfma(acc[n], ttr_std<NP>(dstT, 16 * k, 32 * n, lane), xfr[k]);
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[n][v] *= f;
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int lt = st + t;
      if (lt < nlv) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          mfma(acc[n], ttr_perm<NP>(Ct, 32 * lt, 0, 32 * n, lane), dS16[t][0]);
          mfma(acc[n], ttr_perm<NP>(Ct, 32 * lt, 1, 32 * n, lane), dS16[t][1]);
        }
      }
    }
    relane();
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += PT) {
#pragma unroll
      for (int q = 0; q < PT; ++q)
        if (n0 + q < NT) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[n0 + q < NT ? n0 + q : 0][4 * r + e];
            *reinterpret_cast<bf16x4*>(own + toff<PP>(l32, 32 * q + 8 * r + 4 * hh)) = o;
          }
        }
      store_own(a.dB + (int64_t)ci.row0 * brow + (int64_t)h * d.N + 32 * n0, brow, min(d.N - 32 * n0, 32 * min(PT, NT - n0)));
    }
  } else if (lane == 0) {
    s_dD[st] = 0.0f;
  }
  if (MODE == 3) {  // the gamma path's states over dst (every wave is done with it after the barrier)
    __syncthreads();
    rS.store(dstT, a.hdec + so);
    __syncthreads();
  }

  // ---- 1c ----
  if (!LATE) rC.load(Bg, brow, ci.len, d.N);  // phase 2's B rows
  if (live) {
    relane();
    const int l = 32 * st + l32;
    const float csl2 = s_cs[l], et = exp2_fast(clamp_med3(csl2, -SSD_T2, SSD_T2));
    float osum = 0.0f;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      floatx16 T;
      zero(T);
#pragma unroll
      for (int k = 0; k < 2 * PT; ++k) mfma(T, ttr_std<NP>(hinT, 16 * k, 32 * n, lane), yfr[k]);
      if (MODE != 3 && lo) {
#pragma unroll
        for (int k = 0; k < 2 * PT; ++k) mfma(T, lo_frag(lf[n][k]), yfr[k]);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[n][v] = et * T[v];
      if (MODE == 3) {
        zero(T);
#pragma unroll
        for (int k = 0; k < 2 * PT; ++k) mfma(T, ttr_std<NP>(dstT, 16 * k, 32 * n, lane), yfr[k]);
        if (lo) {
#pragma unroll
          for (int k = 0; k < 2 * PT; ++k) mfma(T, lo_frag(lf[n][k]), yfr[k]);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bf16x4 cv = tld4<NP>(Ct, l, 32 * n + 8 * r + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) osum = fmaf((float)cv[e], T[4 * r + e], osum);
      }
    }
    osum = add_xor32(osum);
    if (hh == 0 && l < ci.len) a.dcs_off[hq + l] = osum * et * (fabsf(csl2) < SSD_T2 ? 1.0f : 0.0f);
  }
  if (LATE) rC.load(Bg, brow, ci.len, d.N);
  __syncthreads();  // C, dy, the states and the scalars are done with; s_dD written
  float dD0 = 0.0f;
  if (threadIdx.x < nl / 2) dD0 = s_dD[2 * threadIdx.x] + s_dD[2 * threadIdx.x + 1];
  __syncthreads();
  if (threadIdx.x < nl / 2) a.dD_part[((int64_t)c * d.H + h) * (Qpad / 64) + threadIdx.x] = dD0;

  // ---- 2 ----
  constexpr int TS = HeadLds<PT, NT>::TS;
  bf16* Bt = base + L.brows();
  rC.store(Bt);
  if (live) {
    relane();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int lt = st + t;
      if (lt < nlv) {
        bf16* T = base + (lt * (lt + 1) / 2 + st) * TS + l32 * TPI + 4 * hh;  // tile [s][l]
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bf16x8 f = dS16[t][r >> 1];
          *reinterpret_cast<bf16x4*>(T + 8 * r) = (r & 1) ? __builtin_shufflevector(f, f, 4, 5, 6, 7)
                                                          : __builtin_shufflevector(f, f, 0, 1, 2, 3);
        }
      }
    }
  }
  __syncthreads();
  if (live) {
    relane();
    for (int q = 0; q <= st; ++q) {
      const bf16* T = base + (st * (st + 1) / 2 + q) * TS;
      const bf16x8 s0 = ttr_std<32>(T, 0, 0, lane), s1 = ttr_std<32>(T, 16, 0, lane);
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        mfma(acc[n], ttr_std<NP>(Bt, 32 * q, 32 * n, lane), s0);
        mfma(acc[n], ttr_std<NP>(Bt, 32 * q + 16, 32 * n, lane), s1);
      }
    }
  }
  __syncthreads();  // the tiles are done with: their place stages dC
  if (live) {
    relane();
    own = base + 32 * st * PPI;
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += PT) {
#pragma unroll
      for (int q = 0; q < PT; ++q)
        if (n0 + q < NT) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[n0 + q < NT ? n0 + q : 0][4 * r + e];
            *reinterpret_cast<bf16x4*>(own + toff<PP>(l32, 32 * q + 8 * r + 4 * hh)) = o;
          }
        }
      store_own(a.dC + (int64_t)ci.row0 * brow + (int64_t)h * d.N + 32 * n0, brow, min(d.N - 32 * n0, 32 * min(PT, NT - n0)));
    }
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
bool bwd_head_supported(int dtype, const SsdDims& d) {
  // (32-bit byte offsets of a chunk's rows)
  return dtype == 1 && d.hpg == 1 && d.Ppad <= 64 && d.Qpad <= 256 && d.P % 8 == 0 && d.N % 8 == 0 &&
         (int64_t)d.Qpad * d.H * (d.P > d.N ? d.P : d.N) * 2 <= INT32_MAX;
}

size_t lds_bwd_head(const SsdDims& d) {
  const int nl = d.Qpad / 32;
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return HeadLds<1, 1>{nl}.bytes();
    case 12: return HeadLds<1, 2>{nl}.bytes();
    case 14: return HeadLds<1, 4>{nl}.bytes();
    case 21: return HeadLds<2, 1>{nl}.bytes();
    case 22: return HeadLds<2, 2>{nl}.bytes();
    default: return HeadLds<2, 4>{nl}.bytes();
  }
}

template <int PT, int NT, int MODE, bool LATE = false>
static hipError_t bwd_head_launch(const SsdDims& d, const BwdHeadArgs& a, hipStream_t s) {
  const size_t lds = lds_bwd_head(d);
  ensure_lds(k_bwd_head<PT, NT, MODE, LATE>, lds);
  hipLaunchKernelGGL((k_bwd_head<PT, NT, MODE, LATE>), dim3((unsigned)d.max_chunks * d.H), dim3(2 * d.Qpad), lds, s, d, a);
  return hipGetLastError();
}

template <int PT, int NT>
static hipError_t bwd_head_t(const SsdDims& d, const BwdHeadArgs& a, hipStream_t s) {
  if (!d.trapz) return bwd_head_launch<PT, NT, 0>(d, a, s);
  if (!d.gdec) return bwd_head_launch<PT, NT, 1>(d, a, s);
  // Six or eight tiles a block: the spills of MODE 3 cost more than a late load (782 -> 768 us, the whole call at chunk
  // 256); two or four: the late load does (chunk 64 1095 / 1108, chunk 128 896 / 900).
  if (NT == 4 && d.Qpad > 128) return bwd_head_launch<PT, NT, 3, NT == 4>(d, a, s);
  return bwd_head_launch<PT, NT, 3>(d, a, s);
}

hipError_t launch_bwd_head(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, void* dB,
                           void* dC, hipStream_t s) {
  BwdHeadArgs a;
  a.chunks = b.chunks;
  a.cs = b.cs;
  a.hin = static_cast<const bf16*>(b.hin);
  a.hin_lo = b.hin_lo;
  a.hdec = static_cast<const bf16*>(b.hdec);
  a.hdec_lo = b.hdec_lo;
  a.dst = b.dst16;
  a.x = static_cast<const bf16*>(in.x);
  a.dt = in.dt;
  a.Bm = static_cast<const bf16*>(in.B);
  a.Cm = static_cast<const bf16*>(in.C);
  a.Dv = in.D;
  a.Dtok = b.Dtok;
  a.gam = b.tz_gam;
  a.dy = static_cast<const bf16*>(dy);
  a.dx = static_cast<bf16*>(dx);
  a.dB = static_cast<bf16*>(dB);
  a.dC = static_cast<bf16*>(dC);
  a.rowG = b.rowG;
  a.colG = b.colG;
  a.eterm = b.eterm;
  a.xdx = b.xdx;
  a.dcs_off = b.dcs_off;
  a.dD_part = b.dD_part;
  a.xdy = b.xdy;
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return bwd_head_t<1, 1>(d, a, s);
    case 12: return bwd_head_t<1, 2>(d, a, s);
    case 14: return bwd_head_t<1, 4>(d, a, s);
    case 21: return bwd_head_t<2, 1>(d, a, s);
    case 22: return bwd_head_t<2, 2>(d, a, s);
    default: return bwd_head_t<2, 4>(d, a, s);
  }
}
