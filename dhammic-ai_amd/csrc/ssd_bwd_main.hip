// Fused backward of the chunked SSD scan for bf16 inputs (gfx950), the work
// that FusedSSDScan.backward (r2/dhammic-ai/src/kernels/ssd_scan.py:467-533)
// gets by re-running the forward under autograd, written out per chunk.
//
// Notation per (chunk, head h); rows l (outputs) and columns s (inputs) of the
// chunk's 64-token blocks, tile (i, j) = rows of block i x columns of block j:
//   S = C B^T (shared by the heads of a group), L[l,s] = exp(clamp(cs_l - cs_s)),
//   M = S*L, dM[l,s] = dy_l . x_s, dm = dM dt_s, G = dm*M*pass(cs_l - cs_s)
// gives per head
//   dX_s   = sum_l M[l,s] dy_l + w_s B_s dst^T           (dx = dt dX + D dy)
//   rowG_l = sum_s G[l,s],  colG_s = sum_l G[l,s]
//   E_s    = pass_w(s) dt_s x_s . (w_s B_s dst^T),  xdx_s = x_s . dX_s
// and, summed over the heads of the group,
//   dS[l,s] = sum_h dm L                   (-> dB = dS^T C, dC = dS B, kernel k_bwd_gemm)
// The head-summed state terms of dB and dC and the Y_off part of the decay
// gradient are k_bwd_gemm's (ssd_bwd_gemm.hip).
//
// k_bwd_main: one block per (column block j, chunk, group, head slice). The
// block owns the 64 columns s of block j, so dX and colG are complete there;
// it walks the tiles (i, j), i >= j, of every head of its
// slice. S for those tiles is computed once per block and kept in registers;
// dS accumulates in registers over the slice's heads. Tiles are computed
// transposed ([s rows][l lanes]): row sums of G are per-lane, column sums are
// reduced across lanes once per head. M goes through a per-wave LDS tile to
// become the B operand of dX^T = dY^T M; every other operand is read from
// natural-layout LDS tiles (ds_read_b64_tr_b16 where the contraction runs over
// the row index).
#include <algorithm>

#include "ssd_launch.h"
#include "ssd_tile.h"

struct BwdMainArgs {
  const ChunkInfo* chunks;
  const float* cs;    // [MC][H][Qpad]
  const bf16* dst;    // [MC][H][Ppad][Npad], gradient leaving each chunk (bf16)
  const bf16* x;
  const float* dt;
  const bf16* Bm;
  const bf16* Cm;
  const float* Dv;
  const bf16* dy;
  bf16* dx;
  float* rowG;        // [nb][MC][H][Qpad], partial per column block (block j covers rows >= 64 j)
  float* colG;        // [MC][H][Qpad]
  float* eterm;
  float* xdx;
  float* dD_part;     // [MC][H][Qpad/64]
  float* dS;          // [nslices][MC][G][nb*nb][64][64], tile (i, j) row-major [l][s]
  const float* Dtok;  // trapezoidal mode: D per token, [R][H]
  // the decay gradient's dt (G's v_s and E's factor): a.dt, or (trapezoidal drop mode) the gamma path's
  // dt per token, [R][H]
  const float* ddec;
  int nslices, hslice;
  // fixup mode (non-null): only the heads flagged 0 here run (the factorised kernel
  // cannot take them); the block skips the others and exits if it has none
  const int32_t* fast;
};

constexpr int kMaxSlots = 4;  // tiles per column block (nb <= 4)

template <int PT, int NT>
struct BwdMainLds {
  static constexpr int PP = 32 * PT, NP = 32 * NT;
  static constexpr int RED = 1024;  // floats of reduction scratch
  static size_t bytes(int Qpad) {
    const size_t xch = 2 * PT * 4096;
    return sizeof(float) * (3 * Qpad + RED) +
           2 * (size_t)(5 * tsize<64, PP>() + tsize<PP, NP>() + tsize<64, NP>() + 4 * tsize<32, 32>()) + xch;
  }
};

// One block per (column block j, group, head slice, chunk); blocks are
// numbered column-major with the heaviest column (j = 0, nb tiles) first, and
// the column blocks of one chunk share an XCD (same block index mod 8).
// The work of block `bid` of that numbering.
template <int PT, int NT>
__device__ __forceinline__ void bwd_main_block(const SsdDims& d, const BwdMainArgs& a, int bid) {
  constexpr int PP = 32 * PT, NP = 32 * NT;
  constexpr int NTW = (NT + 1) / 2;  // n tiles per wave in the state terms
  constexpr int PTW = (PT + 1) / 2;  // p tiles kept per wave after the dX exchange
  extern __shared__ __align__(16) unsigned char smem[];
  const int nb = d.Qpad / 64;

  const int U = d.max_chunks * d.G * a.nslices;
  const int U8 = (U + 7) / 8 * 8;
  const int j = bid / U8;
  const int u = bid % U8;
  if (u >= U) return;
  const int c = u % d.max_chunks;
  const int gsl = u / d.max_chunks;
  const int g = gsl / a.nslices, slc = gsl % a.nslices;
  const ChunkInfo ci = a.chunks[c];
  const int nbl = (ci.len + 63) >> 6;
  if (j >= nbl) return;
  const int nt_i = nbl - j;  // tiles (i, j), i = j .. nbl-1
  const int h_lo = g * d.hpg + slc * a.hslice;
  const int h_hi = min(h_lo + a.hslice, (g + 1) * d.hpg);
  if (h_lo >= h_hi) return;
  if (a.fast) {
    // fixup mode: blocks whose heads all took the factorised path leave at once
    bool need = false;
    for (int h = h_lo + (int)threadIdx.x; h < h_hi; h += 256) need = need || a.fast[(int64_t)c * d.H + h] == 0;
    if (!__syncthreads_or(need)) return;
  }
  // the next head this block runs at or after h (h_hi: none)
  auto next_head = [&](int h) {
    if (a.fast)
      while (h < h_hi && a.fast[(int64_t)c * d.H + h] != 0) ++h;
    return h;
  };
  const int h_first = next_head(h_lo);
  if (h_first >= h_hi) return;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = w & 1, wc = w >> 1;
  int lane = threadIdx.x & 63, hh = lane >> 5, l32 = lane & 31;
  const int Qpad = d.Qpad;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;

  float* s_cs2 = reinterpret_cast<float*>(smem);  // cs * log2(e) of the current head
  float* s_dt = s_cs2 + Qpad;
  float* s_gd = s_dt + Qpad;                       // the decay gradient's dt (a.ddec)
  float* red = s_gd + Qpad;                        // RED floats
  float* red_row = red;                            // [4 blocks][2 wr][64]
  float* red_col = red + 512;                      // [2 wc][64]
  float* red_e = red + 640;                        // [2 wc][64]
  float* red_x = red + 768;                        // [2 wc][64]
  float* red_o = red + 896;                        // [2 wc][64] (the first 4 also hold the dD partials)
  constexpr int XT = tsize<64, PP>(), ST = tsize<PP, NP>(), BTS = tsize<64, NP>(), MT = tsize<32, 32>();
  bf16* xj = reinterpret_cast<bf16*>(red + BwdMainLds<PT, NT>::RED);  // [64][PP]
  bf16* dYt = xj + XT;                             // [4][64][PP] (blocks j .. nbl-1 used)
  bf16* dstT = dYt + 4 * XT;                       // [PP][NP]
  bf16* Bt = dstT + ST;                            // [64][NP]
  bf16* Mb = Bt + BTS + w * MT;                    // this wave's [32][32]
  float* xch = reinterpret_cast<float*>(Bt + BTS + 4 * MT);

  // ---- B tile of column block j ----
  {
    TileStage<64, NP, 256> st;
    tstage_load_v(st, a.Bm + (int64_t)(ci.row0 + 64 * j) * brow + (int64_t)g * d.N, brow,
                min(64, ci.len - 64 * j), d.N);
    tstage_store(st, Bt);
  }
  __syncthreads();

  // ---- S^T tiles (i, j), slot t = i - j: rows s (wr half of block j), lanes l (wc half of block i) ----
  bf16x8 S[kMaxSlots][2];  // kept in bf16: M = S L is rounded to bf16 for the MFMA anyway
  floatx16 dS[kMaxSlots];
#pragma unroll
  for (int t = 0; t < kMaxSlots; ++t) {
    floatx16 sacc;
    zero(sacc);
    zero(dS[t]);
    S[t][0] = acc_frag(sacc, 0);
    S[t][1] = acc_frag(sacc, 1);
    if (t >= nt_i) continue;
    const int i = j + t;
    if (t == 0 && wr == 1 && wc == 0) continue;  // above the diagonal
    const int lrow = 64 * i + 32 * wc + l32;
    const bool lok = lrow < ci.len;
    const bf16* crow = a.Cm + (int64_t)(ci.row0 + (lok ? lrow : 0)) * brow + (int64_t)g * d.N;
#pragma unroll
    for (int kk = 0; kk < NP; kk += 16) {
      const int n0 = kk + 8 * hh;
      bf16x8 cb;
#pragma unroll
      for (int e = 0; e < 8; ++e) cb[e] = (bf16)0.0f;
      if (lok && n0 < d.N) cb = *reinterpret_cast<const bf16x8*>(crow + n0);
      mfma(sacc, tld8<NP>(Bt, 32 * wr + l32, n0), cb);
    }
    S[t][0] = acc_frag(sacc, 0);
    S[t][1] = acc_frag(sacc, 1);
  }

  // per-token lane of the state terms: token 32 wr + l32 of block j
  const int t_loc = 32 * wr + l32;
  const int tg = 64 * j + t_loc;
  const bool t_ok = tg < ci.len;

  // Inputs of the tile phase (x, dy, cs, dt) are loaded during the previous
  // head's state phase; those of the state phase (dst, h_in) during this
  // head's tile phase.
  struct HeadStage {
    TileStage<64, PP, 256> x, y[kMaxSlots];
    float cs, dt, gd;
  } hs;
  auto load_tiles = [&](int h) {
    const int l0 = threadIdx.x;
    hs.cs = 0.0f;
    hs.dt = 1.0f;
    hs.gd = 1.0f;
    if (l0 < Qpad) {
      hs.cs = a.cs[((int64_t)c * d.H + h) * Qpad + l0];
      if (d.has_dt && l0 < ci.len) hs.dt = a.dt[(int64_t)(ci.row0 + l0) * d.H + h];
      if (d.has_dt && l0 < ci.len) hs.gd = a.ddec[(int64_t)(ci.row0 + l0) * d.H + h];
    }
    tstage_load_v(hs.x, a.x + (int64_t)(ci.row0 + 64 * j) * xrow + (int64_t)h * d.P, xrow, min(64, ci.len - 64 * j),
                  d.P);
#pragma unroll
    for (int t = 0; t < kMaxSlots; ++t)
      if (t < nt_i)
        tstage_load_v(hs.y[t], a.dy + (int64_t)(ci.row0 + 64 * (j + t)) * xrow + (int64_t)h * d.P, xrow,
                      min(64, ci.len - 64 * (j + t)), d.P);
  };
  load_tiles(h_first);
  for (int h = h_first; h < h_hi;) {
    const int h_next = next_head(h + 1);
    lane = opaque_lane();
#pragma unroll
    for (int t = 0; t < kMaxSlots; ++t) {
      launder(S[t][0]);
      launder(S[t][1]);
    }
    hh = lane >> 5;
    l32 = lane & 31;
    __syncthreads();  // the previous head's LDS reads are done
    if (threadIdx.x < Qpad) {
      s_cs2[threadIdx.x] = hs.cs * SSD_LOG2E;
      s_dt[threadIdx.x] = hs.dt;
      s_gd[threadIdx.x] = hs.gd;
    }
    for (int e = threadIdx.x; e < 4 * 2 * 64; e += 256) red_row[e] = 0.0f;
    tstage_store(hs.x, xj);
#pragma unroll
    for (int t = 0; t < kMaxSlots; ++t)
      if (t < nt_i) tstage_store(hs.y[t], dYt + (j + t) * XT);
    __syncthreads();
    TileStage<PP, NP, 256> sd;
    tstage_load_v(sd, a.dst + ((int64_t)c * d.H + h) * PP * NP, NP, PP, NP);

    const float cs_last = s_cs2[Qpad - 1];
    const float Dh = d.trapz ? (t_ok ? a.Dtok[(int64_t)(ci.row0 + tg) * d.H + h] : 0.0f) : (d.has_D ? a.Dv[h] : 0.0f);

    float colacc[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) colacc[v] = 0.0f;
    floatx16 dXT[PT];
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) zero(dXT[pt]);

#pragma unroll
    for (int t = 0; t < kMaxSlots; ++t) {
      if (t >= nt_i) continue;
      const int i = j + t;
      const bool diag = t == 0;
      if (diag && wr == 1 && wc == 0) continue;
      const bf16* dyi = dYt + i * XT;
      floatx16 dm;
      zero(dm);
#pragma unroll
      for (int kk = 0; kk < PP; kk += 16)
        mfma(dm, tld8<PP>(xj, 32 * wr + l32, kk + 8 * hh), tld8<PP>(dyi, 32 * wc + l32, kk + 8 * hh));
      const int l_loc = 32 * wc + l32;
      const float cs_l = s_cs2[64 * i + l_loc];
      float cs_s[16], dt_s[16], gd_s[16];
      rows16(s_cs2 + 64 * j + 32 * wr, cs_s);
      rows16(s_dt + 64 * j + 32 * wr, dt_s);
      rows16(s_gd + 64 * j + 32 * wr, gd_s);
      float rsum = 0.0f;
      float Mv[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int s_loc = 32 * wr + acc_row(v, lane);
        const float dd = cs_l - cs_s[v];
        float Lv = exp2_fast(clamp_med3(dd, -SSD_T2, SSD_T2));
        if (diag && s_loc + (d.trapz ? 1 : 0) > l_loc) Lv = 0.0f;  // trapezoidal mode: strictly causal
        const float dmv = dm[v] * dt_s[v];
        const float M = (float)S[t][v >> 3][v & 7] * Lv;
        dS[t][v] = fmaf(dmv, Lv, dS[t][v]);
        const float Mp = fabsf(dd) < SSD_T2 ? M : 0.0f;
        const float gg = dm[v] * gd_s[v] * Mp;
        colacc[v] += gg;
        rsum += gg;
        Mv[v] = M;
      }
      // M^T (rows s, lanes l) -> this wave's LDS tile Mb[l][s]
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        bf16x4 q;
        q[0] = (bf16)Mv[4 * r + 0];
        q[1] = (bf16)Mv[4 * r + 1];
        q[2] = (bf16)Mv[4 * r + 2];
        q[3] = (bf16)Mv[4 * r + 3];
        *reinterpret_cast<bf16x4*>(Mb + toff<32>(l32, 8 * r + 4 * hh)) = q;
      }
      // dX^T[p][s] += sum_l dy_i[l][p] M[l][s]  (l over this wave's 32-row window)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8 mb = ttr_std<32>(Mb, 16 * kk, 0, lane);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) mfma(dXT[pt], ttr_std<PP>(dyi, 32 * wc + 16 * kk, 32 * pt, lane), mb);
      }
      // row sums of G: per lane over its 16 s rows, then the two half-waves
      rsum += __shfl_xor(rsum, 32, 64);
      if (hh == 0) red_row[(i * 2 + wr) * 64 + l_loc] += rsum;
    }

    // ---- column sums of G over l (lanes and the wc pair) ----
    {
      const float cg = half_reduce16(colacc, lane);
      const int idx = (lane >> 1) & 15;
      if ((lane & 1) == 0) red_col[wc * 64 + 32 * wr + 8 * (idx >> 2) + 4 * hh + (idx & 3)] = cg;
    }
    // ---- dX^T exchange: wave (wr, wc) keeps the p tiles pt % 2 == wc ----
#pragma unroll
    for (int pt = 0; pt < PT; ++pt)
      if (pt % 2 != wc) {
        float* o = xch + ((wr * PT + pt) * 16) * 64 + lane;
#pragma unroll
        for (int v = 0; v < 16; ++v) o[v * 64] = dXT[pt][v];
      }
    __syncthreads();
    floatx16 dXk[PTW];
#pragma unroll
    for (int q = 0; q < PTW; ++q) {
      const int pt = 2 * q + wc;
      zero(dXk[q]);
      if (pt >= PT) continue;
      const float* o = xch + ((wr * PT + pt) * 16) * 64 + lane;
#pragma unroll
      for (int v = 0; v < 16; ++v) dXk[q][v] = dXT[pt][v] + o[v * 64];
    }
    if (threadIdx.x < 64) {
      const int sg = 64 * j + threadIdx.x;
      if (sg < ci.len) a.colG[((int64_t)c * d.H + h) * Qpad + sg] = red_col[threadIdx.x] + red_col[64 + threadIdx.x];
    }
    tstage_store(sd, dstT);
    __syncthreads();
    if (h_next < h_hi) load_tiles(h_next);

    // ---- per-token state terms of column block j (lane = token t_loc) ----
    const float cs_t = s_cs2[tg];
    const float dw = cs_last - cs_t;
    const float ws = t_ok ? exp2_fast(clamp_med3(dw, -SSD_T2, SSD_T2)) : 0.0f;
    const float pw = fabsf(dw) < SSD_T2 ? 1.0f : 0.0f;
    const float dts = s_dt[tg], gds = s_gd[tg];
    // dX^T += w_s B_s dst^T; E, x.dX, D.dy, dx
    float esum = 0.0f, xsum = 0.0f, dpart = 0.0f;
    const bf16* dyc = dYt + j * XT;
#pragma unroll
    for (int q = 0; q < PTW; ++q) {
      const int pt = 2 * q + wc;
      if (pt >= PT) continue;
      floatx16 tmp;
      zero(tmp);
#pragma unroll
      for (int kk = 0; kk < NP; kk += 16)
        mfma(tmp, tld8<NP>(dstT, 32 * pt + l32, kk + 8 * hh), tld8<NP>(Bt, t_loc, kk + 8 * hh));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p0 = 32 * pt + 8 * r + 4 * hh;
        const bf16x4 xv = tld4<PP>(xj, t_loc, p0);
        const bf16x4 yv = tld4<PP>(dyc, t_loc, p0);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * r + e;
          const float xf = (float)xv[e], yf = (float)yv[e];
          const float tv = tmp[v] * ws;
          const float dX = dXk[q][v] + tv;
          esum += xf * tv;
          xsum += xf * dX;
          dpart += xf * yf;
          o[e] = (bf16)(dts * dX + Dh * yf);
        }
        if (t_ok && p0 < d.P)
          *reinterpret_cast<bf16x4*>(a.dx + (int64_t)(ci.row0 + tg) * xrow + (int64_t)h * d.P + p0) = o;
      }
    }
    esum += __shfl_xor(esum, 32, 64);
    xsum += __shfl_xor(xsum, 32, 64);

    for (int o = 32; o > 0; o >>= 1) dpart += __shfl_xor(dpart, o, 64);
    if (hh == 0) {
      red_e[wc * 64 + t_loc] = esum * gds * pw;
      red_x[wc * 64 + t_loc] = xsum;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      const int tl = threadIdx.x, tgg = 64 * j + tl;
      if (tgg < ci.len) {
        const int64_t o = ((int64_t)c * d.H + h) * Qpad + tgg;
        a.eterm[o] = red_e[tl] + red_e[64 + tl];
        a.xdx[o] = red_x[tl] + red_x[64 + tl];
      }
    }
    for (int e = threadIdx.x; e < nt_i * 64; e += 256) {
      const int i = j + e / 64, l = e % 64;
      const int lg = 64 * i + l;
      if (lg < ci.len)
        a.rowG[(((int64_t)j * d.max_chunks + c) * d.H + h) * Qpad + lg] =
            red_row[(i * 2 + 0) * 64 + l] + red_row[(i * 2 + 1) * 64 + l];
    }
    __syncthreads();  // red_e / red_o reads done before the dD partials reuse red_o
    if (lane == 0) red_o[w] = dpart;
    __syncthreads();
    if (threadIdx.x == 0) a.dD_part[((int64_t)c * d.H + h) * nb + j] = red_o[0] + red_o[1] + red_o[2] + red_o[3];
    h = h_next;
  }

  // ---- outputs summed over the slice's heads ----
  float* dSbase = a.dS + (((int64_t)slc * d.max_chunks + c) * d.G + g) * (int64_t)(nb * nb) * 4096;
#pragma unroll
  for (int t = 0; t < kMaxSlots; ++t) {
    if (t >= nt_i) continue;
    float* tile = dSbase + (int64_t)((j + t) * nb + j) * 4096;
    const int l_loc = 32 * wc + l32;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      floatx4 q;
      q[0] = dS[t][4 * r + 0];
      q[1] = dS[t][4 * r + 1];
      q[2] = dS[t][4 * r + 2];
      q[3] = dS[t][4 * r + 3];
      *reinterpret_cast<floatx4*>(tile + l_loc * 64 + 32 * wr + 8 * r + 4 * hh) = q;
    }
  }
}

// Full mode: one block per unit of the numbering above. Fixup mode (a.fast): a grid sized to the chip,
// each block taking the units bid = blockIdx.x + k gridDim.x; it reads the flags of all its units at once
// and runs only those holding a head the factorised kernel left (launching one block per unit that
// mostly exits at once cost ~0.8 us per CU-wave of blocks: 26 us for 8 192 units).
template <int PT, int NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_bwd_main(SsdDims d, BwdMainArgs a, int total) {
  if (!a.fast) {
    bwd_main_block<PT, NT>(d, a, blockIdx.x);
    return;
  }
  __shared__ int s_need[SSD_FIX_UNITS];
  const int U = d.max_chunks * d.G * a.nslices;
  const int U8 = (U + 7) / 8 * 8;
  const int per = (total - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;  // <= SSD_FIX_UNITS
  for (int k = threadIdx.x; k < per; k += 256) s_need[k] = 0;
  __syncthreads();
  // (unit k, head) pairs over the block's threads; a unit's head range as bwd_main_block forms it
  const int hs = a.hslice;
  for (int q = threadIdx.x; q < per * hs; q += 256) {
    const int k = q / hs, hq = q % hs;
    const int u = (blockIdx.x + k * gridDim.x) % U8;
    if (u >= U) continue;
    const int c = u % d.max_chunks, gsl = u / d.max_chunks;
    const int g = gsl / a.nslices, slc = gsl % a.nslices;
    const int h = g * d.hpg + slc * hs + hq;
    if (slc * hs + hq < d.hpg && a.fast[(int64_t)c * d.H + h] == 0) s_need[k] = 1;
  }
  __syncthreads();
  for (int k = 0; k < per; ++k) {
    if (!s_need[k]) continue;
    __syncthreads();  // the previous unit's LDS reads are done
    bwd_main_block<PT, NT>(d, a, blockIdx.x + k * gridDim.x);
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// Shapes of the fused path; at launch it also needs 16-byte vector access
// (d.vec_x, d.vec_bc), otherwise ssd_bwd runs the column / row kernels. The kernels address a chunk's B / C
// rows with 32-bit byte offsets (x rows always fit: 255 rows of 65535 heads of 64 columns).
bool bwd_main_supported(int dtype, const SsdDims& d) {
  return dtype == 1 && d.Ppad <= 64 && d.Qpad <= 256 && d.Npad <= 128 && d.P % 8 == 0 && d.N % 8 == 0 &&
         (int64_t)d.Qpad * d.G * d.N * 2 <= INT32_MAX;
}

size_t lds_bwd_main(const SsdDims& d) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return BwdMainLds<1, 1>::bytes(d.Qpad);
    case 12: return BwdMainLds<1, 2>::bytes(d.Qpad);
    case 14: return BwdMainLds<1, 4>::bytes(d.Qpad);
    case 21: return BwdMainLds<2, 1>::bytes(d.Qpad);
    case 22: return BwdMainLds<2, 2>::bytes(d.Qpad);
    default: return BwdMainLds<2, 4>::bytes(d.Qpad);
  }
}

template <int PT, int NT>
static hipError_t bwd_main_t(const SsdDims& d, const BwdMainArgs& a, hipStream_t s) {
  const int U = d.max_chunks * d.G * a.nslices;
  const int blocks = (U + 7) / 8 * 8 * (d.Qpad / 64);
  const size_t lds = BwdMainLds<PT, NT>::bytes(d.Qpad);
  ensure_lds(k_bwd_main<PT, NT>, lds);
  const int grid = a.fast ? std::max(std::min(blocks, 256), (blocks + SSD_FIX_UNITS - 1) / SSD_FIX_UNITS) : blocks;
  hipLaunchKernelGGL((k_bwd_main<PT, NT>), dim3(grid), dim3(256), lds, s, d, a, blocks);
  return hipGetLastError();
}

static BwdMainArgs make_main_args(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx,
                                  bool fixup) {
  BwdMainArgs a;
  a.chunks = b.chunks;
  a.cs = b.cs;
  a.dst = b.dst16;
  a.x = reinterpret_cast<const bf16*>(in.x);
  a.dt = in.dt;
  a.Bm = reinterpret_cast<const bf16*>(in.B);
  a.Cm = reinterpret_cast<const bf16*>(in.C);
  a.Dv = in.D;
  a.dy = reinterpret_cast<const bf16*>(dy);
  a.dx = reinterpret_cast<bf16*>(dx);
  a.rowG = b.rowG;
  a.colG = b.colG;
  a.eterm = b.eterm;
  a.xdx = b.xdx;
  a.dD_part = b.dD_part;
  a.Dtok = b.Dtok;
  a.ddec = d.gdec ? b.tz_gam : in.dt;
  a.dS = fixup ? b.dS_fix : b.dS_tiles;
  a.nslices = fixup ? 1 : b.nslices;
  a.hslice = fixup ? d.hpg : b.hslice;
  a.fast = fixup ? b.fast : nullptr;
  return a;
}

hipError_t launch_bwd_main(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, bool fixup,
                           hipStream_t s) {
  const BwdMainArgs a = make_main_args(d, b, in, dy, dx, fixup);
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return bwd_main_t<1, 1>(d, a, s);
    case 12: return bwd_main_t<1, 2>(d, a, s);
    case 14: return bwd_main_t<1, 4>(d, a, s);
    case 21: return bwd_main_t<2, 1>(d, a, s);
    case 22: return bwd_main_t<2, 2>(d, a, s);
    default: return bwd_main_t<2, 4>(d, a, s);
  }
}

int bwd_main_num_sets(const SsdDims& d) { return d.Qpad / 64; }
