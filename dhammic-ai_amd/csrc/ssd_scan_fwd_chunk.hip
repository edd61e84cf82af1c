// Forward chunk scan for bf16 inputs (gfx950): for every chunk and head
//   Y = (S * L) X~ + exp(cs) C h_in^T (+ D x),   S = C B^T, X~ = dt x,
//   L[l,s] = exp(clamp(cs_l - cs_s)) for s <= l (exact zero above the diagonal)
// (r2/dhammic-ai/src/kernels/ssd_scan.py:370-385 for the diagonal blocks,
// :412-417 for the state term; the reference's acausal e^-20 entries, :111-116,
// are not reproduced: they change Y by at most e^-20 * sum|terms|).
//
// One block (4 waves) per (chunk, group, slice of heads); the block computes
// the whole chunk for each head, so x and h_in of a (chunk, head) are read
// once. Work split: the output is Y^T[p][l]; its l axis is cut into 32-token
// quadrants (i, lh) (64-token block i, half lh). Quadrant (i, lh) needs the
// 32 x 32 units (j, sh) of M^T[s][l] with s in block j half sh, s <= l:
// 2 i + lh + 1 of them. Wave w owns two quadrants, {(3,1),(0,0)}, {(3,0),(0,1)},
// {(2,1),(1,0)}, {(2,0),(1,1)}: nine units each for a full chunk, no unit
// computed twice and no partial sums across waves.
//   S^T units are computed once per block (K = N) and kept in registers (bf16).
//   Per head and unit: M^T = S^T * exp2(clamp(cs_l - cs_s)) * dt_s in registers,
//   used directly as the B operand of Y^T += X~^T M^T (the x tile read
//   transposed in the accumulator's row order); Y_off^T = h_in C^T scaled by
//   exp(clamp(cs_l)) per lane. The next head's x / h_in / cs / dt are loaded
//   into registers while the current head computes.
// This exact per-element form runs as the fixup of the factorised kernel
// (ssd_scan_fwd_fact.hip): with `fast` given, only blocks whose head slice
// holds a (chunk, head) flagged 0 run, and they rewrite their whole slice.
// S32 (halves of wide heads, whole grid): S^T stays in fp32 registers, so M is the only operand that is
// rounded, as in the general kernel that takes such heads whole. The factorised kernel rounds S' and the
// scaled x: y of the reference op with 128-column heads is 2.87e-3 from 64 bits there, 2.37e-3 here.
// Price, forward and backward at B=4 L=2048 H=16 P=128 N=64 chunk 256 with the norm: 254 -> 288 us (whole heads on
// the general kernels: 605). Up to 128-token chunks two blocks share a CU, where a lone one waits for its loads: 8 x 2048
// tokens of 32 heads of 128 columns, 32 groups, N=16, chunk 64, the forward 355 -> 249 us (whole heads 285).
#include <stdint.h>

#include <algorithm>

#include "ssd_launch.h"
#include "ssd_tile.h"

namespace {

constexpr int kUnits = 9;  // S^T units per wave (full 256-token chunk)


template <int PT, int NT>
struct FwdLds {
  static constexpr int PP = 32 * PT, NP = 32 * NT;
  static size_t bytes(int nb) {
    return 2 * (size_t)(nb * tsize<64, NP>() + nb * tsize<64, PP>() + tsize<PP, NP>()) + sizeof(float) * 3 * 64 * nb;
  }
};

template <int PT, int NT, int NB>
struct FwdStage {
  TileStage<64, 32 * PT, 256> x[NB];
  TileStage<32 * PT, 32 * NT, 256> hin;
  float cs, dt, dtk;
};

}  // namespace

#define SSD_FWD_CHUNK_PARAMS                                                                                  \
  SsdDims d, int hslice, int nslices, const ChunkInfo* __restrict__ chunks, const float* __restrict__ cs,         \
      const bf16* __restrict__ hin, const bf16* __restrict__ x, const float* __restrict__ dt,                    \
      const bf16* __restrict__ Bm, const bf16* __restrict__ Cm, const float* __restrict__ Dv,                     \
      bf16* __restrict__ y, const int32_t* __restrict__ fast, const float* __restrict__ Dtok
#define SSD_FWD_CHUNK_ARGS d, hslice, nslices, chunks, cs, hin, x, dt, Bm, Cm, Dv, y, fast, Dtok

// The work of block `bid`: (chunk bid % max_chunks, group and head slice bid / max_chunks).
template <int PT, int NT, int NB, bool S32>
__device__ __forceinline__ void scan_fwd_chunk_block(int bid, SSD_FWD_CHUNK_PARAMS) {
  constexpr int PP = 32 * PT, NP = 32 * NT;
  constexpr int XT = tsize<64, PP>(), CT = tsize<64, NP>();
  extern __shared__ __align__(16) unsigned char smem[];
  const int c = bid % d.max_chunks;
  const int gsl = bid / d.max_chunks;
  const int g = gsl / nslices, slc = gsl % nslices;
  const ChunkInfo ci = chunks[c];
  if (ci.len == 0) return;
  const int nbl = (ci.len + 63) >> 6;
  const int h_lo = g * d.hpg + slc * hslice;
  const int h_hi = min(h_lo + hslice, (g + 1) * d.hpg);
  if (h_lo >= h_hi) return;
  if (fast) {
    // fixup mode: only slices holding a head the factorised kernel cannot take
    bool need = false;
    for (int h = h_lo + (int)threadIdx.x; h < h_hi; h += 256) need = need || fast[(int64_t)c * d.H + h] == 0;
    if (!__syncthreads_or(need)) return;
  }
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;

  bf16* Ct = reinterpret_cast<bf16*>(smem);  // [NB][64][NP]
  bf16* xt = Ct + NB * CT;                   // [NB][64][PP]
  bf16* ht = xt + NB * XT;                   // [PP][NP]
  float* s_cs2 = reinterpret_cast<float*>(ht + tsize<PP, NP>());  // [64 NB]
  float* s_dt = s_cs2 + 64 * NB;
  float* s_dtk = s_dt + 64 * NB;  // trapezoidal mode: D per token

  // quadrants of this wave: slot 0 = (NB - 1 - w/2, 1 - w%2), slot 1 = (w/2, w%2)
  // while w/2 < NB - 2 (beyond that slot 0 of another wave already holds it);
  // a quadrant past the chunk's last block is empty
  int qi[2], qlh[2], qn[2];
  qi[0] = (NB - 1) - (w >> 1);
  qlh[0] = 1 - (w & 1);
  qi[1] = w >> 1;
  qlh[1] = w & 1;
  qn[0] = (qi[0] >= 0 && qi[0] < nbl) ? 2 * qi[0] + qlh[0] + 1 : 0;
  qn[1] = (qi[1] < NB - 2 && qi[1] < nbl) ? 2 * qi[1] + qlh[1] + 1 : 0;
  const int nU = qn[0] + qn[1];

  // ---- C tiles of the chunk ----
#pragma unroll
  for (int i = 0; i < NB; ++i)
    if (i < nbl) {
      TileStage<64, NP, 256> st;
      tstage_load_v(st, Cm + (int64_t)(ci.row0 + 64 * i) * brow + (int64_t)g * d.N, brow, min(64, ci.len - 64 * i),
                    d.N);
      tstage_store(st, Ct + i * CT);
    }
  __syncthreads();

  // ---- S^T units: rows s (block j half sh), lanes l (quadrant) ----
  bf16x8 S[S32 ? 1 : kUnits][2];
  floatx16 Sf[S32 ? kUnits : 1];
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    floatx16 sacc;
    zero(sacc);
    if (u < nU) {
      const int q = u < qn[0] ? 0 : 1;
      const int uu = u < qn[0] ? u : u - qn[0];
      const int j = uu >> 1, sh = uu & 1;
      const int srow = 64 * j + 32 * sh + (lane & 31);
      const bool sok = srow < ci.len;
      const bf16* brp = Bm + (int64_t)(ci.row0 + (sok ? srow : 0)) * brow + (int64_t)g * d.N;
#pragma unroll
      for (int kk = 0; kk < NP; kk += 16) {
        const int n0 = kk + 8 * (lane >> 5);
        bf16x8 bv;
#pragma unroll
        for (int e = 0; e < 8; ++e) bv[e] = (bf16)0.0f;
        if (sok && n0 < d.N) bv = *reinterpret_cast<const bf16x8*>(brp + n0);
        mfma(sacc, bv, tld8<NP>(Ct + qi[q] * CT, 32 * qlh[q] + (lane & 31), n0));
      }
    }
    if constexpr (S32) {
      Sf[u] = sacc;
    } else {
      S[u][0] = acc_frag(sacc, 0);
      S[u][1] = acc_frag(sacc, 1);
    }
  }

  // ---- per-head loop with the next head's inputs in flight ----
  FwdStage<PT, NT, NB> st;
  auto load_head = [&](int h) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i < nbl)
        tstage_load_v(st.x[i], x + (int64_t)(ci.row0 + 64 * i) * xrow + (int64_t)h * d.P, xrow,
                      min(64, ci.len - 64 * i), d.P);
    tstage_load_v(st.hin, hin + ((int64_t)c * d.H + h) * PP * NP, NP, PP, NP);
    st.cs = 0.0f;
    st.dt = 1.0f;
    st.dtk = 0.0f;
    if (threadIdx.x < 64 * NB) {
      st.cs = cs[((int64_t)c * d.H + h) * d.Qpad + threadIdx.x];
      if (d.has_dt && (int)threadIdx.x < ci.len) st.dt = dt[(int64_t)(ci.row0 + threadIdx.x) * d.H + h];
      if (d.trapz && (int)threadIdx.x < ci.len) st.dtk = Dtok[(int64_t)(ci.row0 + threadIdx.x) * d.H + h];
    }
  };
  load_head(h_lo);
  for (int h = h_lo; h < h_hi; ++h) {
    lane = opaque_lane();
    if constexpr (!S32) {
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
        launder(S[u][0]);
        launder(S[u][1]);
      }
    }
    __syncthreads();  // the previous head's LDS reads are done
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (i < nbl) tstage_store(st.x[i], xt + i * XT);
    tstage_store(st.hin, ht);
    if (threadIdx.x < 64 * NB) {
      s_cs2[threadIdx.x] = st.cs * SSD_LOG2E;
      s_dt[threadIdx.x] = st.dt;
      s_dtk[threadIdx.x] = st.dtk;
    }
    __syncthreads();
    if (h + 1 < h_hi) load_head(h + 1);
    const float Dh = d.has_D ? Dv[h] : 0.0f;

#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (qn[q] == 0) continue;
      const int i = qi[q], lh = qlh[q];
      const int l_loc = 32 * lh + (lane & 31);  // lane's token within block i
      const int lg = 64 * i + l_loc;
      const float cs_l = s_cs2[lg];
      // Y_off^T[p][l] = exp(clamp(cs_l)) sum_n h_in[p][n] C[l][n]
      floatx16 acc[PT];
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) {
        zero(acc[pt]);
#pragma unroll
        for (int kk = 0; kk < NP; kk += 16)
          mfma(acc[pt], tld8<NP>(ht, 32 * pt + (lane & 31), kk + 8 * (lane >> 5)),
               tld8<NP>(Ct + i * CT, l_loc, kk + 8 * (lane >> 5)));
        const float e = exp2_fast(clamp_med3(cs_l, -SSD_T2, SSD_T2));
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[pt][v] *= e;
      }
      // Y_diag^T[p][l] += sum_s X~^T[p][s] M^T[s][l]
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
        const int base = q == 0 ? 0 : qn[0];
        if (u < base || u >= base + qn[q]) continue;
        const int uu = u - base;
        const int j = uu >> 1, sh = uu & 1;
        const bool diag = j == i && sh == lh;
        float css[16], dts[16];
        rows16(s_cs2 + 64 * j + 32 * sh, css);
        rows16(s_dt + 64 * j + 32 * sh, dts);
        floatx16 m;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float dd = cs_l - css[v];
          float sv;
          if constexpr (S32)
            sv = Sf[u][v];
          else
            sv = (float)S[u][v >> 3][v & 7];
          float mv = sv * exp2_fast(clamp_med3(dd, -SSD_T2, SSD_T2)) * dts[v];
          if (diag && acc_row(v, lane) + (d.trapz ? 1 : 0) > (lane & 31)) mv = 0.0f;  // trapz: strict
          m[v] = mv;
        }
        const bf16* xj = xt + j * XT;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const bf16x8 mb = acc_frag(m, kk);
#pragma unroll
          for (int pt = 0; pt < PT; ++pt) mfma(acc[pt], ttr_perm<PP>(xj, 32 * sh, kk, 32 * pt, lane), mb);
        }
      }
      // epilogue: + D x, store y[l][p] (lane l writes 4 consecutive p per register group)
      if (lg < ci.len) {
        const bf16* xi = xt + i * XT;
        const float Dl = d.trapz ? s_dtk[lg] : Dh;
        bf16* yrow = y + (int64_t)(ci.row0 + lg) * xrow + (int64_t)h * d.P;
#pragma unroll
        for (int pt = 0; pt < PT; ++pt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int p0 = 32 * pt + 8 * r + 4 * (lane >> 5);
            if (p0 >= d.P) continue;
            const bf16x4 xv = tld4<PP>(xi, l_loc, p0);
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (bf16)(acc[pt][4 * r + e] + Dl * (float)xv[e]);
            *reinterpret_cast<bf16x4*>(yrow + p0) = o;
          }
      }
    }
  }
}

// Full mode: one block per (chunk, group, head slice). Fixup mode (fast): a grid sized to the chip, each
// block taking the units blockIdx.x + k gridDim.x, reading all their flags at once and running only the
// units holding a flagged head (a block per unit that mostly exits at once costs a launch wave per
// 256 of them).
template <int PT, int NT, int NB, bool S32>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, S32 && NB <= 2 ? 2 : 1)))
k_scan_fwd_chunk(int total, SSD_FWD_CHUNK_PARAMS) {
  if (S32 || !fast) {
    scan_fwd_chunk_block<PT, NT, NB, S32>(blockIdx.x, SSD_FWD_CHUNK_ARGS);
    return;
  }
  __shared__ int s_need[SSD_FIX_UNITS];
  const int per = (total - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;  // <= SSD_FIX_UNITS
  for (int k = threadIdx.x; k < per; k += 256) s_need[k] = 0;
  __syncthreads();
  for (int q = threadIdx.x; q < per * hslice; q += 256) {
    const int k = q / hslice, hq = q % hslice;
    const int u = blockIdx.x + k * gridDim.x;
    const int c = u % d.max_chunks, gsl = u / d.max_chunks;
    const int g = gsl / nslices, slc = gsl % nslices;
    if (slc * hslice + hq < d.hpg && fast[(int64_t)c * d.H + g * d.hpg + slc * hslice + hq] == 0) s_need[k] = 1;
  }
  __syncthreads();
  for (int k = 0; k < per; ++k) {
    if (!s_need[k]) continue;
    __syncthreads();  // the previous unit's LDS reads are done
    scan_fwd_chunk_block<PT, NT, NB, S32>(blockIdx.x + k * gridDim.x, SSD_FWD_CHUNK_ARGS);
  }
}

// Shapes of this kernel: bf16, P <= 64 and N <= 128 multiples of 8, chunk <= 256,
// 16-byte vector access (the caller checks d.vec_x / d.vec_bc).
bool scan_fwd_chunk_supported(int dtype, const SsdDims& d) {
  return dtype == 1 && d.Ppad <= 64 && d.Npad <= 128 && d.Qpad <= 256 && d.P % 8 == 0 && d.N % 8 == 0;
}

size_t lds_scan_fwd_chunk(const SsdDims& d) {
  const int nb = d.Qpad / 64;
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return FwdLds<1, 1>::bytes(nb);
    case 12: return FwdLds<1, 2>::bytes(nb);
    case 14: return FwdLds<1, 4>::bytes(nb);
    case 21: return FwdLds<2, 1>::bytes(nb);
    case 22: return FwdLds<2, 2>::bytes(nb);
    default: return FwdLds<2, 4>::bytes(nb);
  }
}

template <int PT, int NT, int NB, bool S32>
static hipError_t scan_fwd_chunk_t(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y,
                                   const int32_t* fast, hipStream_t s) {
  // heads per block: about four blocks per CU over the grid
  const int per = d.max_chunks * d.G;
  int ns = (1024 + per - 1) / per;
  if (ns < 1) ns = 1;
  if (ns > d.hpg) ns = d.hpg;
  int hslice = (d.hpg + ns - 1) / ns;
  if constexpr (S32) {
    // the whole grid runs, each block building S for its heads: the slices whose blocks take the least time in whole
    // passes over the chip, the block's set-up and S at 1 + NT / 4 heads' time. The halves of a head share S. How many chunks packed sequences
    // have the host does not know (chunks start at each sequence, and one a sequence ends short): the mean over 0.3,
    // 0.5 and 0.7 chunks more per sequence than their tokens fill.
    const int64_t slots = NB <= 2 ? 512 : 256, full = (d.seqlen + d.Q - 1) / d.Q;
    int64_t best = INT64_MAX;
    for (int q = 2; q <= std::max(2, d.hpg); ++q) {
      const int64_t slices = (d.hpg + q - 1) / q;
      int64_t passes = 0;
      for (int e = 3; e <= 7; e += 2) {
        const int64_t chunks = d.varlen ? full + (e * (int64_t)d.nseq + 9) / 10 : d.max_chunks;
        passes += (chunks * d.G * slices + slots - 1) / slots;
      }
      if (passes * (4 * q + 4 + NT) < best) {
        best = passes * (4 * q + 4 + NT);
        hslice = q;
      }
    }
  }
  ns = (d.hpg + hslice - 1) / hslice;
  const size_t lds = FwdLds<PT, NT>::bytes(NB);
  ensure_lds(k_scan_fwd_chunk<PT, NT, NB, S32>, lds);
  const int blocks = d.max_chunks * d.G * ns;
  const int grid = fast ? std::max(std::min(blocks, 256), (blocks + SSD_FIX_UNITS - 1) / SSD_FIX_UNITS) : blocks;
  hipLaunchKernelGGL((k_scan_fwd_chunk<PT, NT, NB, S32>), dim3(grid), dim3(256), lds, s, blocks, d, hslice, ns,
                     b.chunks, b.cs, reinterpret_cast<const bf16*>(b.hin), reinterpret_cast<const bf16*>(in.x), in.dt,
                     reinterpret_cast<const bf16*>(in.B), reinterpret_cast<const bf16*>(in.C), in.D,
                     reinterpret_cast<bf16*>(y), fast, b.Dtok);
  return hipGetLastError();
}

template <int PT, int NT, bool S32 = false>
static hipError_t scan_fwd_chunk_nb(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y,
                                    const int32_t* fast, hipStream_t s) {
  switch (d.Qpad / 64) {
    case 1: return scan_fwd_chunk_t<PT, NT, 1, S32>(d, b, in, y, fast, s);
    case 2: return scan_fwd_chunk_t<PT, NT, 2, S32>(d, b, in, y, fast, s);
    case 3: return scan_fwd_chunk_t<PT, NT, 3, S32>(d, b, in, y, fast, s);
    default: return scan_fwd_chunk_t<PT, NT, 4, S32>(d, b, in, y, fast, s);
  }
}

hipError_t launch_scan_fwd_chunk(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, const int32_t* fast,
                                 hipStream_t s) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return scan_fwd_chunk_nb<1, 1>(d, b, in, y, fast, s);
    case 12: return scan_fwd_chunk_nb<1, 2>(d, b, in, y, fast, s);
    case 14: return scan_fwd_chunk_nb<1, 4>(d, b, in, y, fast, s);
    case 21: return scan_fwd_chunk_nb<2, 1>(d, b, in, y, fast, s);
    case 22: return scan_fwd_chunk_nb<2, 2>(d, b, in, y, fast, s);
    default: return scan_fwd_chunk_nb<2, 4>(d, b, in, y, fast, s);
  }
}

// Every (chunk, head) with S in fp32: the halves of 80- to 128-column heads, 40 to 64 columns each.
hipError_t launch_scan_fwd_pairs(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  switch (d.Npad / 32) {
    case 1: return scan_fwd_chunk_nb<2, 1, true>(d, b, in, y, nullptr, s);
    case 2: return scan_fwd_chunk_nb<2, 2, true>(d, b, in, y, nullptr, s);
    default: return scan_fwd_chunk_nb<2, 4, true>(d, b, in, y, nullptr, s);
  }
}
