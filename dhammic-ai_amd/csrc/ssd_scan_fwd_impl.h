// Forward chunk scan kernel template of the general bf16 path (instantiated in ssd_scan_fwd_bf16.hip).
//   Y = (C B^T * L) X + exp(cs) C h_in^T (+ D x)
#pragma once

#include "ssd_launch.h"

// ---------------------------------------------------------------------------
// One block per (row block rb of 64 tokens, slice of HS heads of one group,
// chunk c). Shapes are compile-time: Ppad = 32*PT, Npad = 32*NT. Wave w owns
// rows l in half lh = w/2 and the 32-wide p tiles t with t%2 == w%2 of the
// 64 x Ppad output of every head of the slice.
//   Y_off (ssd_scan.py:412-415): acc_h = C_rb h_in,h^T over K = N (h_in read
//       from global in its [p][n] layout, k-contiguous), rows scaled by exp(cs_l).
//   Y_diag (:370-385): for each column block j <= rb and each 32-row half of
//       it, the wave forms S^T = B_j C_rb^T (K = N) once for the slice, applies
//       exp(clamp(cs_l - cs_s)) * dt_s per head on the causal part (exact zero
//       above the diagonal) in registers, and feeds that tile directly as the
//       A operand of acc_h += M x_j (mma_xt, no LDS round trip for M).
//   The reference's acausal e^-20 entries (the clamped -1e4 fill, :111-116)
//   are not reproduced: they change Y by at most e^-20 * sum|terms|.
// B and x rows of block j+1 are loaded into registers while block j computes.
// ---------------------------------------------------------------------------
template <typename T, int HS, int PT, int NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_chunk_scan_fwd(SsdDims d, const ChunkInfo* __restrict__ chunks,
                                                        const float* __restrict__ cs, const T* __restrict__ hin,
                                                        const T* __restrict__ x, const float* __restrict__ dt,
                                                        const T* __restrict__ Bm, const T* __restrict__ Cm,
                                                        const float* __restrict__ Dv, T* __restrict__ y,
                                                        const float* __restrict__ Dtok) {
  constexpr int PPAD = 32 * PT, NPAD = 32 * NT;
  constexpr int NP = lds_pitch<T>(NPAD), BP = lds_pitch<T>(SSD_BLK);
  constexpr int MYT = (PT + 1) / 2;  // p tiles per wave
  extern __shared__ __align__(16) unsigned char smem[];
  const int rb = blockIdx.x, h0 = blockIdx.y * HS, c = blockIdx.z;
  const ChunkInfo ci = chunks[c];
  const int r0 = rb * SSD_BLK;
  if (r0 >= ci.len) return;
  const int g = h0 / d.hpg;
  const int Qpad = d.Qpad;
  float* s_cs = reinterpret_cast<float*>(smem);  // [HS][Qpad]
  float* s_dt = s_cs + HS * Qpad;                 // [HS][Qpad]
  T* Ci = reinterpret_cast<T*>(s_dt + HS * Qpad);  // [64][NP]
  T* Bj = Ci + SSD_BLK * NP;                       // [64][NP]
  T* xT = Bj + SSD_BLK * NP;                       // [HS][PPAD][BP]

  for (int idx = threadIdx.x; idx < HS * Qpad; idx += blockDim.x) {
    const int k = idx / Qpad, l = idx - k * Qpad;
    s_cs[idx] = cs[((int64_t)c * d.H + h0 + k) * Qpad + l];
    s_dt[idx] = (d.has_dt && l < ci.len) ? dt[(int64_t)(ci.row0 + l) * d.H + h0 + k] : 1.0f;
  }
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  stage_nat<T>(Ci, NP, Cm, brow, (int64_t)g * d.N, ci.row0, r0, ci.len, d.N, NPAD, d.vec_bc);

  TileRegs<T, NPAD> rbj;
  TileRegs<T, PPAD> rxj[HS];
  auto load_blk = [&](int jj) {
    tile_load<T, false>(rbj, Bm, brow, (int64_t)g * d.N, ci.row0, jj * SSD_BLK, ci.len, d.N, NPAD, d.vec_bc);
#pragma unroll
    for (int k = 0; k < HS; ++k)
      tile_load<T, true>(rxj[k], x, xrow, (int64_t)(h0 + k) * d.P, ci.row0, jj * SSD_BLK, ci.len, d.P, PPAD,
                         d.vec_x);
  };
  load_blk(0);
  __syncthreads();

  const int lane = lane_id();
  const int w = threadIdx.x >> 6, lh = w >> 1, ph = w & 1;
  const int l_me = r0 + lh * 32 + (lane & 31);  // this lane's l in the S^T tiles
  const bool l_ok = l_me < ci.len;
  floatx16 acc[HS][MYT];
  float cs_l[HS];
  // Y_off
#pragma unroll
  for (int k = 0; k < HS; ++k) {
    cs_l[k] = s_cs[k * Qpad + l_me];
    const T* hrow = hin + ((int64_t)c * d.H + h0 + k) * PPAD * NPAD;
    float rc[16];
    rows16(s_cs + k * Qpad + r0 + lh * 32, rc);
#pragma unroll
    for (int tt = 0; tt < MYT; ++tt) {
      zero(acc[k][tt]);
      const int t = 2 * tt + ph;
      if (t < PT) mma_k<T, NPAD>(acc[k][tt], Ci + lh * 32 * NP, NP, hrow + t * 32 * NPAD, NPAD);
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[k][tt][v] *= exp_clamp(rc[v]);
    }
  }
  // Y_diag
  for (int j = 0; j <= rb; ++j) {
    __syncthreads();
    tile_store_nat<T, false>(rbj, Bj, NP, NPAD);
#pragma unroll
    for (int k = 0; k < HS; ++k) tile_store_tr<T>(rxj[k], xT + k * PPAD * BP, BP, PPAD);
    __syncthreads();
    if (j < rb) load_blk(j + 1);
#pragma unroll
    for (int sh = 0; sh < 2; ++sh) {
      floatx16 st;
      zero(st);
      mma_k<T, NPAD>(st, Bj + sh * 32 * NP, NP, Ci + lh * 32 * NP, NP);  // S^T[s][l]
      const int sb = j * SSD_BLK + sh * 32;
#pragma unroll
      for (int k = 0; k < HS; ++k) {
        float css[16], dts[16];
        rows16(s_cs + k * Qpad + sb, css);
        rows16(s_dt + k * Qpad + sb, dts);
        floatx16 X;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int s = sb + acc_row(v, lane);
          const float m = st[v] * exp_clamp(cs_l[k] - css[v]) * dts[v];
          X[v] = (s + (d.trapz ? 1 : 0) <= l_me && l_ok) ? m : 0.0f;  // trapezoidal mode: strictly causal
        }
        const AccFrags<T> xf = acc_frags<T>(X);
#pragma unroll
        for (int tt = 0; tt < MYT; ++tt) {
          const int t = 2 * tt + ph;
          if (t < PT) mma_xt_f<T>(acc[k][tt], xf, xT + k * PPAD * BP + t * 32 * BP + sh * 32, BP);
        }
      }
    }
  }
  // epilogue: + D x, store
#pragma unroll
  for (int k = 0; k < HS; ++k) {
    const int h = h0 + k;
    const float Dh = d.has_D ? Dv[h] : 0.0f;
#pragma unroll
    for (int tt = 0; tt < MYT; ++tt) {
      const int t = 2 * tt + ph;
      const int p = t * 32 + (lane & 31);
      if (t >= PT || p >= d.P) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int l = r0 + lh * 32 + acc_row(v, lane);
        if (l >= ci.len) continue;
        const int64_t o = (int64_t)(ci.row0 + l) * xrow + (int64_t)h * d.P + p;
        float yv = acc[k][tt][v];
        // trapezoidal mode: D per token
        if (d.has_D || d.trapz) yv += (d.trapz ? Dtok[(int64_t)(ci.row0 + l) * d.H + h] : Dh) * to_f(x[o]);
        y[o] = from_f<T>(yv);
      }
    }
  }
}

inline size_t lds_scan_fwd_hs(size_t es, const SsdDims& d, size_t hs) {
  const size_t NP = d.Npad + 16 / es, BP = SSD_BLK + 16 / es;
  return 2 * sizeof(float) * hs * d.Qpad + es * (2 * SSD_BLK * NP + hs * d.Ppad * BP);
}

// Heads per block: 2 when the heads of a group allow it and two blocks then fit
// one CU's LDS (80 KiB each), else 1. All heads of a block share B and C; two
// heads keep the register count low enough for two blocks per CU, whose
// interleaving hides the barrier and load latency of each.
inline int fwd_heads_per_block(size_t es, const SsdDims& d) {
  if (d.hpg % 2 == 0 && lds_scan_fwd_hs(es, d, 2) <= 80 * 1024) return 2;
  return 1;
}

template <typename T, int HS, int PT, int NT>
hipError_t scan_fwd_t(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  dim3 grid(d.Qpad / SSD_BLK, d.H / HS, d.max_chunks);
  const size_t lds = lds_scan_fwd_hs(sizeof(T), d, HS);
  ensure_lds(k_chunk_scan_fwd<T, HS, PT, NT>, lds);
  hipLaunchKernelGGL((k_chunk_scan_fwd<T, HS, PT, NT>), grid, dim3(256), lds, s, d, b.chunks, b.cs,
                     reinterpret_cast<const T*>(b.hin), reinterpret_cast<const T*>(in.x), in.dt,
                     reinterpret_cast<const T*>(in.B), reinterpret_cast<const T*>(in.C), in.D,
                     reinterpret_cast<T*>(y), b.Dtok);
  return hipGetLastError();
}

template <typename T, int HS, int PT>
hipError_t scan_fwd_n(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  switch (d.Npad) {
    case 32: return scan_fwd_t<T, HS, PT, 1>(d, b, in, y, s);
    case 64: return scan_fwd_t<T, HS, PT, 2>(d, b, in, y, s);
    default: return scan_fwd_t<T, HS, PT, 4>(d, b, in, y, s);
  }
}

template <typename T, int HS>
hipError_t scan_fwd_p(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  switch (d.Ppad) {
    case 32: return scan_fwd_n<T, HS, 1>(d, b, in, y, s);
    case 64: return scan_fwd_n<T, HS, 2>(d, b, in, y, s);
    default: return scan_fwd_n<T, HS, 4>(d, b, in, y, s);
  }
}

template <typename T>
hipError_t scan_fwd_dispatch(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s) {
  const int hs = fwd_heads_per_block(sizeof(T), d);
  if (hs == 2) return scan_fwd_p<T, 2>(d, b, in, y, s);
  return scan_fwd_p<T, 1>(d, b, in, y, s);
}
