// Trapezoidal two-SSD mode: the coefficient kernels around the one scan that
// computes both SSD calls of r2/dhammic-ai/src/mamba_base_engine.py:167-183,
//   y = SSD(gamma x, a, B, C) + SSD(beta x_prev, a, B_prev, C),
// x_prev[t] = x[t-1], B_prev[t] = B[t-1], both zero at a sequence's first token.
//
// With rho[t] = beta[t+1] exp(-a[t+1]) (zero at a sequence's last token), the
// state h~[t] = exp(a[t]) h~[t-1] + (gamma[t] + rho[t]) x[t] B[t]^T equals the
// sum of the two paths' states plus rho[t] x[t] B[t]^T, the beta input of token
// t+1 taken in one step early (exp(a[t+1]) rho[t] = beta[t+1]). So
//   y[t] = C[t] h~[t] - rho[t] (C[t] . B[t]) x[t]
//        = sum_{s < t} (C[t] . B[s]) L[t, s] (gamma + rho)[s] x[s] + state term + gamma[t] (C[t] . B[t]) x[t]:
// the scan runs once, strictly causal, with dt = gamma + rho, and the diagonal
// term is a per-token D, D[t] = D + gamma (C . B). The gradient at dt of the
// strict scan is drho, dgamma = drho + (C . B)(x . dy), dbeta[t+1] =
// drho[t] exp(-a[t+1]) and, through both paths (EXACT_DA), da[t+1] -= drho[t]
// rho[t]; d(C . B) = sum_h gamma (x . dy) enters dB and dC as the diagonal of
// dS. Nothing is subtracted, so no gradient loses digits to cancellation.
//
// The reference's second call reuses the first call's cache (L, decay_chunk,
// A_cumsum), so the beta path contributes nothing to dA (ssd_scan.py:476-533);
// DROP_BETA_DA keeps that: its dA is the gamma path's alone, from a second
// backward of SSD(gamma x, a, B, C) over the gamma path's states.
//
// Steep decays. The fold's factor exp(-a[t+1]) is taken with its exponent
// capped at 20 (so it cannot overflow; beta = (1 - lam) dt e^a has then
// underflowed below the reference's e^-20 floor, and rho x B with it), the
// same cap in dbeta. Where a[t+1] < -8 the fold's dbeta is not the beta call's:
// its decays are anchored at t, where the reference's clamp binds, instead of
// t+1. There k_trapz_dbeta_steep evaluates dbeta from the beta call's own
// definition (intra-chunk terms and the chunk state's gradient). Every other
// output takes the beta path's inputs only through beta x_prev and beta B_prev,
// so the fold's error there is below beta e^-8 times its terms.
#include "ssd_mi355x.h"
#include "ssd_launch.h"
#include "ssd_tile.h"

// Decay below which the fold's dbeta is replaced by the beta call's own (k_trapz_dbeta_steep): above it
// the fold's clamp mismatch moves a dbeta term by less than e^(-20 - a) <= e^-12 of its size.
#define SSD_TRAPZ_STEEP (-8.0f)

namespace {

// [start, end) of the sequence holding `row` and its index (end = start: row is in none)
__device__ __forceinline__ int tz_seq(const SsdDims& d, const int32_t* __restrict__ cu, int64_t row, int64_t& start,
                                      int64_t& end) {
  if (!d.varlen) {
    const int s = (int)(row / d.seqlen);
    start = (int64_t)s * d.seqlen;
    end = start + d.seqlen;
    return s;
  }
  const int64_t R = d.R;
  int lo = 0, hi = d.nseq - 1;  // last s with cu[s] <= row (offsets clamped as the chunk table does)
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (min<int64_t>(max(cu[mid], 0), R) <= row) lo = mid; else hi = mid - 1;
  }
  start = min<int64_t>(max(cu[lo], 0), R);
  end = min<int64_t>(max<int64_t>(cu[lo + 1], start), R);
  if (row < start || row >= end) end = start = row;
  return lo;
}

// Index of `row` (in sequence `seq` starting at `start`) in the [max_chunks][H][Qpad] per-position
// arrays, head 0: chunks restart at every sequence start (k_chunk_table).
__device__ __forceinline__ int64_t tz_pos(const SsdDims& d, const SsdBufs& b, int64_t row, int64_t start, int seq) {
  const int64_t c0 = d.varlen ? b.seq_chunk0[seq] : (int64_t)seq * ((d.seqlen + d.Q - 1) / d.Q);
  const int64_t k = (row - start) / d.Q;
  return (c0 + k) * d.H * d.Qpad + (row - start - k * d.Q);
}

// exp(-a) with the exponent capped at SSD_HI: rho[t] = beta[t+1] e^{-a[t+1]} without overflow.
__device__ __forceinline__ float trapz_unfold(float a) { return exp2_fast(fminf(-a, SSD_HI) * SSD_LOG2E); }

}  // namespace

// cb[row][g] = C[row, g] . B[row, g]; one wave per (row, group), lanes over the state dim.
template <typename T>
__global__ void __launch_bounds__(256) k_trapz_cb(SsdDims d, const T* __restrict__ B, const T* __restrict__ C,
                                                  float* __restrict__ cb) {
  const int64_t row = blockIdx.x;
  const int g = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= d.G) return;
  const int64_t o = (row * d.G + g) * d.N;
  float s = 0.0f;
  for (int n = lane; n < d.N; n += 64) s += to_f(B[o + n]) * to_f(C[o + n]);
  for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
  if (lane == 0) cb[row * d.G + g] = s;
}

// The same with one wave per row reading its G N values as contiguous 16-byte vectors (bf16, N / 8 a
// power of two up to 64, aligned rows): a load instruction covers 1 KB of the row, the N / 8 lanes of
// a group hold its pieces, and their partial sums meet by butterfly shuffles.
__global__ void __launch_bounds__(256) k_trapz_cb_v(SsdDims d, const bf16* __restrict__ B, const bf16* __restrict__ C,
                                                    float* __restrict__ cb) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= d.R) return;
  const int lane = threadIdx.x & 63;
  const int per = d.N >> 3;                     // lanes (16-byte pieces) per group
  const int nq = d.G * per;                     // pieces of the row
  const bf16x8* b8 = reinterpret_cast<const bf16x8*>(B + row * d.G * d.N);
  const bf16x8* c8 = reinterpret_cast<const bf16x8*>(C + row * d.G * d.N);
  for (int q0 = 0; q0 < nq; q0 += 64) {
    const int q = q0 + lane;
    float s = 0.0f;
    if (q < nq) {
      const bf16x8 bv = b8[q], cv = c8[q];
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf((float)bv[e], (float)cv[e], s);
    }
    for (int m = 1; m < per; m <<= 1) s += __shfl_xor(s, m, 64);
    if (q < nq && (q & (per - 1)) == 0) cb[row * d.G + q / per] = s;
  }
}

// Per (row, head): rho, dt = gamma + rho, gamma in fp32, D per token = D + gamma cb.
template <typename T>
__global__ void __launch_bounds__(256) k_trapz_coef(SsdDims d, const int32_t* __restrict__ cu,
                                                    const T* __restrict__ A, const T* __restrict__ gamma,
                                                    const T* __restrict__ beta, const float* __restrict__ D,
                                                    SsdBufs b) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= d.R * d.H) return;
  const int64_t row = id / d.H;
  const int h = (int)(id - row * d.H);
  int64_t start, end;
  const int seq = tz_seq(d, cu, row, start, end);
  float rho = 0.0f;
  const int Hr = d.H >> d.hs;  // the caller's heads
  const int64_t ir = row * Hr + (h >> d.hs);
  if (row + 1 < end) rho = to_f(beta[ir + Hr]) * trapz_unfold(to_f(A[ir + Hr]));
  const float gm = to_f(gamma[ir]);
  b.tz_rho[id] = rho;
  b.tz_gam[id] = gm;
  b.tz_dt[id] = gm + rho;
  if (!b.tz_cb_fwd) b.Dtok[id] = (d.has_D ? D[h] : 0.0f) + gm * b.tz_cb[row * d.G + h / d.hpg];
  // the fused state walks' per-token factors exp(clamp(cs_last - cs_t)) dt_t, with dt = gamma + rho
  // (and dt = gamma for the gamma path's walk); positions past a chunk's end keep the cumsum's zeros
  if (b.fwd_fac && row < end) {
    const int64_t pos = tz_pos(d, b, row, start, seq) + (int64_t)h * d.Qpad;
    const int64_t t = (row - start) % d.Q;
    const float cst = b.cs[pos], tot = b.cs[pos - t + d.Qpad - 1];
    const float e = exp_clamp(tot - cst);
    b.fwd_fac[pos] = e * (gm + rho);
    if (b.fwd_fac2) b.fwd_fac2[pos] = e * gm;
  }
}

// k_trapz_coef over one chunk's 64-token block and all heads (fixed-length or packed batches, through
// the chunk table): the token-major [R][H] inputs and outputs are read and written by consecutive
// threads, and the walks' per-token factors, which are head-major per chunk ([chunk][H][Qpad]), go out
// through an LDS transpose as whole 64-token rows with the cumsum read the same way. Positions past
// the chunk's length keep the cumsum's zeros.
template <typename T>
__global__ void __launch_bounds__(256) k_trapz_coef_blk(SsdDims d, const T* __restrict__ A,
                                                        const T* __restrict__ gamma, const T* __restrict__ beta,
                                                        const float* __restrict__ D, SsdBufs b) {
  extern __shared__ float tz_s[];  // [2][H][65]: dt = gamma + rho, gamma (rows padded: conflict-free writes)
  const int c = blockIdx.x, kb = blockIdx.y;
  const ChunkInfo ci = b.chunks[c];
  const int n = min(64, ci.len - 64 * kb);
  if (n <= 0) return;
  const int H = d.H, Hr = H >> d.hs;  // kernel heads, the caller's heads
  const int64_t r0 = (int64_t)ci.row0 + 64 * kb;
  // the sequence's end: the chunk table restarts chunks at every sequence start, so a chunk that ends
  // short of Q is its sequence's last; a full chunk is the last unless the next entry continues it
  const bool seq_last_chunk = ci.len < d.Q || c + 1 >= d.max_chunks || b.chunks[c + 1].seq != ci.seq ||
                              b.chunks[c + 1].len <= 0;
  const int64_t end = (int64_t)ci.row0 + ci.len;  // rows of this chunk: [row0, end)
  for (int e = threadIdx.x; e < n * H; e += blockDim.x) {
    const int t = e / H, h = e - t * H;
    const int64_t row = r0 + t, id = row * H + h, ir = row * Hr + (h >> d.hs);
    float rho = 0.0f;
    // the next token's beta folds into this one unless this is the sequence's last token
    if (row + 1 < end || (row + 1 == end && !seq_last_chunk))
      rho = to_f(beta[ir + Hr]) * trapz_unfold(to_f(A[ir + Hr]));
    const float gm = to_f(gamma[ir]);
    b.tz_rho[id] = rho;
    b.tz_gam[id] = gm;
    b.tz_dt[id] = gm + rho;
    if (!b.tz_cb_fwd) b.Dtok[id] = (d.has_D ? D[h] : 0.0f) + gm * b.tz_cb[row * d.G + h / d.hpg];
    tz_s[h * 65 + t] = gm + rho;
    tz_s[(H + h) * 65 + t] = gm;
  }
  if (!b.fwd_fac) return;
  __syncthreads();
  for (int e = threadIdx.x; e < n * H; e += blockDim.x) {
    const int h = e / n, t = e - h * n;
    const int64_t cb0 = ((int64_t)c * H + h) * d.Qpad;
    const float tot = b.cs[cb0 + d.Qpad - 1];
    const float ex = exp_clamp(tot - b.cs[cb0 + 64 * kb + t]);
    b.fwd_fac[cb0 + 64 * kb + t] = ex * tz_s[h * 65 + t];
    if (b.fwd_fac2) b.fwd_fac2[cb0 + 64 * kb + t] = ex * tz_s[(H + h) * 65 + t];
  }
}

// Column / row path only (the fused path does this inside k_bwd_fact and k_bwd_gemm): per (row, group)
// xdy = x . dy per head, and d(C . B) = sum_h gamma xdy into dB (+= . C) and dC (+= . B).
template <typename T>
__global__ void __launch_bounds__(256) k_trapz_bc(SsdDims d, const int32_t* __restrict__ cu,
                                                  const T* __restrict__ x, const T* __restrict__ dy,
                                                  const T* __restrict__ B, const T* __restrict__ C,
                                                  T* __restrict__ dB, T* __restrict__ dC, SsdBufs b) {
  const int64_t row = blockIdx.x;
  const int g = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= d.G) return;
  int64_t start, end;
  const int seq = tz_seq(d, cu, row, start, end);
  if (row >= end) return;  // in no sequence
  const int64_t pos = tz_pos(d, b, row, start, seq);
  float dcb = 0.0f;
  for (int h = g * d.hpg; h < (g + 1) * d.hpg; ++h) {
    const int64_t o = (row * d.H + h) * d.P;
    float s = 0.0f;
    for (int p = lane; p < d.P; p += 64) s += to_f(x[o + p]) * to_f(dy[o + p]);
    for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
    if (lane == 0) b.xdy[pos + (int64_t)h * d.Qpad] = s;
    dcb += b.tz_gam[row * d.H + h] * s;
  }
  const int64_t o = (row * d.G + g) * d.N;
  for (int n = lane; n < d.N; n += 64) {
    dB[o + n] = from_f<T>(to_f(dB[o + n]) + dcb * to_f(C[o + n]));
    dC[o + n] = from_f<T>(to_f(dC[o + n]) + dcb * to_f(B[o + n]));
  }
}

// Per (row, head), after the finish kernel: drho = d(dt) of the strict scan, dgamma = drho + cb xdy;
// drho of the previous token gives dbeta = drho exp(-a) and (EXACT_DA) the decay term -drho rho;
// dA = the scan's decay gradient + that.
template <typename T>
__global__ void __launch_bounds__(256) k_trapz_grads(SsdDims d, const int32_t* __restrict__ cu,
                                                     const T* __restrict__ A, SsdBufs b, T* __restrict__ dgamma,
                                                     T* __restrict__ dbeta, T* __restrict__ dA) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Hr = d.H >> d.hs;  // the caller's heads (tz_ddt, tz_da and the outputs are per caller head)
  if (id >= d.R * Hr) return;
  const int64_t row = id / Hr;
  const int h = (int)(id - row * Hr) << d.hs;  // its first kernel head
  int64_t start, end;
  const int seq = tz_seq(d, cu, row, start, end);
  const bool inside = row < end;
  if (dgamma) {
    float xdy = 0.0f;
    if (inside) {
      const float* xd = b.xdy + tz_pos(d, b, row, start, seq) + (int64_t)h * d.Qpad;
      xdy = xd[0];
      if (d.hs) xdy += xd[d.Qpad];
    }
    dgamma[id] = from_f<T>(inside ? b.tz_ddt[id] + b.tz_cb[row * d.G + h / d.hpg] * xdy : 0.0f);
  }
  float drho = 0.0f, rho = 0.0f;
  if (row > start && inside) {
    drho = b.tz_ddt[id - Hr];
    rho = b.tz_rho[(row - 1) * d.H + h];
  }
  // (steep tokens: overwritten by k_trapz_dbeta_steep)
  if (dbeta) dbeta[id] = from_f<T>(drho * trapz_unfold(to_f(A[id])));
  if (dA) dA[id] = from_f<T>(inside ? b.tz_da[id] - (d.trapz == 2 ? drho * rho : 0.0f) : 0.0f);
}

// dbeta at the tokens r whose decay a[r] is below SSD_TRAPZ_STEEP, from the beta call's definition:
// its input at r is beta[r] x[s] B[s]^T, s = r - 1, at position i of chunk c, so
//   dbeta[r] = sum_{t = i}^{len-1} e^{clamp(cs_t - cs_i)} (C_t . B_s)(x_s . dy_t)
//              + e^{clamp(cs_last - cs_i)} x_s^T dst[c] B_s,
// dst[c] the gradient of the state leaving chunk c (the reference's acausal e^-20 entries left out,
// as everywhere in this build). One block per (chunk, head); a block without a steep token exits
// after one flag reduction. Per steep token: x_s and B_s in LDS, one thread per t for the
// intra-chunk terms, all threads over (p, n) for the state term, one block sum.
template <typename T, typename DS>
__global__ void __launch_bounds__(256) k_trapz_dbeta_steep(SsdDims d, const SsdBufs b, const T* __restrict__ A,
                                                           const T* __restrict__ x, const T* __restrict__ dy,
                                                           const T* __restrict__ B, const T* __restrict__ C,
                                                           const DS* __restrict__ dst, T* __restrict__ dbeta) {
  __shared__ float xs[SSD_MAX_HEADDIM], bs[SSD_MAX_DSTATE], csl[SSD_MAX_CHUNK], red[4];
  __shared__ unsigned char steep[SSD_MAX_CHUNK];
  // (with two kernel heads per caller head, the block's head is the caller's and its terms sum over both)
  const int c = blockIdx.x, hr = blockIdx.y, tid = threadIdx.x;
  const int Hr = d.H >> d.hs, nk = 1 << d.hs, h = hr << d.hs;
  const ChunkInfo ci = b.chunks[c];
  const int len = min(ci.len, d.Q);
  if (len <= 0) return;
  const int g = h / d.hpg;
  const float* cs = b.cs + ((int64_t)c * d.H + h) * d.Qpad;
  const int64_t row0 = ci.row0;
  bool mine = false;
  if (tid < len) {
    csl[tid] = cs[tid];
    // a sequence's first token has no beta input (x_prev = 0 there)
    mine = !(ci.idx_in_seq == 0 && tid == 0) && to_f(A[(row0 + tid) * Hr + hr]) < SSD_TRAPZ_STEEP;
    steep[tid] = mine ? 1 : 0;
  }
  if (!__syncthreads_or(mine)) return;
  const float cs_last = cs[d.Qpad - 1];
  const int PN = d.P * d.N;
  for (int i = 0; i < len; ++i) {
    if (!steep[i]) continue;  // block-uniform (LDS)
    const int64_t s = row0 + i - 1;
    const int PW = d.P << d.hs;  // the caller head's width: its kernel heads side by side
    for (int p = tid; p < PW; p += 256) xs[p] = to_f(x[(s * d.H + h) * d.P + p]);
    for (int n = tid; n < d.N; n += 256) bs[n] = to_f(B[(s * d.G + g) * d.N + n]);
    __syncthreads();
    float acc = 0.0f;
    if (tid >= i && tid < len) {
      const int64_t t = row0 + tid;
      const T* ct = C + (t * d.G + g) * d.N;
      const T* dyt = dy + (t * d.H + h) * d.P;
      float cb = 0.0f, xd = 0.0f;
      for (int n = 0; n < d.N; ++n) cb += to_f(ct[n]) * bs[n];
      for (int p = 0; p < PW; ++p) xd += xs[p] * to_f(dyt[p]);
      acc = exp_clamp(csl[tid] - csl[i]) * cb * xd;
    }
    float sacc = 0.0f;
    for (int k = 0; k < nk; ++k) {
      const DS* dsc = dst + ((int64_t)c * d.H + h + k) * d.Ppad * d.Npad;
      for (int e = tid; e < PN; e += 256) {
        const int p = e / d.N, n = e - p * d.N;
        sacc += xs[k * d.P + p] * bs[n] * to_f(dsc[p * d.Npad + n]);
      }
    }
    acc += exp_clamp(cs_last - csl[i]) * sacc;
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) dbeta[(row0 + i) * Hr + hr] = from_f<T>(red[0] + red[1] + red[2] + red[3]);
    __syncthreads();  // xs, bs and red are reused by the next steep token
  }
}

template <typename T>
static hipError_t trapz_prep_t(const SsdDims& d, const SsdBufs& b, const void* A, const void* gamma, const void* beta,
                               const void* B, const void* C, const float* D, const int32_t* cu, hipStream_t s) {
  const int per = d.N / 8;
  if (b.tz_cb_fwd) {
    // cb and D per token come from the factorised forward scan
  } else if (sizeof(T) == 2 && d.vec_bc && per <= 64 && (per & (per - 1)) == 0)
    hipLaunchKernelGGL(k_trapz_cb_v, dim3((unsigned)((d.R + 3) / 4)), dim3(256), 0, s, d,
                       reinterpret_cast<const bf16*>(B), reinterpret_cast<const bf16*>(C), b.tz_cb);
  else
    hipLaunchKernelGGL(k_trapz_cb<T>, dim3((unsigned)d.R, (d.G + 3) / 4), dim3(256), 0, s, d,
                       reinterpret_cast<const T*>(B), reinterpret_cast<const T*>(C), b.tz_cb);
  // chunk-ordered form when its transpose tile fits (2 H 65 fp32), else one thread per (row, head)
  const size_t lds = 2 * (size_t)d.H * 65 * sizeof(float);
  if (lds <= 64 * 1024) {
    hipLaunchKernelGGL(k_trapz_coef_blk<T>, dim3((unsigned)d.max_chunks, (unsigned)(d.Qpad / 64)), dim3(256), lds, s,
                       d, reinterpret_cast<const T*>(A), reinterpret_cast<const T*>(gamma),
                       reinterpret_cast<const T*>(beta), D, b);
  } else {
    const int64_t n = d.R * d.H;
    hipLaunchKernelGGL(k_trapz_coef<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d, cu,
                       reinterpret_cast<const T*>(A), reinterpret_cast<const T*>(gamma),
                       reinterpret_cast<const T*>(beta), D, b);
  }
  return hipGetLastError();
}

hipError_t launch_trapz_prep(int dtype, const SsdDims& d, const SsdBufs& b, const void* A, const void* gamma,
                             const void* beta, const void* B, const void* C, const float* D, const int32_t* cu,
                             hipStream_t s) {
  return dtype == 1 ? trapz_prep_t<bf16>(d, b, A, gamma, beta, B, C, D, cu, s)
                    : trapz_prep_t<float>(d, b, A, gamma, beta, B, C, D, cu, s);
}

// D per token, D + gamma cb, once the factorised forward scan has written cb (tz_cb_fwd): one thread per
// (row, head), the [R][H] arrays read and written by consecutive threads.
__global__ void __launch_bounds__(256) k_trapz_dtok(SsdDims d, const float* __restrict__ D, SsdBufs b) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= d.R * d.H) return;
  const int64_t row = id / d.H;
  const int h = (int)(id - row * d.H);
  b.Dtok[id] = (d.has_D ? D[h] : 0.0f) + b.tz_gam[id] * b.tz_cb[row * d.G + h / d.hpg];
}

hipError_t launch_trapz_dtok(const SsdDims& d, const SsdBufs& b, const float* D, hipStream_t s) {
  const int64_t n = d.R * d.H;
  hipLaunchKernelGGL(k_trapz_dtok, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d, D, b);
  return hipGetLastError();
}

hipError_t launch_trapz_bc(int dtype, const SsdDims& d, const SsdBufs& b, const void* x, const void* dy,
                           const void* B, const void* C, void* dB, void* dC, const int32_t* cu, hipStream_t s) {
  const dim3 grid((unsigned)d.R, (d.G + 3) / 4);
  if (dtype == 1)
    hipLaunchKernelGGL(k_trapz_bc<bf16>, grid, dim3(256), 0, s, d, cu, reinterpret_cast<const bf16*>(x),
                       reinterpret_cast<const bf16*>(dy), reinterpret_cast<const bf16*>(B),
                       reinterpret_cast<const bf16*>(C), reinterpret_cast<bf16*>(dB), reinterpret_cast<bf16*>(dC), b);
  else
    hipLaunchKernelGGL(k_trapz_bc<float>, grid, dim3(256), 0, s, d, cu, reinterpret_cast<const float*>(x),
                       reinterpret_cast<const float*>(dy), reinterpret_cast<const float*>(B),
                       reinterpret_cast<const float*>(C), reinterpret_cast<float*>(dB), reinterpret_cast<float*>(dC),
                       b);
  return hipGetLastError();
}

template <typename T>
static hipError_t trapz_grads_t(const SsdDims& d, const SsdBufs& b, const void* A, const int32_t* cu, const void* x,
                                const void* dy, const void* B, const void* C, void* dgamma, void* dbeta, void* dA,
                                hipStream_t s) {
  const int64_t n = d.R * (d.H >> d.hs);
  hipLaunchKernelGGL(k_trapz_grads<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d, cu,
                     reinterpret_cast<const T*>(A), b, reinterpret_cast<T*>(dgamma), reinterpret_cast<T*>(dbeta),
                     reinterpret_cast<T*>(dA));
  if (!dbeta) return hipGetLastError();
  const dim3 grid((unsigned)d.max_chunks, (unsigned)(d.H >> d.hs));
  const T *tA = reinterpret_cast<const T*>(A), *tx = reinterpret_cast<const T*>(x),
          *tdy = reinterpret_cast<const T*>(dy), *tB = reinterpret_cast<const T*>(B),
          *tC = reinterpret_cast<const T*>(C);
  // the gradient leaving each chunk: bf16 on the fused path, else fp32 in place
  if (b.dst16)
    hipLaunchKernelGGL((k_trapz_dbeta_steep<T, bf16>), grid, dim3(256), 0, s, d, b, tA, tx, tdy, tB, tC,
                       (const bf16*)b.dst16, reinterpret_cast<T*>(dbeta));
  else
    hipLaunchKernelGGL((k_trapz_dbeta_steep<T, float>), grid, dim3(256), 0, s, d, b, tA, tx, tdy, tB, tC,
                       (const float*)b.dst, reinterpret_cast<T*>(dbeta));
  return hipGetLastError();
}

hipError_t launch_trapz_grads(int dtype, const SsdDims& d, const SsdBufs& b, const void* A, const int32_t* cu,
                              const void* x, const void* dy, const void* B, const void* C, void* dgamma, void* dbeta,
                              void* dA, hipStream_t s) {
  return dtype == 1 ? trapz_grads_t<bf16>(d, b, A, cu, x, dy, B, C, dgamma, dbeta, dA, s)
                    : trapz_grads_t<float>(d, b, A, cu, x, dy, B, C, dgamma, dbeta, dA, s);
}
