// Chunk table, in-chunk cumsum of the log-decay, and the reference cache
// tensors (L, decay_chunk).
#include "ssd_launch.h"

// ---------------------------------------------------------------------------
// Chunk table: chunks restart at every sequence start, so each chunk lies in
// one sequence (the reference pads every sequence to a chunk multiple,
// r2/dhammic-ai/src/mamba_base_engine.py:154-165). One block; the per-sequence
// prefix lives in LDS (nseq <= 16000 is checked on the host).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_chunk_table(const int32_t* __restrict__ cu, int nseq, int seqlen,
                                                     int Q, int max_chunks, ChunkInfo* __restrict__ chunks,
                                                     int32_t* __restrict__ seq_chunk0, int32_t* __restrict__ seq_order) {
  extern __shared__ int32_t s_first[];  // [nseq + 1]
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int s = 0; s < nseq; ++s) {
      int start, end;
      if (cu) {
        start = min(max(cu[s], 0), seqlen);
        end = min(max(cu[s + 1], start), seqlen);
      } else {
        start = s * seqlen;
        end = start + seqlen;
      }
      // clamped so that malformed offsets can never index past the table
      s_first[s] = min(acc, max_chunks);
      acc += (end - start + Q - 1) / Q;
    }
    s_first[nseq] = min(acc, max_chunks);
  }
  __syncthreads();
  for (int s = threadIdx.x; s <= nseq; s += blockDim.x) seq_chunk0[s] = s_first[s];
  // the state walks' order: most chunks first, ties by index (each sequence's rank counts the ones before
  // it), so that the longest walks start first and the short ones fill in behind them; in order beyond
  // kSortSeqs sequences (the rank count is quadratic)
  if (seq_order) {
    constexpr int kSortSeqs = 1024;
    for (int s = threadIdx.x; s < nseq; s += blockDim.x) {
      int rank = s;
      if (nseq <= kSortSeqs) {
        const int ns = s_first[s + 1] - s_first[s];
        rank = 0;
        for (int t = 0; t < nseq; ++t) {
          const int nt = s_first[t + 1] - s_first[t];
          rank += (nt > ns || (nt == ns && t < s)) ? 1 : 0;
        }
      }
      seq_order[rank] = s;
    }
  }
  const int total = s_first[nseq];
  for (int c = threadIdx.x; c < max_chunks; c += blockDim.x) {
    ChunkInfo ci;
    ci.row0 = 0; ci.len = 0; ci.seq = -1; ci.idx_in_seq = 0;
    if (c < total) {
      int lo = 0, hi = nseq - 1;  // last s with s_first[s] <= c
      while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (s_first[mid] <= c) lo = mid; else hi = mid - 1;
      }
      int start, end;
      if (cu) {
        start = min(max(cu[lo], 0), seqlen);
        end = min(max(cu[lo + 1], start), seqlen);
      } else {
        start = lo * seqlen;
        end = start + seqlen;
      }
      const int k = c - s_first[lo];
      ci.row0 = start + k * Q;
      ci.len = min(Q, end - ci.row0);
      ci.seq = lo;
      ci.idx_in_seq = k;
    }
    chunks[c] = ci;
  }
}

hipError_t launch_chunk_table(const SsdDims& d, const SsdBufs& b, const int32_t* cu, hipStream_t s) {
  const int seqlen = d.varlen ? (int)d.R : d.seqlen;
  hipLaunchKernelGGL(k_chunk_table, dim3(1), dim3(256), (d.nseq + 1) * sizeof(int32_t), s,
                     d.varlen ? cu : nullptr, d.nseq, seqlen, d.Q, d.max_chunks, b.chunks, b.seq_chunk0,
                     b.seq_order);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// In-chunk inclusive cumsum of a (ssd_scan.py:364-368), one wave per
// (chunk, head), fp32. Positions past the chunk's length carry a = 0, so
// cs[Qpad-1] is the chunk total. Optionally writes the reference's
// A_cumsum (b, h, c, Q) in the input dtype, and the fused state walks'
// per-token factors (0 past the chunk's length): bfac = exp(clamp(cs_t)),
// ffac = exp(clamp(cs_last - cs_t)) dt_t (trapezoidal mode: zeros here, the
// coefficient kernel writes the chunk's positions with its own dt), ffac2
// (trapezoidal gamma walk: zeros here likewise). For a fixed-length batch it
// also writes the chunk table (no k_chunk_table launch). With two kernel heads per caller head (d.hs) it
// also writes dt and D per kernel head.
// ---------------------------------------------------------------------------
// One row of Qpad fp32 values, `per` consecutive positions per lane: a 16-byte store per lane when
// each lane holds four and the row is 16-byte aligned.
__device__ __forceinline__ void store_row(float* __restrict__ p, int lane, int per, const float (&v)[4]) {
  if (per == 4 && (reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    *reinterpret_cast<float4*>(p + lane * 4) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    for (int e = 0; e < per; ++e) p[lane * per + e] = v[e];
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_chunk_cumsum(SsdDims d, ChunkInfo* __restrict__ chunks,
                                                      int32_t* __restrict__ seq_chunk0, int build_table,
                                                      const void* __restrict__ Av, const float* __restrict__ dt,
                                                      float* __restrict__ cs, T* __restrict__ acs_out,
                                                      int32_t* __restrict__ fast, float* __restrict__ ffac,
                                                      float* __restrict__ ffac2, float* __restrict__ bfac,
                                                      float* __restrict__ dt_rep, const float* __restrict__ Dv,
                                                      float* __restrict__ D_rep) {
  // dt of the block's four heads, [head][position] (Qpad <= 256)
  __shared__ float s_dt[4][256];
  const int c = blockIdx.x;
  const int h0 = blockIdx.y * 4, hw = threadIdx.x >> 6;
  const int h = h0 + hw;
  const int hs = d.hs, Hr = d.H >> hs, hr = h >> hs;  // the caller's heads
  const int lane = lane_id();
  ChunkInfo ci;
  if (build_table) {
    // Fixed-length batch (max_chunks = nseq * nch, every chunk valid): chunk c is chunk c % nch of
    // sequence c / nch, the entry k_chunk_table writes for it; the blocks of head group 0 write the table.
    const int nch = (d.seqlen + d.Q - 1) / d.Q;
    const int sq = c / nch, k = c - sq * nch;
    ci.row0 = sq * d.seqlen + k * d.Q;
    ci.len = min(d.Q, d.seqlen - k * d.Q);
    ci.seq = sq;
    ci.idx_in_seq = k;
    if (blockIdx.y == 0) {
      if (threadIdx.x == 0) chunks[c] = ci;
      if (c == 0)
        for (int q = threadIdx.x; q <= d.nseq; q += blockDim.x) seq_chunk0[q] = q * nch;
    }
  } else {
    ci = chunks[c];
  }
  if (ci.len == 0) return;  // the whole block
  const bool use_dt = d.has_dt && !d.trapz;
  if (use_dt) {
    // dt is token-major ([R][H]): one thread per position reads the four heads' values, one 16-byte
    // load when they are in range and aligned, where a lane per head would touch a line per position
    const int l = threadIdx.x;
    if (l < d.Qpad) {
      float q[4] = {1.0f, 1.0f, 1.0f, 1.0f};
      if (l < ci.len) {
        const float* p = dt + ((int64_t)ci.row0 + l) * Hr + (h0 >> hs);
        if (hs) {
          // two kernel heads per caller head: their dt per kernel head goes out for the scan kernels, in
          // whole vectors (d.H is even; dword stores a row apart took the launch from 7 to 13 us at 7368
          // tokens of 32 heads)
          float2* o = reinterpret_cast<float2*>(dt_rep + ((int64_t)ci.row0 + l) * d.H + h0);
          const bool two = h0 + 2 < d.H;
          float2 f = {0.0f, 0.0f};
          if (two && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
            f = *reinterpret_cast<const float2*>(p);
          } else {
            f.x = p[0];
            if (two) f.y = p[1];
          }
          if ((d.H & 3) == 0) {
            *reinterpret_cast<float4*>(o) = float4{f.x, f.x, f.y, f.y};
          } else {
            o[0] = float2{f.x, f.x};
            if (two) o[1] = float2{f.y, f.y};
          }
          q[0] = q[1] = f.x;
          q[2] = q[3] = f.y;
        } else if ((d.H & 3) == 0 && (reinterpret_cast<uintptr_t>(dt) & 15) == 0) {
          const float4 f = *reinterpret_cast<const float4*>(p);
          q[0] = f.x; q[1] = f.y; q[2] = f.z; q[3] = f.w;
        } else {
          for (int k = 0; k < 4; ++k)
            if (h0 + k < d.H) q[k] = p[k];
        }
      }
      for (int k = 0; k < 4; ++k) s_dt[k][l] = q[k];
    }
    __syncthreads();
  }
  if (h >= d.H) return;
  if (D_rep && c == 0 && lane == 0) D_rep[h] = Dv[hr];
  const int per = d.Qpad / 64;  // 1 to 4 consecutive positions per lane
  float v[4] = {}, dtv[4] = {};
  float run = 0.0f;
  for (int e = 0; e < per; ++e) {
    const int l = lane * per + e;
    float a = 0.0f;
    dtv[e] = (use_dt && l < ci.len) ? s_dt[hw][l] : 1.0f;
    if (d.a_mode == 2) {
      // the caller's inclusive cumsum: differences are not needed, keep it as is
      const int nch = d.seqlen / d.Q;
      const T* A = reinterpret_cast<const T*>(Av);
      const int ll = min(l, ci.len - 1);
      v[e] = to_f(A[(((int64_t)ci.seq * Hr + hr) * nch + ci.idx_in_seq) * d.Q + ll]);
      continue;
    }
    if (l < ci.len) {
      const int64_t row = ci.row0 + l;
      if (d.a_mode == 0) {
        const float* A = reinterpret_cast<const float*>(Av);
        a = dtv[e] * A[hr];
      } else {
        const T* A = reinterpret_cast<const T*>(Av);
        a = to_f(A[row * Hr + hr]);
      }
    }
    run += a;
    v[e] = run;
  }
  if (d.a_mode != 2) {
    // exclusive scan of the lane totals across the wave
    float incl = run;
    for (int off = 1; off < 64; off <<= 1) {
      float o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    const float excl = incl - run;
    for (int e = 0; e < per; ++e) v[e] += excl;
  }
  const int64_t o = ((int64_t)c * d.H + h) * d.Qpad;
  store_row(cs + o, lane, per, v);
  if (ffac) {
    const float tot = __shfl(v[per - 1], 63, 64);  // cs[Qpad - 1], the chunk total
    float f[4] = {}, g[4] = {};
    const float zero[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int e = 0; e < per; ++e) {
      const bool in = lane * per + e < ci.len;
      f[e] = (in && !d.trapz) ? exp_clamp(tot - v[e]) * dtv[e] : 0.0f;
      g[e] = in ? exp_clamp(v[e]) : 0.0f;
    }
    store_row(ffac + o, lane, per, f);
    if (ffac2) store_row(ffac2 + o, lane, per, zero);
    store_row(bfac + o, lane, per, g);
  }
  if (fast) {
    // Factorised-decay guard: cs non-increasing over the chunk (every a <= 0, up to the scan's
    // rounding: SSD_FACT_RISE) and each 64-token block's drop cs[64 j] - cs[64 j + 63] at most
    // 2 SSD_FACT_RANGE, so exp(cs_l - c) and exp(c - cs_s) around the block's
    // midpoint reference c stay within e^{+-SSD_FACT_RANGE} (see the factorised kernels).
    bool ok = true;
    for (int e = 1; e < per; ++e) ok = ok && v[e] <= v[e - 1] + SSD_FACT_RISE;
    const float prev = __shfl_up(v[per - 1], 1, 64);
    if (lane > 0) ok = ok && v[0] <= prev + SSD_FACT_RISE;
    // Lane j < Qpad / 64 checks block j from its exact end positions 64 j and 64 j + 63, fetched
    // from the lanes and elements that own them (with per = 3 a block does not start on a lane).
    const int jb = lane < per ? lane : 0;
    const int ptop = 64 * jb, pbot = 64 * jb + 63;
    float top = 0.0f, bot = 0.0f;
    for (int e = 0; e < per; ++e) {
      const float a1 = __shfl(v[e], ptop / per, 64);
      const float a2 = __shfl(v[e], pbot / per, 64);
      if (e == ptop % per) top = a1;
      if (e == pbot % per) bot = a2;
    }
    if (lane < per) ok = ok && (top - bot) <= 2.0f * SSD_FACT_RANGE;
    const bool all_ok = __all(ok);
    if (lane == 0) fast[(int64_t)c * d.H + h] = all_ok ? 1 : 0;
  }
  if (acs_out && (h & ((1 << hs) - 1)) == 0) {
    const int nch = d.seqlen / d.Q;
    T* o = acs_out + (((int64_t)ci.seq * Hr + hr) * nch + ci.idx_in_seq) * d.Q;
    for (int e = 0; e < per; ++e) {
      const int l = lane * per + e;
      if (l < d.Q) o[l] = from_f<T>(v[e]);
    }
  }
}

hipError_t launch_chunk_cumsum(int dtype, const SsdDims& d, const SsdBufs& b, const void* A,
                               const float* dt, const float* D, void* A_cumsum_out, hipStream_t s) {
  dim3 grid(d.max_chunks, (d.H + 3) / 4);
  const int build = d.varlen ? 0 : 1;  // fixed-length batches: the chunk table is written here
  if (dtype == 1)
    hipLaunchKernelGGL(k_chunk_cumsum<bf16>, grid, dim3(256), 0, s, d, b.chunks, b.seq_chunk0, build, A, dt, b.cs,
                       reinterpret_cast<bf16*>(A_cumsum_out), b.fast, b.fwd_fac, b.fwd_fac2, b.bwd_fac, b.dt_rep, D,
                       b.D_rep);
  else
    hipLaunchKernelGGL(k_chunk_cumsum<float>, grid, dim3(256), 0, s, d, b.chunks, b.seq_chunk0, build, A, dt, b.cs,
                       reinterpret_cast<float*>(A_cumsum_out), b.fast, b.fwd_fac, b.fwd_fac2, b.bwd_fac, b.dt_rep, D,
                       b.D_rep);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// decay_chunk = exp(clamp(segsum(pad(A_cumsum[..., -1], (1, 0))))) in the
// input dtype (ssd_scan.py:402-406): the segsum is accumulated in fp32 down
// each column from j+1 (:104-116), rounded to the dtype, then exp-clamped and
// rounded again, as the reference's two kernels do. One block per (b, h).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_decay_chunk(int nch, int Q, const T* __restrict__ Acs, T* __restrict__ out) {
  const int bh = blockIdx.x;
  const int n = nch + 1;
  const T* a = Acs + (int64_t)bh * nch * Q;
  T* o = out + (int64_t)bh * n * n;
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    float acc = 0.0f;
    for (int i = 0; i < n; ++i) {
      float seg;
      if (i < j) {
        seg = -1e4f;
      } else {
        if (i > j) acc += to_f(a[(int64_t)(i - 1) * Q + (Q - 1)]);  // v_i = A_cumsum[i-1, Q-1]
        seg = acc;
      }
      seg = to_f(from_f<T>(fminf(fmaxf(seg, SSD_LO), SSD_HI)));
      o[(int64_t)i * n + j] = from_f<T>(__expf(fminf(fmaxf(seg, SSD_LO), SSD_HI)));
    }
  }
}

hipError_t launch_decay_chunk(int dtype, int batch, int H, int nch, int Q, const void* Acs, void* out,
                              hipStream_t s) {
  if (dtype == 1)
    hipLaunchKernelGGL(k_decay_chunk<bf16>, dim3(batch * H), dim3(256), 0, s, nch, Q,
                       reinterpret_cast<const bf16*>(Acs), reinterpret_cast<bf16*>(out));
  else
    hipLaunchKernelGGL(k_decay_chunk<float>, dim3(batch * H), dim3(256), 0, s, nch, Q,
                       reinterpret_cast<const float*>(Acs), reinterpret_cast<float*>(out));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// L = exp(clamp(segsum(a))) per (b, h, chunk), a permuted to (b, h, c, l)
// (ssd_scan.py:380-382). Thread per column j, walking rows i: the same fp32
// accumulation order as the reference segsum kernel (:104-116).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_materialize_L(int seqlen, int H, int Q, const T* __restrict__ a, T* __restrict__ L) {
  const int nch = seqlen / Q;
  const int k = blockIdx.x % nch;
  const int h = (blockIdx.x / nch) % H;
  const int b = blockIdx.x / (nch * H);
  T* o = L + (int64_t)blockIdx.x * Q * Q;  // (b, h, c) major order matches blockIdx
  for (int j = threadIdx.x; j < Q; j += blockDim.x) {
    float acc = 0.0f;
    for (int i = 0; i < Q; ++i) {
      float seg;
      if (i < j) {
        seg = -1e4f;
      } else {
        if (i > j) acc += to_f(a[((int64_t)b * seqlen + (int64_t)k * Q + i) * H + h]);
        seg = acc;
      }
      seg = to_f(from_f<T>(fminf(fmaxf(seg, SSD_LO), SSD_HI)));
      o[(int64_t)i * Q + j] = from_f<T>(__expf(fminf(fmaxf(seg, SSD_LO), SSD_HI)));
    }
  }
}

hipError_t launch_materialize_L(int dtype, int batch, int seqlen, int H, int Q, const void* a, void* L,
                                hipStream_t s) {
  const int blocks = batch * H * (seqlen / Q);
  if (dtype == 1)
    hipLaunchKernelGGL(k_materialize_L<bf16>, dim3(blocks), dim3(256), 0, s, seqlen, H, Q,
                       reinterpret_cast<const bf16*>(a), reinterpret_cast<bf16*>(L));
  else
    hipLaunchKernelGGL(k_materialize_L<float>, dim3(blocks), dim3(256), 0, s, seqlen, H, Q,
                       reinterpret_cast<const float*>(a), reinterpret_cast<float*>(L));
  return hipGetLastError();
}
