// Launch parameters shared by the host entry points and the kernels.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "ssd_common.h"


struct SsdDims {
  int batch, seqlen, H, P, G, N, Q;  // Q: tokens per chunk
  int Ppad, Npad, Qpad;              // P, N padded to 32, 64 or 128; Q rounded up to 64
  int nseq, max_chunks, hpg;         // hpg: heads per group
  int64_t R;                         // rows of the packed token axis (batch * seqlen)
  int a_mode, has_dt, has_D, has_z, has_init, has_dfinal, varlen;
  float eps;
  int dA_skip;                       // enum ssd_dA_skip bits (terms left out of the decay gradient)
  int trapz;                         // enum ssd_trapz: dt is gamma + rho, D per token, strictly causal
  int da_only;                       // backward for the decay gradient only (no dx / dB / dC / dS written)
  int gdec;                          // trapezoidal drop mode: the column kernels' decay terms (G, E) take the
                                     // gamma path's dt (b.tz_gam); dS, dX and dx keep dt = gamma + rho
  // 16-byte global loads allowed for x/dy/z-shaped tensors and for B/C (set per call
  // from the feature widths and the pointers' alignment)
  bool vec_x, vec_bc;
  // log2 of the kernel heads per caller head: 1 where a bf16 head wider than 64 runs as two heads of half its
  // width (plan() in ssd_capi.hip). H, P and hpg are then the kernels' (2 H heads of P / 2); the caller's
  // per-head tensors (dt, A, D, gamma, beta and their gradients) have H >> hs heads.
  int hs;
};

// Internal buffers (all inside the caller's workspaces).
struct SsdBufs {
  ChunkInfo* chunks;       // [max_chunks]
  int32_t* seq_chunk0;     // [nseq + 1] first chunk of each sequence
  int32_t* seq_order;      // packed sequences: [nseq] sequence indices, most chunks first (the state walks take
                           // the longest sequences first); nullptr for fixed-length batches
  float* cs;               // [max_chunks][H][Qpad] in-chunk inclusive cumsum of a
  int32_t* fast;           // [max_chunks][H] 1: the factorised-decay kernels are exact enough
                           // for this (chunk, head) (see k_chunk_cumsum), 0: exact-path fixup
  void* hin;               // [max_chunks][H][Ppad][Npad] (T) state entering each chunk
  // bf16 storage: the rounding residual hin - bf16(hin) (fp8, lo_pack4), [max_chunks][H][Ppad * Npad]
  // bytes in the row kernel's MFMA fragment order (hin_lo_off), read where the decay gradient takes hin
  // (the row kernel's Y_off term); nullptr for fp32
  uint8_t* hin_lo;
  // the row kernel's decay term over other states than h_in (k_bwd_rows; nullptr: h_in): the trapezoidal
  // drop setting's gamma-path states hgam and their residual
  const void* hdec;
  const uint8_t* hdec_lo;
  void* ypre;              // [R][H][P] (T) y before the gated norm (has_z)
  float* rstd;             // [R] (has_z)
  float* st;               // fwd scratch: [max_chunks][H][Ppad][Npad] chunk-local states
  // per-token factors of the fused state walks, [max_chunks][H][Qpad] (0 past a chunk's end):
  // fwd_fac = exp(clamp(cs_last - cs_t)) dt_t (fwd scratch; fwd_fac2 with dt = gamma, the trapezoidal
  // gamma walk); bwd_fac = exp(clamp(cs_t)) (saved)
  float* fwd_fac;
  float* fwd_fac2;
  float* bwd_fac;
  // backward scratch
  void* dyp;               // [R][H][P] (T) gradient at y before the gated norm (has_z)
  float* dst;              // [max_chunks][H][Ppad][Npad] local dh, then gradient leaving each chunk
  bf16* dst16;             // fused path: the gradient leaving each chunk in bf16 (dst keeps the local dh)
  float* dtot_part;        // [max_chunks][H][npass_blk]
  float* rowG;             // [nrowg][max_chunks][H][Qpad] (partials summed by the finish kernel)
  float* colG;             // [max_chunks][H][Qpad]
  float* eterm;            // [max_chunks][H][Qpad]
  float* dcs_off;          // [ndcs][max_chunks][H][Qpad] (partials summed by the finish kernel)
  float* xdx;              // [max_chunks][H][Qpad]
  float* dD_part;          // [max_chunks][H][Qpad/64]
  float* dA_part;          // [max_chunks][H]
  float* dB_part;          // [head slices][R][G][N] (bf16 column / row kernels, fp32 rows, k_bwd_gemm)
  float* dC_part;          // the same
  float* dS_tiles;         // fused path: [nslices][max_chunks][G][nb*nb][64][64] head-summed dS
  bf16* dS_tiles16;        // the same in bf16 when one head slice covers each group (nslices == 1; the row
                           // kernel rounds the tiles to bf16 for its products anyway); dS_tiles then nullptr
  float* dS_fix;           // fused path: [max_chunks][G][nb*nb][64][64] dS of the heads the exact fixup runs
  float* dw_part;          // [norm_blocks][H*P]
  // trapezoidal mode (saved): rho = beta[t+1] exp(-a[t+1]); dt = gamma + rho; cb = C_t . B_t;
  // Dtok = D + gamma cb (D per token; the scan is then strictly causal); gam = gamma in fp32;
  // hgam = the gamma path's states (DROP_BETA_DA)
  float* tz_dt;            // [R][H]
  float* tz_rho;           // [R][H]
  float* tz_gam;           // [R][H]
  float* tz_cb;            // [R][G]
  float* Dtok;             // [R][H] (nullptr outside trapezoidal mode)
  // hs = 1 (saved): the caller's dt and D per kernel head, written by the cumsum launch
  float* dt_rep;           // [R][H]
  float* D_rep;            // [H]
  int tz_cb_fwd;           // 1: cb and Dtok are written by the factorised forward scan (the diagonal of its
                           // C B^T units), not by the trapezoidal prep kernels
  void* hgam;              // [max_chunks][H][Ppad][Npad] (T)
  uint8_t* hgam_lo;        // its rounding residual, as hin_lo
  // trapezoidal mode (backward scratch)
  float* xdy;              // [max_chunks][H][Qpad] x_t . dy_t per head (the layout of xdx)
  float* tz_ddt;           // [R][H] gradient at dt = gamma + rho
  float* tz_da;            // [R][H] decay gradient of the scan (fp32)
  // fp32 path (scratch), units (chunk, group) in batches of f32_batch: the S tiles, the dS tiles per head
  // slice (ssd_f32.hip)
  float* f32_cb;
  float* f32_dS;
  int f32_batch;
  int f32_rhs, f32_rsl;    // the row kernel's heads per slice and its slices (the tile term's among them)
  int npass_blk, nslices, hslice, norm_blocks;
  int fused_bwd;           // 1: k_bwd_main + k_bwd_gemm (bf16), 0: column / row kernels
  int ndcs;                // dcs_off partials
  int gemm_hslice, gemm_tsteps, gemm_parts;  // k_bwd_gemm: heads and tile steps per block, partial sums (1: none)
  int rows_chunk;          // fused path: k_bwd_rows builds dB / dC (else k_bwd_gemm)
  int nrowg;               // rowG partials (column sets of the fused path, else 1)
};

// Elements per thread block in the state passes.
#define SSD_PASS_THREADS 256
