// Host-side launchers of the SSD kernels (one per kernel family; each
// dispatches on the storage dtype, 0 = fp32, 1 = bf16). All return the
// hipError_t of their launches.
#pragma once

#include <hip/hip_runtime.h>

#include "ssd_params.h"

// Lift the default dynamic-LDS cap for kernels that stage more than 64 KiB
// (gfx950 offers 160 KiB per workgroup).
template <typename K>
inline void ensure_lds(K kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)bytes);
}

struct SsdIn {
  const void* x; const float* dt; const void* A; const void* B; const void* C;
  const float* D; const void* z; const float* w; const void* init; const int32_t* cu;
};

// ssd_prep.hip
// packed sequences (d.varlen) only: a fixed-length batch's table is written by launch_chunk_cumsum
hipError_t launch_chunk_table(const SsdDims& d, const SsdBufs& b, const int32_t* cu, hipStream_t s);
hipError_t launch_chunk_cumsum(int dtype, const SsdDims& d, const SsdBufs& b, const void* A,
                               const float* dt, const float* D, void* A_cumsum_out, hipStream_t s);
hipError_t launch_decay_chunk(int dtype, int batch, int H, int nch, int Q, const void* Acs,
                              void* out, hipStream_t s);
hipError_t launch_materialize_L(int dtype, int batch, int seqlen, int H, int Q, const void* a,
                                void* L, hipStream_t s);

// ssd_state.hip (fp32: launch_chunk_state runs ssd_f32.hip's)
// mode 0: st[c][h] = sum_l x_l^T (exp(cs_last - cs_l) dt_l B_l)      (forward chunk states)
// mode 1: dst[c][h] = sum_l dy_l^T (exp(cs_l) C_l)                    (backward local dh)
hipError_t launch_chunk_state(int dtype, int mode, const SsdDims& d, const SsdBufs& b,
                              const void* U, const void* V, const float* dt, float* out, hipStream_t s);
hipError_t launch_state_pass_fwd(int dtype, int state_dtype, const SsdDims& d, const SsdBufs& b,
                                 const void* init, void* final_state, hipStream_t s);
hipError_t launch_state_pass_bwd(int dtype, int state_dtype, const SsdDims& d, const SsdBufs& b,
                                 const void* dfinal, void* dinit, hipStream_t s);

// ssd_state_fused.hip (bf16 with 16-byte vector access): chunk states and the
// recurrence in one pass; the backward one writes b.dst16 and b.npass_blk partials
bool state_fused_supported(int dtype, const SsdDims& d);
int state_fused_slices(const SsdDims& d);
hipError_t launch_state_fwd_fused(const SsdDims& d, const SsdBufs& b, const void* x, const void* B, const float* fac,
                                  const void* init, void* final_state, int state_dtype, hipStream_t s);
// The same with a second forward walk in the same launch (no initial or final state): fac2, its states hst2
// and their residual hlo2 (the trapezoidal gamma path's beside the scan's).
hipError_t launch_state_fwd_fused2(const SsdDims& d, const SsdBufs& b, const void* x, const void* B, const float* fac,
                                   const float* fac2, void* hst2, uint8_t* hlo2, int state_dtype, hipStream_t s);
hipError_t launch_state_bwd_fused(const SsdDims& d, const SsdBufs& b, const void* dy, const void* C,
                                  const void* dfinal, void* dinit, int state_dtype, hipStream_t s);

// ssd_scan_fwd_chunk.hip (bf16 with 16-byte vector access): one block per (chunk, head slice)
bool scan_fwd_chunk_supported(int dtype, const SsdDims& d);
size_t lds_scan_fwd_chunk(const SsdDims& d);
// with `fast` (the k_chunk_cumsum flags) only slices holding a flagged (chunk, head) run: the fixup
// of the factorised kernel
hipError_t launch_scan_fwd_chunk(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, const int32_t* fast,
                                 hipStream_t s);
hipError_t launch_scan_fwd_pairs(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s);

// ssd_scan_fwd_fact.hip (same shapes): the factorised-decay forward scan, exact for the (chunk, head)
// pairs k_chunk_cumsum flags 1; the others are rewritten by launch_scan_fwd_chunk(..., b.fast, ...)
size_t lds_scan_fwd_fact(const SsdDims& d);
hipError_t launch_scan_fwd_fact(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s);

// ssd_scan_fwd.hip (bf16 shapes outside the fused path)
hipError_t launch_chunk_scan_fwd(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s);
size_t lds_chunk_scan_fwd(const SsdDims& d);

// ssd_f32.hip (fp32): the forward chunk scan, the chunk states (modes of launch_chunk_state), and the
// backward of units [u0, u0 + n) (units: chunk * G + group), column side then row side
size_t f32_unit_floats(const SsdDims& d);  // S (or dS) tiles of one unit
bool f32_supported(const SsdDims& d, size_t max_lds);
bool f32_self(const SsdDims& d);  // S is multiplied where it is used: no tiles of it
hipError_t launch_f32_scan(const SsdDims& d, const SsdBufs& b, const SsdIn& in, void* y, hipStream_t s);
hipError_t launch_f32_state(int mode, const SsdDims& d, const SsdBufs& b, const void* U, const void* V, const float* dt,
                            float* out, hipStream_t s);
hipError_t launch_f32_col(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, int u0, int n,
                          hipStream_t s);
hipError_t launch_f32_row(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC, int u0,
                          int n, hipStream_t s);

// ssd_bwd_bf16.hip (bf16 shapes outside the fused path)
hipError_t launch_bwd_col(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, void* dB,
                          hipStream_t s);
hipError_t launch_bwd_row(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dC, hipStream_t s);
// ssd_bwd.hip
// ddt and da32 (fp32 per-token decay gradient, a_mode PER_TOKEN) are optional
hipError_t launch_bwd_finish(int dtype, const SsdDims& d, const SsdBufs& b, const SsdIn& in,
                             float* ddt, void* dA_tok, float* da32, hipStream_t s);
size_t lds_bwd_col(const SsdDims& d);
size_t lds_bwd_row(const SsdDims& d);

// Fixup launches (k_scan_fwd_chunk, k_bwd_main with the k_chunk_cumsum flags): at most this many units per
// block of their chip-sized grid
#define SSD_FIX_UNITS 64

// ssd_bwd_main.hip (fused backward, bf16, Ppad <= 64, Qpad <= 256)
bool bwd_main_supported(int dtype, const SsdDims& d);
size_t lds_bwd_main(const SsdDims& d);
int bwd_main_num_sets(const SsdDims& d);
// fixup: only the (chunk, head) pairs b.fast flags 0, dS into b.dS_fix (the exact path behind k_bwd_fact)
hipError_t launch_bwd_main(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, bool fixup,
                           hipStream_t s);

// ssd_bwd_head.hip (fused path, one head per group): the whole of a (chunk, head)'s backward but the walks and the
// finish: dx, dB, dC, the decay gradient's terms (one rowG and one dcs_off partial), exact decays (no fixup).
// b.hdec / b.hdec_lo: the decay term's states with d.gdec
bool bwd_head_supported(int dtype, const SsdDims& d);
size_t lds_bwd_head(const SsdDims& d);
hipError_t launch_bwd_head(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx, void* dB,
                           void* dC, hipStream_t s);

// ssd_bwd_fact.hip (same shapes and grid as k_bwd_main): the factorised-decay column kernel
size_t lds_bwd_fact(const SsdDims& d);
hipError_t launch_bwd_fact(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dx,
                           hipStream_t s);

// ssd_bwd_gemm.hip (fused path): dB, dC and the Y_off part of the decay gradient
size_t lds_bwd_gemm(const SsdDims& d);
hipError_t launch_bwd_gemm(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                           hipStream_t s);

// ssd_bwd_rows.hip (fused path, groups of at most SSD_ROWS_MAX_HPG heads at 256-token chunks): the same
// outputs as launch_bwd_gemm, one block per (chunk, group, role) with the chunk's B / C rows in LDS; its
// decay term fills one dcs_off partial (b.ndcs == 1)
#define SSD_ROWS_MAX_HPG 8
bool bwd_rows_supported(const SsdDims& d, int nslices, bool any_hpg = false);
size_t lds_bwd_rows(const SsdDims& d);
hipError_t launch_bwd_rows(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                           hipStream_t s);

// ssd_norm.hip
hipError_t launch_gated_norm_fwd(int dtype, const SsdDims& d, const SsdBufs& b, const SsdIn& in,
                                 void* y, hipStream_t s);
hipError_t launch_gated_norm_bwd(int dtype, const SsdDims& d, const SsdBufs& b, const SsdIn& in,
                                 const void* dout, void* dz, hipStream_t s);

// ssd_trapz.hip (trapezoidal mode): rho, dt = gamma + rho, C.B and D per token into b.tz_* / b.Dtok;
// the column / row path's d(C.B) terms of dB and dC (and b.xdy); dgamma, dbeta, dA per token
hipError_t launch_trapz_prep(int dtype, const SsdDims& d, const SsdBufs& b, const void* A, const void* gamma,
                             const void* beta, const void* B, const void* C, const float* D, const int32_t* cu,
                             hipStream_t s);
// D per token from gamma and the forward scan's cb (tz_cb_fwd), between the factorised scan and its fixup.
hipError_t launch_trapz_dtok(const SsdDims& d, const SsdBufs& b, const float* D, hipStream_t s);
hipError_t launch_trapz_bc(int dtype, const SsdDims& d, const SsdBufs& b, const void* x, const void* dy,
                           const void* B, const void* C, void* dB, void* dC, const int32_t* cu, hipStream_t s);
hipError_t launch_trapz_grads(int dtype, const SsdDims& d, const SsdBufs& b, const void* A, const int32_t* cu,
                              const void* x, const void* dy, const void* B, const void* C, void* dgamma, void* dbeta,
                              void* dA, hipStream_t s);

// ssd_reduce.hip
hipError_t launch_reduce_slices(int dtype, int64_t nelem, int nslices, const float* part0, const float* part1,
                                void* out0, void* out1, hipStream_t s);
// dA / dD per head and the norm weight's gradient (out = sum of part's nblocks rows of width) in one launch;
// either side may be absent (dA_head = dD = nullptr, or out = nullptr)
hipError_t launch_reduce_tail(const SsdDims& d, const SsdBufs& b, float* dA_head, float* dD, int nblocks, int width,
                              const float* part, float* out, hipStream_t s);
hipError_t launch_reduce_rows(int nblocks, int width, const float* part, float* out, hipStream_t s);
