// extern "C" entry points: validation, workspace layout, launch sequences.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <initializer_list>
#include <mutex>

#include "ssd_mi355x.h"
#include "ssd_launch.h"

namespace {

constexpr size_t kAlign = 256;
constexpr size_t kMaxLds = 160 * 1024;   // LDS per workgroup on gfx950
constexpr int kMaxSeq = 16000;           // chunk-table prefix kept in LDS
constexpr int kMaxGrid = 65535;          // grid.y / grid.z limit used by the launches
constexpr int kNormMaxHP = 16384;        // dw partial row kept in LDS

size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

struct Plan {
  SsdDims d;
  int dtype, state_dtype;
  int64_t nslices, hslice, npass_blk, norm_blocks;
  // byte offsets inside each workspace
  size_t o_chunks, o_seq0, o_cs, o_bfac, o_ffac, o_ffac2, o_fast, o_hin, o_hinlo, o_ypre, o_rstd, o_tzdt, o_tzrho, o_tzgam,
      o_tzcb, o_Dtok, o_hgam, o_hgamlo, o_dtrep, o_Drep, saved_bytes;
  size_t o_st, fwd_bytes;
  size_t o_dyp, o_dst, o_dtot, o_rowG, o_colG, o_eterm, o_dcs, o_xdx, o_dD, o_dA, o_dBp, o_dCp, o_dw, o_dS, o_dSf, o_dst16,
      o_xdy, o_tzddt, o_tzda, o_bcb, o_fdS, bwd_bytes;
  int f32_fbatch, f32_bbatch, f32_rhs, f32_rsl;  // fp32: units per batch (forward, backward), row slices
  int fused_bwd, nrowg;
  int rows_chunk;  // fused path: the chunk-resident row kernel (k_bwd_rows) instead of k_bwd_gemm
  int gemm_hslice, gemm_tsteps, gemm_parts;  // fused path: SsdBufs
  int head_bwd;    // fused path, one head per group: k_bwd_head in place of the column and row kernels
};

// k_bwd_gemm's slices. Its blocks (one per CU) walk a group's heads one after the other and then the chunk's tile
// terms; where they fill a quarter of the chip or less, slices of the heads and the tile terms run side by side and
// one more launch sums their partials. Forward and backward at P = 64, N = 128, whole / sliced, us:
//   up to 32 blocks, four slices (more cost more to sum than they save) and one per tile step: 24 heads, chunk 256:
//     256 tokens 117 / 81, 2048 tokens 146 / 120; 64 heads, 64 tokens 136 / 72; 8 heads, 512 tokens 78 / 69; below 6
//     heads nothing (49 / 49 at 4)
//   up to 64, two slices or three and one for the tile terms: 24 heads 160 / 141 (8 x 512 tokens 140 / 122), 64 heads
//     277 / 229; 8 heads 97 / 99, so from 16 heads
//   more: 96 blocks of 16 heads 140 / 142, 120 of 12 heads 119 / 126, 128 of 64 heads 425 / 407: whole
// With several groups (one chunk of 256 tokens, 64 heads in 2 / 4 / 8 groups 160 / 93, 119 / 90, 103 / 90; four
// chunks in 4 groups 130 / 120) this holds because the kernel spreads groups and slices over the XCDs: on the chunks'
// own XCDs the slices queued up (8 groups 153).
void gemm_slices(const SsdDims& d, int* hslice, int* tsteps, int* parts) {
  const int nb = d.Qpad / SSD_BLK;
  const int64_t blocks = (int64_t)d.max_chunks * d.G * nb;
  const bool few = blocks <= 32 && d.hpg >= 6;
  int nz = few ? std::min(4, d.hpg / 2) : blocks <= 64 && d.hpg >= 16 ? (d.hpg >= 36 ? 3 : 2) : 1;
  *hslice = (d.hpg + nz - 1) / nz;
  nz = (d.hpg + *hslice - 1) / *hslice;
  *tsteps = few ? 1 : nb;
  *parts = nz > 1 ? nz + (nb + *tsteps - 1) / *tsteps : 1;
}

// `tight`: the plan with the smallest forward workspaces (wide bf16 heads whole, fp32 S tiles in the chunk
// states' place).
int plan(const ssd_desc_t* s, Plan* p, bool tight = false) {
  if (!s || !p) return SSD_ERR_INVALID;
  memset(p, 0, sizeof(*p));
  if (s->batch < 1 || s->seqlen < 1 || s->nheads < 1 || s->headdim < 1 || s->ngroups < 1 || s->dstate < 1 ||
      s->chunk < 1)
    return SSD_ERR_INVALID;
  if (s->nheads % s->ngroups) return SSD_ERR_INVALID;
  if ((s->dtype != SSD_DTYPE_F32 && s->dtype != SSD_DTYPE_BF16) ||
      (s->state_dtype != SSD_DTYPE_F32 && s->state_dtype != SSD_DTYPE_BF16))
    return SSD_ERR_INVALID;
  if (s->a_mode != SSD_A_PER_HEAD && s->a_mode != SSD_A_PER_TOKEN && s->a_mode != SSD_A_CUMSUM)
    return SSD_ERR_INVALID;
  if (s->a_mode != SSD_A_PER_HEAD && s->has_dt) return SSD_ERR_INVALID;
  if (s->varlen && (s->batch != 1 || s->nseq < 1)) return SSD_ERR_INVALID;
  if ((s->a_mode == SSD_A_CUMSUM || s->want_A_cumsum) && (s->varlen || s->seqlen % s->chunk)) return SSD_ERR_INVALID;
  if (s->has_z && !(s->norm_eps >= 0.0f)) return SSD_ERR_INVALID;
  if (s->dA_skip & ~(SSD_DA_SKIP_INTRA | SSD_DA_SKIP_CUMSUM | SSD_DA_SKIP_CHUNK)) return SSD_ERR_INVALID;
  // a cached A_cumsum carries no gradient, and neither does the decay_chunk built from it
  if (s->a_mode == SSD_A_CUMSUM && (~s->dA_skip & (SSD_DA_SKIP_CUMSUM | SSD_DA_SKIP_CHUNK))) return SSD_ERR_INVALID;
  // trapezoidal mode: per-token decay; dt, the initial / final state and the cache options are not part of it
  if (s->trapz != SSD_TRAPZ_OFF && s->trapz != SSD_TRAPZ_DROP_BETA_DA && s->trapz != SSD_TRAPZ_EXACT_DA)
    return SSD_ERR_INVALID;
  if (s->trapz && (s->a_mode != SSD_A_PER_TOKEN || s->has_dt || s->has_init || s->has_dfinal || s->want_final ||
                   s->want_A_cumsum || s->dA_skip))
    return SSD_ERR_INVALID;
  if (s->chunk > SSD_MAX_CHUNK || s->headdim > SSD_MAX_HEADDIM || s->dstate > SSD_MAX_DSTATE)
    return SSD_ERR_UNSUPPORTED;
  if (s->varlen && s->nseq > kMaxSeq) return SSD_ERR_UNSUPPORTED;
  // each factor bounded before the products below (which then fit in int64)
  if (s->batch > INT32_MAX || s->seqlen > INT32_MAX) return SSD_ERR_UNSUPPORTED;
  const int64_t R = s->batch * s->seqlen;
  if (R > INT32_MAX / 2 || s->nheads > kMaxGrid) return SSD_ERR_UNSUPPORTED;
  const int64_t cps = (s->seqlen + s->chunk - 1) / s->chunk;
  const int64_t nseq = s->varlen ? s->nseq : s->batch;
  const int64_t max_chunks = s->varlen ? cps + nseq : s->batch * cps;
  if (max_chunks > kMaxGrid) return SSD_ERR_UNSUPPORTED;
  if (s->has_z && s->nheads * s->headdim > kNormMaxHP) return SSD_ERR_UNSUPPORTED;

  SsdDims& d = p->d;
  d.batch = (int)s->batch; d.seqlen = (int)s->seqlen; d.H = (int)s->nheads; d.P = (int)s->headdim;
  d.G = (int)s->ngroups; d.N = (int)s->dstate; d.Q = (int)s->chunk;
  // The fused bf16 kernels hold heads of up to 64 columns. A head's P channels are independent given its dt,
  // A, B, C and D, so a wider one whose half is a whole number of 16-byte vectors runs as two kernel heads of
  // P / 2 that share them: x, y, z, the states and their gradients keep their layout (heads are the slower
  // dimension), the cumsum launch repeats dt and D, and the finish sums the gradients of the pair.
  // Past two limits the head stays whole on the general kernels, whose grids have three axes and whose backward
  // keeps no tiles of dS: the pairs' grids on one axis (at most 1024 threads per chunk and kernel head; a launch takes
  // 2^32), and dS tiles of 16 GiB.
  const int64_t nbk = round_up(d.Q, SSD_BLK) / SSD_BLK, pair_tiles = max_chunks * d.G * nbk * nbk * 4096 * 6;
  if (!tight && s->dtype == SSD_DTYPE_BF16 && d.P > 64 && d.P % 16 == 0 && d.N % 8 == 0 && 2 * s->nheads <= kMaxGrid &&
      max_chunks * s->nheads * 2 * 1024 <= (int64_t)UINT32_MAX && pair_tiles <= 16ll << 30) {
    d.H *= 2;
    d.P /= 2;
    d.hs = 1;
  }
  // feature widths padded to 32, 64 or 128 (the tile shapes the kernels are built for)
  d.Ppad = d.P <= 32 ? 32 : (d.P <= 64 ? 64 : 128);
  d.Npad = d.N <= 32 ? 32 : (d.N <= 64 ? 64 : 128);
  d.Qpad = round_up(d.Q, SSD_BLK);
  d.nseq = (int)nseq; d.max_chunks = (int)max_chunks; d.hpg = d.H / d.G; d.R = R;
  d.a_mode = s->a_mode; d.has_dt = s->has_dt != 0; d.has_D = s->has_D != 0; d.has_z = s->has_z != 0;
  d.has_init = s->has_init != 0; d.has_dfinal = s->has_dfinal != 0; d.varlen = s->varlen != 0;
  d.eps = s->norm_eps;
  d.dA_skip = s->dA_skip;
  d.trapz = s->trapz;
  if (d.trapz) d.has_dt = 1;  // the scan's dt is gamma + rho (k_trapz_coef)
  p->dtype = s->dtype;
  p->state_dtype = s->state_dtype;
  p->fused_bwd = bwd_main_supported(p->dtype, d) ? 1 : 0;
  if (p->dtype == SSD_DTYPE_F32) {
    if (!f32_supported(d, kMaxLds)) return SSD_ERR_UNSUPPORTED;
  } else if ((scan_fwd_chunk_supported(p->dtype, d) ? std::max(lds_scan_fwd_chunk(d), lds_scan_fwd_fact(d))
                                                    : lds_chunk_scan_fwd(d)) > kMaxLds ||
             (p->fused_bwd ? (lds_bwd_main(d) > kMaxLds || lds_bwd_fact(d) > kMaxLds || lds_bwd_gemm(d) > kMaxLds)
                           : (lds_bwd_col(d) > kMaxLds || lds_bwd_row(d) > kMaxLds))) {
    return SSD_ERR_UNSUPPORTED;
  }

  // head slices of the backward: enough blocks to fill the chip, fewest partials
  int64_t ns;
  if (p->fused_bwd) {
    // one block per (chunk, group, slice, column set); about one block per CU
    p->nrowg = bwd_main_num_sets(d);
    const int64_t per_slice = max_chunks * d.G * p->nrowg;
    ns = (256 + per_slice - 1) / per_slice;
  } else if (s->dtype == SSD_DTYPE_F32) {
    // four waves per SIMD in the column kernel (its waves are a unit's 32-token tiles; rowG in one partial per
    // block of a unit)
    p->nrowg = d.Qpad >= 192 ? 2 : 1;
    const int64_t per_slice = max_chunks * d.G * (d.Qpad / 32);
    ns = (4096 + per_slice - 1) / per_slice;
  } else {
    p->nrowg = 1;
    const int64_t per_slice = max_chunks * d.G * (d.Qpad / SSD_BLK);
    // at least ~1024 column blocks (32 heads per slice at config 2: fewer dS partials than 16, and the
    // block's S and B set-up spread over more heads)
    ns = (1024 + per_slice - 1) / per_slice;
  }
  if (ns < 1) ns = 1;
  if (ns > d.hpg) ns = d.hpg;
  p->hslice = (d.hpg + ns - 1) / ns;
  p->nslices = (d.hpg + p->hslice - 1) / p->hslice;
  gemm_slices(d, &p->gemm_hslice, &p->gemm_tsteps, &p->gemm_parts);
  // the row kernel of the fused path; SSD_ROW_KERNEL=block or =chunk in the environment overrides the choice
  // (block: k_bwd_gemm everywhere; chunk: k_bwd_rows wherever its shape limits allow, any heads per group)
  const char* rk = getenv("SSD_ROW_KERNEL");
  const bool force_block = rk && !strcmp(rk, "block"), force_chunk = rk && !strcmp(rk, "chunk");
  p->rows_chunk = p->fused_bwd && !force_block && bwd_rows_supported(d, (int)p->nslices, force_chunk) &&
                          lds_bwd_rows(d) <= kMaxLds
                      ? 1
                      : 0;
  // the fp32 path: tiles of S and dS per unit (chunk, group), in batches that bound their memory, and the row
  // kernel's head slices (up to two waves per SIMD over both roles, the tile term a slice of its own)
  const int64_t units = max_chunks * d.G;
  const bool f32 = s->dtype == SSD_DTYPE_F32;
  const size_t unit_bytes = f32 ? f32_unit_floats(d) * sizeof(float) : 0;
  const size_t s_bytes = f32 && !f32_self(d) ? unit_bytes : 0;  // S tiles of a unit
  if (f32) {
    constexpr int64_t kFwdTiles = 512ll << 20, kBwdTiles = 1ll << 30;
    const int64_t st_bytes = max_chunks * d.H * d.Ppad * d.Npad * 4;
    const int64_t fb = s_bytes ? (tight ? st_bytes : std::max(st_bytes, kFwdTiles)) / (int64_t)s_bytes : units;
    const int64_t bb = kBwdTiles / (int64_t)(p->nslices * unit_bytes + s_bytes);
    // the grids are on one axis of 2^32 threads: per unit the scan's heads of a group and 64-column parts of a head,
    // and the S tiles' waves
    const int64_t unit_threads = std::max<int64_t>((int64_t)d.hpg * ((d.P + 63) / 64) * 64 * ((d.Qpad / 32 + 1) / 2),
                                                   (int64_t)(unit_bytes / 4096 + 3) / 4 * 256);
    p->f32_fbatch = (int)std::max<int64_t>(1, std::min({units, fb, (int64_t)UINT32_MAX / unit_threads}));
    p->f32_bbatch = (int)std::max<int64_t>(1, std::min(units, bb));
    int64_t nhs = 2048 / (units * 2 * (d.Qpad / 32)) - 1;
    nhs = std::min<int64_t>(std::max<int64_t>(nhs, 1), d.hpg);
    p->f32_rhs = (int)((d.hpg + nhs - 1) / nhs);
    nhs = (d.hpg + p->f32_rhs - 1) / p->f32_rhs;
    p->f32_rsl = nhs == 1 ? 1 : (int)nhs + 1;
  }
  p->head_bwd = p->fused_bwd && !force_block && !force_chunk && bwd_head_supported(p->dtype, d) &&
                lds_bwd_head(d) <= kMaxLds && max_chunks * d.H <= INT32_MAX;
  p->npass_blk = ((int64_t)d.Ppad * d.Npad + SSD_PASS_THREADS - 1) / SSD_PASS_THREADS;
  p->norm_blocks = R < 512 ? R : 512;

  const size_t es = p->dtype == SSD_DTYPE_BF16 ? 2 : 4;
  const size_t MC = (size_t)max_chunks, H = (size_t)d.H, PN = (size_t)d.Ppad * d.Npad;
  size_t off = 0;
  auto take = [&off](size_t bytes) { size_t o = off; off = align_up(off + bytes); return o; };
  p->o_chunks = take(MC * sizeof(ChunkInfo));
  p->o_seq0 = take((nseq + 1 + (d.varlen ? nseq : 0)) * sizeof(int32_t));  // + the walks' sequence order
  p->o_cs = take(MC * H * d.Qpad * sizeof(float));
  p->o_bfac = take(MC * H * d.Qpad * sizeof(float));
  p->o_fast = take(MC * H * sizeof(int32_t));
  p->o_hin = take(MC * H * PN * es);
  // bf16 states: their rounding residuals (fp8 bytes), for the decay gradient's Y_off term, where that
  // term feeds an output (not with a cached A_cumsum, and not the trapezoidal scan whose dA is the gamma
  // path's alone: there only the gamma path's states need it)
  const bool lo = p->dtype == SSD_DTYPE_BF16;
  p->o_hinlo = (lo && !(d.dA_skip & SSD_DA_SKIP_CUMSUM) && d.trapz != SSD_TRAPZ_DROP_BETA_DA) ? take(MC * H * PN) : 0;
  p->o_ypre = d.has_z ? take((size_t)R * H * d.P * es) : 0;
  p->o_rstd = d.has_z ? take((size_t)R * sizeof(float)) : 0;
  const size_t rh = (size_t)R * H * sizeof(float);
  p->o_tzdt = d.trapz ? take(rh) : 0;
  p->o_tzrho = d.trapz ? take(rh) : 0;
  p->o_tzgam = d.trapz ? take(rh) : 0;
  p->o_Dtok = d.trapz ? take(rh) : 0;
  p->o_tzcb = d.trapz ? take((size_t)R * d.G * sizeof(float)) : 0;
  p->o_hgam = d.trapz == SSD_TRAPZ_DROP_BETA_DA ? take(MC * H * PN * es) : 0;
  p->o_hgamlo = (d.trapz == SSD_TRAPZ_DROP_BETA_DA && lo) ? take(MC * H * PN) : 0;
  p->o_dtrep = (d.hs && d.has_dt && !d.trapz) ? take(rh) : 0;
  p->o_Drep = (d.hs && d.has_D) ? take(H * sizeof(float)) : 0;
  p->saved_bytes = off;
  off = 0;
  // (fp32: the scan's S tiles, once the chunk states have been used)
  p->o_st = take(std::max(MC * H * PN * sizeof(float), p->f32_fbatch * s_bytes));
  p->o_ffac = take(MC * H * d.Qpad * sizeof(float));
  p->o_ffac2 = d.trapz == SSD_TRAPZ_DROP_BETA_DA ? take(MC * H * d.Qpad * sizeof(float)) : 0;
  p->fwd_bytes = off;
  off = 0;
  p->o_dyp = d.has_z ? take((size_t)R * H * d.P * es) : 0;
  p->o_dst = take(MC * H * PN * sizeof(float));
  p->o_dtot = take(MC * H * p->npass_blk * sizeof(float));
  p->o_rowG = take((size_t)p->nrowg * MC * H * d.Qpad * sizeof(float));
  p->o_colG = take(MC * H * d.Qpad * sizeof(float));
  p->o_eterm = take(MC * H * d.Qpad * sizeof(float));
  p->o_dcs = take((p->fused_bwd ? 2 : 1) * MC * H * d.Qpad * sizeof(float));
  p->o_xdx = take(MC * H * d.Qpad * sizeof(float));
  p->o_dD = take(MC * H * (d.Qpad / SSD_BLK) * sizeof(float));
  p->o_dA = take(MC * H * sizeof(float));
  const size_t bcn = (size_t)R * d.G * d.N * sizeof(float);
  // (a fused plan's general kernels, for rows off the 16-byte grid, have nslices partials)
  const int64_t nparts = f32 ? p->f32_rsl : std::max<int64_t>(p->nslices, p->fused_bwd ? p->gemm_parts : 1);
  p->o_dBp = nparts > 1 ? take(nparts * bcn) : 0;
  p->o_dCp = nparts > 1 ? take(nparts * bcn) : 0;
  p->o_bcb = s_bytes ? take(p->f32_bbatch * s_bytes) : 0;
  p->o_fdS = f32 ? take(p->nslices * p->f32_bbatch * unit_bytes) : 0;
  const size_t nbq = (size_t)(d.Qpad / SSD_BLK);
  const bool tiles = p->fused_bwd;
  // one head slice: the tiles in bf16 (each is rounded to bf16 for the row kernel's products anyway)
  p->o_dS = tiles ? take((size_t)p->nslices * MC * d.G * nbq * nbq * 4096 * (p->nslices == 1 ? 2 : 4)) : 0;
  p->o_dSf = tiles ? take(MC * d.G * nbq * nbq * 4096 * sizeof(float)) : 0;
  p->o_dst16 = tiles ? take(MC * H * PN * 2) : 0;
  p->o_dw = d.has_z ? take((size_t)p->norm_blocks * d.H * d.P * sizeof(float)) : 0;
  p->o_xdy = d.trapz ? take(MC * H * d.Qpad * sizeof(float)) : 0;
  p->o_tzddt = d.trapz ? take(rh) : 0;
  p->o_tzda = d.trapz ? take(rh) : 0;
  p->bwd_bytes = off;
  return SSD_OK;
}

void bind_saved(const Plan& p, void* saved, SsdBufs* b) {
  unsigned char* s = static_cast<unsigned char*>(saved);
  b->chunks = reinterpret_cast<ChunkInfo*>(s + p.o_chunks);
  b->seq_chunk0 = reinterpret_cast<int32_t*>(s + p.o_seq0);
  b->seq_order = p.d.varlen ? b->seq_chunk0 + p.d.nseq + 1 : nullptr;
  b->cs = reinterpret_cast<float*>(s + p.o_cs);
  b->bwd_fac = reinterpret_cast<float*>(s + p.o_bfac);
  b->fast = reinterpret_cast<int32_t*>(s + p.o_fast);
  b->hin = s + p.o_hin;
  b->hin_lo = p.o_hinlo ? s + p.o_hinlo : nullptr;
  b->ypre = p.d.has_z ? s + p.o_ypre : nullptr;
  b->rstd = p.d.has_z ? reinterpret_cast<float*>(s + p.o_rstd) : nullptr;
  b->npass_blk = (int)p.npass_blk;
  b->nslices = (int)p.nslices;
  b->hslice = (int)p.hslice;
  b->norm_blocks = (int)p.norm_blocks;
  b->fused_bwd = p.fused_bwd;
  b->nrowg = p.nrowg;
  b->gemm_hslice = p.gemm_hslice;
  b->gemm_tsteps = p.gemm_tsteps;
  b->gemm_parts = p.gemm_parts;
  b->ndcs = p.fused_bwd && !p.rows_chunk ? 2 : 1;
  b->rows_chunk = p.rows_chunk;
  b->dt_rep = p.o_dtrep ? reinterpret_cast<float*>(s + p.o_dtrep) : nullptr;
  b->D_rep = p.o_Drep ? reinterpret_cast<float*>(s + p.o_Drep) : nullptr;
  if (p.d.trapz) {
    b->tz_dt = reinterpret_cast<float*>(s + p.o_tzdt);
    b->tz_rho = reinterpret_cast<float*>(s + p.o_tzrho);
    b->tz_gam = reinterpret_cast<float*>(s + p.o_tzgam);
    b->Dtok = reinterpret_cast<float*>(s + p.o_Dtok);
    b->tz_cb = reinterpret_cast<float*>(s + p.o_tzcb);
    b->hgam = p.d.trapz == SSD_TRAPZ_DROP_BETA_DA ? s + p.o_hgam : nullptr;
    b->hgam_lo = p.o_hgamlo ? s + p.o_hgamlo : nullptr;
  }
}

void bind_bwd(const Plan& p, void* scratch, SsdBufs* b) {
  unsigned char* s = static_cast<unsigned char*>(scratch);
  b->dyp = p.d.has_z ? s + p.o_dyp : nullptr;
  b->dst = reinterpret_cast<float*>(s + p.o_dst);
  b->dtot_part = reinterpret_cast<float*>(s + p.o_dtot);
  b->rowG = reinterpret_cast<float*>(s + p.o_rowG);
  b->colG = reinterpret_cast<float*>(s + p.o_colG);
  b->eterm = reinterpret_cast<float*>(s + p.o_eterm);
  b->dcs_off = reinterpret_cast<float*>(s + p.o_dcs);
  b->xdx = reinterpret_cast<float*>(s + p.o_xdx);
  b->dD_part = reinterpret_cast<float*>(s + p.o_dD);
  b->dA_part = reinterpret_cast<float*>(s + p.o_dA);
  b->dB_part = p.o_dBp ? reinterpret_cast<float*>(s + p.o_dBp) : nullptr;
  b->dC_part = p.o_dCp ? reinterpret_cast<float*>(s + p.o_dCp) : nullptr;
  b->f32_cb = reinterpret_cast<float*>(s + p.o_bcb);
  b->f32_dS = reinterpret_cast<float*>(s + p.o_fdS);
  b->f32_batch = p.f32_bbatch;
  b->f32_rhs = p.f32_rhs;
  b->f32_rsl = p.f32_rsl;
  const bool tiles = p.fused_bwd;
  b->dS_tiles = (tiles && p.nslices > 1) ? reinterpret_cast<float*>(s + p.o_dS) : nullptr;
  b->dS_tiles16 = (tiles && p.nslices == 1) ? reinterpret_cast<bf16*>(s + p.o_dS) : nullptr;
  b->dS_fix = tiles ? reinterpret_cast<float*>(s + p.o_dSf) : nullptr;
  b->dst16 = tiles ? reinterpret_cast<bf16*>(s + p.o_dst16) : nullptr;
  b->dw_part = p.d.has_z ? reinterpret_cast<float*>(s + p.o_dw) : nullptr;
  if (p.d.trapz) {
    b->xdy = reinterpret_cast<float*>(s + p.o_xdy);
    b->tz_ddt = reinterpret_cast<float*>(s + p.o_tzddt);
    b->tz_da = reinterpret_cast<float*>(s + p.o_tzda);
  }
}

bool aligned16(const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Vector-load flags for this call: widths and row strides multiples of one
// 16-byte vector, every pointer of that shape 16-byte aligned.
void set_vec_flags(SsdDims* d, int dtype, std::initializer_list<const void*> xs,
                   std::initializer_list<const void*> bcs) {
  const int V = dtype == SSD_DTYPE_BF16 ? 8 : 4;
  bool vx = d->P % V == 0, vbc = d->N % V == 0;
  for (const void* p : xs) vx = vx && aligned16(p);
  for (const void* p : bcs) vbc = vbc && aligned16(p);
  d->vec_x = vx;
  d->vec_bc = vbc;
}

#define SSD_TRY(expr)                          \
  do {                                         \
    if ((expr) != hipSuccess) return SSD_ERR_HIP; \
  } while (0)

// Brackets the launches of one phase with the caller's events (if any).
struct PhaseTimer {
  void* const* ev;
  hipStream_t s;
  hipError_t begin(int ph) const {
    return ev ? hipEventRecord(static_cast<hipEvent_t>(ev[2 * ph]), s) : hipSuccess;
  }
  hipError_t end(int ph) const {
    return ev ? hipEventRecord(static_cast<hipEvent_t>(ev[2 * ph + 1]), s) : hipSuccess;
  }
};

#define SSD_PHASE(tm, ph, expr)   \
  do {                            \
    SSD_TRY((tm).begin(ph));      \
    SSD_TRY(expr);                \
    SSD_TRY((tm).end(ph));        \
  } while (0)

int fwd_impl(Plan& p, const ssd_desc_t* desc, const ssd_fwd_args_t* a, void* saved, size_t saved_bytes, void* scratch,
             size_t scratch_bytes, void* stream) {
  SsdDims& d = p.d;
  if (!a || !a->x || !a->A || !a->B || !a->C || !a->y) return SSD_ERR_INVALID;
  if ((d.has_dt && !d.trapz && !a->dt) || (d.has_D && !a->D) || (d.has_z && (!a->z || !a->norm_weight)) ||
      (d.has_init && !a->init) || (d.varlen && !a->cu_seqlens) || (desc->want_final && !a->final_state) ||
      (desc->want_A_cumsum && !a->A_cumsum_out) || (d.trapz && (!a->gamma || !a->beta)))
    return SSD_ERR_INVALID;
  if (!saved || saved_bytes < p.saved_bytes || !scratch || scratch_bytes < p.fwd_bytes) return SSD_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  set_vec_flags(&p.d, p.dtype, {a->x, a->y, a->z}, {a->B, a->C});
  SsdBufs b;
  memset(&b, 0, sizeof(b));
  bind_saved(p, saved, &b);
  b.st = reinterpret_cast<float*>(scratch);
  b.f32_cb = b.st;
  b.f32_batch = p.f32_fbatch;
  b.fwd_fac = reinterpret_cast<float*>(static_cast<unsigned char*>(scratch) + p.o_ffac);
  b.fwd_fac2 = p.o_ffac2 ? reinterpret_cast<float*>(static_cast<unsigned char*>(scratch) + p.o_ffac2) : nullptr;
  // trapezoidal mode: the scan's dt is gamma + rho, written by the coefficient kernel; dt and D per kernel
  // head where a caller head is two of them
  const float* dt = d.trapz ? b.tz_dt : (b.dt_rep ? b.dt_rep : a->dt);
  const float* Dk = b.D_rep ? b.D_rep : a->D;
  SsdIn in = {a->x, dt, a->A, a->B, a->C, Dk, a->z, a->norm_weight, a->init, a->cu_seqlens};
  const PhaseTimer tm{a->events, s};
  const bool fused_state = state_fused_supported(p.dtype, d);
  // packed sequences: the chunk table from cu_seqlens; fixed-length batches: written by the cumsum launch
  if (d.varlen) SSD_PHASE(tm, SSD_PH_CHUNK_TABLE, launch_chunk_table(d, b, a->cu_seqlens, s));
  SSD_PHASE(tm, SSD_PH_CUMSUM,
            launch_chunk_cumsum(p.dtype, d, b, a->A, a->dt, a->D, desc->want_A_cumsum ? a->A_cumsum_out : nullptr, s));
  // the factorised forward scan (bf16, 16-byte rows) computes S = C B^T per chunk and group anyway: in the
  // trapezoidal mode it also writes the per-token cb = C_t . B_t (S's diagonal) and D per token
  // Halves of wide heads take the exact kernel with S in fp32 (ssd_scan_fwd_chunk.hip): the factorised one would
  // round S and x once more than the general kernel does for the whole head.
  const bool fwd_fused = scan_fwd_chunk_supported(p.dtype, d) && d.vec_x && d.vec_bc;
  const bool fwd_pairs = fwd_fused && d.hs, fwd_fact = fwd_fused && !d.hs;
  b.tz_cb_fwd = d.trapz && fwd_fact ? 1 : 0;
  if (d.trapz) {
    SSD_TRY(tm.begin(SSD_PH_TRAPZ_PREP));
    SSD_TRY(launch_trapz_prep(p.dtype, d, b, a->A, a->gamma, a->beta, a->B, a->C, Dk, a->cu_seqlens, s));
    if (d.trapz == SSD_TRAPZ_DROP_BETA_DA && !fused_state) {
      // the gamma path's own states, for the backward's gamma-path decay gradient (the fused walk computes
      // them in the scan's forward walk launch)
      SsdBufs bg = b;
      bg.hin = b.hgam;
      bg.hin_lo = b.hgam_lo;
      SSD_TRY(launch_chunk_state(p.dtype, 0, d, bg, a->x, a->B, b.tz_gam, b.st, s));
      SSD_TRY(launch_state_pass_fwd(p.dtype, p.state_dtype, d, bg, nullptr, nullptr, s));
    }
    SSD_TRY(tm.end(SSD_PH_TRAPZ_PREP));
  }
  if (fused_state && d.trapz == SSD_TRAPZ_DROP_BETA_DA) {
    // the scan's states and the gamma path's own (for the backward's gamma-path decay gradient), one launch
    SSD_PHASE(tm, SSD_PH_FWD_PASS,
              launch_state_fwd_fused2(d, b, a->x, a->B, b.fwd_fac, b.fwd_fac2, b.hgam, b.hgam_lo, p.state_dtype, s));
  } else if (fused_state) {
    SSD_PHASE(tm, SSD_PH_FWD_PASS,
              launch_state_fwd_fused(d, b, a->x, a->B, b.fwd_fac, d.has_init ? a->init : nullptr,
                                     desc->want_final ? a->final_state : nullptr, p.state_dtype, s));
  } else {
    SSD_PHASE(tm, SSD_PH_FWD_STATE, launch_chunk_state(p.dtype, 0, d, b, a->x, a->B, dt, b.st, s));
    SSD_PHASE(tm, SSD_PH_FWD_PASS,
              launch_state_pass_fwd(p.dtype, p.state_dtype, d, b, d.has_init ? a->init : nullptr,
                                    desc->want_final ? a->final_state : nullptr, s));
  }
  void* yout = d.has_z ? b.ypre : a->y;
  if (fwd_fact) {
    // factorised decay, then the exact kernel on the (chunk, head) pairs it cannot take
    SSD_TRY(tm.begin(SSD_PH_FWD_SCAN));
    SSD_TRY(launch_scan_fwd_fact(d, b, in, yout, s));
    if (b.tz_cb_fwd) SSD_TRY(launch_trapz_dtok(d, b, Dk, s));
    SSD_TRY(launch_scan_fwd_chunk(d, b, in, yout, b.fast, s));
    SSD_TRY(tm.end(SSD_PH_FWD_SCAN));
  } else if (fwd_pairs)
    SSD_PHASE(tm, SSD_PH_FWD_SCAN, launch_scan_fwd_pairs(d, b, in, yout, s));
  else if (p.dtype == SSD_DTYPE_F32)
    SSD_PHASE(tm, SSD_PH_FWD_SCAN, launch_f32_scan(d, b, in, yout, s));
  else
    SSD_PHASE(tm, SSD_PH_FWD_SCAN, launch_chunk_scan_fwd(d, b, in, yout, s));
  if (d.has_z) SSD_PHASE(tm, SSD_PH_NORM_FWD, launch_gated_norm_fwd(p.dtype, d, b, in, a->y, s));
  return SSD_OK;
}

// ---------------------------------------------------------------------------
// Workspace of ssd_fwd_noalloc: one file-scope device array per GPU, allocated
// with the code object when the library is first used on that GPU and held
// until the process ends. Host code never passes the array's name to a kernel
// (on the host it is a stand-in, not a device address): each device's address
// comes from hipGetSymbolAddress, taken once with that device current.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[SSD_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (nullptr on a HIP error).
void* scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

// Shape checks of the cache helpers (ssd_materialize_L, ssd_decay_chunk), before their pointers: each
// extent goes to the launch as an int, and the grid (batch x heads, times the chunks for L) is one
// dimension; every factor is bounded before a product.
int cache_helper_shape(const ssd_desc_t* d) {
  if (!d) return SSD_ERR_INVALID;
  if (d->batch < 1 || d->seqlen < 1 || d->nheads < 1 || d->chunk < 1 || d->seqlen % d->chunk || d->varlen ||
      (d->dtype != SSD_DTYPE_F32 && d->dtype != SSD_DTYPE_BF16))
    return SSD_ERR_INVALID;
  if (d->batch > INT32_MAX || d->nheads > INT32_MAX || d->seqlen > INT32_MAX) return SSD_ERR_UNSUPPORTED;
  const int64_t bh = d->batch * d->nheads;
  if (bh > INT32_MAX || bh * (d->seqlen / d->chunk) > INT32_MAX) return SSD_ERR_UNSUPPORTED;
  return SSD_OK;
}

}  // namespace

extern "C" {

int ssd_validate(const ssd_desc_t* desc) {
  Plan p;
  return plan(desc, &p);
}

size_t ssd_workspace_bytes(const ssd_desc_t* desc, int kind) {
  Plan p;
  if (plan(desc, &p) != SSD_OK) return 0;
  switch (kind) {
    case SSD_WS_SAVED: return p.saved_bytes;
    case SSD_WS_FWD_SCRATCH: return p.fwd_bytes;
    case SSD_WS_BWD_SCRATCH: return p.bwd_bytes;
    default: return 0;
  }
}

int ssd_fwd(const ssd_desc_t* desc, const ssd_fwd_args_t* a, void* saved, size_t saved_bytes, void* scratch,
            size_t scratch_bytes, void* stream) {
  Plan p;
  const int st = plan(desc, &p);
  if (st != SSD_OK) return st;
  return fwd_impl(p, desc, a, saved, saved_bytes, scratch, scratch_bytes, stream);
}

int ssd_fwd_noalloc(const ssd_desc_t* desc, const ssd_fwd_args_t* a, void* stream) {
  Plan p;
  int st = plan(desc, &p);
  if (st != SSD_OK) return st;
  // both forward workspaces, one after the other (the saved part is not kept for a backward); near the limit
  // the plan with the smallest ones (a wide head's pair takes a little more than the head itself)
  if (align_up(p.saved_bytes) + p.fwd_bytes > (size_t)SSD_NOALLOC_SCRATCH_BYTES) {
    st = plan(desc, &p, true);
    if (st != SSD_OK) return st;
  }
  const size_t off = align_up(p.saved_bytes);
  if (off + p.fwd_bytes > (size_t)SSD_NOALLOC_SCRATCH_BYTES) return SSD_ERR_TOO_LARGE;
  unsigned char* base = static_cast<unsigned char*>(scratch_on_current_device());
  if (!base) return SSD_ERR_HIP;
  return fwd_impl(p, desc, a, base, p.saved_bytes, base + off, p.fwd_bytes, stream);
}

int ssd_bwd(const ssd_desc_t* desc, const ssd_bwd_args_t* a, const void* saved, size_t saved_bytes, void* scratch,
            size_t scratch_bytes, void* stream) {
  Plan p;
  int st = plan(desc, &p);
  if (st != SSD_OK) return st;
  SsdDims& d = p.d;
  if (!a || !a->x || !a->A || !a->B || !a->C || !a->dy || !a->dx || !a->dB || !a->dC) return SSD_ERR_INVALID;
  if ((d.has_dt && !d.trapz && !a->dt) || (d.has_D && !a->D) || (d.has_z && (!a->z || !a->norm_weight || !a->dz)) ||
      (d.varlen && !a->cu_seqlens) || (d.has_dfinal && !a->dfinal))
    return SSD_ERR_INVALID;
  if (!saved || saved_bytes < p.saved_bytes || !scratch || scratch_bytes < p.bwd_bytes) return SSD_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  set_vec_flags(&p.d, p.dtype, {a->x, a->z, a->dy, a->dx, a->dz}, {a->B, a->C, a->dB, a->dC});
  SsdBufs b;
  memset(&b, 0, sizeof(b));
  bind_saved(p, const_cast<void*>(saved), &b);
  bind_bwd(p, scratch, &b);
  const float* dt = d.trapz ? b.tz_dt : (b.dt_rep ? b.dt_rep : a->dt);
  SsdIn in = {a->x, dt, a->A, a->B, a->C, b.D_rep ? b.D_rep : a->D, a->z, a->norm_weight, a->init, a->cu_seqlens};
  const PhaseTimer tm{a->events, s};
  // the fused backward needs 16-byte vector access; otherwise the column / row kernels run
  const bool fused = p.fused_bwd && d.vec_x && d.vec_bc;
  if (!fused) {
    b.ndcs = 1;
    if (p.dtype != SSD_DTYPE_F32) b.nrowg = 1;  // the bf16 column / row kernels write one rowG partial
    b.dst16 = nullptr;     // and read dst in fp32
  }
  const bool head = fused && p.head_bwd;
  if (head) b.nrowg = b.ndcs = 1;  // (its row sums of G and its decay term are whole)
  const bool fused_state = fused && state_fused_supported(p.dtype, d);
  if (fused_state) b.npass_blk = state_fused_slices(d);  // dtot partials: one per 32 x 32 state tile
  const void* dY = a->dy;
  if (d.has_z) {
    // (its weight gradient's partials are reduced by the backward's last launch, with dA / dD)
    SSD_PHASE(tm, SSD_PH_NORM_BWD, launch_gated_norm_bwd(p.dtype, d, b, in, a->dy, a->dz, s));
    dY = b.dyp;
  }
  // dB / dC of the head slices
  const int nparts = p.dtype == SSD_DTYPE_F32    ? p.f32_rsl
                     : !fused                    ? (int)p.nslices
                     : (head || b.rows_chunk)    ? 1
                                                 : p.gemm_parts;
  auto reduce_bc = [&](const PhaseTimer& t) -> int {
    if (nparts > 1)
      SSD_PHASE(t, SSD_PH_BWD_REDUCE_BC,
                launch_reduce_slices(p.dtype, d.R * d.G * d.N, nparts, b.dB_part, b.dC_part, a->dB, a->dC, s));
    return SSD_OK;
  };
  // One backward of the scan for (dd, bb, ii): the state pass (unless skipped: dst is then the one a
  // previous pass left in the scratch), the column / row phases and the finish.
  auto scan_bwd = [&](const SsdDims& dd, const SsdBufs& bb, const SsdIn& ii, const PhaseTimer& t, bool state_pass,
                      float* ddt, void* dA_tok, float* da32) -> int {
    if (state_pass) {
      if (fused_state) {
        SSD_PHASE(t, SSD_PH_BWD_PASS,
                  launch_state_bwd_fused(dd, bb, dY, a->C, dd.has_dfinal ? a->dfinal : nullptr,
                                         dd.has_init ? a->dinit : nullptr, p.state_dtype, s));
      } else {
        SSD_PHASE(t, SSD_PH_BWD_STATE, launch_chunk_state(p.dtype, 1, dd, bb, dY, a->C, ii.dt, bb.dst, s));
        SSD_PHASE(t, SSD_PH_BWD_PASS,
                  launch_state_pass_bwd(p.dtype, p.state_dtype, dd, bb, dd.has_dfinal ? a->dfinal : nullptr,
                                        dd.has_init ? a->dinit : nullptr, s));
      }
    }
    if (head) {
      SSD_PHASE(t, SSD_PH_BWD_COL, launch_bwd_head(dd, bb, ii, dY, a->dx, a->dB, a->dC, s));
    } else if (fused) {
      // factorised column kernel, then the exact one on the (chunk, head) pairs it cannot take;
      // the row phase builds dB / dC
      SSD_TRY(t.begin(SSD_PH_BWD_COL));
      SSD_TRY(launch_bwd_fact(dd, bb, ii, dY, a->dx, s));
      SSD_TRY(launch_bwd_main(dd, bb, ii, dY, a->dx, true, s));
      SSD_TRY(t.end(SSD_PH_BWD_COL));
      SSD_PHASE(t, SSD_PH_BWD_ROW,
                bb.rows_chunk ? launch_bwd_rows(dd, bb, ii, dY, a->dB, a->dC, s)
                              : launch_bwd_gemm(dd, bb, ii, dY, a->dB, a->dC, s));
    } else if (p.dtype == SSD_DTYPE_F32) {
      // both sides per batch of units (one batch up to 1 GiB of tiles; past it the column phase's events
      // bracket both)
      const int units = dd.max_chunks * dd.G;
      SSD_TRY(t.begin(SSD_PH_BWD_COL));
      for (int u0 = 0; u0 < units; u0 += bb.f32_batch) {
        const int n = std::min(bb.f32_batch, units - u0);
        SSD_TRY(launch_f32_col(dd, bb, ii, dY, a->dx, u0, n, s));
        if (u0 + n == units) {
          SSD_TRY(t.end(SSD_PH_BWD_COL));
          SSD_TRY(t.begin(SSD_PH_BWD_ROW));
        }
        SSD_TRY(launch_f32_row(dd, bb, ii, dY, a->dB, a->dC, u0, n, s));
      }
      SSD_TRY(t.end(SSD_PH_BWD_ROW));
    } else {
      SSD_PHASE(t, SSD_PH_BWD_COL, launch_bwd_col(dd, bb, ii, dY, a->dx, a->dB, s));
      SSD_PHASE(t, SSD_PH_BWD_ROW, launch_bwd_row(dd, bb, ii, dY, a->dC, s));
    }
    SSD_PHASE(t, SSD_PH_BWD_FINISH, launch_bwd_finish(p.dtype, dd, bb, ii, ddt, dA_tok, da32, s));
    return reduce_bc(t);
  };
  // The reference's dA in the drop setting: the gamma path's alone, the decay gradient of
  // SSD(gamma x, a, B, C) over its own states (h_in of the gamma path, hgam).
  SsdDims dg = d;
  dg.trapz = SSD_TRAPZ_OFF;
  dg.has_D = 0;
  dg.has_z = 0;
  dg.da_only = 1;
  SsdBufs bg = b;
  bg.hin = b.hgam;
  bg.hin_lo = b.hgam_lo;
  bg.Dtok = nullptr;
  SsdIn ig = in;
  ig.dt = b.tz_gam;
  if (d.trapz == SSD_TRAPZ_DROP_BETA_DA && fused) {
    // Inside the scan's own backward: the walk takes dtot from the gamma path's states (its dst is the
    // same for both paths), the column kernel and the exact fixup weight their decay terms by gamma
    // (SsdDims.gdec: G's v_s = gamma_s g_s, E's gamma_s) while dS, dX and dx keep dt = gamma + rho, the
    // row kernel's decay term reads hgam (the chunk-resident kernel in the same blocks; the other in a
    // decay-only pass after the scan's, rewriting dcs_off), and one finish gives d(dt) (x . dX, for
    // drho, dgamma and dbeta) and the gamma path's da.
    SsdDims dm = d;
    dm.gdec = 1;
    SsdBufs bw = b;
    bw.hin = b.hgam;
    bw.hin_lo = b.hgam_lo;
    if (fused_state) {
      SSD_PHASE(tm, SSD_PH_BWD_PASS, launch_state_bwd_fused(dm, bw, dY, a->C, nullptr, nullptr, p.state_dtype, s));
    } else {
      SSD_PHASE(tm, SSD_PH_BWD_STATE, launch_chunk_state(p.dtype, 1, dm, bw, dY, a->C, in.dt, bw.dst, s));
      SSD_PHASE(tm, SSD_PH_BWD_PASS, launch_state_pass_bwd(p.dtype, p.state_dtype, dm, bw, nullptr, nullptr, s));
    }
    SsdBufs br = b;  // the decay term over hgam in the same blocks (head kernel, chunk-resident row kernel)
    br.hdec = b.hgam;
    br.hdec_lo = b.hgam_lo;
    if (head) {
      SSD_PHASE(tm, SSD_PH_BWD_COL, launch_bwd_head(dm, br, in, dY, a->dx, a->dB, a->dC, s));
    } else {
      SSD_TRY(tm.begin(SSD_PH_BWD_COL));
      SSD_TRY(launch_bwd_fact(dm, b, in, dY, a->dx, s));
      SSD_TRY(launch_bwd_main(dm, b, in, dY, a->dx, true, s));
      SSD_TRY(tm.end(SSD_PH_BWD_COL));
    }
    if (head) {
    } else if (b.rows_chunk) {
      SSD_PHASE(tm, SSD_PH_BWD_ROW, launch_bwd_rows(dm, br, in, dY, a->dB, a->dC, s));
    } else {
      SSD_PHASE(tm, SSD_PH_BWD_ROW, launch_bwd_gemm(dm, b, in, dY, a->dB, a->dC, s));
      SSD_PHASE(tm, SSD_PH_TRAPZ_GAMMA, launch_bwd_gemm(dg, bg, ig, dY, a->dB, a->dC, s));
    }
    SSD_PHASE(tm, SSD_PH_BWD_FINISH, launch_bwd_finish(p.dtype, dm, b, in, b.tz_ddt, nullptr, b.tz_da, s));
    st = reduce_bc(tm);
  } else {
    if (d.trapz == SSD_TRAPZ_DROP_BETA_DA) {
      // (the column / row path) a backward of the gamma path that computes the decay gradient only (the
      // exact kernels still write dx / dB / dC, which the pass below overwrites), then the scan's own
      const PhaseTimer none{nullptr, s};
      SSD_TRY(tm.begin(SSD_PH_TRAPZ_GAMMA));
      st = scan_bwd(dg, bg, ig, none, true, nullptr, nullptr, b.tz_da);
      if (st != SSD_OK) return st;
      SSD_TRY(tm.end(SSD_PH_TRAPZ_GAMMA));
    }
    // the scan of both paths (dt = gamma + rho, D per token); its dst equals the gamma pass's, which
    // differs only in the decay term it feeds (h_in of the gamma path)
    st = scan_bwd(d, b, in, tm, d.trapz != SSD_TRAPZ_DROP_BETA_DA, d.trapz ? b.tz_ddt : (d.has_dt ? a->ddt : nullptr),
                  d.trapz ? nullptr
                          : ((d.a_mode == SSD_A_PER_TOKEN ||
                              (d.a_mode == SSD_A_CUMSUM && !(d.dA_skip & SSD_DA_SKIP_INTRA)))
                                 ? a->dA
                                 : nullptr),
                  d.trapz == SSD_TRAPZ_EXACT_DA ? b.tz_da : nullptr);
  }
  if (st != SSD_OK) return st;
  if (d.trapz) {
    SSD_TRY(tm.begin(SSD_PH_TRAPZ_POST));
    if (!fused) SSD_TRY(launch_trapz_bc(p.dtype, d, b, a->x, dY, a->B, a->C, a->dB, a->dC, a->cu_seqlens, s));
    SSD_TRY(launch_trapz_grads(p.dtype, d, b, a->A, a->cu_seqlens, a->x, dY, a->B, a->C, a->dgamma, a->dbeta, a->dA,
                               s));
    SSD_TRY(tm.end(SSD_PH_TRAPZ_POST));
  }
  float* dA_head = d.a_mode == SSD_A_PER_HEAD ? reinterpret_cast<float*>(a->dA) : nullptr;
  float* dD = d.has_D ? a->dD : nullptr;
  float* dw = d.has_z ? a->dnorm_weight : nullptr;
  if (dA_head || dD || dw)
    SSD_PHASE(tm, SSD_PH_BWD_REDUCE_HEADS,
              launch_reduce_tail(d, b, dA_head, dD, (int)p.norm_blocks, d.H * d.P, b.dw_part, dw, s));
  return SSD_OK;
}

int ssd_materialize_L(const ssd_desc_t* desc, const void* a, void* L, void* stream) {
  const int st = cache_helper_shape(desc);
  if (st != SSD_OK) return st;
  if (!a || !L) return SSD_ERR_INVALID;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SSD_TRY(launch_materialize_L(desc->dtype, (int)desc->batch, (int)desc->seqlen, (int)desc->nheads,
                               (int)desc->chunk, a, L, s));
  return SSD_OK;
}

int ssd_decay_chunk(const ssd_desc_t* desc, const void* A_cumsum, void* decay_chunk, void* stream) {
  const int st = cache_helper_shape(desc);
  if (st != SSD_OK) return st;
  if (!A_cumsum || !decay_chunk) return SSD_ERR_INVALID;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SSD_TRY(launch_decay_chunk(desc->dtype, (int)desc->batch, (int)desc->nheads, (int)(desc->seqlen / desc->chunk),
                             (int)desc->chunk, A_cumsum, decay_chunk, s));
  return SSD_OK;
}

const char* ssd_status_string(int status) {
  switch (status) {
    case SSD_OK: return "ok";
    case SSD_ERR_INVALID: return "invalid argument";
    case SSD_ERR_UNSUPPORTED: return "unsupported shape or option";
    case SSD_ERR_WORKSPACE: return "workspace missing or too small";
    case SSD_ERR_HIP: return "HIP launch error";
    case SSD_ERR_TOO_LARGE: return "input exceeds the no-allocation scratch (SSD_NOALLOC_SCRATCH_BYTES)";
    default: return "unknown status";
  }
}

int ssd_abi_version(void) { return 4; }

}  // extern "C"
