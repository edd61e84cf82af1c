// Chunk states and the inter-chunk recurrence in one pass (bf16 inputs).
//
// Forward (ssd_scan.py:387-410): per sequence and head, walking the chunks in
// order,
//   hin[c] = run;  run = exp(clamp(total_c)) * run + st_c,
//   st_c[p][n] = sum_s x[s][p] * exp(clamp(cs_last - cs_s)) * dt_s * B[s][n]
// and final = run. Backward (the reverse recurrence for the gradient leaving
// each chunk, the adjoint of the above plus the Y_off term :412-415):
//   dst[c] = run;  dtot_c = sum run * exp(clamp(total_c)) * hin[c] * pass(total_c);
//   run = exp(clamp(total_c)) * run + dh_c,
//   dh_c[p][n] = sum_l dy[l][p] * exp(clamp(cs_l)) * C[l][n]
// and dinit = run. The running state stays in the MFMA accumulator registers;
// nothing but hin / dst (bf16) and the final / initial state is written.
//
// One block per (head, sequence) over all Npad = 32 NT state columns (over half of them, two blocks per
// unit, when there are at most 128 units; packed sequences longest first; the trapezoidal gamma path's
// forward walk in the same launch as the scan's), with PT NT waves:
// the walk is bound by its DMA stream (without the B / C columns it runs in 79 % of
// the time, without the x / dy rows in 73 %), so each x / dy row is loaded once per
// head, not once per group of columns. In the forward walk with head dims 33..64
// (PT = 2) wave w owns all 64 rows p of the 16 columns 16 w .. 16 w + 15 (four 16 x 16
// MFMA tiles), so each B element is scaled by the per-token factor once per block;
// otherwise wave w owns the 32 x 32 tile (p tile w % PT, n tile w / PT). Tokens go 64
// at a time through a ring of three LDS slots filled by
// buffer_load ... lds (x or dy rows, the pair's B or C columns, and the tokens'
// precomputed factors exp(clamp(cs_last - cs_t)) dt_t or exp(clamp(cs_t))),
// issued two steps ahead with explicit vmcnt waits, so no register holds
// staged data and every step's wait counts exactly. Both MFMA operands are
// read with ds_read_b64_tr_b16 from granule-permuted rows (the contraction is
// over tokens, the tiles' row index); the per-token factor is applied to the
// B / C operand in registers after the read.
#include "ssd_launch.h"
#include "ssd_tile.h"

namespace {

template <int PT, int NT>
struct StateCfg {
  static constexpr int PP = 32 * PT;            // state rows per block
  static constexpr int NC = 32 * NT;            // state columns per block (all of Npad)
  static constexpr int NW = PT * NT;            // compute waves: (p tile, n tile)
  static constexpr int NPW = 4;                 // DMA waves (one more per SIMD), after the compute waves
  static constexpr int NTHR = 64 * (NW + NPW);
  static constexpr int R = (PT == 2 && NT == 4) ? 4 : 3;  // ring slots
  static constexpr int UB = 64 * PP * 2;        // x / dy rows of a step
  static constexpr int VB = 64 * NC * 2;        // B / C rows of a step
  static constexpr int SLOT = UB + VB + 256;    // + the step's 64 per-token factors (loaded by wave 0)
  static constexpr int UI = UB / 1024, VI = VB / 1024;  // 1 KB DMA instructions
  static constexpr int PERW = (UI + VI) / NPW;  // row DMAs per DMA wave and step
  static constexpr int D = PERW, D0 = PERW + 1; // DMAs per step: any DMA wave, DMA wave 0 (+ the factor row)
  static_assert(UI % NPW == 0 && VI % NPW == 0, "DMA split");
  static_assert(NTHR <= 1024, "the largest block a launch takes");
  static constexpr int TP = 40;                 // s_tile row pitch (elements), 32 x 32 tiles
  // PT = 2: each wave owns all 64 p of 16 columns of the pair (four 16 x 16 MFMA tiles), so every
  // B / C element is scaled by one wave, not by both p-tile waves; other PT use 32 x 32 tiles
  static constexpr int TW = 24;                 // s_tile row pitch (elements), 64 x 16 tiles
  static constexpr int TWE = PT == 2 ? 64 * TW : 32 * TP;  // s_tile elements per wave
  // The backward walk's h_in tile of a chunk (2 KB per wave) shares the wave's state tile: the tile is
  // written and read at the chunk's first step before the h_in DMAs are issued into it, which are read
  // at the chunk's end, before the next chunk's first step.
  static constexpr int TILE = TWE * 2 > 2048 ? TWE * 2 : 2048;  // bytes per wave
  static size_t bytes(bool) { return (size_t)R * SLOT + (size_t)NW * TILE; }
  // waves per SIMD a block brings (its compute waves and one DMA wave per SIMD), at least two
  static constexpr int WPE = (NW + NPW + 3) / 4 > 2 ? (NW + NPW + 3) / 4 : 2;
  // ... and at most: two blocks per CU of a two-wave block where their LDS fits. (With WPE as the limit the register
  // allocation was padded until one block filled a CU: 128 one-token sequences of 16 heads of 128 columns, 4096 walks
  // over 64 state columns, 74 -> 43 us.)
  static constexpr int WPX = 2 * (R * SLOT + NW * TILE) <= 160 * 1024 && WPE == 2 ? 4 : WPE;
};

// Whether the walk uses the 64 x 16 wave tiles: the forward walk at PT = 2. The backward walk
// keeps 32 x 32 tiles: with 64 x 16 it ran 11 us slower at config 2 on the same box (199 against
// 188 us) despite 25 % fewer VALU instructions, while the forward walk gained 6-10 us.
template <int PT, bool FWD>
constexpr bool state_wide() {
  return PT == 2 && FWD;
}
// Row (p, within the wave's tile) of accumulator register v, and column (n) of lane L.
template <bool WIDE>
__device__ __forceinline__ int state_row(int v, int L) {
  return WIDE ? 16 * (v >> 2) + 4 * (L >> 4) + (v & 3) : acc_row(v, L);
}
template <bool WIDE>
__device__ __forceinline__ int state_col(int L) {
  return WIDE ? (L & 15) : (L & 31);
}

}  // namespace

// Everything a step needs besides LDS (wave-uniform unless noted).
struct StateCtx {
  SsdDims d;
  const ChunkInfo* chunks;
  const float* cs;
  const float* fac;  // per-token factors [max_chunks][H][Qpad] (0 past a chunk's end)
  const bf16* U;
  const bf16* V;
  bf16* hst;
  uint8_t* hlo;  // forward: the residual hin - bf16(hin) (fp8, lo_pack4), in hin_lo_off order (or nullptr)
  const bf16* hin_in;
  float* dtot_part;
  int64_t urow, vrow, ucol, vcol;
  int h, w, pw, pt, ntl, nt, NTn, c0, c1, nch;  // pw: index of a DMA wave
  int ncol0;  // first state column (n) of this wave's tile
  int cofs;   // first state column of the block (a column half when the walk splits the columns)
  bool nt_ok;
};

// Chunk-table index of walk position k (clamped to the sequence's last chunk).
template <bool FWD>
__device__ __forceinline__ int walk_chunk(const StateCtx& x, int k) {
  const int kc = min(k, x.nch - 1);
  return __builtin_amdgcn_readfirstlane(FWD ? x.c0 + kc : x.c1 - 1 - kc);
}
// Total log-decay (cs at the last padded position) of chunk c for the walk's head.
__device__ __forceinline__ float chunk_total(const StateCtx& x, int c) {
  return x.cs[((int64_t)c * x.d.H + x.h) * x.d.Qpad + x.d.Qpad - 1];
}

// A walk position: chunk index k of the sequence, token offset t in it, the chunk's table
// entry and total log-decay, and those of the next chunk, loaded a whole chunk before use so
// that entering a chunk waits on no scalar load.
struct Cursor {
  int k, t, c;
  ChunkInfo ci, nci;
  float tot, ntot;
};

template <bool FWD>
__device__ __forceinline__ void cursor_init(const StateCtx& x, Cursor& u) {
  u.c = walk_chunk<FWD>(x, 0);
  u.ci = x.chunks[u.c];
  u.tot = chunk_total(x, u.c);
  const int cn = walk_chunk<FWD>(x, 1);
  u.nci = x.chunks[cn];
  u.ntot = chunk_total(x, cn);
}
// Enter chunk u.k (the one after the current) and load the entry and total of the chunk after it.
template <bool FWD>
__device__ __forceinline__ void cursor_next(const StateCtx& x, Cursor& u) {
  u.c = walk_chunk<FWD>(x, u.k);
  u.ci = u.nci;
  u.tot = u.ntot;
  const int cn = walk_chunk<FWD>(x, u.k + 1);
  u.nci = x.chunks[cn];
  u.ntot = chunk_total(x, cn);
}

// Advance the compute cursor past one 64-token step.
template <bool FWD>
__device__ __forceinline__ void cursor_step(const StateCtx& x, Cursor& u) {
  u.t += 64;
  if (u.t >= u.ci.len) {
    ++u.k;
    u.t = 0;
    cursor_next<FWD>(x, u);
  }
}

// The issue cursor: the walk position whose rows the next DMAs fetch, with the bases of its
// chunk's rows (set when the cursor enters a chunk; a step's rows are then the soffset t * pitch)
// and the next chunk's table entry (loaded a chunk ahead).
struct IssueCur {
  int k, t;
  ChunkInfo ci, nci;
  const bf16* bu;
  const bf16* bv;
  const float* bs;
};

// Per-wave loop invariants of the ring DMAs. Every DMA wave issues UPW row DMAs of x / dy and VPW of
// B / C per step (the same split in every DMA wave, so no wave branches on its share); DMA wave 0
// also the step's row of per-token factors.
template <int PT, int NT>
struct IssueLanes {
  using Cfg = StateCfg<PT, NT>;
  static constexpr int UPW = Cfg::UI / Cfg::NPW, VPW = Cfg::VI / Cfg::NPW;
  int ou[UPW], ov[VPW];  // lane's byte offset within the step's rows (SSD_BUF_SIZE: column outside)
  int lu[UPW], lv[VPW];  // lane's row within the step
};

template <int PT, int NT, bool FWD>
__device__ __forceinline__ IssueLanes<PT, NT> issue_lanes(const StateCtx& x, int lane) {
  using Cfg = StateCfg<PT, NT>;
  using IL = IssueLanes<PT, NT>;
  constexpr int PP = Cfg::PP, UG = PP / 8, URI = 64 / UG;  // granules per U row, U rows per DMA
  constexpr int NC = Cfg::NC, VG = NC / 8, VRI = 64 / VG;  // ... and per V row
  const SsdDims& d = x.d;
  IL il;
#pragma unroll
  for (int q = 0; q < IL::UPW; ++q) {
    const int qq = x.pw * IL::UPW + q;
    const int r = qq * URI + lane / UG, gcol = swz_tr<PP>(r, lane % UG) << 3;
    il.lu[q] = r;
    il.ou[q] = gcol < d.P ? (int)((r * x.urow + gcol) * 2) : SSD_BUF_SIZE;
  }
#pragma unroll
  for (int q = 0; q < IL::VPW; ++q) {
    const int vi = x.pw * IL::VPW + q;
    const int r = vi * VRI + lane / VG, gcol = swz_tr<NC>(r, lane % VG) << 3;
    il.lv[q] = r;
    il.ov[q] = x.cofs + gcol < d.N ? (int)((r * x.vrow + gcol) * 2) : SSD_BUF_SIZE;
  }
  return il;
}

// Enter the issue cursor's chunk u.k (its table entry is u.nci, or loaded here at the first
// chunk): the bases of its rows, and the next chunk's entry.
template <int PT, int NT, bool FWD>
__device__ __forceinline__ void issue_fetch(const StateCtx& x, const IssueLanes<PT, NT>& il, IssueCur& u, bool first) {
  const SsdDims& d = x.d;
  const int c = walk_chunk<FWD>(x, u.k);
  u.ci = first ? x.chunks[c] : u.nci;
  u.nci = x.chunks[walk_chunk<FWD>(x, u.k + 1)];
  u.bu = x.U + (int64_t)u.ci.row0 * x.urow + x.ucol;
  u.bv = x.V + (int64_t)u.ci.row0 * x.vrow + x.vcol;
  u.bs = x.fac + ((int64_t)c * d.H + x.h) * d.Qpad;
}

// One step's DMAs into ring slot `nxt`: StateCfg::D per DMA wave (D0 in DMA wave 0), also past the
// last step (then masked to zeros), so that every step issues the same count. Advances the
// issue cursor.
template <int PT, int NT, bool FWD>
__device__ __forceinline__ void state_issue(const StateCtx& x, const IssueLanes<PT, NT>& il, unsigned char* __restrict__ nxt,
                                            IssueCur& u, int lane) {
  using Cfg = StateCfg<PT, NT>;
  using IL = IssueLanes<PT, NT>;
  const bool live = u.k < x.nch;
  const int t0i = live ? u.t : 0;
  const int nrows = live ? min(64, u.ci.len - t0i) : 0;
  const int su = t0i * (int)x.urow * 2, sv = t0i * (int)x.vrow * 2;
  const __amdgpu_buffer_rsrc_t ru = buf_rsrc(u.bu), rv = buf_rsrc(u.bv), rs = buf_rsrc(u.bs);
  // (each offset goes through a plain int: an argument whose type depends on the template would
  // make the target builtin's call dependent, which the host pass cannot resolve)
#pragma unroll
  for (int q = 0; q < IL::UPW; ++q) {
    const int vo = il.lu[q] < nrows ? il.ou[q] : SSD_BUF_SIZE;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        ru, (__attribute__((address_space(3))) void*)(nxt + (x.pw * IL::UPW + q) * 1024), 16, vo, su, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < IL::VPW; ++q) {
    const int vo = il.lv[q] < nrows ? il.ov[q] : SSD_BUF_SIZE;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rv, (__attribute__((address_space(3))) void*)(nxt + Cfg::UB + (x.pw * IL::VPW + q) * 1024), 16, vo, sv, 0, 0);
  }
  if (x.pw == 0) {
    const int vo = lane * 4, so = t0i * 4;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void*)(nxt + Cfg::UB + Cfg::VB), 4, vo, so, 0, 0);
  }
  if (live) {
    u.t += 64;
    if (u.t >= u.ci.len) {
      ++u.k;
      u.t = 0;
      issue_fetch<PT, NT, FWD>(x, il, u, false);
    }
  }
}

// vmcnt wait until at most n steps' ring DMAs of DMA wave pw are outstanding (n <= 3)
template <int D0, int D>
__device__ __forceinline__ void wait_ring(int pw, int n) {
  if (pw == 0) {
    switch (n) {
      case 0: wait_vm<0>(); break;
      case 1: wait_vm<D0>(); break;
      case 2: wait_vm<2 * D0>(); break;
      default: wait_vm<3 * D0>(); break;
    }
  } else {
    switch (n) {
      case 0: wait_vm<0>(); break;
      case 1: wait_vm<D>(); break;
      case 2: wait_vm<2 * D>(); break;
      default: wait_vm<3 * D>(); break;
    }
  }
}

// One 64-token step of a compute wave: consume slot `cur` (filled by the DMA waves).
template <int PT, int NT, bool FWD>
__device__ __forceinline__ void state_step(const StateCtx& x, const unsigned char* __restrict__ cur,
                                           bf16* __restrict__ tw, Cursor& uc, floatx16& acc, floatx16& run) {
  using Cfg = StateCfg<PT, NT>;
  constexpr int PP = Cfg::PP, TP = Cfg::TP;
  constexpr bool WIDE = state_wide<PT, FWD>();
  const SsdDims& d = x.d;
  const int lane = threadIdx.x & 63;
  const int c = uc.c;
  const int clen = uc.ci.len;
  const int t0 = uc.t;
  const int64_t soff = ((int64_t)c * d.H + x.h) * d.Ppad * d.Npad;
  const int prow0 = 32 * x.pt;
  // tile geometry: rows (p) x columns (n) per wave, and the 16-byte pieces per row
  constexpr int TR = WIDE ? 64 : 32, TC = WIDE ? 16 : 32, TPR = WIDE ? Cfg::TW : TP;
  constexpr int GPR = TC / 8;
  if (t0 == 0) {
    // state entering (forward) / gradient leaving (backward) chunk c: accumulator layout
    // -> this wave's LDS tile -> 16-byte row pieces (two per lane)
#pragma unroll
    for (int v = 0; v < 16; ++v) tw[state_row<WIDE>(v, lane) * TPR + state_col<WIDE>(lane)] = (bf16)run[v];
    __builtin_amdgcn_wave_barrier();
    if (x.nt_ok) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int id = lane + 64 * q, r = id / GPR, c8 = (id % GPR) * 8;
        const int64_t o = soff + (int64_t)(prow0 + r) * d.Npad + x.ncol0 + c8;
        *reinterpret_cast<bf16x8*>(x.hst + o) = *reinterpret_cast<const bf16x8*>(tw + r * TPR + c8);
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (FWD && x.hlo) {
      // the residual of the bf16 rounding (fp8, lo_pack4): a lane's registers 4 m .. 4 m + 3 are four
      // consecutive rows p of its column n, i.e. half of an 8-byte piece (n, p .. p + 7) of hin_lo's
      // fragment order (hin_lo_off), so one 4-byte store each, straight from registers
      if (x.nt_ok) {
        const int64_t tb = ((int64_t)c * d.H + x.h) * d.Npad * d.Ppad;
        const int nn = x.ncol0 + state_col<WIDE>(lane);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int p0 = prow0 + state_row<WIDE>(4 * m, lane);
          *reinterpret_cast<unsigned*>(x.hlo + tb + hin_lo_off(d.Ppad, nn, p0 & ~7) + (p0 & 7)) =
              lo_pack4(run[4 * m], run[4 * m + 1], run[4 * m + 2], run[4 * m + 3]);
        }
      }
    }
    if (!FWD) {
      // this wave's tile of h_in[c] ([TR][TC], 2 KB), consumed at the end of the chunk
      const __amdgpu_buffer_rsrc_t rh = buf_rsrc(x.hin_in + soff);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int r = (TR / 2) * q + lane / GPR, c8 = (lane % GPR) * 8;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rh, (__attribute__((address_space(3))) void*)(tw + q * 512), 16,
            x.nt_ok ? (int)(((prow0 + r) * d.Npad + x.ncol0 + c8) * 2) : SSD_BUF_SIZE, 0, 0, 0);
      }
    }
  }
  const bf16* tu = reinterpret_cast<const bf16*>(cur);
  const bf16* tv = reinterpret_cast<const bf16*>(cur + Cfg::UB);
  // the step's per-token factors of the B / C rows (precomputed, 0 past the chunk's end): read
  // straight from the slot, eight consecutive tokens per lane
  const float* fac = reinterpret_cast<const float*>(cur + Cfg::UB + Cfg::VB);
  if constexpr (WIDE) {
    // 64 p x 16 n: the scaled B / C operand is shared by the four p blocks
#pragma unroll
    for (int kk = 0; kk < 64; kk += 32) {
      const floatx4 f0 = *reinterpret_cast<const floatx4*>(fac + kk + 8 * (lane >> 4));
      const floatx4 f1 = *reinterpret_cast<const floatx4*>(fac + kk + 8 * (lane >> 4) + 4);
      bf16x8 b = swz_tr8_16<Cfg::NC>(tv, kk, 16 * x.w, lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        b[e] = (bf16)((float)b[e] * f0[e]);
        b[4 + e] = (bf16)((float)b[4 + e] * f1[e]);
      }
      mfma16<0>(acc, swz_tr8_16<PP>(tu, kk, 0, lane), b);
      mfma16<1>(acc, swz_tr8_16<PP>(tu, kk, 16, lane), b);
      mfma16<2>(acc, swz_tr8_16<PP>(tu, kk, 32, lane), b);
      mfma16<3>(acc, swz_tr8_16<PP>(tu, kk, 48, lane), b);
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < 64; kk += 16) {
      const floatx4 f0 = *reinterpret_cast<const floatx4*>(fac + kk + 8 * (lane >> 5));
      const floatx4 f1 = *reinterpret_cast<const floatx4*>(fac + kk + 8 * (lane >> 5) + 4);
      bf16x8 b = swz_tr8<Cfg::NC>(tv, kk, 32 * x.ntl, lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        b[e] = (bf16)((float)b[e] * f0[e]);
        b[4 + e] = (bf16)((float)b[4 + e] * f1[e]);
      }
      mfma(acc, swz_tr8<PP>(tu, kk, prow0, lane), b);
    }
  }
  if (t0 + 64 >= clen) {
    // end of chunk c
    const float tot = uc.tot;
    const float dec = exp_clamp(tot);
    if (!FWD) {
      // the h_in tile's DMAs (issued at the chunk's first step) are the wave's only loads
      wait_vm<0>();
      float contrib = 0.0f;
#pragma unroll
      for (int v = 0; v < 16; ++v) contrib += run[v] * (float)tw[state_row<WIDE>(v, lane) * TC + state_col<WIDE>(lane)];
      contrib *= dec * clamp_pass(tot);
      contrib = wave_sum(contrib);
      // one partial per wave, (32-wide n tile, p tile or 16-wide half) in order: no block
      // synchronisation at the chunk's end, and the reader sums them in a fixed order
      const int part = x.nt * PT + (WIDE ? (x.w & 1) : x.pt);
      if (x.nt_ok && lane == 0) x.dtot_part[((int64_t)c * d.H + x.h) * x.NTn * PT + part] = contrib;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) run[v] = dec * run[v] + acc[v];
    zero(acc);
  }
  cursor_step<FWD>(x, uc);
}

// StateCfg::WPE to WPX waves per SIMD: the block's compute and DMA waves, once or twice
template <int PT, int NT, bool FWD>
__global__ void __launch_bounds__((StateCfg<PT, NT>::NTHR)) __attribute__((amdgpu_waves_per_eu(StateCfg<PT, NT>::WPE, StateCfg<PT, NT>::WPX)))
k_state_fused(SsdDims d, const ChunkInfo* __restrict__ chunks,
                                                         const int32_t* __restrict__ seq_chunk0,
                                                         const int32_t* __restrict__ seq_order,
                                                         const float* __restrict__ cs, const float* __restrict__ fac,
                                                         const bf16* __restrict__ U, const bf16* __restrict__ V,
                                                         bf16* __restrict__ hst, uint8_t* __restrict__ hlo,
                                                         const bf16* __restrict__ hin_in,
                                                         const void* __restrict__ s_in, void* __restrict__ s_out,
                                                         int state_bf16, float* __restrict__ dtot_part, int nsplit,
                                                         const float* __restrict__ fac2, bf16* __restrict__ hst2,
                                                         uint8_t* __restrict__ hlo2) {
  using Cfg = StateCfg<PT, NT>;
  constexpr int TP = Cfg::TP, SLOT = Cfg::SLOT;
  constexpr bool WIDE = state_wide<PT, FWD>();
  extern __shared__ __align__(16) unsigned char smem[];
  // [NW][TILE bytes]: each wave's state tile, and in the backward walk its h_in tile
  unsigned char* s_tile = smem + Cfg::R * SLOT;

  // block -> unit = (head, sequence)
  StateCtx x;
  x.d = d;
  x.NTn = d.Npad / 32;
  // two walks in one launch (fac2 given: the trapezoidal gamma path's states beside the scan's): the
  // blocks past the first walk's run the second with its own factors and outputs
  const int units = d.H * d.nseq;
  const int per_walk = nsplit == 1 ? units : (units + 7) / 8 * 16;
  int b = blockIdx.x;
  if (fac2 && b >= per_walk) {
    b -= per_walk;
    fac = fac2;
    hst = hst2;
    hlo = hlo2;
  }
  // with the columns split in two (few units: each half is a block of 32 NT columns), the halves of a unit
  // are 8 blocks apart, on one XCD, where they share the unit's x / dy rows in L2
  const int unit = nsplit == 1 ? b : (b >> 4) * 8 + (b & 7);
  x.cofs = nsplit == 1 ? 0 : ((b >> 3) & 1) * 32 * NT;
  if (unit >= units) return;
  x.h = unit % d.H;
  // packed sequences: the longest first (seq_order), so that the last walks to start are short ones
  const int sq = seq_order ? seq_order[unit / d.H] : unit / d.H;
  const int g = x.h / d.hpg;
  x.w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool dma_wave = x.w >= Cfg::NW;
  x.pw = dma_wave ? x.w - Cfg::NW : -1;
  if constexpr (WIDE) {  // wave w: all p, columns 16 w .. 16 w + 15
    x.pt = 0;
    x.ntl = x.w >> 1;
    x.ncol0 = x.cofs + 16 * x.w;
  } else {                    // wave w: p tile w % PT, 32-wide column tile w / PT
    x.pt = x.w % PT;
    x.ntl = x.w / PT;
    x.ncol0 = x.cofs + 32 * x.ntl;
  }
  x.nt = x.ncol0 / 32;
  x.nt_ok = x.nt < x.NTn;
  x.chunks = chunks;
  x.cs = cs;
  x.fac = fac;
  x.U = U;
  x.V = V;
  x.hst = hst;
  x.hlo = FWD ? hlo : nullptr;
  x.hin_in = hin_in;
  x.dtot_part = dtot_part;
  x.urow = (int64_t)d.H * d.P;
  x.vrow = (int64_t)d.G * d.N;
  x.ucol = (int64_t)x.h * d.P;
  x.vcol = (int64_t)g * d.N + x.cofs;
  const int lane = threadIdx.x & 63;
  x.c0 = seq_chunk0[sq];
  x.c1 = seq_chunk0[sq + 1];
  x.nch = x.c1 - x.c0;
  // Step st of both roles: the DMA waves wait for their DMAs of slot st % R, all waves meet at the
  // step's barrier (step st - 1 is then done everywhere and its slot free), the DMA waves refill that
  // slot with step st + R - 1 while the compute waves consume slot st % R. The loops are unrolled R
  // times so that every slot address is a constant (the LDS accesses carry it in their offset field);
  // both roles follow the same cursor, so they meet at the same number of barriers.
  static_assert(Cfg::R == 3 || Cfg::R == 4, "three- or four-slot ring");
  auto ring = [&](auto&& step) {
    Cursor uc{};
    if (x.nch > 0) cursor_init<FWD>(x, uc);
    if constexpr (Cfg::R == 4) {
      while (uc.k < x.nch) {
        step(uc, smem, smem + 3 * SLOT);
        if (uc.k >= x.nch) break;
        step(uc, smem + SLOT, smem);
        if (uc.k >= x.nch) break;
        step(uc, smem + 2 * SLOT, smem + SLOT);
        if (uc.k >= x.nch) break;
        step(uc, smem + 3 * SLOT, smem + 2 * SLOT);
      }
    } else {
      while (uc.k < x.nch) {
        step(uc, smem, smem + 2 * SLOT);
        if (uc.k >= x.nch) break;
        step(uc, smem + SLOT, smem);
        if (uc.k >= x.nch) break;
        step(uc, smem + 2 * SLOT, smem + SLOT);
      }
    }
  };

  if (dma_wave) {
    const IssueLanes<PT, NT> il = issue_lanes<PT, NT, FWD>(x, lane);
    IssueCur ui{};  // issue cursor, R - 1 steps ahead of the compute cursor
    if (x.nch > 0) {  // (an empty sequence passes its state through)
      issue_fetch<PT, NT, FWD>(x, il, ui, true);
      for (int q = 0; q < Cfg::R - 1; ++q) state_issue<PT, NT, FWD>(x, il, smem + q * SLOT, ui, lane);
    }
    ring([&](Cursor& uc, unsigned char* __restrict__, unsigned char* __restrict__ nxt) {
      // this wave's DMAs of slot st are done (those of the next R - 2 slots may still fly)
      wait_ring<Cfg::D0, Cfg::D>(x.pw, Cfg::R - 2);
      lds_barrier();
      state_issue<PT, NT, FWD>(x, il, nxt, ui, lane);
      cursor_step<FWD>(x, uc);
    });
    wait_vm<0>();  // the trailing (masked) DMAs land before the block's LDS is released
    return;
  }

  const int n = x.ncol0 + state_col<WIDE>(lane);
  const int prow0 = 32 * x.pt;
  // running state: rows p = 32 pt + acc_row(v), column n
  floatx16 run;
  zero(run);
  if (s_in) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int p = prow0 + state_row<WIDE>(v, lane);
      if (p < d.P && n < d.N) {
        const int64_t o = (((int64_t)sq * d.H + x.h) * d.P + p) * d.N + n;
        run[v] = state_bf16 ? (float)reinterpret_cast<const bf16*>(s_in)[o] : reinterpret_cast<const float*>(s_in)[o];
      }
    }
  }
  floatx16 acc;
  zero(acc);
  bf16* tw = reinterpret_cast<bf16*>(s_tile + x.w * Cfg::TILE);
  ring([&](Cursor& uc, unsigned char* __restrict__ cur, unsigned char* __restrict__) {
    lds_barrier();  // the DMA waves' loads of slot st have landed; step st - 1 is done everywhere
    state_step<PT, NT, FWD>(x, cur, tw, uc, acc, run);
  });
  // final state (forward) / gradient of the initial state (backward)
  if (s_out) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int p = prow0 + state_row<WIDE>(v, lane);
      if (p < d.P && n < d.N) {
        const int64_t o = (((int64_t)sq * d.H + x.h) * d.P + p) * d.N + n;
        if (state_bf16) reinterpret_cast<bf16*>(s_out)[o] = (bf16)run[v];
        else reinterpret_cast<float*>(s_out)[o] = run[v];
      }
    }
  }
}

bool state_fused_supported(int dtype, const SsdDims& d) {
  return dtype == 1 && d.P % 8 == 0 && d.N % 8 == 0 && d.vec_x && d.vec_bc;
}

// dtot partials per (chunk, head) of the backward walk: one per wave, i.e. per 32 x 32 tile
int state_fused_slices(const SsdDims& d) { return d.Npad / 32 * (d.Ppad / 32); }

// The second walk (W2.fac given) runs in the same launch, after the first's blocks.
struct Walk2 {
  const float* fac;
  bf16* hst;
  uint8_t* hlo;
};

template <int PT, int NT, bool FWD>
static void state_fused_launch(const SsdDims& d, const SsdBufs& b, const bf16* u, const bf16* v, const float* fac,
                               bf16* hst, uint8_t* hlo, const bf16* hin_in, const void* s_in, void* s_out,
                               int state_bf16, hipStream_t s, int nsplit, const Walk2& w2) {
  using Cfg = StateCfg<PT, NT>;
  const int units = d.H * d.nseq;
  const int per_walk = nsplit == 1 ? units : (units + 7) / 8 * 16;
  const dim3 grid(per_walk * (w2.fac ? 2 : 1));
  // One block per CU (by asking for more than half its LDS) for packed sequences of up to three walks a CU: the longest
  // walks, which start first, are what the launch waits for, and a second block slows them (65 536 tokens of 32 heads,
  // forward and backward, one / two: 15 sequences 1414 / 1435 us, 24 1431 / 1443; 32 768 tokens of 64 heads in 15, 960
  // walks: 1239 / 1224).
  const size_t lone = 81 * 1024, need = Cfg::bytes(!FWD);
  const size_t lds = d.varlen && grid.x > 256 && grid.x <= 768 && need < lone ? lone : need;
  ensure_lds(k_state_fused<PT, NT, FWD>, lds);
  hipLaunchKernelGGL((k_state_fused<PT, NT, FWD>), grid, dim3(Cfg::NTHR), lds, s, d, b.chunks, b.seq_chunk0,
                     b.seq_order, b.cs, fac, u, v, hst, hlo, hin_in, s_in, s_out, state_bf16, b.dtot_part, nsplit,
                     w2.fac, w2.hst, w2.hlo);
}
template <int PT, bool FWD>
static void state_fused_nt(const SsdDims& d, const SsdBufs& b, const bf16* u, const bf16* v, const float* fac,
                           bf16* hst, uint8_t* hlo, const bf16* hin_in, const void* s_in, void* s_out, int state_bf16,
                           hipStream_t s, const Walk2& w2) {
  // at most half the CUs' worth of (head, sequence) walks: two blocks per unit, each over half the state
  // columns (each reads the unit's x / dy rows; every walk is serial, so idle CUs are the larger loss). States of
  // 128 x 128 always: one block's compute and DMA waves would be 20.
  const bool few = (w2.fac ? 2 : 1) * d.H * d.nseq <= 128 && d.Npad / 32 >= 2;
  const int nsplit = few || (PT == 4 && d.Npad == 128) ? 2 : 1;
  switch (d.Npad / 32 / nsplit) {
    case 1: state_fused_launch<PT, 1, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, nsplit, w2); break;
    case 2: state_fused_launch<PT, 2, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, nsplit, w2); break;
    default:
      if constexpr (PT < 4)
        state_fused_launch<PT, 4, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, nsplit, w2);
  }
}

template <bool FWD>
static hipError_t state_fused_t(const SsdDims& d, const SsdBufs& b, const void* U, const void* V, const float* fac,
                                bf16* hst, uint8_t* hlo, const bf16* hin_in, const void* s_in, void* s_out,
                                int state_bf16, hipStream_t s, const Walk2& w2 = Walk2{}) {
  const bf16* u = reinterpret_cast<const bf16*>(U);
  const bf16* v = reinterpret_cast<const bf16*>(V);
  switch (d.Ppad / 32) {
    case 1: state_fused_nt<1, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, w2); break;
    case 2: state_fused_nt<2, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, w2); break;
    default: state_fused_nt<4, FWD>(d, b, u, v, fac, hst, hlo, hin_in, s_in, s_out, state_bf16, s, w2);
  }
  return hipGetLastError();
}
hipError_t launch_state_fwd_fused(const SsdDims& d, const SsdBufs& b, const void* x, const void* B, const float* fac,
                                  const void* init, void* final_state, int state_dtype, hipStream_t s) {
  return state_fused_t<true>(d, b, x, B, fac, reinterpret_cast<bf16*>(b.hin), b.hin_lo, nullptr, init, final_state,
                             state_dtype == 1, s);
}

hipError_t launch_state_fwd_fused2(const SsdDims& d, const SsdBufs& b, const void* x, const void* B, const float* fac,
                                   const float* fac2, void* hst2, uint8_t* hlo2, int state_dtype, hipStream_t s) {
  return state_fused_t<true>(d, b, x, B, fac, reinterpret_cast<bf16*>(b.hin), b.hin_lo, nullptr, nullptr, nullptr,
                             state_dtype == 1, s, Walk2{fac2, reinterpret_cast<bf16*>(hst2), hlo2});
}

hipError_t launch_state_bwd_fused(const SsdDims& d, const SsdBufs& b, const void* dy, const void* C,
                                  const void* dfinal, void* dinit, int state_dtype, hipStream_t s) {
  return state_fused_t<false>(d, b, dy, C, b.bwd_fac, b.dst16, nullptr, reinterpret_cast<const bf16*>(b.hin), dfinal,
                              dinit, state_dtype == 1, s);
}
