// dB and dC of the chunked SSD scan backward (bf16 fused path, gfx950) for groups of few heads
// (B / C per head, G = H, and small H / G) at 256-token chunks, and the Y_off part of the decay
// gradient. The terms are those of k_bwd_gemm, per chunk and group g, with the head-summed dS tiles:
//   dC_t = sum_{s <= t} dS[t,s] B_s + sum_h exp(clamp(cs_t)) (dy_t h_in^T)
//   dB_s = sum_{l >= s} dS[l,s] C_l + sum_h w_s dt_s (x_s dst^T)
//   dcs_off_t = pass(cs_t) exp(clamp(cs_t)) C_t . (dy_t h_in^T)        (per head)
// (r2/dhammic-ai/src/kernels/ssd_scan.py:389-392 and :412-415 are the forward terms whose adjoints
// these are; w_s = exp(clamp(cs_last - cs_s)).)
//
// k_bwd_gemm gives each 64-token block of a chunk its own block and streams the group's heads
// through it, so with one head per group each block is one head's state term and then a chain of
// up to four dependent tile steps. Here a block owns a whole chunk of one group and one role, with
// the chunk's B rows (dC role) or C rows (dB role) resident in LDS for every tile product:
//   - wave w owns the 32 tokens 32 w .. 32 w + 31 and all n tiles (results kept transposed,
//     [n rows][token lanes], as the MFMA writes them);
//   - the heads' h_in (dC) or dst (dB) tiles pass through two LDS slots by buffer_load ... lds, the
//     token rows (dy, x) are loaded straight into MFMA operand registers (a token's head row is
//     contiguous along the contraction index p);
//   - dC role: the dS rows of a token are its B operand as stored ([t][s], s contiguous), all of the
//     wave's tiles loaded into registers at once after the head loop; dB role: the chunk's ten tiles
//     (i, j <= i) are loaded with the first head (one 8-element piece per thread of each), stored to LDS
//     over the head slots after the head loop and read transposed (rows l). Each block then waits on
//     memory about once for its tile terms instead of once per tile.
// The two role blocks of a (chunk, group) are 8 apart in dispatch order, so they run together on one
// XCD and the dS tiles and C rows that both read come from HBM once; consecutive blocks step through
// the groups (see k_bwd_rows).
// With bf16 states the decay term takes h_in = hi + lo, lo the fp8 rounding residual the forward walk
// stores in MFMA fragment order (see k_bwd_gemm).
#include "ssd_launch.h"
#include "ssd_tile.h"

namespace {

constexpr int kRowsQ = 256;  // chunk positions (Qpad) this kernel is built for: 8 token tiles of 32

template <int PT, int NT>
struct RowsCfg {
  static constexpr int PP = 32 * PT, NP = 32 * NT;
  static constexpr int HIN = PP * NP;       // elements of one head's h_in or dst tile
  static constexpr int CH = kRowsQ * NP;    // elements of the chunk's B or C rows
  // after the chunk rows: the two head slots, and over them after the head loop the dB role's ten dS tiles
  // (i, j <= i) of 64 x 64; then the trapezoidal diagonal values
  static constexpr size_t o_slot = (size_t)CH * 2;
  static constexpr size_t kTiles = 10 * 4096 * 2;
  // four head slots: h_in / dst of two heads, and (dC role, decay states apart from h_in) those states
  static constexpr size_t o_dcb = o_slot + (4 * (size_t)HIN * 2 > kTiles ? 4 * (size_t)HIN * 2 : kTiles);
  static constexpr size_t bytes = o_dcb + kRowsQ * 4;
  // buffer_load ... lds instructions (1 KB each) per wave: a head tile, the chunk rows
  static constexpr int kHeadDma = HIN * 2 / 1024 / 8;
  static constexpr int kChunkDma = CH * 2 / 1024 / 8;
  static_assert(kHeadDma >= 1 && HIN * 2 % 8192 == 0, "head tile split over 8 waves");
  static_assert(CH * 2 % 8192 == 0, "chunk rows split over 8 waves");
};

}  // namespace

#define SSD_ROWS_PARAMS                                                                                       \
  SsdDims d, const ChunkInfo* __restrict__ chunks, const float* __restrict__ cs, const float* __restrict__ dt,    \
      const bf16* __restrict__ x, const bf16* __restrict__ dy, const bf16* __restrict__ hin,                     \
      const uint8_t* __restrict__ hin_lo, const bf16* __restrict__ hdec, const uint8_t* __restrict__ hdec_lo,   \
      const bf16* __restrict__ dst, const bf16* __restrict__ Bm,                                                 \
      const bf16* __restrict__ Cm, const bf16* __restrict__ dS16, const float* __restrict__ dS_fix,              \
      const int32_t* __restrict__ fast, float* __restrict__ dcs_off, bf16* __restrict__ dB, bf16* __restrict__ dC, \
      const float* __restrict__ tz_gam, float* __restrict__ xdy
#define SSD_ROWS_ARGS \
  d, chunks, cs, dt, x, dy, hin, hin_lo, hdec, hdec_lo, dst, Bm, Cm, dS16, dS_fix, fast, dcs_off, dB, dC, tz_gam, xdy

// One role's block (the role is a template parameter so that each role's code is register-allocated on
// its own: the roles keep different operands live across the head loop). DEC (dC role): the decay term
// takes other states than dC's state term, hdec (and its residual hdec_lo) in place of h_in: the
// trapezoidal scan's drop setting, whose decay gradient is the gamma path's (states hgam) while dC is the
// scan's; their tiles come through two more slots.
template <int PT, int NT, bool brole, bool DEC>
__device__ __forceinline__ void bwd_rows_role(int c, int g, SSD_ROWS_PARAMS) {
  using Cfg = RowsCfg<PT, NT>;
  constexpr int PP = Cfg::PP, NP = Cfg::NP, NK = PP / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  const ChunkInfo ci = chunks[c];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  const int hh = lane >> 5, l32 = lane & 31;
  const int t = 32 * w + l32;  // this lane's token (MFMA output column) within the chunk
  const bool tok = t < ci.len;
  const int ib = w >> 1;       // its 64-token block
  const int nb = kRowsQ / 64;
  const int nbl = (ci.len + 63) >> 6;
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const int Qpad = kRowsQ;
  const int h0 = g * d.hpg, nhd = d.hpg;
  const bool tiles = !d.da_only;
  const uint8_t* lo_src = DEC ? hdec_lo : hin_lo;  // the decay term's residual
  const bool use_lo = !brole && lo_src != nullptr;

  bf16* chunk_rows = reinterpret_cast<bf16*>(smem);                 // [256][NP] B (dC role) or C rows
  unsigned char* slot0 = smem + Cfg::o_slot;                        // head tiles [PP][NP], two slots
  unsigned char* slot1 = slot0 + Cfg::HIN * 2;
  float* s_dcb = reinterpret_cast<float*>(smem + Cfg::o_dcb);       // [256] trapezoidal diagonal of dS

  // ---- DMA: one head's h_in / dst tile, and the chunk's B / C rows (granules permuted per row for
  // the transposed operand reads; rows past the chunk's end and columns past N read as zeros) ----
  constexpr int TG = NP / 8, TRI = 64 / TG;
  const bf16* tsrc = (brole ? dst : hin) + (int64_t)c * d.H * Cfg::HIN;
  const bf16* dsrc = DEC ? hdec + (int64_t)c * d.H * Cfg::HIN : tsrc;
  auto issue_head = [&](int h, unsigned char* slot) {
    const __amdgpu_buffer_rsrc_t rt = buf_rsrc(tsrc);
    const int so = h * Cfg::HIN * 2;
#pragma unroll
    for (int q = 0; q < Cfg::kHeadDma; ++q) {
      const int qi = w * Cfg::kHeadDma + q, r = qi * TRI + lane / TG;
      const int vo = (r * NP + (swz_tr<NP>(r, lane % TG) << 3)) * 2;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (__attribute__((address_space(3))) void*)(slot + qi * 1024), 16,
                                               vo, so, 0, 0);
      if constexpr (DEC) {  // the decay states' tile, two slots on
        const __amdgpu_buffer_rsrc_t rd = buf_rsrc(dsrc);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rd, (__attribute__((address_space(3))) void*)(slot + 2 * Cfg::HIN * 2 + qi * 1024), 16, vo, so, 0, 0);
      }
    }
  };
  auto issue_chunk = [&]() {
    const __amdgpu_buffer_rsrc_t rc = buf_rsrc((brole ? Cm : Bm) + (int64_t)ci.row0 * brow + (int64_t)g * d.N);
    unsigned char* base = reinterpret_cast<unsigned char*>(chunk_rows);
#pragma unroll
    for (int q = 0; q < Cfg::kChunkDma; ++q) {
      const int qi = w * Cfg::kChunkDma + q, r = qi * TRI + lane / TG;
      const int col = swz_tr<NP>(r, lane % TG) << 3;
      const int vo = (r < ci.len && col < d.N) ? (int)((r * brow + col) * 2) : SSD_BUF_SIZE;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rc, (__attribute__((address_space(3))) void*)(base + qi * 1024), 16,
                                               vo, 0, 0, 0);
    }
  };

  // ---- per-head register operands: the token's head row (dy for dC, x for dB; B[k = p][j = t]), the
  // other row in trapezoidal mode (x . dy), the residual fragments (dC), the per-token scalars ----
  const __amdgpu_buffer_rsrc_t rrow = buf_rsrc((brole ? x : dy) + (int64_t)ci.row0 * xrow);
  const __amdgpu_buffer_rsrc_t rrow2 = buf_rsrc((brole ? dy : x) + (int64_t)ci.row0 * xrow);
  const __amdgpu_buffer_rsrc_t rcs = buf_rsrc(cs + (int64_t)c * d.H * Qpad);
  const __amdgpu_buffer_rsrc_t rdt = buf_rsrc(d.has_dt ? dt + (int64_t)ci.row0 * d.H : cs);
  const __amdgpu_buffer_rsrc_t rgm = buf_rsrc(d.trapz ? tz_gam + (int64_t)ci.row0 * d.H : cs);
  bf16x8 rf[NK], rx[NK];
  uint2 lf[NT][NK];
  float s_cs = 0.0f, s_csl = 0.0f, s_dt = 1.0f, s_gm = 0.0f;
  auto load_head = [&](int h) {
    const int ln = opaque_lane(), lt = 32 * w + (ln & 31), lh = ln >> 5;
    const bool ok = lt < ci.len;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const int p0 = 16 * kk + 8 * lh;
      const int vo = (int)((lt * xrow + p0) * 2);
      rf[kk] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                                              rrow, ok && p0 < d.P ? vo : SSD_BUF_SIZE, h * d.P * 2, 0));
      if (d.trapz)
        rx[kk] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                                                rrow2, ok && p0 < d.P ? vo : SSD_BUF_SIZE, h * d.P * 2, 0));
    }
    if (use_lo) {
      const __amdgpu_buffer_rsrc_t rl = buf_rsrc(lo_src + ((int64_t)c * d.H + h) * Cfg::HIN);
#pragma unroll
      for (int q = 0; q < NT; ++q)
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
          lf[q][kk] = __builtin_bit_cast(
              uint2, __builtin_amdgcn_raw_buffer_load_b64(rl, (int)hin_lo_off(PP, 32 * q, 16 * kk) + ln * 8, 0, 0));
    }
    s_cs = buf_ldf(rcs, (h * Qpad + lt) * 4, true);
    if (brole) {
      s_csl = buf_ldf(rcs, (h * Qpad + Qpad - 1) * 4, true);
      if (d.has_dt) s_dt = buf_ldf(rdt, (int)((lt * (int64_t)d.H + h) * 4), ok);
    }
    if (d.trapz) s_gm = buf_ldf(rgm, (int)((lt * (int64_t)d.H + h) * 4), ok);
  };

  // C[t][n] at this lane's accumulator rows n (the Y_off part of the decay gradient), dC role
  const __amdgpu_buffer_rsrc_t rC = buf_rsrc(Cm + (int64_t)ci.row0 * brow + (int64_t)g * d.N);
  bf16x4 Cv[NT][4];
#pragma unroll
  for (int q = 0; q < NT; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n0 = 32 * q + 8 * r + 4 * hh;
      const bool ok = !brole && tok && n0 < d.N;
      Cv[q][r] = __builtin_bit_cast(
          bf16x4, __builtin_amdgcn_raw_buffer_load_b64(rC, ok ? (int)(t * brow + n0) * 2 : SSD_BUF_SIZE, 0, 0));
    }

  floatx16 acc[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) zero(acc[q]);
  float dcb = 0.0f;  // trapezoidal mode: sum_h gamma (x_t . dy_t), the diagonal of dS

  // the dS operands of every tile term, all in flight at once: dC role, the token's rows of tiles
  // (ib, j <= ib) as B operands (sf[j]), issued after the head loop (whose registers they take); dB role,
  // one 8-element piece per thread of each tile (i, j <= i) of the chunk (pc[i (i + 1) / 2 + j]), issued
  // with the first head's loads and stored to LDS after the head loop
  const int64_t tile0 = ((int64_t)c * d.G + g) * nb * nb * 4096;
  const __amdgpu_buffer_rsrc_t rS = buf_rsrc(dS16 + tile0);
  const int pid = threadIdx.x, pr = pid >> 3, pk = (pid & 7) * 8;  // dB role: this thread's piece of a tile
  bf16x8 sf[4][4];
  bf16x8 pc[10];
  issue_head(h0, slot0);
  load_head(h0);
  if (tiles) {
    issue_chunk();
    if (brole) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j)
          pc[i * (i + 1) / 2 + j] = buf_ld16(rS, (int)((((int64_t)i * nb + j) * 4096 + pr * 64 + pk) * 2), i < nbl);
    }
  }

  auto head_step = [&](int k, const unsigned char* __restrict__ cur, unsigned char* __restrict__ nxt) {
    const int h = h0 + k;
    wait_vm<0>();
    lds_barrier();  // head k's tile in LDS (every wave's DMAs); the other slot's reads (head k - 1) done
    ring_step(cur, nxt, k + 1 < nhd, [&](unsigned char* nx) { issue_head(h + 1, nx); },
              [&](const unsigned char* base) {
      lane = opaque_lane();
      if (!brole) {
        // C_t stays bf16 across heads (its fp32 conversion hoisted out of the head loop would double it)
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(Cv[q][r]));
      }
      const bf16* tile = reinterpret_cast<const bf16*>(base);
      const float et = exp_clamp(s_cs);
      // dC role: T = h_in^T dy_t^T per n tile (+ the residual), dC += exp(clamp(cs_t)) T, decay term
      // C_t . T; dB role: U = dst^T x_t^T, dB += w_t dt_t U
      const float sc = brole ? exp_clamp(s_csl - s_cs) * s_dt : et;
      float osum = 0.0f;
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        floatx16 T;
        zero(T);
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) mfma(T, swz_tr8<NP>(tile, 16 * kk, 32 * q, lane), rf[kk]);
        if (!DEC && use_lo) {
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) mfma(T, lo_frag(lf[q][kk]), rf[kk]);
        }
        if (tiles) {
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[q][v] = fmaf(sc, T[v], acc[q][v]);
        }
        if constexpr (DEC) {
          // the decay term's product over the decay states (+ their residual)
          zero(T);
          const bf16* tdec = tile + 2 * Cfg::HIN;
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) mfma(T, swz_tr8<NP>(tdec, 16 * kk, 32 * q, lane), rf[kk]);
          if (use_lo) {
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) mfma(T, lo_frag(lf[q][kk]), rf[kk]);
          }
        }
        if (!brole) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) osum += (float)Cv[q][r][e] * T[4 * r + e];
        }
      }
      if (!brole) {
        osum = add_xor32(osum);
        if (hh == 0 && tok)
          dcs_off[((int64_t)c * d.H + h) * Qpad + t] = osum * et * clamp_pass(s_cs);
      }
      if (d.trapz) {
        // x_t . dy_t (dy and x rows, in either order), for dgamma (dC role) and the diagonal of dS
        float xd = 0.0f;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
#pragma unroll
          for (int e = 0; e < 8; ++e) xd = fmaf((float)rx[kk][e], (float)rf[kk][e], xd);
        xd = add_xor32(xd);
        if (!brole && hh == 0 && tok) xdy[((int64_t)c * d.H + h) * Qpad + t] = xd;
        dcb = fmaf(s_gm, xd, dcb);
      }
    });
    if (k + 1 < nhd) load_head(h + 1);
  };
  for (int k = 0; k < nhd; k += 2) {
    head_step(k, slot0, slot1);
    if (k + 1 < nhd) head_step(k + 1, slot1, slot0);
  }
  if (!tiles) return;  // decay gradient only: the Y_off term above is all it needs

  // ---- tile terms ----
  // heads of the group the factorised kernel left to the exact fixup: their dS is in dS_fix
  bool slow = false;
  if (fast)
    for (int hq = h0 + (int)threadIdx.x; hq < h0 + nhd; hq += 512) slow = slow || fast[(int64_t)c * d.H + hq] == 0;
  const int tb = (32 * w + (opaque_lane() & 31)) & 63;  // dC role: the lane's token within block ib
  if (!brole) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        sf[j][kk] = buf_ld16(rS, (int)((((int64_t)ib * nb + j) * 4096 + tb * 64 + 16 * kk + 8 * hh) * 2), j <= ib);
  }
  if (d.trapz && hh == 0) s_dcb[t] = dcb;
  wait_vm<0>();
  // every wave's chunk rows and s_dcb in LDS, every wave done with the head slots
  const bool any_fix = __syncthreads_or(slow);
  // one 8-element dS piece as stored, plus the fixup heads' dS and (trapezoidal mode, diagonal tile) the
  // diagonal sum_h gamma (x_t . dy_t) at element e0 (the per-token D part), rounded to bf16 once
  auto adjust = [&](bf16x8& o, const float* fx, bool diag, int e0, float dv) {
    if (!any_fix && !diag) return;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)o[e];
    if (any_fix) {
      const floatx4 f0 = *reinterpret_cast<const floatx4*>(fx), f1 = *reinterpret_cast<const floatx4*>(fx + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += f0[e];
        v[4 + e] += f1[e];
      }
    }
    if (diag) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e == e0) v[e] += dv;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)v[e];
  };

  if (!brole) {
    // dC role: tiles (ib, j), j <= ib: A = B^T (rows s of the chunk), B[k = s][j = t] = dS[t][s]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j > ib) continue;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        adjust(sf[j][kk], dS_fix + tile0 + ((int64_t)ib * nb + j) * 4096 + tb * 64 + 16 * kk + 8 * hh,
               d.trapz && j == ib, tb - 16 * kk - 8 * hh, dcb);
      lane = opaque_lane();
#pragma unroll
      for (int q = 0; q < NT; ++q)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          mfma(acc[q], swz_tr8<NP>(chunk_rows, 64 * j + 16 * kk, 32 * q, lane), sf[j][kk]);
    }
  } else {
    // dB role: every tile (i, j <= i) of the chunk into LDS (over the head slots, free now), then the waves
    // of column block ib take tiles (i >= ib, ib): A = C^T (rows l), B[k = l][j = s] = dS[l][s] (transposed)
    bf16* tls = reinterpret_cast<bf16*>(smem + Cfg::o_slot);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        if (i >= nbl) continue;
        const int li = i * (i + 1) / 2 + j;
        // row pr is token 64 i + pr; the diagonal element sits in this piece when pk <= pr < pk + 8
        adjust(pc[li], dS_fix + tile0 + ((int64_t)i * nb + j) * 4096 + pr * 64 + pk, d.trapz && i == j, pr - pk,
               s_dcb[64 * i + pr]);
        *reinterpret_cast<bf16x8*>(tls + li * 4096 + pr * 64 + (swz_tr<64>(pr, pk >> 3) << 3)) = pc[li];
      }
    lds_barrier();
    lane = opaque_lane();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < ib || i >= nbl) continue;
      const bf16* ts = tls + (i * (i + 1) / 2 + ib) * 4096;
#pragma unroll
      for (int q = 0; q < NT; ++q)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          mfma(acc[q], swz_tr8<NP>(chunk_rows, 64 * i + 16 * kk, 32 * q, lane),
               swz_tr8<64>(ts, 16 * kk, 32 * (w & 1), lane));
    }
  }

  if (tok) {
    const int64_t row = (int64_t)(ci.row0 + t) * brow + (int64_t)g * d.N;
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n0 = 32 * q + 8 * r + 4 * hh;
        if (n0 >= d.N) continue;
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[q][4 * r + e];
        *reinterpret_cast<bf16x4*>((brole ? dB : dC) + row + n0) = o;
      }
  }
}

template <int PT, int NT>
__global__ void __launch_bounds__(512) k_bwd_rows(SSD_ROWS_PARAMS) {
  // block -> (chunk, group, role): block 16 (G q + g) + 8 r + x8 takes role r of chunk 8 q + x8, group g.
  // The two role blocks of a (chunk, group) are 8 apart (one XCD, dispatched together); consecutive
  // blocks step through the groups, so the resident blocks read the B / C and x / dy columns of many
  // groups at once (rows of G N and H P elements: one group's columns alone would load few HBM channels)
  const int b = blockIdx.x, x8 = b & 7;
  const bool brole = ((b >> 3) & 1) != 0;  // dB role (else dC and the decay term)
  const int rest = b >> 4, g = rest % d.G;
  const int c = (rest / d.G) * 8 + x8;
  if (c >= d.max_chunks) return;
  if (brole) {
    if (!d.da_only) bwd_rows_role<PT, NT, true, false>(c, g, SSD_ROWS_ARGS);
  } else if (hdec) {
    bwd_rows_role<PT, NT, false, true>(c, g, SSD_ROWS_ARGS);
  } else {
    bwd_rows_role<PT, NT, false, false>(c, g, SSD_ROWS_ARGS);
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
bool bwd_rows_supported(const SsdDims& d, int nslices, bool any_hpg) {
  // 256-token chunks, one head slice (bf16 dS tiles), few heads per group (beyond that the
  // per-block kernel's head stream already amortises its set-up), and tiles of at least 8 KB
  const int key = d.Ppad / 32 * 10 + d.Npad / 32;
  const int64_t blocks = ((int64_t)d.max_chunks + 7) / 8 * 16 * d.G;  // one-dimensional grid
  return d.Qpad == kRowsQ && nslices == 1 && (any_hpg || d.hpg <= SSD_ROWS_MAX_HPG) &&
         (key == 24 || key == 22 || key == 14) && blocks <= INT32_MAX;
}

size_t lds_bwd_rows(const SsdDims& d) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 14: return RowsCfg<1, 4>::bytes;
    case 22: return RowsCfg<2, 2>::bytes;
    default: return RowsCfg<2, 4>::bytes;
  }
}

template <int PT, int NT>
static hipError_t bwd_rows_t(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                             hipStream_t s) {
  ensure_lds(k_bwd_rows<PT, NT>, RowsCfg<PT, NT>::bytes);
  hipLaunchKernelGGL((k_bwd_rows<PT, NT>), dim3((d.max_chunks + 7) / 8 * 16 * d.G), dim3(512), (RowsCfg<PT, NT>::bytes),
                     s, d, b.chunks, b.cs, in.dt, reinterpret_cast<const bf16*>(in.x),
                     reinterpret_cast<const bf16*>(dy), reinterpret_cast<const bf16*>(b.hin), b.hin_lo,
                     reinterpret_cast<const bf16*>(b.hdec), b.hdec_lo, b.dst16,
                     reinterpret_cast<const bf16*>(in.B), reinterpret_cast<const bf16*>(in.C), b.dS_tiles16, b.dS_fix,
                     b.fast, b.dcs_off, reinterpret_cast<bf16*>(dB), reinterpret_cast<bf16*>(dC), b.tz_gam, b.xdy);
  return hipGetLastError();
}

hipError_t launch_bwd_rows(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                           hipStream_t s) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 14: return bwd_rows_t<1, 4>(d, b, in, dy, dB, dC, s);
    case 22: return bwd_rows_t<2, 2>(d, b, in, dy, dB, dC, s);
    case 24: return bwd_rows_t<2, 4>(d, b, in, dy, dB, dC, s);
    default: return hipErrorInvalidValue;
  }
}
