// dB and dC of the chunked SSD scan backward (bf16 fused path, gfx950), and
// the Y_off part of the decay gradient. Per chunk, 64-token block kb and
// group g, with the head-summed dS tiles of k_bwd_main:
//   dC_t = sum_{j <= kb} sum_s dS[t,s] B_s + sum_h exp(clamp(cs_t)) (dy_t h_in^T)
//   dB_t = sum_{i >= kb} sum_l dS[l,t] C_l + sum_h w_t dt_t (x_t dst^T)
//   dcs_off_t = pass(cs_t) exp(clamp(cs_t)) C_t . (dy_t h_in^T)        (per head)
// With bf16 states, the decay term takes h_in = hi + lo: hi is the staged bf16 state and lo its
// rounding residual (fp8, written by the forward walk in MFMA fragment order), loaded by the dC
// waves straight from global memory as MFMA operands one head ahead. The decay gradient is a
// per-head sum over every token whose terms largely cancel, and one chunk's rounding of h_in
// enters all of that chunk's tokens alike, so the bf16 state alone moves dA by about 1e-2
// where the sum is small. (The same work in the dB waves, which wait at each head's barrier,
// measured slower: their residual loads then sit behind the ring's DMAs in the in-order vmcnt.)
// (r2/dhammic-ai/src/kernels/ssd_scan.py:389-392 and :412-415 are the
// forward terms whose adjoints these are; w_t = exp(clamp(cs_last - cs_t)).)
//
// The state terms are GEMMs over the group's heads, K = P per head. Their
// per-token factors are applied to the per-head products (which the decay
// gradient needs unscaled), results kept transposed ([n rows][token lanes]).
// Each head's inputs (h_in, dst, the block's x and dy rows, cs, dt) are moved
// into LDS by buffer_load ... lds, two heads ahead through a ring of three
// slots, so no register holds staged data and the loads of two heads are in
// flight while one computes. The ring allows one block per CU, so its 8 waves
// take two roles that share each SIMD and overlap: waves 0-3 build dC and the
// decay gradient, waves 4-7 build dB (the shorter work) and issue the ring loads,
// whose issue waits for room in the texture unit's queue. LDS rows are unpadded; 16-byte granules are
// permuted per row so that transposed reads (h_in, dst) and row reads (x, dy)
// hit distinct banks.
//
// Few blocks (a short batch of one or two groups): the walk over the heads is a serial chain of ~2.2 us each and the
// tile terms another one (each step sums the column slices' dS partials, several in flight: 70 -> 58 us for 24 heads of
// one 256-token chunk), so both go to slices with fp32 partials of dB / dC (58 -> 22 us with the launch that sums
// them; gemm_slices in ssd_capi.hip has the rule).
#include <type_traits>

#include "ssd_launch.h"
#include "ssd_tile.h"

namespace {

template <int PT, int NT>
struct GemmCfg {
  static constexpr int PP = 32 * PT, NP = 32 * NT;
  static constexpr int HIN = PP * NP;           // elements of h_in (and of dst)
  static constexpr int XT = 64 * PP;            // elements of the x (and dy) rows
  // bytes of one ring slot: h_in, dst, x, dy, then cs, dt, cs_last, spare (64 floats each)
  static constexpr size_t kSlot = (size_t)(2 * HIN + 2 * XT) * 2 + 4 * 256;
  static constexpr size_t bytes = 3 * kSlot;
  // DMA instructions per issuing wave and head (waves 4-7)
  static constexpr int kTileDma = HIN / 512;    // 1 KB per instruction
  static constexpr int kRowDma = XT / 512;
  static constexpr int kPerWave = (2 * kTileDma + 2 * kRowDma) / 4 + 1;
  static_assert((2 * kTileDma + 2 * kRowDma) % 4 == 0, "DMA split");
  // Waves per SIMD to leave registers for: two blocks per CU (at most 128 VGPRs) where two rings fit its 160 KB of LDS
  // and the registers suffice (the 128-column dC / dB accumulators of NT = 4 take 158 and more).
  static constexpr int kWaves = NT <= 2 && 2 * (bytes + 256) <= 160 * 1024 ? 4 : 2;
};

}  // namespace

// MULTI: fp32 dS partials of several column slices (nslices > 1), summed here, and this kernel's own slices. Whole
// bf16 dS tiles (one column slice) take the other variant, which holds none of the registers the partials need.
template <int PT, int NT, bool MULTI>
__global__ void __launch_bounds__(512, (GemmCfg<PT, NT>::kWaves)) k_bwd_gemm(SsdDims d, const ChunkInfo* __restrict__ chunks,
                                                  const float* __restrict__ cs, const float* __restrict__ dt,
                                                  const bf16* __restrict__ x, const bf16* __restrict__ dy,
                                                  const bf16* __restrict__ hin, const uint8_t* __restrict__ hin_lo,
                                                  const bf16* __restrict__ dst,
                                                  const bf16* __restrict__ Bm, const bf16* __restrict__ Cm,
                                                  const float* __restrict__ dS, const bf16* __restrict__ dS16,
                                                  int nslices,
                                                  const float* __restrict__ dS_fix, const int32_t* __restrict__ fast,
                                                  float* __restrict__ dcs_off, bf16* __restrict__ dB,
                                                  bf16* __restrict__ dC, const float* __restrict__ tz_gam,
                                                  float* __restrict__ xdy, int hslice, int tsteps,
                                                  float* __restrict__ dB_part,
                                                  float* __restrict__ dC_part) {
  using Cfg = GemmCfg<PT, NT>;
  constexpr int PP = Cfg::PP, NP = Cfg::NP, NTW = (NT + 1) / 2, NK = PP / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  // block -> (chunk, 64-token block kb): the nb blocks of a chunk are consecutive in
  // dispatch order and share an XCD (same index mod 8), so each head's h_in / dst
  // tiles come from HBM once and from that XCD's L2 for the other blocks. The chunks of
  // the next group or slice go on where the last one's ended, mod 8: all XCDs get as many, also of few chunks.
  const int nbq = d.Qpad / 64;
  const int x8 = (blockIdx.x - d.max_chunks * (blockIdx.y + d.G * blockIdx.z)) & 7, rr = blockIdx.x >> 3;
  const int kb = rr % nbq;
  const int c = (rr / nbq) * 8 + x8, g = blockIdx.y;
  if (c >= d.max_chunks) return;
  const ChunkInfo ci = chunks[c];
  if (64 * kb >= ci.len) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool brole = w >= 4;  // dB waves, which also issue the ring loads (else dC waves)
  const int wi = w & 3;       // index among the issuing (dB) waves
  const int th = w & 1, nh = (w >> 1) & 1;
  int lane = threadIdx.x & 63, hh = lane >> 5, l32 = lane & 31;
  const int t_loc = 32 * th + l32;         // token of this lane within block kb
  const int t = 64 * kb + t_loc;           // ... within the chunk
  const bool tok = t < ci.len;
  const int nrows = min(64, ci.len - 64 * kb);
  const int64_t brow = (int64_t)d.G * d.N, xrow = (int64_t)d.H * d.P;
  const int MC = d.max_chunks, Qpad = d.Qpad;
  // this block's heads: all of the group's, then the tile terms; or (dB_part set) slice z of hslice heads, with more
  // slices for tsteps steps of the tile terms each
  const bool sliced = MULTI && dB_part != nullptr;
  const int hz = blockIdx.z * hslice, nhd = max(0, min(hslice, d.hpg - hz));
  const int h0 = g * d.hpg + hz;

  // ---- one head's inputs into a ring slot (kPerWave DMA instructions per issuing wave) ----
  // Issuing waves 0-1 (waves 4-5) load h_in and the x rows, 2-3 dst and the dy rows, each its own fixed
  // share, and one scalar row each (0 cs of the block's tokens, 1 dt, 2 cs of the chunk's last position,
  // 3 gamma in trapezoidal mode). Every per-lane offset and every base is fixed for
  // the block; a head only moves the bases by a wave-uniform soffset.
  constexpr int TPW = Cfg::kTileDma / 2, RPW = Cfg::kRowDma / 2;  // tile / row DMAs per issuing wave
  constexpr int TG = NP / 8, TRI = 64 / TG;  // h_in / dst rows of NP elements: granules per row, rows per DMA
  constexpr int XG = PP / 8, XRI = 64 / XG;  // x / dy rows of PP elements
  const bool second = wi >= 2;
  int vt[TPW], vr[RPW];
#pragma unroll
  for (int q = 0; q < TPW; ++q) {
    const int qi = (wi & 1) * TPW + q, r = qi * TRI + lane / TG;
    vt[q] = (r * NP + (swz_tr<NP>(r, lane % TG) << 3)) * 2;
  }
#pragma unroll
  for (int q = 0; q < RPW; ++q) {
    const int qi = (wi & 1) * RPW + q, r = qi * XRI + lane / XG;
    const int gcol = swz_nat<PP>(r, lane % XG) << 3;
    vr[q] = (r < nrows && gcol < d.P) ? (int)((r * xrow + gcol) * 2) : SSD_BUF_SIZE;
  }
  const int64_t row_b = (int64_t)(ci.row0 + 64 * kb);
  const bf16* tile_base = (second ? dst : hin) + (int64_t)c * d.H * Cfg::HIN;
  const bf16* rows_base = (second ? dy : x) + row_b * xrow;
  const bool s_tok = (wi == 1 && d.has_dt) || (wi == 3 && d.trapz);  // a per-token [R][H] row
  const float* scal_base = wi == 1 && d.has_dt ? dt + row_b * d.H
                         : wi == 3 && d.trapz ? tz_gam + row_b * d.H : cs + (int64_t)c * d.H * Qpad;
  const int s_vo = s_tok ? (lane < nrows ? lane * d.H * 4 : SSD_BUF_SIZE)
                 : wi == 0 ? (64 * kb + lane) * 4 : wi == 1 ? SSD_BUF_SIZE : (Qpad - 1) * 4;
  const int s_str = s_tok ? 4 : Qpad * 4;  // soffset bytes per head
  auto issue = [&](int h, unsigned char* base) {
    const __amdgpu_buffer_rsrc_t rt = buf_rsrc(tile_base), rr = buf_rsrc(rows_base), rs = buf_rsrc(scal_base);
    const int so_t = h * Cfg::HIN * 2, so_r = h * d.P * 2;
    unsigned char* bt = base + (second ? Cfg::HIN * 2 : 0);
    unsigned char* br = base + (2 * Cfg::HIN + (second ? Cfg::XT : 0)) * 2;
    // (each offset goes through a plain int, so that the target builtins' calls stay non-dependent)
#pragma unroll
    for (int q = 0; q < TPW; ++q) {
      const int vo = vt[q];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (__attribute__((address_space(3))) void*)(bt + ((wi & 1) * TPW + q) * 1024),
                                               16, vo, so_t, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
      const int vo = vr[q];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rr, (__attribute__((address_space(3))) void*)(br + ((wi & 1) * RPW + q) * 1024),
                                               16, vo, so_r, 0, 0);
    }
    {
      const int vo = s_vo, so = h * s_str;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void*)(base + (2 * Cfg::HIN + 2 * Cfg::XT) * 2 + wi * 256), 4, vo, so, 0,
          0);
    }
  };

  // trapezoidal mode: sum_h gamma (x_t . dy_t), the diagonal of dS (dC waves)
  float dcb = 0.0f;
  // dC (waves 0-3) or dB (waves 4-7) rows t, columns n of the wave's n tiles
  floatx16 acc[NTW];
#pragma unroll
  for (int q = 0; q < NTW; ++q) zero(acc[q]);
  // C[t][n] at this lane's accumulator rows n (the Y_off part of the decay gradient)
  const __amdgpu_buffer_rsrc_t rC = buf_rsrc(Cm + (int64_t)ci.row0 * brow + (int64_t)g * d.N);
  bf16x4 Cv[NTW][4];
#pragma unroll
  for (int q = 0; q < NTW; ++q) {
    const int nt = nh * NTW + q;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n0 = 32 * nt + 8 * r + 4 * hh;
      const bool ok = !brole && tok && nt < NT && n0 < d.N;
      Cv[q][r] = __builtin_bit_cast(
          bf16x4, __builtin_amdgcn_raw_buffer_load_b64(rC, ok ? (int)(t * brow + n0) * 2 : SSD_BUF_SIZE, 0, 0));
    }
  }
  wait_vm<0>();  // the ring's waits below count the ring's DMAs only

  // the tile terms' operands (fetched below the head loop)
  const int nb = Qpad / 64;
  const int nbl = (ci.len + 63) >> 6;
  const int64_t sstride = (int64_t)MC * d.G * nb * nb * 4096;
  const int64_t tile0 = ((int64_t)c * d.G + g) * nb * nb * 4096;
  const int pid = threadIdx.x, pr = pid >> 3, pk = (pid & 7) * 8;  // this thread's piece of a tile
  const int nsteps = max(kb + 1, nbl - kb);
  const __amdgpu_buffer_rsrc_t rS = buf_rsrc(MULTI ? (const void*)dS : (const void*)(dS16 + tile0));
  bf16x8 pS0, pS1;
  TileStage<64, NP, 512> sB, sC;
  auto fetch = [&](int st) {
    const bool ok0 = st <= kb, ok1 = kb + st < nbl;
    if (!MULTI) {
      pS0 = buf_ld16(rS, (int)((((int64_t)kb * nb + st) * 4096 + pr * 64 + pk) * 2), ok0);
      pS1 = buf_ld16(rS, (int)((((int64_t)(kb + st) * nb + kb) * 4096 + pr * 64 + pk) * 2), ok1);
    }
    tstage_load_v(sB, Bm + (int64_t)(ci.row0 + (ok0 ? 64 * st : 0)) * brow + (int64_t)g * d.N, brow,
                  ok0 ? min(64, ci.len - 64 * st) : 0, d.N);
    tstage_load_v(sC, Cm + (int64_t)(ci.row0 + (ok1 ? 64 * (kb + st) : 0)) * brow + (int64_t)g * d.N, brow,
                  ok1 ? min(64, ci.len - 64 * (kb + st)) : 0, d.N);
  };

  // dC waves: the h_in residual's MFMA fragments ([n = 32 nt + l32][p = 16 kk + 8 hh ..], fp8, stored in
  // that order: each is a contiguous 512 bytes) of the head being computed, loaded one head ahead
  uint2 lf[NTW][NK];
  const bool use_lo = !brole && hin_lo != nullptr;
  auto load_lo = [&](int hq) {
    const int ln = opaque_lane();
    const __amdgpu_buffer_rsrc_t rl = buf_rsrc(hin_lo + ((int64_t)c * d.H + hq) * Cfg::HIN);
#pragma unroll
    for (int q = 0; q < NTW; ++q)
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const bool ok = nh * NTW + q < NT;
        lf[q][kk] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(
            rl, ok ? (int)hin_lo_off(PP, 32 * (nh * NTW + q), 16 * kk) + ln * 8 : SSD_BUF_SIZE, 0, 0));
      }
  };
  // head order rotated per chunk (the blocks of one chunk keep the same order, so they still share each
  // head's tiles through L2): the resident blocks then read different 128-byte columns of the 8 KB token
  // rows at any moment instead of all the same one (HBM channel spread)
  const int hrot = nhd ? c % nhd : 0;
  auto head = [&](int k) { const int m = k + hrot; return h0 + (m >= nhd ? m - nhd : m); };
  if (brole) {
    if (0 < nhd) issue(head(0), smem);
    if (1 < nhd) issue(head(1), smem + Cfg::kSlot);
  }
  if (use_lo && 0 < nhd) load_lo(head(0));
  // head k reads slot k % 3 and refills slot (k + 2) % 3; the loop below is unrolled over the three
  // slots, so every slot address is a constant
  auto head_step = [&](int k, const unsigned char* __restrict__ cur, unsigned char* __restrict__ nxt) {
    const int h = head(k);
    // this wave's loads of head k are done (those of k + 1 may still fly); then every wave's
    if (brole) {
      if (k + 1 < nhd) wait_vm<Cfg::kPerWave>();
      else wait_vm<0>();
    }
    lds_barrier();  // head k visible in LDS; slot (k + 2) % 3 is free (head k - 1 done)
    ring_step(cur, nxt, brole && k + 2 < nhd,
              [&](unsigned char* nxt) { issue(head(k + 2), nxt); }, [&](const unsigned char* base) {
    if (brole && d.da_only) return;  // decay gradient only: no dB
    lane = opaque_lane();
    hh = lane >> 5;
    l32 = lane & 31;
    const bf16* th_ = reinterpret_cast<const bf16*>(base);
    const bf16* td_ = th_ + Cfg::HIN;
    const bf16* tx = td_ + Cfg::HIN;
    const bf16* ty = tx + Cfg::XT;
    const float* scal = reinterpret_cast<const float*>(ty + Cfg::XT);
    const float cst = scal[t_loc], csl = scal[128];
    const float dtt = d.has_dt ? scal[64 + t_loc] : 1.0f;
    const float et = exp_clamp(cst), pt_ = clamp_pass(cst);
    const float wdt = exp_clamp(csl - cst) * dtt;
    // dC waves: T = h_in dy_t^T (per n tile), dC += exp(clamp(cs_t)) T, decay term C_t . T;
    // dB waves: U = dst x_t^T, dB += w_t dt_t U
    const bf16* tile = brole ? td_ : th_;
    const bf16* rows = brole ? tx : ty;
    const float sc = brole ? wdt : et;
    bf16x8 rf[NK];
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) rf[kk] = swz_nat8<PP>(rows, t_loc, 16 * kk + 8 * hh);
    float osum = 0.0f;
#pragma unroll
    for (int q = 0; q < NTW; ++q) {
      const int nt = nh * NTW + q;
      if (nt >= NT) continue;
      floatx16 T;
      zero(T);
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) mfma(T, swz_tr8<NP>(tile, 16 * kk, 32 * nt, lane), rf[kk]);
      if (use_lo) {  // + lo dy_t^T: dC and the decay term take h_in = hi + lo
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) mfma(T, lo_frag(lf[q][kk]), rf[kk]);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[q][v] = fmaf(sc, T[v], acc[q][v]);
      if (!brole) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) osum += (float)Cv[q][r][e] * T[4 * r + e];
      }
    }
    if (use_lo && k + 1 < nhd) load_lo(head(k + 1));  // a whole head ahead of its use
    if (!brole) {
      osum = add_xor32(osum);
      if (hh == 0 && tok) dcs_off[((int64_t)nh * MC * d.H + (int64_t)c * d.H + h) * Qpad + t] = osum * et * pt_;
      if (d.trapz) {
        // x_t . dy_t from the staged rows (rf holds dy_t), for dgamma and the diagonal of dS
        float xd = 0.0f;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const bf16x8 xr = swz_nat8<PP>(tx, t_loc, 16 * kk + 8 * hh);
#pragma unroll
          for (int e = 0; e < 8; ++e) xd = fmaf((float)xr[e], (float)rf[kk][e], xd);
        }
        xd = add_xor32(xd);
        if (nh == 0 && hh == 0 && tok) xdy[((int64_t)c * d.H + h) * Qpad + t] = xd;
        dcb = fmaf(scal[192 + t_loc], xd, dcb);
      }
    }
    });
  };
  for (int k = 0; k < nhd; k += 3) {
    head_step(k, smem, smem + 2 * Cfg::kSlot);
    if (k + 1 < nhd) head_step(k + 1, smem + Cfg::kSlot, smem);
    if (k + 2 < nhd) head_step(k + 2, smem + 2 * Cfg::kSlot, smem + Cfg::kSlot);
  }

  if (d.da_only) return;  // decay gradient only: the Y_off term above is all it needs
  // dC (dC waves) / dB rows t: bf16, or a slice's partial sums
  auto put = [&]() {
    if (!tok) return;
    const int64_t row = (int64_t)(ci.row0 + t) * brow + (int64_t)g * d.N;
    float* part = sliced ? (brole ? dB_part : dC_part) + (int64_t)blockIdx.z * d.R * brow + row : nullptr;
    bf16* out = (brole ? dB : dC) + row;
#pragma unroll
    for (int q = 0; q < NTW; ++q) {
      const int nt = nh * NTW + q;
      if (nt >= NT) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n0 = 32 * nt + 8 * r + 4 * hh;
        if (n0 >= d.N) continue;
        if (sliced) {
          floatx4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = acc[q][4 * r + e];
          *reinterpret_cast<floatx4*>(part + n0) = o;
        } else {
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (bf16)acc[q][4 * r + e];
          *reinterpret_cast<bf16x4*>(out + n0) = o;
        }
      }
    }
  };
  // ---- tile terms, both roles at once: step m of the dC waves takes tile (kb, m), m <= kb, with the B
  // rows of block m (dC += dS B); step m of the dB waves tile (kb + m, kb), kb + m < nbl, with the C rows
  // of block kb + m (dB += dS^T C). Each role has its LDS buffer pair; every thread stages one 8-element
  // piece of each tile and its share of both row blocks. With bf16 dS tiles (one head slice) the next
  // step's pieces are in flight in registers while a step computes ----
  constexpr int PI = tpitch_tr<NP>();
  bf16* tBC0 = reinterpret_cast<bf16*>(smem);                // dC waves: B rows of block m   [64][NP]
  bf16* tS0 = tBC0 + tsize<64, NP, PI>();                    //           dS tile (kb, m)     [64][64]
  bf16* tBC1 = tS0 + tsize<64, 64, tpitch<64>()>();          // dB waves: C rows of block m'
  bf16* tS1 = tBC1 + tsize<64, NP, PI>();                    //           dS tile (m', kb)
  float* s_dcb = reinterpret_cast<float*>(smem + Cfg::bytes) - 64;  // [64] (trapezoidal mode), past them
  static_assert(4 * (tsize<64, NP, PI>() + tsize<64, 64, tpitch<64>()>()) + 256 <= Cfg::bytes, "tile buffers");
  if (d.trapz) {
    __syncthreads();  // the ring's last reads are done
    if (!brole && nh == 0 && hh == 0) s_dcb[t_loc] = dcb;
  }
  if (sliced && nhd > 0) {
    if (d.trapz) {  // the slice's part of dS's diagonal: dC_t += dcb B_t, dB_t += dcb C_t
      __syncthreads();
      const float dg = s_dcb[t_loc];
      const __amdgpu_buffer_rsrc_t rg = buf_rsrc((brole ? Cm : Bm) + (int64_t)ci.row0 * brow + (int64_t)g * d.N);
#pragma unroll
      for (int q = 0; q < NTW; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n0 = 32 * (nh * NTW + q) + 8 * r + 4 * hh;
          const bool ok = tok && n0 < d.N;
          const bf16x4 v = __builtin_bit_cast(bf16x4, __builtin_amdgcn_raw_buffer_load_b64(
              rg, ok ? (int)(t * brow + n0) * 2 : SSD_BUF_SIZE, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[q][4 * r + e] = fmaf(dg, (float)v[e], acc[q][4 * r + e]);
        }
    }
    put();
    return;
  }
  // heads of the group the factorised kernel left to the exact fixup: their dS is in dS_fix
  bool slow = false;
  if (fast)
    for (int hq = g * d.hpg + (int)threadIdx.x; hq < (g + 1) * d.hpg; hq += 512) slow = slow || fast[(int64_t)c * d.H + hq] == 0;
  const bool any_fix = __syncthreads_or(slow);
  const int st0 = sliced ? (blockIdx.z - (d.hpg + hslice - 1) / hslice) * tsteps : 0;
  const int st1 = sliced ? min(nsteps, st0 + tsteps) : nsteps;
  if (st0 < st1) fetch(st0);
  // one tile's piece: the fetched bf16 values, or the fp32 slice partials summed here; plus the fixup
  // heads' dS and (trapezoidal mode, tile (kb, kb)) the diagonal sum_h gamma (x_t . dy_t)
  auto store_piece = [&](bf16* tS, int ti, int tj, const bf16x8& pre) {
    float v[8];
    if constexpr (!MULTI) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (float)pre[e];
    } else {
      // (uniform bases, one per slice: the lane's offset is the same in all of them)
      const float* src = dS + tile0 + ((int64_t)ti * nb + tj) * 4096;
      const int po = (pr * 64 + pk) * 4;
      auto ld = [&](int slc, floatx4& a0, floatx4& a1) {
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(src + slc * sstride);
        a0 = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, po, 0, 0));
        a1 = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, po + 16, 0, 0));
      };
      floatx4 s0, s1;
      ld(0, s0, s1);
      // the other slices in order, up to six of them in flight (eight take 135 VGPRs: one block per CU)
      int sl = 1;
      auto add = [&](auto n) {
        constexpr int U = decltype(n)::value;
#pragma unroll 1
        for (; sl + U <= nslices; sl += U) {
          floatx4 u0[U], u1[U];
#pragma unroll
          for (int u = 0; u < U; ++u) ld(sl + u, u0[u], u1[u]);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            s0 += u0[u];
            s1 += u1[u];
          }
        }
      };
      add(std::integral_constant<int, 6>{});
      add(std::integral_constant<int, 3>{});
      add(std::integral_constant<int, 2>{});
      add(std::integral_constant<int, 1>{});
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = s0[e];
        v[4 + e] = s1[e];
      }
    }
    if (any_fix) {
      const float* fx = dS_fix + tile0 + ((int64_t)ti * nb + tj) * 4096 + pr * 64 + pk;
      const floatx4 f0 = *reinterpret_cast<const floatx4*>(fx), f1 = *reinterpret_cast<const floatx4*>(fx + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += f0[e];
        v[4 + e] += f1[e];
      }
    }
    // trapezoidal mode: the scan is strictly causal and the diagonal term is the per-token D part
    // gamma (C_t . B_t) x_t, so the diagonal of dS is sum_h gamma (x_t . dy_t)
    if (d.trapz && ti == tj && (pr >> 3) == (pid & 7)) v[pr & 7] += s_dcb[pr];  // row pr is token 64 kb + pr
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (bf16)v[e];
    *reinterpret_cast<bf16x8*>(tS + toff<64, tpitch<64>()>(pr, pk)) = o;
  };
  for (int st = st0; st < st1; ++st) {
    lds_barrier();  // the previous step's reads of both buffers are done (st = 0: the ring's, and s_dcb)
    if (st <= kb) {
      store_piece(tS0, kb, st, pS0);
      tstage_store<64, NP, 512, PI>(sB, tBC0);
    }
    if (kb + st < nbl) {
      store_piece(tS1, kb + st, kb, pS1);
      tstage_store<64, NP, 512, PI>(sC, tBC1);
    }
    if (st + 1 < st1) fetch(st + 1);
    lds_barrier();
    lane = opaque_lane();
    hh = lane >> 5;
    const bool mine = brole ? kb + st < nbl : st <= kb;
    if (!mine) continue;
    const bf16* tBC = brole ? tBC1 : tBC0;
    const bf16* tS = brole ? tS1 : tS0;
#pragma unroll
    for (int q = 0; q < NTW; ++q) {
      const int nt = nh * NTW + q;
      if (nt >= NT) continue;
#pragma unroll
      for (int kk = 0; kk < 64; kk += 16) {
        const bf16x8 av = ttr_std<NP, PI>(tBC, kk, 32 * nt, lane);
        // dC waves: B[k = s][j = t] = dS[t][s] (row t, natural); dB waves: B[k = l][j = t] (transposed)
        if (!brole)
          mfma(acc[q], av, tld8<64, tpitch<64>()>(tS, t_loc, kk + 8 * hh));
        else
          mfma(acc[q], av, ttr_std<64, tpitch<64>()>(tS, kk, 32 * th, lane));
      }
    }
  }
  put();
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
size_t lds_bwd_gemm(const SsdDims& d) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return GemmCfg<1, 1>::bytes;
    case 12: return GemmCfg<1, 2>::bytes;
    case 14: return GemmCfg<1, 4>::bytes;
    case 21: return GemmCfg<2, 1>::bytes;
    case 22: return GemmCfg<2, 2>::bytes;
    default: return GemmCfg<2, 4>::bytes;
  }
}

template <int PT, int NT, bool MULTI>
static hipError_t bwd_gemm_m(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                             hipStream_t s) {
  ensure_lds(k_bwd_gemm<PT, NT, MULTI>, GemmCfg<PT, NT>::bytes);
  const int nbq = d.Qpad / 64, nz = (d.hpg + b.gemm_hslice - 1) / b.gemm_hslice;
  const bool sliced = MULTI && nz > 1 && !d.da_only;  // (a decay-only pass has no tile terms and nothing to sum)
  hipLaunchKernelGGL((k_bwd_gemm<PT, NT, MULTI>), dim3((d.max_chunks + 7) / 8 * 8 * nbq, d.G, sliced ? b.gemm_parts : nz),
                     dim3(512), (GemmCfg<PT, NT>::bytes), s,
                     d, b.chunks, b.cs, in.dt, reinterpret_cast<const bf16*>(in.x),
                     reinterpret_cast<const bf16*>(dy), reinterpret_cast<const bf16*>(b.hin), b.hin_lo, b.dst16,
                     reinterpret_cast<const bf16*>(in.B), reinterpret_cast<const bf16*>(in.C), b.dS_tiles,
                     b.dS_tiles16, b.nslices, b.dS_fix, b.fast, b.dcs_off, reinterpret_cast<bf16*>(dB),
                     reinterpret_cast<bf16*>(dC), b.tz_gam, b.xdy, b.gemm_hslice, b.gemm_tsteps, sliced ? b.dB_part : nullptr,
                     sliced ? b.dC_part : nullptr);
  return hipGetLastError();
}

// (the row kernel's slices come with several column slices: gemm_slices splits at 64 blocks or fewer and 6 heads or
// more, where the column side has four slices or one per head)
template <int PT, int NT>
static hipError_t bwd_gemm_t(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                             hipStream_t s) {
  return b.dS_tiles ? bwd_gemm_m<PT, NT, true>(d, b, in, dy, dB, dC, s) : bwd_gemm_m<PT, NT, false>(d, b, in, dy, dB, dC, s);
}

hipError_t launch_bwd_gemm(const SsdDims& d, const SsdBufs& b, const SsdIn& in, const void* dy, void* dB, void* dC,
                           hipStream_t s) {
  switch (d.Ppad / 32 * 10 + d.Npad / 32) {
    case 11: return bwd_gemm_t<1, 1>(d, b, in, dy, dB, dC, s);
    case 12: return bwd_gemm_t<1, 2>(d, b, in, dy, dB, dC, s);
    case 14: return bwd_gemm_t<1, 4>(d, b, in, dy, dB, dC, s);
    case 21: return bwd_gemm_t<2, 1>(d, b, in, dy, dB, dC, s);
    case 22: return bwd_gemm_t<2, 2>(d, b, in, dy, dB, dC, s);
    default: return bwd_gemm_t<2, 4>(d, b, in, dy, dB, dC, s);
  }
}
