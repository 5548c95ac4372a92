// One output tile of the bf16 matrix-core GEMM as device code shared by the kernels that run it: the batched /
// grouped GEMM kernel (one workgroup per tile, gemm_bf16.hip) and the persistent Newton-Schulz kernel (a workgroup
// takes tile after tile of the products of a whole iteration sequence, ns_flow.hip).
//
// Work decomposition, LDS layouts, direct-to-LDS staging, operand-swapped MFMA and the epilogue through LDS are
// described at the top of gemm_bf16.hip.
#pragma once
#include "common.h"
#include "mfma_tile.h"
#include <type_traits>

namespace {

template <int BT_, int WGM_, int WGN_>
struct Cfg {
  static constexpr int BT = BT_, WGM = WGM_, WGN = WGN_;
  static constexpr int NT = 64 * WGM * WGN;        // threads
  static constexpr int TMI = BT / (16 * WGM);      // 16 x 16 accumulator blocks per wavefront, row direction
  static constexpr int TNJ = BT / (16 * WGN);      // ... column direction
  static constexpr int NCH = BT * 8 / NT;          // 16-byte chunks per thread per operand stage
  static constexpr int WROWS = BT / WGM, WCOLS = BT / WGN;
  // the last row and column of tiles lies against the matrix's end, over part of its neighbour (gemm_bf16.hip, Mid)
  static constexpr bool SLIDE = BT == 192;
  // interior and edge tiles run gemm_tile_k_loop_quad
  static constexpr bool QUAD = WGM == 2 && WGN == 2;
  // A k-strided operand of 128-tiles there: a wavefront has two runs of 32 rows (columns) 64 apart, so that what it reads in one phase
  // is half a k-row of the tile, a whole cache line (two half lines otherwise: both operands k-strided 1720 - 1880 clocks a stage).
  static constexpr bool split(bool full, bool ks) { return QUAD && full && BT == 128 && ks; }
  typedef f32x4_t acc_t;
};

template <int BT, bool KS>
struct Tile {
  static constexpr int bytes = BT * BK * 2;   // either layout: 64 x BT bf16
};

// Per-thread addressing of the NCH 16-byte chunks a thread moves per operand stage.
//   Register-staged path (bounds-checked): chunk i lies at global `g + i * gstep` (elements)
//   and goes to LDS byte offset `l + i * lstep`.
//   Direct-to-LDS path: wave-instruction i of wavefront w fills the 1024-byte LDS block
//   (i * NW + w); lane p of it fetches the chunk whose *physical* position is p, i.e. the
//   swizzle is applied to the global address, which is kept as a wave-uniform base pointer
//   (`dbase`) plus a 32-bit byte offset (`doff + i * dstep`, per lane and loop invariant, plus
//   the stage's offset, a scalar) so that the loads use SGPR-base addressing.
template <typename C, bool KS>
struct StageAddr {
  const bf16_t* g;
  const char* dbase;
  unsigned doff, dstep;
  long long gstep, tstep;   // per chunk and per stage, in elements
  int l, lstep;
  int row, col;             // first chunk's (row within tile, k offset) resp. (k row, row offset)
  // `dim`: extent of the operand in the tile's row direction (M or N); the direct-to-LDS addresses of a
  // k-strided operand keep their 16-byte chunks inside it (an edge tile then fetches a neighbouring chunk for the
  // columns it does not own: finite values that the bounds-checked epilogue never stores).
  __device__ __forceinline__ StageAddr(const bf16_t* base, int ld, int row0, int tid, int dim) {
    constexpr int NW = C::NT / 64;
    const int lane = tid & 63, wave = tid >> 6;
    if (!KS) {
      row = tid >> 3;
      col = (tid & 7) * 8;
      g = base + (long long)(row0 + row) * ld + col;
      gstep = (long long)(C::NT / 8) * ld;
      tstep = BK;
      l = row * 128 + kc_swizzle(tid & 7, row) * 16;
      lstep = (C::NT / 8) * 128;   // NT/8 is a multiple of 16: the swizzle term is the same for all chunks
      const int drow = wave * 8 + (lane >> 3);             // block (0 * NW + wave), 8 rows per block
      dbase = reinterpret_cast<const char*>(base + (long long)row0 * ld);
      doff = (unsigned)(drow * ld + kc_swizzle(lane & 7, drow) * 8) * 2u;
      dstep = (unsigned)(NW * 8 * ld) * 2u;                // NW * 8 is a multiple of 16
    } else {
      constexpr int CPR = C::BT / 8;                       // chunks per k-row
      constexpr int RPB = 64 / CPR;                        // k-rows per 1024-byte block
      row = tid / CPR;
      col = (tid % CPR) * 8;
      g = base + (long long)row * ld + row0 + col;
      gstep = (long long)(C::NT / CPR) * ld;
      tstep = (long long)BK * ld;
      l = row * (C::BT * 2) + ks_swizzle(tid % CPR, row) * 16;
      lstep = (C::NT / CPR) * (C::BT * 2);                 // NT / CPR = 16: swizzle term unchanged
      const int drow = wave * RPB + lane / CPR;
      dbase = reinterpret_cast<const char*>(base + row0);
      int dcol = ks_swizzle(lane % CPR, drow) * 8;
      if (row0 + dcol > dim - 8) dcol = dim - 8 - row0;
      doff = (unsigned)(drow * ld + dcol) * 2u;
      dstep = (unsigned)(NW * RPB * ld) * 2u;              // NW * RPB = 16
    }
  }
};

// The accumulators go through LDS (the stage buffers are free by now), one 32-row band of the
// wavefront's sub-tile at a time, so that C and E move as 16-byte row segments.  Each wavefront
// stages through its own LDS region, so only wavefront-level ordering is needed inside.
// Output dtype, epilogue form and rounding mode are compile-time here: evaluated per element at
// run time they cost more than the MFMAs of a short-K product.
// The weight update of the reference's post-orthogonalisation pass on 8 consecutive elements of the weights at `Wp`
// (dion/muon.py:569-573): W <- r_W(r_W(W * decay) - r_bf16(U * step)), U = the eight bf16 results in `pk`; the old
// weights come in x0 (bf16: all eight) resp. x0, x1 (fp32), requested a band earlier.
__device__ __forceinline__ void update_weights8(char* Wp, bool w_f32, u32x4_t x0, u32x4_t x1, u32x4_t pk, float decay,
                                                float step) {
  if (!w_f32) {
    u32x4_t o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned x = x0[q], u = pk[q];
      const unsigned xd = cvt_pk_bf16(lo_f(x) * decay, hi_f(x) * decay);
      const unsigned t = cvt_pk_bf16(lo_f(u) * step, hi_f(u) * step);
      o[q] = cvt_pk_bf16(lo_f(xd) - lo_f(t), hi_f(xd) - hi_f(t));
    }
    stg16(Wp, o);
  } else {
    u32x4_t o0, o1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned u = pk[q];
      const unsigned t = cvt_pk_bf16(lo_f(u) * step, hi_f(u) * step);
      const unsigned xa = q < 2 ? x0[2 * q] : x1[2 * q - 4], xb = q < 2 ? x0[2 * q + 1] : x1[2 * q - 3];
      const float ra = __builtin_bit_cast(float, xa) * decay - lo_f(t);
      const float rb = __builtin_bit_cast(float, xb) * decay - hi_f(t);
      if (q < 2) { o0[2 * q] = __builtin_bit_cast(unsigned, ra); o0[2 * q + 1] = __builtin_bit_cast(unsigned, rb); }
      else { o1[2 * q - 4] = __builtin_bit_cast(unsigned, ra); o1[2 * q - 3] = __builtin_bit_cast(unsigned, rb); }
    }
    stg16(Wp, o0);
    stg16(Wp + 16, o1);
  }
}

// LDS bytes of the epilogue: a band of fp32 results and one of bf16 results (to be turned) for each wavefront.
template <typename C> constexpr int epilogue_lds() {
  return (C::NT / 64) * 32 * ((C::WCOLS + 4) * 4 + (C::WCOLS <= 64 ? 128 : 256));
}
// UPD: 0 the result is stored in C; 1 / 2 it is not stored but updates the weights d.upd_tab[b] in place (2: those are
// stored transposed), see GemmDesc.
// RSPLIT, CSPLIT: a wavefront's rows (columns) are two runs, see Cfg::split.
template <typename C, bool SYM, bool FULL, bool CF32, bool HAS_E, bool FAITHFUL, bool S1_ONE, int UPD = 0, bool WF32 = false,
          bool RSPLIT = false, bool CSPLIT = false>
__device__ __forceinline__ void epilogue_impl(typename C::acc_t (&acc)[C::TMI][C::TNJ], const GemmDesc& d, char* lds, int b,
                                              bool mirror, int m0, int n0, int wave, int lane, int wm, int wn) {
  constexpr int W = C::WCOLS;        // columns of a wavefront's sub-tile
  constexpr int PITCH = W + 4;       // floats; 16-byte aligned rows, conflict-free float4 writes
  constexpr int CPR = W / 8;         // 8-column chunks per row
  constexpr int RPP = 64 / CPR;      // rows per pass of the wavefront
  constexpr bool PIPE = C::QUAD && !(SYM && CF32);   // (see below)
  // rows of a band; 16 of 128 columns, for the registers' sake: two staging areas then, taken in turns
  constexpr int BR = PIPE && W == 128 ? 16 : 32, NB = C::WROWS / BR;
  constexpr int NPASS = (BR + RPP - 1) / RPP;
  constexpr bool ODD = 64 % CPR != 0;   // (twelve chunks to a row: five rows a pass, four lanes and most of the last pass idle)
  constexpr int CSZ = CF32 ? 4 : 2;
  constexpr int NV = CF32 ? 2 : 1;   // 16-byte vectors per 8 elements
  // TURN: the bf16 results go through LDS a second time, to be stored transposed: 32 rows of the band as a k-strided tile ([32][W] in
  // 32-byte slots, read_frag16), whose transpose read hands a lane eight consecutive rows of a column.
  constexpr bool TURN = (SYM && !CF32) || UPD == 2;
  constexpr int TPITCH = W <= 64 ? 128 : 256;
  // PIPE: a band is written to LDS and requested back before the arithmetic of the one before it (with one wavefront to a SIMD
  // nothing else covers the round trip; a wavefront's LDS operations run in order).
  float* stg = reinterpret_cast<float*>(lds) + wave * (32 * PITCH);
  char* const trn = lds + (C::NT / 64) * (32 * PITCH * 4) + wave * (32 * TPITCH);
  // the descriptor lives in the kernel-argument segment: fields read inside the band loop would be fetched
  // again after every store (scalar load + a full wait in the middle of the band), so they are copied first
  const float s0 = d.s0, s1 = d.s1;
  const long long c2 = (!HAS_E && !FAITHFUL && !SYM && !CF32) ? d.c2_off * 2 : 0;   // bytes to the second output
  const int dM = d.M, dN = d.N;
  const long long ldc = d.ldc, lde = d.lde;
  const int wm0 = m0 + wm * (RSPLIT ? 32 : C::WROWS), wn0 = n0 + wn * (CSPLIT ? 32 : W);
  auto row_of = [&](int band) { return wm0 + (RSPLIT ? band * 64 : band * BR); };        // first row of a band
  auto col_of = [&](int c) { return wn0 + (CSPLIT ? (c & 31) + (c >> 5) * 64 : c); };   // column c of the wavefront's
  char* const Cbase = d.Ctab ? static_cast<char*>(d.Ctab[b]) : static_cast<char*>(d.C) + (long long)b * d.sC * CSZ;
  const char* const Ebase = !HAS_E ? nullptr
                            : d.Etab ? static_cast<const char*>(d.Etab[b])
                                     : static_cast<const char*>(d.E) + (long long)b * d.sE * CSZ;
  const int lr = lane / CPR, c8 = (lane % CPR) * 8, cn = col_of(c8);
  const bool col_ok = (FULL || cn < dN) && (!ODD || lane < RPP * CPR);
  char* const Wbase = UPD ? static_cast<char*>(d.upd_tab[b]) : nullptr;
  constexpr bool w_f32 = WF32;   // (a compile-time variant: the prefetch buffers differ in size)
  constexpr int wsz = w_f32 ? 4 : 2;
  const long long ldw = d.upd_ld;
  const float w_decay = d.upd_decay, w_step = d.upd_step;
  // E is requested up to three bands ahead (registers that the K loop's fragments no longer need), so that a
  // tile's epilogue pays one memory latency and not one per band; an fp32 E (twice the registers) one band ahead.
  constexpr int DEPTH = (!HAS_E || CF32) ? 1 : BR == 16 ? (UPD ? 2 : 4) : (UPD ? 2 : (NB < 3 ? NB : 3));
  u32x4_t ev[DEPTH][NPASS][NV];
  // the weights a band updates are requested when the band starts, ahead of its staging through LDS and of the
  // arithmetic on E (two vectors per 8 elements when they are fp32)
  constexpr int NWP = UPD == 2 ? W / 16 : NPASS;
  constexpr int NWV = WF32 ? 2 : 1;
  u32x4_t wv[NWP][NWV];
  auto weight_ptr = [&](int band, int pass) -> char* {
    if (UPD == 2) {
      const int n = col_of(pass * 16 + (lane & 15)), m = row_of(band / (32 / BR) * (32 / BR)) + (lane >> 4) * 8;
      return Wbase + ((long long)n * ldw + m) * wsz;
    }
    const int m = row_of(band) + pass * RPP + lr;
    return Wbase + ((long long)m * ldw + cn) * wsz;
  };
  auto load_w = [&](int band, u32x4_t (&dst)[NWP][NWV]) {
#pragma unroll
    for (int pass = 0; pass < NWP; ++pass) {
      const char* p = weight_ptr(band, pass);
#pragma unroll
      for (int h = 0; h < NWV; ++h) dst[pass][h] = ldg16(p + 16 * h);
    }
  };

  auto load_e = [&](int band, u32x4_t (&dst)[NPASS][NV]) {
#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) {
      const int m = row_of(band) + pass * RPP + lr;
      const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int h = 0; h < NV; ++h) dst[pass][h] = z;
      if (col_ok && (FULL || m < dM) && (!ODD || pass * RPP + lr < BR)) {
        const char* Ep = Ebase + ((long long)m * lde + cn) * CSZ;
#pragma unroll
        for (int h = 0; h < NV; ++h) dst[pass][h] = ldg16(Ep + 16 * h);
      }
    }
  };
  if (HAS_E) {
#pragma unroll
    for (int q = 0; q < DEPTH; ++q) load_e(q, ev[q]);
  }
  auto put_band = [&](int i) {
    // a lane holds, for row (lane & 15) of a block, the four columns 4 (lane >> 4) .. + 3
    float* row = stg + (BR == 16 ? (i & 1) * 16 * PITCH : 0) + (lane & 15) * PITCH + (lane >> 4) * 4;
#pragma unroll
    for (int ib = 0; ib < BR / 16; ++ib)
#pragma unroll
      for (int j = 0; j < C::TNJ; ++j) {
        const typename C::acc_t& a = acc[(BR / 16 * i + ib) % C::TMI][j];
        *reinterpret_cast<float4*>(row + ib * 16 * PITCH + j * 16) = make_float4(a[0], a[1], a[2], a[3]);
      }
    wave_sync_lds();
  };
  float4 raw[PIPE ? 2 : 1][NPASS][2];
  auto get_pass = [&](int i, int pass, float4 (&dst)[2]) {
    if (!ODD || pass * RPP + lr < BR) {
      const float* sp = stg + (BR == 16 ? (i & 1) * 16 * PITCH : 0) + (pass * RPP + lr) * PITCH + c8;
      dst[0] = *reinterpret_cast<const float4*>(sp);
      dst[1] = *reinterpret_cast<const float4*>(sp + 4);
    }
  };
  auto get_band = [&](int i, float4 (&dst)[NPASS][2]) {
#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) get_pass(i, pass, dst[pass]);
    wave_sync_lds();
  };
  if (PIPE) {
    put_band(0);
    get_band(0, raw[0]);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (UPD == 1 || (UPD == 2 && i % (32 / BR) == 0)) load_w(i, wv);
    if (!PIPE) put_band(i);
    else if (i + 1 < NB) {
      put_band(i + 1);
      get_band(i + 1, raw[(i + 1) & (PIPE ? 1 : 0)]);
    }
    const int band_m = row_of(i);
    u32x4_t ec[NPASS][NV];
    if (HAS_E) {
#pragma unroll
      for (int pass = 0; pass < NPASS; ++pass)
#pragma unroll
        for (int h = 0; h < NV; ++h) ec[pass][h] = ev[i % DEPTH][pass][h];
      if (i + DEPTH < NB) load_e(i + DEPTH, ev[i % DEPTH]);
    }

#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) {
      const int r = pass * RPP + lr;
      const int m = band_m + r;
      if (col_ok && (FULL || m < dM) && (!ODD || r < BR)) {
        float* sp = stg + r * PITCH + c8;
        if (!PIPE) get_pass(i, pass, raw[0][pass]);
        const float4 a0 = raw[PIPE ? i & 1 : 0][pass][0], a1 = raw[PIPE ? i & 1 : 0][pass][1];
        float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        float e[8];
        char* Cp = Cbase + ((long long)m * ldc + cn) * CSZ;
        if (CF32) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const unsigned w = HAS_E ? ec[pass][q >> 2][q & 3] : 0u;  // (bit_cast of a vector element lvalue reads element 0)
            e[q] = __builtin_bit_cast(float, w);
          }
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = epi_value<HAS_E, FAITHFUL, true>(s0, s1, v[q], e[q]);
          const u32x4_t o0 = {__builtin_bit_cast(unsigned, v[0]), __builtin_bit_cast(unsigned, v[1]),
                              __builtin_bit_cast(unsigned, v[2]), __builtin_bit_cast(unsigned, v[3])};
          const u32x4_t o1 = {__builtin_bit_cast(unsigned, v[4]), __builtin_bit_cast(unsigned, v[5]),
                              __builtin_bit_cast(unsigned, v[6]), __builtin_bit_cast(unsigned, v[7])};
          stg16(Cp, o0);
          stg16(Cp + 16, o1);
        } else {
          u32x4_t pk;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const unsigned w = HAS_E ? ec[pass][0][q] : 0u;   // (copied out: see the note on bit_cast above)
            const unsigned o = epi_pair<HAS_E, FAITHFUL, S1_ONE>(s0, s1, v[2 * q], v[2 * q + 1], w);
            pk[q] = o;
          }
          if (UPD == 0) stg16(Cp, pk);
          if (UPD == 1) update_weights8(weight_ptr(i, pass), w_f32, wv[pass][0], wv[pass][NWV - 1], pk, w_decay, w_step);
          if (TURN && (UPD == 2 || mirror))
            *reinterpret_cast<u32x4_t*>(trn + (r + i % (32 / BR) * BR) * TPITCH + (((c8 >> 4) ^ (r & 3)) * 32 + (c8 & 8) * 2)) = pk;
          if (!HAS_E && !FAITHFUL && !SYM && c2) {
            // what the stored bf16 leaves of s1 * acc, as a second bf16 matrix
            u32x4_t lo;
#pragma unroll
            for (int q = 0; q < 4; ++q) lo[q] = cvt_pk_bf16(s1 * v[2 * q] - lo_f(pk[q]), s1 * v[2 * q + 1] - hi_f(pk[q]));
            stg16(Cp + c2, lo);
          }
        }
        if (SYM && CF32 && mirror) {  // keep the final values for the transposed store
          *reinterpret_cast<float4*>(sp) = make_float4(v[0], v[1], v[2], v[3]);
          *reinterpret_cast<float4*>(sp + 4) = make_float4(v[4], v[5], v[6], v[7]);
        }
      }
    }
    // Transposed: row n of the mirrored tile (of the weights) holds 32 consecutive m of this band.  Where sliding tiles overlap, what a
    // diagonal tile stores (from E itself) is left to it: with E(m, n) here and E(n, m) there, an E that is not symmetric would leave either.
    const int n_own = C::SLIDE && n0 + C::BT >= dN ? (dN - 1) / C::BT * C::BT : 0;
    const int m_end = C::SLIDE ? dM - C::BT : 0;
    if (TURN && (UPD == 2 || mirror) && (i + 1) % (32 / BR) == 0) {
      wave_sync_lds();
#pragma unroll
      for (int slot = 0; slot < W / 16; ++slot) {
        const int g = lane >> 4, q = (lane & 15) >> 2;
        const char* p = trn + (g * 8 + q) * TPITCH + (slot ^ q) * 32 + (lane & 3) * 8;
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(DA_LDS_PTR(s16x4_t, p));
        const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(DA_LDS_PTR(s16x4_t, p + 4 * TPITCH));
        typedef short s16x8_t __attribute__((ext_vector_type(8)));
        const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        const u32x4_t pk = __builtin_bit_cast(u32x4_t, v);
        const int n = col_of(slot * 16 + (lane & 15)), m = row_of(i + 1 - 32 / BR) + g * 8;
        if (C::SLIDE && (n < n_own || m >= m_end)) continue;
        if (FULL || (n < dN && m < dM)) {   // M is a multiple of 8 for symmetric outputs
          if (UPD == 2) update_weights8(weight_ptr(i, slot), w_f32, wv[slot][0], wv[slot][NWV - 1], pk, w_decay, w_step);
          else stg16(Cbase + ((long long)n * ldc + m) * CSZ, pk);
        }
      }
    }
    if (SYM && CF32 && mirror) {
      wave_sync_lds();
#pragma unroll
      for (int pass = 0; pass < (W + 63) / 64 * 4; ++pass) {
        const int nl = (pass >> 2) * 64 + lane;
        const int mg = (pass & 3) * 8;
        const int n = wn0 + nl, m = band_m + mg;
        if (C::SLIDE && (n < n_own || m >= m_end)) continue;
        if ((FULL || (n < dN && m < dM)) && (W % 64 == 0 || nl < W)) {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = stg[(mg + q) * PITCH + nl];
          char* Cp = Cbase + ((long long)n * ldc + m) * CSZ;
          const u32x4_t o0 = {__builtin_bit_cast(unsigned, v[0]), __builtin_bit_cast(unsigned, v[1]),
                              __builtin_bit_cast(unsigned, v[2]), __builtin_bit_cast(unsigned, v[3])};
          const u32x4_t o1 = {__builtin_bit_cast(unsigned, v[4]), __builtin_bit_cast(unsigned, v[5]),
                              __builtin_bit_cast(unsigned, v[6]), __builtin_bit_cast(unsigned, v[7])};
          stg16(Cp, o0);
          stg16(Cp + 16, o1);
        }
      }
    }
    wave_sync_lds();
  }
}

template <typename C, bool SYM, bool FULL, bool RSPLIT = false, bool CSPLIT = false>
__device__ __forceinline__ void epilogue(typename C::acc_t (&acc)[C::TMI][C::TNJ], const GemmDesc& d, char* lds, int b, int ti,
                                         int tj, int m0, int n0, int wave, int lane, int wm, int wn) {
  const bool mirror = SYM && (ti != tj);
  const bool cf32 = d.c_dtype == DA_F32, has_e = d.epilogue == DA_EPI_AXPBY, fa = d.faithful != 0;
  const bool one = d.s1 == 1.f;   // rounding-faithful bf16 output: the exact multiplication by 1 is left out
#define DA_EPI(CF, HE, FA, S1) \
  epilogue_impl<C, SYM, FULL, CF, HE, FA, S1, 0, false, RSPLIT, CSPLIT>(acc, d, lds, b, mirror, m0, n0, wave, lane, wm, wn)
#define DA_EPI_UPD(FA, S1, U, WF) \
  epilogue_impl<C, false, FULL, false, true, FA, S1, U, WF, RSPLIT, CSPLIT>(acc, d, lds, b, false, m0, n0, wave, lane, wm, wn)
#define DA_EPI_UPD_FA(U, WF)                                                              \
  do {                                                                                    \
    if (fa) { if (one) DA_EPI_UPD(true, true, U, WF); else DA_EPI_UPD(true, false, U, WF); } \
    else DA_EPI_UPD(false, false, U, WF);                                                 \
  } while (0)
  if (!SYM && FULL && !cf32 && has_e && d.upd_tab) {
    // (the launcher only sets upd_tab where these conditions hold)
    const bool wf = d.upd_dtype == DA_F32;
    if (d.upd_transposed) { if (wf) DA_EPI_UPD_FA(2, true); else DA_EPI_UPD_FA(2, false); }
    else                  { if (wf) DA_EPI_UPD_FA(1, true); else DA_EPI_UPD_FA(1, false); }
    return;
  }
  if (!cf32) {
    if (has_e) {
      if (fa) { if (one) DA_EPI(false, true, true, true); else DA_EPI(false, true, true, false); }
      else DA_EPI(false, true, false, false);
    } else {
      if (fa) { if (one) DA_EPI(false, false, true, true); else DA_EPI(false, false, true, false); }
      else DA_EPI(false, false, false, false);
    }
  } else {
    if (has_e) { if (fa) DA_EPI(true, true, true, false); else DA_EPI(true, true, false, false); }
    else       { if (fa) DA_EPI(true, false, true, false); else DA_EPI(true, false, false, false); }
  }
#undef DA_EPI
#undef DA_EPI_UPD
#undef DA_EPI_UPD_FA
}


constexpr int DA_LOOP_CHECKED = 0, DA_LOOP_INTERIOR = 1, DA_LOOP_EDGE = 2;

__device__ __forceinline__ unsigned long long wave_uniform64(unsigned long long x) {
  return ((unsigned long long)(unsigned)wave_uniform((int)(x >> 32)) << 32) | (unsigned)wave_uniform((int)x);
}
template <int N> __device__ __forceinline__ void dma_wait_all_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// 16 bytes per lane from a raw buffer into LDS at `lbase` + `l` + 16 * lane (dma16, addressed by scalars: a request costs the wavefront
// three instructions).  From a buffer of no records nothing is fetched, the request is counted all the same.  The wait states between
// the vector unit's scalars and the request are the caller's (buffers_ready): five in every request, as in dma16, cost 2 to 4 % of a step
// of large products, one set of them a stage 0.3 %.  tests/test_wait_states.py looks for a scalar that the compiler moves in between.
__device__ __forceinline__ void dma16_buf(u32x4_t buf, unsigned off, unsigned soff, unsigned lbase, unsigned l) {
  asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(off), "s"(buf), "s"(soff), "s"(lbase), "s"(l)
               : "memory", "scc");
}

__device__ __forceinline__ void buffers_ready(u32x4_t& a, u32x4_t& b) { asm volatile("s_nop 4" : "+s"(a), "+s"(b)); }

// One product added to accumulators that stay in their AGPRs.  As assembly: the compiler, given 256 of them, moved some about on every
// pass of the loop (56 v_accvgpr_mov a stage with both operands k-contiguous, 3400 clocks instead of 2600).  It does not know the
// instruction's hazards then: no accumulator is touched again within four products, mfma_drain() comes before they are read, and no
// fragment is moved by the vector unit within two wait states of its product, which tests/test_wait_states.py holds the build to.
__device__ __forceinline__ void mfma16_in_place(f32x4_t& c, bf16x8_t col, bf16x8_t row) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(col), "v"(row));
}
// The accumulators' start: zeros times zeros.  Assembly as well, so that it stays behind the first stage's requests: as assignments the
// compiler had put 256 register moves, half a microsecond, in front of them where an operand is k-strided (a tile of 768 = 12 stages
// 19.9 -> 18.9 us in its K loop, of 384 42.9 -> 42.4 a launch; Newton-Schulz of 4096 x 14336 3425 -> 3398, GPT-small Muon 1575 -> 1563).
__device__ __forceinline__ void mfma16_clear(f32x4_t& c, u32x4_t zeros) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "=a"(c) : "v"(zeros));
}
__device__ __forceinline__ void mfma_drain() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// Addresses of one operand in gemm_tile_k_loop_quad.  The unit of a request is half an operand stage, what every wavefront reads in one
// phase: H rows of each of the two wavefronts along the operand.  In LDS a k-contiguous operand has the layout of read_frag16
// ([BT][64], the halves are blocks of its rows), a k-strided one two tiles [64][BT / 2], a unit each.
template <typename C, bool KS>
struct UnitAddr {
  static constexpr int H = C::BT / 4;
  static constexpr int NU = H / 16;                      // wave instructions (1024 bytes) of a wavefront per unit
  static constexpr int LHALF = KS ? H * 2 * BK * 2 : H * 128;
  unsigned long long base;                               // bytes; wave-uniform, as step and l
  unsigned step[2][NU], l[NU];                           // to the instructions' blocks, in memory (both units) and in LDS
  unsigned off[KS ? 2 : 1];                              // per lane
  __device__ __forceinline__ UnitAddr(const bf16_t* P, int ld, int row0, int dim, int lane, int wave) {
    const unsigned pitch = (unsigned)ld * 2u;
    if (!KS) {
      constexpr int HB = H / 8;                          // blocks of eight rows in a half
      const int r = lane >> 3;
      base = wave_uniform64(reinterpret_cast<unsigned long long>(P + (long long)row0 * ld));
      off[0] = (unsigned)r * pitch + (unsigned)kc_swizzle(lane & 7, (wave & 1) * 8 + r) * 16u;   // (a block's parity is the wavefront's)
#pragma unroll
      for (int e = 0; e < NU; ++e) {
        const int q = e * 4 + wave, blk = q / HB * (2 * HB) + q % HB;
        step[0][e] = (unsigned)wave_uniform((int)((unsigned)blk * 8u * pitch));
        step[1][e] = (unsigned)wave_uniform((int)((unsigned)(blk * 8 + H) * pitch));
        l[e] = (unsigned)blk * 1024u;
      }
    } else {
      constexpr int CPR = H / 4, RPB = 64 / CPR;         // chunks of a unit's k-row, k-rows of an instruction
      const int kr = lane / CPR, c = ks_swizzle(lane % CPR, kr) * 8;
      base = wave_uniform64(reinterpret_cast<unsigned long long>(P + row0));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int col = C::split(true, true) ? h * (2 * H) + c : c / H * (2 * H) + h * H + c % H;
        if (row0 + col > dim - 8) col = dim - 8 - row0;  // (StageAddr: an edge tile stays inside the matrix)
        off[h] = (unsigned)kr * pitch + (unsigned)col * 2u;
      }
#pragma unroll
      for (int e = 0; e < NU; ++e) {
        step[0][e] = step[1][e] = (unsigned)wave_uniform((int)((unsigned)((e * 4 + wave) * RPB) * pitch));
        l[e] = (unsigned)(e * 4 + wave) * 1024u;
      }
    }
  }
};
template <typename C, bool KS>
__device__ __forceinline__ bf16x8_t unit_frag(const char* op, int w, int h, int i, int ks, int lane) {
  constexpr int H = C::BT / 4;
  if (!KS) return read_frag16<C::BT, false>(op, w * (2 * H) + h * H + i * 16, ks, lane);
  return read_frag16<C::BT / 2, true>(op + h * UnitAddr<C, true>::LHALF, w * H + i * 16, ks, lane);
}

// The direct-to-LDS K loop of four wavefronts, a quarter of the tile each (of a 256-tile 128 x 128: 256 accumulators, in AGPRs).
// A wavefront's results are four quadrants; a 64-deep stage is four phases, a quadrant's products each:
//   phase            0              1              2                3
//   products         A0 B0          A0 B1          A1 B0            A1 B1          (A0, A1: halves of the wavefront's rows; B: of its columns)
//   LDS reads        B1             A1             A0 of the next   B0 of the next stage
//   requests         A0 of t + 2    B0 of t + 2    B1 of t + 2      A1 of t + 2    (into the buffer of stage t)
// Two barriers to a stage, behind phases 1 and 3: what the next two phases read has landed (four to six phases after its request; the
// wait leaves the 16 younger requests in flight) and what they request anew has been read.  Reads and requests stand singly between
// products, in a fixed order: with one wavefront to a SIMD nothing else covers them, and a product covers three instructions.  The loop
// has no branches: the two stages past the last one are requested from a buffer of no records.
// What bounds it: eight wavefronts of 128 x 64 read 192 KB a stage from LDS (128 bytes a clock) and the requests write 64 KB, 2048 clocks
// of the matrix cores' 2048; four of 128 x 128 read 128 KB.  Clocks per stage of a 256-tile on every CU, eight wavefronts -> four: both
// operands k-contiguous 2990 -> 2610, one k-strided 3130 -> 2640, both - -> 2690 (products and barriers alone 2180).  Under random data
// the chip lowers its clock as the loop gets denser (2.2 GHz for zeros, 1.7 here): 1.21-1.26 -> 1.32-1.39 PFLOP/s.
// `hook`, `a_wrap`, `b_jump`: gemm_tile_k_loop.
template <typename C, bool A_KS, bool B_KS, typename Hook>
__device__ __forceinline__ void gemm_tile_k_loop_quad(typename C::acc_t (&acc)[C::TMI][C::TNJ], const GemmDesc& d, const bf16_t* A,
                                                      const bf16_t* B, int dK, int m0, int n0, char* lds, int lane, int wave,
                                                      int wm, int wn, Hook hook, int a_wrap, unsigned b_jump) {
  static_assert(C::QUAD && (C::BT == 256 || C::BT == 128 || (C::BT == 192 && !A_KS && !B_KS)), "");
  constexpr int OP = C::BT * BK * 2, STAGE = 2 * OP;
  constexpr int HI = C::BT / 64;                         // 16-row blocks of a half
  constexpr int NR = 2 * HI, NU = UnitAddr<C, false>::NU;
  typedef UnitAddr<C, A_KS> UA;
  typedef UnitAddr<C, B_KS> UB;
  const int KT = wave_uniform(dK / BK);
  const unsigned wrap = (unsigned)wave_uniform(a_wrap < 0 ? d.a_kwrap : a_wrap) * 2u;
  const unsigned jump = (unsigned)wave_uniform((int)b_jump);
  const UA ua(A, d.lda, m0, d.M, lane, wave);
  const UB ub(B, d.ldb, n0, d.N, lane, wave);
  const unsigned long long a_stage = wave_uniform64(A_KS ? (unsigned long long)d.lda * (BK * 2) : BK * 2);
  const unsigned long long b_stage = wave_uniform64(B_KS ? (unsigned long long)d.ldb * (BK * 2) : BK * 2);
  const unsigned l0 = lds_addr(lds);
  unsigned long long pa = ua.base, pb = ub.base;         // the stage being requested
  unsigned in_turn = 0;
  u32x4_t ba, bb;
  // `more` >= 0: the stage exists.  (Left to the compiler the choice of the record count ends up on the vector unit.)
  auto set_buffers = [&](int more) {
    unsigned n;
    asm("s_cmp_ge_i32 %1, 0\n\ts_cselect_b32 %0, -1, 0" : "=s"(n) : "s"(more) : "scc");
    ba = u32x4_t{(unsigned)wave_uniform((int)pa), (unsigned)wave_uniform((int)(pa >> 32)), n, 0x00020000u};
    bb = u32x4_t{(unsigned)wave_uniform((int)pb), (unsigned)wave_uniform((int)(pb >> 32)), n, 0x00020000u};
  };
  auto load_a = [&](int h, int e, unsigned l) { dma16_buf(ba, ua.off[A_KS ? h : 0], ua.step[h][e], l + h * UA::LHALF, ua.l[e]); };
  auto load_b = [&](int h, int e, unsigned l) { dma16_buf(bb, ub.off[B_KS ? h : 0], ub.step[h][e], l + OP + h * UB::LHALF, ub.l[e]); };
  auto next_stage = [&](int more) {
    pa += a_stage;
    pb += b_stage;
    in_turn += BK * 2;
    if (in_turn == wrap) { pa = ua.base; in_turn = 0; pb += jump; }   // (0: never, in_turn > 0 here)
    set_buffers(more);
  };

  bf16x8_t a0[HI][2], a1[HI][2], b0[HI][2], b1[HI][2];
  // the products of quadrant (ah, bh), the NR reads and NU requests of the phase at fixed places between them
  auto phase = [&](auto ah, auto bh, bf16x8_t (&a)[HI][2], bf16x8_t (&b)[HI][2], auto read, auto request) {
    int n = 0;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < HI; ++i)
#pragma unroll
        for (int j = 0; j < HI; ++j) {
          constexpr int EVERY = HI == 4 ? 3 : HI == 3 ? 2 : 1;   // (early: the barrier waits for the last of them)
          if (n % EVERY == 0 && n / EVERY < NR) {
            read((n / EVERY) % HI, (n / EVERY) / HI);
            __builtin_amdgcn_sched_barrier(0);
          }
          const int e = HI == 4   ? (n == 1 ? 0 : n == 8 ? 1 : n == 16 ? 2 : n == 23 ? 3 : -1)
                        : HI == 3 ? (n == 1 ? 0 : n == 7 ? 1 : n == 13 ? 2 : -1)
                                  : (n == 4 ? 0 : n == 6 ? 1 : -1);
          if (e >= 0) {
            request(e);
            __builtin_amdgcn_sched_barrier(0);
          }
          mfma16_in_place(acc[decltype(ah)::value * HI + i][decltype(bh)::value * HI + j], b[j][ks], a[i][ks]);
          __builtin_amdgcn_sched_barrier(0);
          ++n;
        }
  };
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  set_buffers(0);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    buffers_ready(ba, bb);   // (in the loop a barrier, its waits and a product stand between the buffers and the first request)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int e = 0; e < NU; ++e) load_a(h, e, l0 + s * STAGE);
#pragma unroll
      for (int e = 0; e < NU; ++e) load_b(h, e, l0 + s * STAGE);
    }
    next_stage(KT - 2 - s);
  }
  __builtin_amdgcn_sched_barrier(0);   // (256 registers are cleared while the first stage is on its way)
  u32x4_t zeros = {0u, 0u, 0u, 0u};
  asm volatile("s_nop 1" : "+v"(zeros));
#pragma unroll
  for (int i = 0; i < C::TMI; ++i)
#pragma unroll
    for (int j = 0; j < C::TNJ; ++j) mfma16_clear(acc[i][j], zeros);
  __builtin_amdgcn_sched_barrier(0);
  dma_wait_all_but<6 * NU>();   // A0, B0
  meet();
  hook();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < HI; ++i) {
      a0[i][ks] = unit_frag<C, A_KS>(lds, wm, 0, i, ks, lane);
      b0[i][ks] = unit_frag<C, B_KS>(lds + OP, wn, 0, i, ks, lane);
    }
  dma_wait_all_but<4 * NU>();   // the rest of stage 0
  meet();
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  for (int left = KT - 1, buf = 0; left >= 0; --left, buf ^= STAGE) {   // (`left` stages follow this one)
    const char* const cur = lds + buf;
    const char* const nxt = lds + (buf ^ STAGE);
    const unsigned l = l0 + buf;
    phase(I0(), I0(), a0, b0, [&](int i, int ks) { b1[i][ks] = unit_frag<C, B_KS>(cur + OP, wn, 1, i, ks, lane); },
          [&](int e) { load_a(0, e, l); });
    phase(I0(), I1(), a0, b1, [&](int i, int ks) { a1[i][ks] = unit_frag<C, A_KS>(cur, wm, 1, i, ks, lane); },
          [&](int e) { load_b(0, e, l); });
    dma_wait_all_but<4 * NU>();
    meet();
    // (behind the last stage these reads return what lies in the other buffer, for no product)
    phase(I1(), I0(), a1, b0, [&](int i, int ks) { a0[i][ks] = unit_frag<C, A_KS>(nxt, wm, 0, i, ks, lane); },
          [&](int e) { load_b(1, e, l); });
    phase(I1(), I1(), a1, b1, [&](int i, int ks) { b0[i][ks] = unit_frag<C, B_KS>(nxt + OP, wn, 0, i, ks, lane); },
          [&](int e) { load_a(1, e, l); });
    next_stage(left - 3);
    dma_wait_all_but<4 * NU>();
    meet();
  }
  dma_wait();   // (requests of no records: what they leave in LDS comes before the epilogue's use of it)
  mfma_drain();
  meet();
}

// K loop of one BT x BT tile: acc += sum over dK elements of k of A-rows (m0 ...) x B-rows (n0 ...).  `A`, `B`: the
// matrix's operands at the first k of the sum.  Three forms (MODE):
//   DA_LOOP_INTERIOR: every tile is interior (M, N multiples of BT, K a multiple of 64): gemm_tile_k_loop_quad.  No
//     bounds checks anywhere.
//   DA_LOOP_EDGE: the same K loop for products whose ragged dimension belongs to a k-strided operand (its chunks
//     are kept inside the matrix) and whose other operand has whole tiles; the epilogue checks bounds.  Dion's
//     rank-r products at a rank that is not a multiple of the tile edge (r = 192).
//   DA_LOOP_CHECKED: bounds-checked 16-byte loads into registers (out-of-range chunks zero filled),
//     written to LDS after the stage's MFMAs.
// Ends with a workgroup barrier: the stage buffers are free for the epilogue.
// `after_first_stage` (direct-to-LDS forms) is called once, behind the loop's first barrier.  Every wavefront has waited there until no
// more than its youngest requests of this loop are outstanding (loads and stores count down in the order they were issued): whatever it
// issued before the loop, stores of earlier work included, has completed; most of the first two stages is still on its way.
// `a_wrap`, `b_jump` (direct-to-LDS forms): A is read again from its first column after a_wrap of its columns instead of
// GemmDesc::a_kwrap of them, and B then goes on b_jump bytes further.
struct DaNoHook { __device__ __forceinline__ void operator()() const {} };
template <typename C, bool A_KS, bool B_KS, int MODE, typename Hook = DaNoHook>
__device__ __forceinline__ void gemm_tile_k_loop(typename C::acc_t (&acc)[C::TMI][C::TNJ], const GemmDesc& d, const bf16_t* A,
                                                 const bf16_t* B, int dK, int m0, int n0, char* lds, int tid, int lane,
                                                 int wave, int wm, int wn, Hook after_first_stage = Hook(),
                                                 int a_wrap = -1, unsigned b_jump = 0) {
  constexpr bool FULL = MODE != DA_LOOP_CHECKED;   // the direct-to-LDS K loop
  static_assert(!FULL || C::QUAD, "");
  if constexpr (FULL) {
    gemm_tile_k_loop_quad<C, A_KS, B_KS>(acc, d, A, B, dK, m0, n0, lds, lane, wave, wm, wn, after_first_stage, a_wrap, b_jump);
    return;
  }
  constexpr int BT = C::BT, TMI = C::TMI, TNJ = C::TNJ, NCH = C::NCH;
  constexpr int A_BYTES = Tile<BT, A_KS>::bytes;
  constexpr int B_BYTES = Tile<BT, B_KS>::bytes;
  constexpr int STAGE = A_BYTES + B_BYTES;
#pragma unroll
  for (int i = 0; i < TMI; ++i)
#pragma unroll
    for (int j = 0; j < TNJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;

  StageAddr<C, A_KS> sa(A, d.lda, m0, tid, d.M);
  StageAddr<C, B_KS> sb(B, d.ldb, n0, tid, d.N);
  const int ar0 = wm * C::WROWS, br0 = wn * C::WCOLS;
  const int KT = (dK + BK - 1) / BK;
  // bounds-checked: a stage is two 32-deep k-steps of TMI row fragments (in two halves) and TNJ column fragments
  constexpr int TH = TMI / 2;
#define DA16_RA(FA, st, ks, h)                                                                     \
  do {                                                                                             \
    _Pragma("unroll") for (int i = 0; i < TH; ++i)                                                 \
        FA[i] = read_frag16<BT, A_KS>((st), ar0 + ((h) * TH + i) * 16, (ks), lane);                \
  } while (0)
#define DA16_RB(FB, st, ks)                                                                        \
  do {                                                                                             \
    _Pragma("unroll") for (int j = 0; j < TNJ; ++j)                                                \
        FB[j] = read_frag16<BT, B_KS>((st) + A_BYTES, br0 + j * 16, (ks), lane);                      \
  } while (0)
#define DA16_MMA(FA, FB, h)                                                                        \
  do {                                                                                             \
    _Pragma("unroll") for (int i = 0; i < TH; ++i)                                                 \
        _Pragma("unroll") for (int j = 0; j < TNJ; ++j)                                            \
            acc[(h) * TH + i][j] =                                                                 \
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(FB[j], FA[i], acc[(h) * TH + i][j], 0, 0, 0); \
  } while (0)
  u32x4_t ra[NCH], rb[NCH];
  constexpr int A_RSTEP = A_KS ? C::NT / (BT / 8) : C::NT / 8;
  constexpr int B_RSTEP = B_KS ? C::NT / (BT / 8) : C::NT / 8;
  auto gload = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int r_ = sa.row + i * A_RSTEP;
      const bool ok = A_KS ? (kt * BK + r_ < dK && m0 + sa.col < d.M) : (m0 + r_ < d.M && kt * BK + sa.col < dK);
      const u32x4_t z_ = {0u, 0u, 0u, 0u};
      ra[i] = ok ? *reinterpret_cast<const u32x4_t*>(sa.g + i * sa.gstep) : z_;
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int r_ = sb.row + i * B_RSTEP;
      const bool ok = B_KS ? (kt * BK + r_ < dK && n0 + sb.col < d.N) : (n0 + r_ < d.N && kt * BK + sb.col < dK);
      const u32x4_t z_ = {0u, 0u, 0u, 0u};
      rb[i] = ok ? *reinterpret_cast<const u32x4_t*>(sb.g + i * sb.gstep) : z_;
    }
    sa.g += sa.tstep;
    if (!A_KS && d.a_kwrap && ((kt + 1) * BK) % d.a_kwrap == 0) sa.g -= d.a_kwrap;   // A again from its first column
    sb.g += sb.tstep;
  };
  auto lstore = [&](char* st) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) *reinterpret_cast<u32x4_t*>(st + sa.l + i * sa.lstep) = ra[i];
#pragma unroll
    for (int i = 0; i < NCH; ++i) *reinterpret_cast<u32x4_t*>(st + A_BYTES + sb.l + i * sb.lstep) = rb[i];
  };
  bf16x8_t a0[TH], a1[TH], b0[TNJ];
  gload(0);
  lstore(lds);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    char* cur = lds + (kt & 1) * STAGE;
    char* nxt = lds + ((kt + 1) & 1) * STAGE;
    const bool more = kt + 1 < KT;
    if (more) gload(kt + 1);
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      DA16_RB(b0, cur, ks);
      DA16_RA(a0, cur, ks, 0);
      DA16_RA(a1, cur, ks, 1);
      DA16_MMA(a0, b0, 0);
      DA16_MMA(a1, b0, 1);
    }
    if (more) lstore(nxt);
    __syncthreads();
  }
#undef DA16_RA
#undef DA16_RB
#undef DA16_MMA
}

// K loop of one BT x BT tile whose row operand is the SUM of two bf16 matrices of the same layout, formed on the way
// into LDS:  acc += sum_k r_bf16(M + G)(m0 + i, k) * B(n0 + j, k).  The row operand goes through registers (16-byte
// loads of M and of G one stage ahead, eight additions with one rounding each, one 16-byte LDS store per chunk); the
// column operand is k-strided and staged with direct-to-LDS loads as in the DA_LOOP_EDGE form (its ragged dimension
// is kept inside the matrix).  `writeback`: the sums are also stored over M (each element by exactly one tile).
// `any` is or-ed with "some sum is not zero".  M: whole tiles of rows (no checks), dK a multiple of 64.
// Ends with a workgroup barrier; stores of the last stage may still be in flight.
template <typename C, bool A_KS>
__device__ __forceinline__ void gemm_tile_k_loop_sum(typename C::acc_t (&acc)[C::TMI][C::TNJ], const GemmDesc& d, bf16_t* M,
                                                     const bf16_t* G, const bf16_t* B, int dK, int m0, int n0,
                                                     char* lds, int tid, int lane, int wave, int wm, int wn,
                                                     bool writeback, bool& any) {
  constexpr bool B_KS = true;
  constexpr int BT = C::BT, TMI = C::TMI, TNJ = C::TNJ, NCH = C::NCH, NW = C::NT / 64;
  constexpr int A_BYTES = Tile<BT, A_KS>::bytes;
  constexpr int B_BYTES = Tile<BT, B_KS>::bytes;
  constexpr int STAGE = A_BYTES + B_BYTES;
  static_assert(NCH == 4, "the stage barrier's wait count below is written for four stores per stage");
#pragma unroll
  for (int i = 0; i < TMI; ++i)
#pragma unroll
    for (int j = 0; j < TNJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;

  StageAddr<C, A_KS> sa(M, d.lda, m0, tid, d.M);
  StageAddr<C, B_KS> sb(B, d.ldb, n0, tid, d.N);
  // the thread's chunks as 32-bit byte offsets from the matrix's first element (wave-uniform base + lane offset: the
  // launcher keeps the matrix below 4 GiB)
  const char* const Mc = reinterpret_cast<const char*>(M);
  const char* const Gc = reinterpret_cast<const char*>(G);
  const unsigned gs2 = (unsigned)(sa.gstep * 2), ts2 = (unsigned)(sa.tstep * 2);
  const int ar0 = wm * C::WROWS, br0 = wn * C::WCOLS;
  const int KT = dK / BK;
  bf16x8_t fa[TMI / 2], fb[TNJ];
  u32x4_t rm[NCH], rg[NCH];
  unsigned nz = 0u;
  unsigned koff_b = 0;
  unsigned aoff = (unsigned)((sa.g - M) * 2);   // chunk 0 of the stage being loaded

#define DA_SUM_LOAD()                                                                              \
  do {                                                                                             \
    _Pragma("unroll") for (int i = 0; i < NCH; ++i)                                                \
        rm[i] = ldg16(Mc + (size_t)(aoff + i * gs2));                                              \
    _Pragma("unroll") for (int i = 0; i < NCH; ++i)                                                \
        rg[i] = ldg16(Gc + (size_t)(aoff + i * gs2));                                              \
  } while (0)
#define DA_SUM_DMA(st)                                                                             \
  do {                                                                                             \
    _Pragma("unroll") for (int i = 0; i < NCH; ++i)                                                \
        dma16(sb.dbase, sb.doff + i * sb.dstep + koff_b, lds_addr(st) + A_BYTES + (i * NW + wave) * 1024); \
    koff_b += (unsigned)(sb.tstep * 2);                                                            \
  } while (0)
// (the stage loaded last: its chunks lie at aoff; the sums go to LDS and, with writeback, over M)
#define DA_SUM_STORE(st)                                                                           \
  do {                                                                                             \
    _Pragma("unroll") for (int i = 0; i < NCH; ++i) {                                              \
      u32x4_t o;                                                                                   \
      _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                              \
        const unsigned x = rm[i][q], y = rg[i][q];                                                 \
        o[q] = cvt_pk_bf16(lo_f(x) + lo_f(y), hi_f(x) + hi_f(y));                                  \
        nz |= o[q] & 0x7fff7fffu;                                                                  \
      }                                                                                            \
      *reinterpret_cast<u32x4_t*>((st) + sa.l + i * sa.lstep) = o;                                 \
      if (writeback) stg16(const_cast<char*>(Mc) + (size_t)(aoff + i * gs2), o);                   \
    }                                                                                              \
    aoff += ts2;                                                                                   \
  } while (0)
  // (fragments are not double buffered here: the registers hold a stage of M and of G instead, and the loop is
  // bound by the stream of M and G from HBM, not by the matrix cores)
  DA_SUM_LOAD();
  DA_SUM_DMA(lds);
  DA_SUM_STORE(lds);
  dma_wait();
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    char* cur = lds + (kt & 1) * STAGE;
    char* nxt = lds + ((kt + 1) & 1) * STAGE;
    const bool more = kt + 1 < KT;
    if (more) {
      DA_SUM_LOAD();
      DA_SUM_DMA(nxt);
    }
    // (the row fragments of a 32-deep k-step in two halves through the same registers)
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
#pragma unroll
      for (int j = 0; j < TNJ; ++j) fb[j] = read_frag16<BT, B_KS>(cur + A_BYTES, br0 + j * 16, ks, lane);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < TMI / 2; ++i) fa[i] = read_frag16<BT, A_KS>(cur, ar0 + (h * (TMI / 2) + i) * 16, ks, lane);
#pragma unroll
        for (int i = 0; i < TMI / 2; ++i)
#pragma unroll
          for (int j = 0; j < TNJ; ++j) acc[h * (TMI / 2) + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[h * (TMI / 2) + i][j], 0, 0, 0);
      }
    }
    if (more) DA_SUM_STORE(nxt);
    // the direct-to-LDS loads of the next stage must have landed; the (up to four) stores issued behind them may
    // stay in flight: memory operations of a wavefront complete in the order issued
    if (writeback) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else dma_wait();
    __syncthreads();
  }
  any = any || nz != 0u;
#undef DA_SUM_LOAD
#undef DA_SUM_DMA
#undef DA_SUM_STORE
}

}  // namespace
