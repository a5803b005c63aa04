// Newton-Schulz quintic as a chain of batched gfx950 MFMA GEMM stages.
//
// One Newton-Schulz iteration over a stack of N blocks X (m x n, m <= n):
//   SYRK : A = s^2 * X X^T                      (m x m, symmetric, K = n)
//   POLY : P = a I + b A + c A A                (m x m, symmetric, K = m)
//   PX   : X' = s * P X                         (m x n, K = m)
//   PX_APPLY (last iteration): param += alpha * bf16(X') written straight into
//          the parameter blocks, un-transposed for tall blocks.
//   SYMM : C = S1 S2 of two symmetric stacks that commute (the Gram form of the
//          rectangular groups: iterations on m x m polynomials of X0 X0^T; the
//          launch plans are built in abi.hip)
// s = 1/(||X0||_F + 1e-7) on the first iteration (the Frobenius normalisation
// folded into the products: (sX)(sX)^T = s^2 XX^T and P(sX) = s PX), 1
// afterwards.  The a X term of the quintic is carried by P's diagonal: POLY adds
// a to its fp32 diagonal before the one bf16 rounding of P (the reference rounds
// a X to bf16 in the same way), so PX is a plain product.
//
// bf16 kernels: v_mfma_f32_32x32x16_bf16, fp32 accumulation, bf16 stage outputs.
// One 512-thread workgroup (8 waves, 2 per SIMD) per CU computes 256 x 256
// output tiles, each wave a 128 x 64 sub-tile (4 x 2 MFMA tiles, 128
// accumulators).  K advances 32 at a time through a 4-slot LDS ring filled by
// direct global->LDS loads (global_load_lds_dwordx4), two slices in flight
// behind the one being read; the loads of a step are interleaved with its
// MFMAs.  The workgroups are persistent and walk the tiles in rounds, all tiles
// of one block on one XCD.  Every bf16 stack is stored in 32-column panels
// (panel_off), so a K slice is one contiguous run in HBM.  The symmetric A and
// P stacks hold only their tiles on and above the diagonal: SYRK and POLY
// compute and store just those, and their consumers read the missing part as
// the transpose of the stored part (ds_read_b64_tr_b16), as PX reads X.
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "kernels.hpp"
#include "mfma_tile.hpp"

namespace mmuon {
namespace {

// Tiles of a symmetric m x m product: BM-row band ti, BN-column band tc with
// tc >= R ti, R = BM / BN (the upper triangle and the diagonal blocks), ti-major.
constexpr int R_SYM = BM / BN;
// 256-wide tiles over an extent (a multiple of 64), the last one possibly partial
__host__ __device__ __forceinline__ int tiles_of(int extent) { return (extent + BM - 1) / BM; }
__device__ __forceinline__ void sym_tile(int t, int nc, int& ti, int& tc) {
  int i = 0;
  while (t >= nc - R_SYM * i) {
    t -= nc - R_SYM * i;
    ++i;
  }
  ti = i;
  tc = R_SYM * i + t;
}

// ---------------------------------------------------------------------------
// The pipelined main loop shared by every stage.  Each operand slice (256
// operand rows x 32 k) is read in one of two forms:
//   K: K-major, rows of the operand itself (one contiguous 16 KiB run of a panel);
//   T: transposed, 32 rows of the 8 panels whose columns are the operand's rows
//      (2 KiB runs), read with ds_read_b64_tr_b16.
// The X operand of PX is always T.  Gram and polynomial stacks store only the
// tiles on and above the diagonal, so an operand band R of them is T for the
// K slices left of its diagonal block (from the stored tile (kb, R)) and K from
// there on.  A slice pair (row operand, column operand) is KK, KT or TT.
// ---------------------------------------------------------------------------
// Identity term folded into the accumulation: IDENT_COL adds v A (A: the row
// operand) over the K slices that cross the tile's diagonal columns.  The
// values are taken from the slice in LDS and enter the fp32 accumulators by
// FMA (Pipe::ident_add).
enum { IDENT_NONE = 0, IDENT_COL = 2 };

enum { OP_K = 0, OP_T = 1, OP_SPLIT = 2 };  // operand form over K: always K, always T, T then K
enum { M_KK = 0, M_KT = 1, M_TT = 2 };        // forms of one slice pair (row, column)
constexpr bool row_t(int m) { return m == M_TT; }
constexpr bool col_t(int m) { return m != M_KK; }

// MASK: the wave's 32x32 MFMA tiles (bit i*TMJ + j) that are computed; the
// others, and the fragment reads only they need, are left out.
// SHARED: the row and column operands are the same rows (a diagonal tile of a
// symmetric product): only the row-operand slice is loaded, and the column
// fragments are read from it.
template <int RK, int CK, int IDENT, int MASK = 0xFF, bool SHARED = false>
struct Pipe {
  static_assert(RDMA == 2 && CDMA == 2, "two direct loads per thread and operand slice");
  static constexpr int DMA = SHARED ? RDMA : SLICE_DMA;  // direct loads per thread and slice
  static constexpr bool tile_on(int i, int j) { return (MASK >> (i * TMJ + j)) & 1; }
  // fragment read G (column fragments first, then row fragments) feeds a computed tile
  static constexpr bool frag_on(int G) {
    bool on = false;
    if (G < TMJ) {
      for (int i = 0; i < TMI; ++i) on = on || tile_on(i, G);
    } else {
      for (int j = 0; j < TMJ; ++j) on = on || tile_on(G - TMJ, j);
    }
    return on;
  }
  static_assert(RK != OP_T && (RK == OP_K || CK != OP_K), "row T only where the column is T");
  // the last run of slices: column T throughout (PX), else both K
  static constexpr int ML = CK == OP_T ? M_KT : M_KK;
  const uint16_t* rsrc_k;  // row operand K form: panel 0 at the operand's first row
  const uint16_t* rsrc_t;  // row operand T form: row 0 of the first panel holding its rows
  const uint16_t* csrc_k;
  const uint16_t* csrc_t;
  int thr_r, thr_c;        // OP_SPLIT: slices kt < thr are T
  uint32_t pstride_b;      // bytes per panel (rows * 32 * 2; a block is below 2^31 bytes)
  // this wave's loads, byte offsets within a slice's source: K form, its two 16-row
  // chunks; T form, its panel.  Beyond the stack's extent (a partial tile) the last
  // chunk or panel is loaded again; it feeds outputs that are not stored.
  uint32_t rk[2], ck[2], rt, ct;
  int KT;
  int wave, lane, wm, wn;
  uint16_t* lds;  // ring slot s at lds + s*SLOT: row-operand slice, then column-operand slice
  uint32_t lds0;  // LDS byte address of lds
  uint32_t k_loff;                // per-lane direct-load byte offset of the K form (T form: 16 * lane)
  uint32_t kfrag[BK / 16];        // per-lane K-form fragment bases
  uint32_t tfrag_r, tfrag_c;      // per-lane T-form fragment bases of the wave's first row / column tile
  int diag0;                      // K index of this wave's first identity column
  float id_v;                     // identity scalar

  __device__ __forceinline__ uint16_t* rslot(int kt) const { return lds + (uint32_t(kt) % NSTAGE) * SLOT; }

  __device__ __forceinline__ bool row_is_t(int kt) const { return RK == OP_SPLIT && kt < thr_r; }
  __device__ __forceinline__ bool col_is_t(int kt) const {
    return CK == OP_T || (CK == OP_SPLIT && kt < thr_c);
  }

  // Direct load Q (0, 1: row operand; 2, 3: column operand) of slice src_kt into
  // the ring slot of slice slot_kt (the same slice, except for the harmless
  // refill of a consumed slot at the end of the loop).  K form: wave w, load q
  // covers operand rows 16 (2w + q) .. +15 of the panel (1 KiB); T form: panel
  // w of the operand, k rows 16q .. 16q+15 of the slice (1 KiB).  Either way the
  // load lands at byte (2w + q) * 1024 of the operand's slice.
  // RF >= 0: the slice pair is in form RF (known when the slice lies in the same
  // run as the step that loads it); RF < 0: decided from the slice index.
  template <int Q, int RF = -1>
  __device__ __forceinline__ void issue_one(int src_kt, int slot_kt) const {
    constexpr int q = Q & 1;
    const uint32_t dst =
        lds0 + (uint32_t(slot_kt) % NSTAGE) * SLOT * 2 + (Q < 2 ? 0 : RSLICE * 2) + (2 * wave + q) * 1024;
    bool t;
    if constexpr (RF >= 0) t = Q < 2 ? row_t(RF) : col_t(RF);
    else t = Q < 2 ? row_is_t(src_kt) : col_is_t(src_kt);
    const uint16_t* srck = Q < 2 ? rsrc_k : csrc_k;
    const uint16_t* srct = Q < 2 ? rsrc_t : csrc_t;
    // 32-bit byte offsets from the operand's base
    const uint32_t ks = uint32_t(src_kt);
    if (t)
      dma16(reinterpret_cast<const char*>(srct) + (ks * (BK * PANEL * 2) + (Q < 2 ? rt : ct) + q * 16 * PANEL * 2),
            uint32_t(lane) << 4, dst);
    else
      dma16(reinterpret_cast<const char*>(srck) + (ks * pstride_b + (Q < 2 ? rk[q] : ck[q])), k_loff, dst);
  }
  __device__ __forceinline__ void issue(int src_kt, int slot_kt) const {
    issue_one<0>(src_kt, slot_kt);
    issue_one<1>(src_kt, slot_kt);
    if constexpr (!SHARED) {
      issue_one<2>(src_kt, slot_kt);
      issue_one<3>(src_kt, slot_kt);
    }
  }

  // Fragment read G (column fragments first, then row fragments) of k step KK
  // of slice kt in slice-pair form M.
  template <int KK, int G, int M>
  __device__ __forceinline__ void load_one(int kt, Frags& f) const {
    const uint16_t* sr = rslot(kt);
    const uint16_t* sc = SHARED ? sr : sr + RSLICE;
    if constexpr (G < TMJ)
      f.c[G] = col_t(M) ? frag_rowmajor_tr(sc, tfrag_c + G * 2048, KK) : frag_kmajor(sc, kfrag[KK], wn * WN + G * 32);
    else
      f.r[G - TMJ] = row_t(M) ? frag_rowmajor_tr(sr, tfrag_r + (G - TMJ) * 2048, KK)
                              : frag_kmajor(sr, kfrag[KK], wm * WM + (G - TMJ) * 32);
  }
  template <int KK, int M>
  __device__ __forceinline__ void load(int kt, Frags& f) const {
    if constexpr (frag_on(0)) load_one<KK, 0, M>(kt, f);
    if constexpr (frag_on(1)) load_one<KK, 1, M>(kt, f);
    if constexpr (frag_on(2)) load_one<KK, 2, M>(kt, f);
    if constexpr (frag_on(3)) load_one<KK, 3, M>(kt, f);
    if constexpr (frag_on(4)) load_one<KK, 4, M>(kt, f);
    if constexpr (frag_on(5)) load_one<KK, 5, M>(kt, f);
  }

  // Identity term of slice kt, which crosses this wave's identity at tile F:
  // acc[i][F] += v A[r][k], k = the accumulator column, from the A slice in K
  // form (byte r*64 + ((k/8) ^ ((r/4)%4))*16 + (k%8)*2, the same chunk order
  // for the four rows r of a read).  The accumulator of a 32 x 32 tile holds,
  // in lane l, column l%32 and rows 8q + 4(l/32) + e (value 4q + e);
  // ds_read_b64_tr_b16 gives lane l of a 16-lane group the four values of one
  // column in four consecutive rows, so one read per q delivers the lane's
  // four rows.
  template <int F, int I0 = 0, int I1 = TMI>
  __device__ __forceinline__ void ident_add(int kt, f32x16 (&acc)[TMI][TMJ]) const {
    static_assert(IDENT == IDENT_COL, "the column identity is the only one");
    const int l16 = lane & 15, g = lane >> 4;
    const int k16 = 16 * (g & 1) + 4 * (l16 & 3);  // first column of the lane's 8-byte chunk
    // The read of rows rb = wm WM + 32 i + 8 q + 4 (g/2) + l16/4 sits at
    // base + (32 i + 8 q) 64 + ((k16/8) ^ ((rb/4) % 4)) 16, and (rb/4) % 4 =
    // (2 q + g/2) % 4 only depends on q's parity: two per-lane bases, the rest
    // an immediate offset of the read.
    const int rlane = wm * WM + 4 * (g >> 1) + (l16 >> 2);
    const uint32_t base = uint32_t(rlane * 64 + (k16 & 7) * 2);
    const uint32_t b0 = base + uint32_t(((k16 >> 3) ^ ((g >> 1) & 3)) << 4);
    const uint32_t b1 = base + uint32_t(((k16 >> 3) ^ ((2 + (g >> 1)) & 3)) << 4);
    {
      const char* sr = reinterpret_cast<const char*>(rslot(kt));
#pragma unroll
      for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (!tile_on(i, F)) continue;
          const uint32_t off = ((q & 1) ? b1 : b0) + uint32_t((32 * i + 8 * q) * 64);
          const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(sr + off));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][F][4 * q + e] = fmaf(id_v, bf2f(uint16_t(v[e])), acc[i][F][4 * q + e]);
        }
    }
  }

  // Step kt: slice kt is consumed in form M, slice kt+1 (its k step 0 fragments)
  // is read in form MN, and slice kt+NSTAGE-1 is loaded in form RF (RF < 0:
  // decided from its index).  Fragments ping-pong at half-slice granularity: the k
  // step 1 reads of slice kt go out one per MFMA of its k step 0, and (after
  // the slice-kt+1 barrier) the k step 0 reads of slice kt+1 one per MFMA of
  // the k step 1.  At the barrier of step kt every wave has consumed slice
  // kt-1, so its slot takes slice kt+NSTAGE-1; those direct loads are
  // interleaved one by one with the k step 1 MFMAs as well.  F >= 0: the
  // slice crosses this wave's identity at tile F (ident_add).
  template <int M, int MN, int F, int RF = -1, int G = -1>
  __device__ __forceinline__ void body(int kt, Frags& fa, Frags& fb, f32x16 (&acc)[TMI][TMJ]) const {
    static_assert(TMI * TMJ == 8 && SLICE_DMA <= 8 && TMI + TMJ <= 8, "one read / direct load per MFMA");
#define MMUON_MFMA(f, g)                                                                          \
    if constexpr (tile_on((g) / TMJ, (g) % TMJ))                                                  \
      acc[(g) / TMJ][(g) % TMJ] = mfma(f.r[(g) / TMJ], f.c[(g) % TMJ], acc[(g) / TMJ][(g) % TMJ]);
#define MMUON_STEP0(g)                                                           \
    MMUON_MFMA(fa, g)                                                            \
    if constexpr ((g) < TMI + TMJ && frag_on(g)) load_one<1, (g), M>(kt, fb);    \
    __builtin_amdgcn_sched_barrier(0);
    MMUON_STEP0(0) MMUON_STEP0(1) MMUON_STEP0(2) MMUON_STEP0(3)
    MMUON_STEP0(4) MMUON_STEP0(5) MMUON_STEP0(6) MMUON_STEP0(7)
#undef MMUON_STEP0
    // G >= 0: the second half of the identity term of slice kt-1 (tile G), whose
    // slot is refilled only after this step's barrier
    if constexpr (G >= 0) ident_add<G, TMI / 2, TMI>(kt - 1, acc);
    wait_vm<(NSTAGE - 3) * DMA>();  // slice kt+1; the later ones may stay in flight
    barrier();
    // on the last step slice kt+1 does not exist and the reads of its slot go
    // unused; near the end a consumed slot is refilled with slice KT-1 so every
    // step has the same shape
    const int src = kt + NSTAGE - 1 < KT ? kt + NSTAGE - 1 : KT - 1;
    const int slot = kt + NSTAGE - 1;
#define MMUON_STEP1(g)                                                               \
    MMUON_MFMA(fb, g)                                                                \
    if constexpr ((g) < TMI + TMJ && frag_on(g)) load_one<0, (g), MN>(kt + 1, fa);   \
    if constexpr ((g) < DMA) issue_one<(g), RF>(src, slot);                          \
    __builtin_amdgcn_sched_barrier(0);
    // Raised wave priority from the barrier to the end of k step 1: a wave
    // still in this phase (reads of slice kt+1, direct loads) wins issue over
    // the SIMD's other wave once that one has moved on to the next step's
    // k step 0, so the wave behind catches up before the next barrier
    // (measured: Newton-Schulz 1-2% faster on the 6.89B groups).
    __builtin_amdgcn_s_setprio(1);
    MMUON_STEP1(0) MMUON_STEP1(1) MMUON_STEP1(2) MMUON_STEP1(3)
    MMUON_STEP1(4) MMUON_STEP1(5) MMUON_STEP1(6) MMUON_STEP1(7)
#undef MMUON_STEP1
#undef MMUON_MFMA
    __builtin_amdgcn_s_setprio(0);
    // the first half of slice kt's identity term (the slot of slice kt is
    // refilled only after the next barrier)
    if constexpr (F >= 0) ident_add<F, 0, TMI / 2>(kt, acc);
  }

  // Slices a .. b-1 in form M (b > a), the last of them reading slice b in form
  // MN.  Runs start and end at multiples of BM / BK = 8 slices, so the slices the
  // last NSTAGE - 1 steps load lie in the next run (form MN) and every load's
  // form is known at compile time.
  static_assert(BM / BK >= NSTAGE - 1, "a run is longer than the loads in flight");
  template <int M, int MN>
  __device__ __forceinline__ void run_span(int a, int b, Frags& fa, Frags& fb, f32x16 (&acc)[TMI][TMJ]) const {
    int kt = a;
    for (; kt < b - (NSTAGE - 1); ++kt) body<M, M, -1, M>(kt, fa, fb, acc);
    for (; kt < b - 1; ++kt) body<M, M, -1, MN>(kt, fa, fb, acc);
    body<M, MN, -1, MN>(b - 1, fa, fb, acc);
  }

  __device__ __forceinline__ void run(f32x16 (&acc)[TMI][TMJ]) const {
#pragma unroll
    for (int i = 0; i < TMI; ++i)
#pragma unroll
      for (int j = 0; j < TMJ; ++j) acc[i][j] = f32x16{};
    // slice runs: TT [0, t1), KT [t1, t2), then ML to the end
    const int t1 = RK == OP_SPLIT ? thr_r : 0;
    const int t2 = CK == OP_SPLIT ? thr_c : (CK == OP_T ? t1 : 0);
    // slices 0 .. NSTAGE-2 (beyond the last slice: refills with slice KT-1)
#pragma unroll
    for (int q = 0; q < NSTAGE - 1; ++q) issue(q < KT ? q : KT - 1, q);
    wait_vm<(NSTAGE - 2) * DMA>();  // slice 0 visible, the others may stay in flight
    barrier();
    Frags fa, fb;
    if (t1 > 0) load<0, M_TT>(0, fa);
    else if (CK == OP_SPLIT && t2 > 0) load<0, M_KT>(0, fa);
    else load<0, ML>(0, fa);
    if constexpr (RK == OP_SPLIT) {
      if (t1 > 0) {
        if (CK == OP_SPLIT && t2 == t1) run_span<M_TT, M_KK>(0, t1, fa, fb, acc);
        else run_span<M_TT, M_KT>(0, t1, fa, fb, acc);
      }
    }
    if constexpr (CK == OP_SPLIT) {
      if (t2 > t1) run_span<M_KT, M_KK>(t1, t2, fa, fb, acc);
    }
    // the last run (every remaining slice in form ML), with the identity steps
    const int k0 = t2;
    // every slice this run loads is in form ML
    if constexpr (IDENT == IDENT_NONE) {
      for (int kt = k0; kt < KT; ++kt) body<ML, ML, -1, ML>(kt, fa, fb, acc);
    } else {
      // the slices starting at diag0 cross this wave's identity tiles in
      // order (diag0 is a multiple of the wave's extent along K and lies in
      // the last run)
      static_assert(TMJ == 2, "a wave's identity columns span two slices");
      const int kd = diag0 / BK;
      for (int kt = k0; kt < kd; ++kt) body<ML, ML, -1, ML>(kt, fa, fb, acc);
      body<ML, ML, 0, ML>(kd, fa, fb, acc);
      body<ML, ML, 1, ML, 0>(kd + 1, fa, fb, acc);
      if (kd + TMJ < KT) {
        body<ML, ML, -1, ML, 1>(kd + TMJ, fa, fb, acc);
        for (int kt = kd + TMJ + 1; kt < KT; ++kt) body<ML, ML, -1, ML>(kt, fa, fb, acc);
      } else {
        // the last slice crossed the identity; the final refills go to other slots
        ident_add<1, TMI / 2, TMI>(KT - 1, acc);
      }
    }
    wait_vm<0>();  // the refills of the last two steps land before the ring is reused
  }
};

// Wave plan of a diagonal tile of a symmetric product.  Only its 36 32 x 32
// MFMA tiles on or above the diagonal (R <= C, units of 32 rows / columns) are
// computed; they are dealt to the 8 waves so that the two waves of every SIMD
// (waves w and w + 4) hold 9 between them, against 16 per SIMD in a full tile.
// Wave w computes, inside the 128 x 64 window (vwm, vwn) of the regular wave
// grid (rows 128 vwm.., columns 64 vwn..), the 32 x 32 tiles of its mask
// (bit i * TMJ + j: window tile row i, column j):
//   w0 (0,2) all 8      w4 (0,1) tile (3,1) = (R 3, C 3)
//   w1 (0,3) all 8      w5 (1,3) tile (3,1) = (R 7, C 7)
//   w2 (0,0) j >= i: 3  w6 (0,1) rows 0-2: 6
//   w3 (1,2) j >= i: 3  w7 (1,3) rows 0-2: 6
// Every tile on or above the diagonal is computed by exactly one wave and no
// tile below it by any; the staging fills those from their transposes.
constexpr int mask_upper() {
  int m = 0;
  for (int i = 0; i < TMI; ++i)
    for (int j = 0; j < TMJ; ++j)
      if (j >= i) m |= 1 << (i * TMJ + j);
  return m;
}
constexpr int MASK_FULL = 0xFF;
constexpr int MASK_UPPER = mask_upper();        // (0,0), (0,1), (1,1)
constexpr int MASK_LAST = 1 << (3 * TMJ + 1);   // (3,1)
constexpr int MASK_FIRST6 = (1 << (3 * TMJ)) - 1;  // rows 0-2
static_assert(TMI == 4 && TMJ == 2 && BM == 8 * 32 && WM == 4 * 32 && WN == 2 * 32,
              "the plan deals the 8 x 8 grid of 32 x 32 tiles of a 256 x 256 tile");

struct WavePlan {
  int vwm, vwn, mask;
};
__device__ __forceinline__ WavePlan diag_plan(int wave) {
  switch (wave) {
    case 0: return {0, 2, MASK_FULL};
    case 1: return {0, 3, MASK_FULL};
    case 2: return {0, 0, MASK_UPPER};
    case 3: return {1, 2, MASK_UPPER};
    case 4: return {0, 1, MASK_LAST};
    case 5: return {1, 3, MASK_LAST};
    case 6: return {0, 1, MASK_FIRST6};
    default: return {1, 3, MASK_FIRST6};
  }
}
// Full tile: the 2 x 4 grid of 128 x 64 windows, the two waves of one column
// window (wave 2 wn and 2 wn + 1) on different SIMDs (a SIMD runs waves w and
// w + 4): a K slice that crosses a window's identity columns (POLY) then
// gives each SIMD one wave of identity work beside its other wave's MFMAs,
// instead of both of one SIMD's waves while the others wait at the barrier.
// A tile with at most 128 valid rows keeps only its upper windows busy: there the
// four busy waves go to four SIMDs instead of two.
__device__ __forceinline__ WavePlan full_plan(int wave, int rows) {
  return rows > WM ? WavePlan{wave & 1, wave >> 1, MASK_FULL} : WavePlan{wave >> 2, wave & 3, MASK_FULL};
}

template <int RK, int CK, int IDENT, int MASK, bool SHARED>
__device__ __forceinline__ void mainloop_run(const uint16_t* rsrc_k, const uint16_t* rsrc_t, int thr_r,
                                             const uint16_t* csrc_k, const uint16_t* csrc_t, int thr_c,
                                             int64_t pstride, int KT, uint16_t* lds, f32x16 (&acc)[TMI][TMJ],
                                             int rows, int cols, float ident_v, int diag, int vwm, int vwn) {
  Pipe<RK, CK, IDENT, MASK, SHARED> p;
  p.rsrc_k = rsrc_k;
  p.rsrc_t = rsrc_t;
  p.csrc_k = csrc_k;
  p.csrc_t = csrc_t;
  p.thr_r = thr_r;
  p.thr_c = thr_c;
  p.pstride_b = uint32_t(pstride) * 2;
  p.KT = KT;
  p.lane = threadIdx.x & 63;
  p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // its share of the direct loads
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int u = 2 * p.wave + q;
    p.rk[q] = uint32_t(rows >= BM ? u : min(u, rows / 16 - 1)) * (16 * PANEL * 2);
    p.ck[q] = uint32_t(cols >= BN ? u : min(u, cols / 16 - 1)) * (16 * PANEL * 2);
  }
  p.rt = uint32_t(rows >= BM ? p.wave : min(p.wave, rows / PANEL - 1)) * p.pstride_b;
  p.ct = uint32_t(cols >= BN ? p.wave : min(p.wave, cols / PANEL - 1)) * p.pstride_b;
  p.wm = vwm;                                                 // its window of the output tile
  p.wn = vwn;
  p.lds = lds;
  p.lds0 = lds_addr(lds);
  p.k_loff = kmajor_lane_offset(p.lane);
#pragma unroll
  for (int kk = 0; kk < BK / 16; ++kk) p.kfrag[kk] = kmajor_frag_base(kk, p.lane);
  p.tfrag_r = rowmajor_frag_base(p.wm * TMI, p.lane);
  p.tfrag_c = rowmajor_frag_base(p.wn * TMJ, p.lane);
  p.diag0 = diag + p.wn * WN;
  p.id_v = ident_v;
  p.run(acc);
}

// Operand sources: *_k the K form (panel 0 at the operand's first row), *_t the
// T form (row 0 of the first panel holding the operand's rows); thr_*: slices
// kt < thr are T (OP_SPLIT); pstride: elements per panel.  ident_v: the identity
// scalar; diag: K index of the tile's first column (IDENT_COL).
// sym_diag (workgroup-uniform): a diagonal tile of a symmetric product, whose
// work is dealt by diag_plan; SHARE: its row and column operands are the same
// rows (SYRK, POLY: loaded once, Pipe SHARED), else two stacks' bands of the
// same rows (SYMM).  rows, cols: rows of the two operands that the stack holds
// from the tile's first on (a multiple of 32; at most the tile's matter).  mv, nv:
// those that are not padding; a wave whose window lies beyond them (as every window
// whose identity columns lie beyond K does) issues its share of the direct loads and
// leaves its accumulators zero (EDGE: there may be such windows).
template <int RK, int CK, bool EDGE, int IDENT = IDENT_NONE, bool SHARE = true>
__device__ __forceinline__ void mainloop(const uint16_t* rsrc_k, const uint16_t* rsrc_t, int thr_r,
                                         const uint16_t* csrc_k, const uint16_t* csrc_t, int thr_c,
                                         int64_t pstride, int KT, uint16_t* lds, f32x16 (&acc)[TMI][TMJ],
                                         int rows, int cols, int mv, int nv, float ident_v = 0.f, int diag = 0,
                                         bool sym_diag = false) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WavePlan plan = sym_diag ? diag_plan(wave) : full_plan(wave, mv);
  const bool idle = EDGE && (plan.vwm * WM >= mv || plan.vwn * WN >= nv);
#define MMUON_RUN(MASK, SH)                                                                                  \
  mainloop_run<RK, CK, (MASK) != 0 ? IDENT : IDENT_NONE, MASK, SH>(rsrc_k, rsrc_t, thr_r, csrc_k, csrc_t, thr_c, \
                                                                   pstride, KT, lds, acc, rows, cols, ident_v, diag, \
                                                                   plan.vwm, plan.vwn)
  if constexpr (EDGE) {
    if (idle) {
      if (sym_diag) MMUON_RUN(0, SHARE);
      else MMUON_RUN(0, false);
      return;
    }
  }
  if (!sym_diag) MMUON_RUN(MASK_FULL, false);
  else if (plan.mask == MASK_FULL) MMUON_RUN(MASK_FULL, SHARE);
  else if (plan.mask == MASK_UPPER) MMUON_RUN(MASK_UPPER, SHARE);
  else if (plan.mask == MASK_LAST) MMUON_RUN(MASK_LAST, SHARE);
  else MMUON_RUN(MASK_FIRST6, SHARE);
#undef MMUON_RUN
}

// D[i][j] accumulators of this wave -> T[j][i] in the staging area, each value
// scaled by f before the bf16 rounding.  Lane geometry: the lane holds column
// j = 64 wn + 32 tj + lane%32 and rows i = 128 wm + 32 ti + 8 qg + 4 (lane/32) + e,
// (wm, wn) the wave's window.  diag: a diagonal tile of a symmetric product
// computed by diag_plan; every computed tile above the diagonal also fills its
// mirror below it, T[i][j] = D[i][j] (copied from the staged tile), and so does
// the upper triangle of each 32 x 32 tile on the diagonal (written after, and
// so replacing, the values the lane pairs computed below it: equal bits when
// both operands are one symmetric matrix, rounding-level apart for SYMM's two
// commuting ones); its diagonal entries i = j < dlim get dadd added (in fp32,
// before the rounding).
__device__ __forceinline__ void stage_tile(char* stage, const f32x16 (&acc)[TMI][TMJ], float f, int mv,
                                           bool diag = false, float dadd = 0.f, int dlim = 0) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const WavePlan plan = diag ? diag_plan(wave) : full_plan(wave, mv);
  const int wm = plan.vwm, wn = plan.vwn;
#pragma unroll
  for (int i = 0; i < TMI; ++i) {
#pragma unroll
    for (int j = 0; j < TMJ; ++j) {
      const int R = wm * (WM / 32) + i, C = wn * (WN / 32) + j;
      if (!((plan.mask >> (i * TMJ + j)) & 1)) continue;
#pragma unroll
      for (int qg = 0; qg < 4; ++qg) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f * acc[i][j][qg * 4 + e];
        if (diag && R == C) {
          // the 32 x 32 tile on the diagonal: lane l holds entry (l%32, l%32)
          // at qg = (l%32)/8, e = l%8 - 4 (l/32) when that lies in [0, 4)
          const int d = lane & 31, e = (d & 7) - 4 * (lane >> 5);
          if ((d >> 3) == qg && e >= 0 && e < 4 && 32 * R + d < dlim) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
              if (x == e) v[x] += dadd;
          }
        }
        const int row = wn * WN + j * 32 + (lane & 31);
        const int col = wm * WM + i * 32 + qg * 8 + (lane >> 5) * 4;
        *reinterpret_cast<uint2*>(stage + tile_off(row, col)) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
      }
      if (diag && C == R) {
        // a 32 x 32 tile on the diagonal: its upper triangle replaces the
        // values just staged below it
#pragma unroll
        for (int qg = 0; qg < 4; ++qg)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = wm * WM + i * 32 + qg * 8 + (lane >> 5) * 4 + e;
            const int col = wn * WN + j * 32 + (lane & 31);
            if (row < col) *reinterpret_cast<uint16_t*>(stage + tile_off(row, col)) = f2bf(f * acc[i][j][qg * 4 + e]);
          }
      }
    }
  }
  if (!diag) return;
  // The mirrors of this wave's tiles above the diagonal (C > R): the tile it
  // has just staged, T[32C + r][32R + i] = D[32R + i][32C + r], read
  // transposed (ds_read_b64_tr_b16, as stage_cols reads) gives rows of D,
  // stored as 16-B chunks at T[32R + i][32C + r] -- four reads and two writes
  // per lane and tile, the staged bf16 values copied bit for bit.  The wave's
  // LDS operations complete in order, and no other wave writes or reads
  // either region.
  asm volatile("" ::: "memory");
  const int l16 = lane & 15, grp = lane >> 4;
#pragma unroll
  for (int i = 0; i < TMI; ++i) {
#pragma unroll
    for (int j = 0; j < TMJ; ++j) {
      const int R = wm * (WM / 32) + i, C = wn * (WN / 32) + j;
      if (!((plan.mask >> (i * TMJ + j)) & 1) || C <= R) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r0 = 32 * C + grp * 8, i0 = 32 * R + 16 * h;
        const int tr = r0 + (l16 >> 2), tc = i0 + ((l16 & 3) << 2);
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr, tc)));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr + 4, tc)));
        uint4 v;
        v.x = uint32_t(uint16_t(lo[0])) | (uint32_t(uint16_t(lo[1])) << 16);
        v.y = uint32_t(uint16_t(lo[2])) | (uint32_t(uint16_t(lo[3])) << 16);
        v.z = uint32_t(uint16_t(hi[0])) | (uint32_t(uint16_t(hi[1])) << 16);
        v.w = uint32_t(uint16_t(hi[2])) | (uint32_t(uint16_t(hi[3])) << 16);
        *reinterpret_cast<uint4*>(stage + tile_off(i0 + l16, r0)) = v;
      }
    }
  }
}

// Staged rows -> a panel-layout destination with the same rows: dst[r][i] =
// T[r][i] for the BN staged rows, dst at the first staged row of the tile's
// first column panel (panel stride pstride).  One wave instruction writes rows
// 16u .. 16u+15 of one panel (1 KiB contiguous).
template <bool PART>
__device__ __forceinline__ void stage_rows(const char* stage, uint16_t* dst, int64_t pstride, int rows) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll 4
  for (int it = 0; it < 8 * (BN / 16) / NWAVES; ++it) {
    const int u = wave + NWAVES * it;  // 8 panels x BN/16 row blocks
    const int q = u & 7, r = (u >> 3) * 16 + (lane >> 2);
    const int i = q * 32 + (lane & 3) * 8;
    if (PART && (i >= rows || r >= rows)) continue;  // beyond a partial tile
    const uint4 v = *reinterpret_cast<const uint4*>(stage + tile_off(r, i));
    *reinterpret_cast<uint4*>(dst + q * pstride + r * PANEL + (lane & 3) * 8) = v;
  }
}

// Staged columns -> rows of the destination: dst[i][r] = T[r][i] (256 rows i,
// BN columns r).  ds_read_b64_tr_b16 (16-lane groups): lane l of a group
// addresses T row r0 + l/4 at column i0 + 4*(l%4) and receives T[r0..r0+3][i0 + l];
// two reads give 8 consecutive r of destination row i0 + l.  The four groups of
// a wave take consecutive 8-column chunks, so one wave instruction covers
// destination rows i0 .. i0+15, columns 32t .. 32t+31: one panel's contiguous
// 1 KiB.  `fn(i, r, uint4)` consumes destination row i, columns r..r+7.
template <class Fn>
__device__ __forceinline__ void stage_cols(const char* stage, Fn&& fn) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
#pragma unroll 2
  for (int it = 0; it < 16 * (BN / 32) / NWAVES; ++it) {
    const int task = wave + NWAVES * it;
    const int i0 = (task & 15) * 16, r0 = (task >> 4) * 32 + grp * 8;
    const int tr = r0 + (l16 >> 2), tc = i0 + ((l16 & 3) << 2);
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr, tc)));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr + 4, tc)));
    uint4 v;
    v.x = uint32_t(uint16_t(lo[0])) | (uint32_t(uint16_t(lo[1])) << 16);
    v.y = uint32_t(uint16_t(lo[2])) | (uint32_t(uint16_t(lo[3])) << 16);
    v.z = uint32_t(uint16_t(hi[0])) | (uint32_t(uint16_t(hi[1])) << 16);
    v.w = uint32_t(uint16_t(hi[2])) | (uint32_t(uint16_t(hi[3])) << 16);
    fn(i0 + l16, r0, v);
  }
}

// ---------------------------------------------------------------------------
// SYRK / POLY / SYMM: symmetric m x m outputs of which only the 256 x 256
// tiles on and above the diagonal are computed and stored (tile ti x tc,
// tc >= ti; a diagonal tile in full).  SYRK reads X (K form); POLY reads the
// stored upper tiles of A (operand band R: T form left of its diagonal block,
// K form from there on); SYMM (C = S1 S2 of two symmetric stacks that commute,
// as polynomials in one Gram matrix do, so C is symmetric) reads its row band
// from S1 and its column band from S2 in the same way.
// ---------------------------------------------------------------------------
static_assert(BM == BN, "square tiles: a symmetric tile is either diagonal or strictly upper");
// PART: the stacks' extents are no multiples of the tile, so tiles at their ends are
// partial; without it those checks are compiled out, of the stores too, where the compiler
// cannot see that a lane's row lies in a whole tile (loads and waves' windows cost the
// 1024 x 1024 blocks 1%, the stores SYRK 0.4%: 41 branches in its epilogue).
template <int STAGE, bool PART>
__device__ __forceinline__ void sym_work(const NsArgs& a, uint16_t* lds, int v) {
  const int nt = tiles_of(a.mp), nc = nt;
  const int tiles = nt * nc - R_SYM * nt * (nt - 1) / 2;
  int b, t;
  if (!decode_tile(v, tiles, a.N, b, t)) return;
  int ti, tc;
  sym_tile(t, nc, ti, tc);

  const uint16_t* src;
  int K;
  if (STAGE == NS_SYRK) {
    src = static_cast<const uint16_t*>(a.x_in) + int64_t(b) * a.mp * a.np;
    K = a.kx;
  } else {
    src = static_cast<const uint16_t*>(a.a_in) + int64_t(b) * a.mp * a.mp;
    K = a.mp;
  }
  // SYMM: the column operand's stack (POLY: the row operand's own)
  const uint16_t* src2 = STAGE == NS_SYMM ? static_cast<const uint16_t*>(a.b_in) + int64_t(b) * a.mp * a.mp : src;
  const int64_t pstride = int64_t(a.mp) * PANEL;
  const int r0 = ti * BM, c0 = tc * BN;
  // on a diagonal tile only the 32 x 32 tiles on or above the diagonal are
  // computed; the others are staged from their transposes
  const bool diag = tc == ti;
  const int rows = PART ? a.mp - r0 : BM, cols = PART ? a.mp - c0 : BN;
  const int mv = PART ? a.m - r0 : BM, nv = PART ? a.m - c0 : BN;
  f32x16 acc[TMI][TMJ];
  if (STAGE == NS_SYRK)
    mainloop<OP_K, OP_K, PART>(src + r0 * PANEL, nullptr, 0, src + c0 * PANEL, nullptr, 0, pstride, K / BK, lds, acc, rows,
                         cols, mv, nv, 0.f, 0, diag);
  else if (STAGE == NS_POLY)  // acc = A A + (b/c) A, so P = c acc + a I = a I + b A + c A A
    mainloop<OP_SPLIT, OP_SPLIT, PART, IDENT_COL>(src + r0 * PANEL, src + (r0 / PANEL) * pstride, r0 / BK,
                                            src + c0 * PANEL, src + (c0 / PANEL) * pstride, c0 / BK,
                                            pstride, K / BK, lds, acc, rows, cols, mv, nv, a.cb / a.cc, c0, diag);
  else  // SYMM: acc = S1 S2; a diagonal tile loads both operands' bands
    mainloop<OP_SPLIT, OP_SPLIT, PART, IDENT_NONE, false>(src + r0 * PANEL, src + (r0 / PANEL) * pstride, r0 / BK,
                                                    src2 + c0 * PANEL, src2 + (c0 / PANEL) * pstride, c0 / BK,
                                                    pstride, K / BK, lds, acc, rows, cols, mv, nv, 0.f, 0, diag);

  float f = STAGE == NS_POLY ? a.cc : 1.f;  // SYRK: s^2 on the first iteration
  if (STAGE == NS_SYRK && a.scale != nullptr) {
    const float s = a.scale[b];
    f = s * s;
  }
  uint16_t* out = static_cast<uint16_t*>(a.out) + int64_t(b) * a.mp * a.mp;
  char* stage = reinterpret_cast<char*>(lds);
  barrier();  // every wave is done with the ring
  // POLY: a on the diagonal of the m valid rows (the padding stays zero)
  stage_tile(stage, acc, f, mv, diag, STAGE == NS_POLY ? a.ca : 0.f, STAGE == NS_POLY ? a.m - r0 : 0);
  barrier_after_lds_writes();
  if (!diag) {
    // upper tile C[r0 + i][c0 + r] = T[r][i]
    uint16_t* dst = out + (c0 / PANEL) * pstride + int64_t(r0) * PANEL;
    stage_cols(stage, [&](int i, int r, const uint4& u) {
      if (!PART || (i < rows && r < cols)) *reinterpret_cast<uint4*>(dst + (r >> 5) * pstride + i * PANEL + (r & 31)) = u;
    });
  } else {
    // diagonal tile in full, through its mirror C[r0 + r][r0 + i] = T[r][i]
    stage_rows<PART>(stage, out + (r0 / PANEL) * pstride + int64_t(r0) * PANEL, pstride, rows);
  }
}

template <int STAGE>
__global__ __launch_bounds__(NT, WG_PER_CU) void ns_sym_bf16(NsArgs a, int total) {
  __shared__ __attribute__((aligned(1024))) uint16_t lds[LDS_ELEMS];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    sym_work<STAGE, false>(a, lds, v);
    barrier();  // the staging area is read before the next tile's loads refill the ring
  }
}
template <int STAGE>
__global__ __launch_bounds__(NT, WG_PER_CU) void ns_sym_edge_bf16(NsArgs a, int total) {
  __shared__ __attribute__((aligned(1024))) uint16_t lds[LDS_ELEMS];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    sym_work<STAGE, true>(a, lds, v);
    barrier();
  }
}

// ---------------------------------------------------------------------------
// PX / PX_APPLY: X' = s P X (P = a I + b A + c A A from POLY), m x n output
// tile (256 x 256), K = m.  D[i][j] in registers (lane holds column j, rows
// i..i+3).  T[j][i] = X'[r0 + i][c0 + j] is staged in LDS;
// X' rows (PX, and the parameter rows of an untransposed block) are T's
// columns, the parameter rows of a tall block (param[j][i]) are T's rows.
// ---------------------------------------------------------------------------

// param[o .. o+valid) += alpha * u (u = 8 bf16 in u8); one rounding to the
// parameter dtype per element, as torch's foreach add with alpha.  `vec`:
// 16-B aligned full chunk (8 bf16 = 16 B, 8 fp32 = 32 B).
template <class TP>
__device__ __forceinline__ void apply_chunk(typename TP::storage* prm, int64_t o, const uint4& u8, float alpha,
                                            int valid, bool vec) {
  const uint32_t w[4] = {u8.x, u8.y, u8.z, u8.w};
  float u[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) u[e] = __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
  if (vec && valid == 8) {
    if constexpr (sizeof(typename TP::storage) == 2) {
      uint4 pv = *reinterpret_cast<const uint4*>(prm + o);
      uint32_t pw[4] = {pv.x, pv.y, pv.z, pv.w};
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float p0 = __uint_as_float(pw[h] << 16), p1 = __uint_as_float(pw[h] & 0xffff0000u);
        pw[h] = f2bf2(fmaf(alpha, u[2 * h], p0), fmaf(alpha, u[2 * h + 1], p1));
      }
      *reinterpret_cast<uint4*>(prm + o) = make_uint4(pw[0], pw[1], pw[2], pw[3]);
    } else {
      float4* q = reinterpret_cast<float4*>(prm + o);
      float4 a0 = q[0], a1 = q[1];
      a0.x = fmaf(alpha, u[0], a0.x); a0.y = fmaf(alpha, u[1], a0.y);
      a0.z = fmaf(alpha, u[2], a0.z); a0.w = fmaf(alpha, u[3], a0.w);
      a1.x = fmaf(alpha, u[4], a1.x); a1.y = fmaf(alpha, u[5], a1.y);
      a1.z = fmaf(alpha, u[6], a1.z); a1.w = fmaf(alpha, u[7], a1.w);
      q[0] = a0;
      q[1] = a1;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e < valid) TP::store(prm, o + e, fmaf(alpha, u[e], TP::load(prm, o + e)));
}

template <int STAGE, bool PART, bool TRANS, class TP>
__device__ __forceinline__ void px_work(const NsArgs& a, uint16_t* lds, int v) {
  const int tiles_i = tiles_of(a.mp);
  const int tiles = tiles_i * tiles_of(a.np);
  int b, t;
  if (!decode_tile(v, tiles, a.N, b, t)) return;
  // column-band-major: the tiles_i tiles that read one column band of X are
  // consecutive virtual tiles, so they run in the same round on one XCD
  // whenever tiles_i divides the workgroups one XCD runs per round (32 on 256
  // CUs; m <= 1024 at every model size here) and the band is fetched from HBM
  // once.  A block with more tiles than a round (n = 2752: 44) is split
  // between rounds at a column-band boundary, so only its P row bands, the
  // smaller operand, are fetched twice.
  const int tc = t / tiles_i, ti = t % tiles_i;
  const int r0 = ti * BM, c0 = tc * BN;

  const int64_t pstride = int64_t(a.mp) * PANEL;
  const uint16_t* P = static_cast<const uint16_t*>(a.a_in) + int64_t(b) * a.mp * a.mp;
  const uint16_t* X = static_cast<const uint16_t*>(a.x_in) + int64_t(b) * a.mp * a.np + (c0 / PANEL) * pstride;
  f32x16 acc[TMI][TMJ];
  // acc = P X; a wave whose window lies in the zero padding computes nothing: its
  // part of X' stays zero
  const int rows = PART ? a.mp - r0 : BM, cols = PART ? a.np - c0 : BN, mv = PART ? a.m - r0 : BM;
  mainloop<OP_SPLIT, OP_T, true>(P + r0 * PANEL, P + (r0 / PANEL) * pstride, r0 / BK, nullptr, X, 0, pstride, a.mp / BK,
                           lds, acc, rows, cols, mv, a.n - c0);

  const float s = a.scale != nullptr ? a.scale[b] : 1.f;
  char* stage = reinterpret_cast<char*>(lds);
  // apply: param += alpha * u; the parameter block is stored (m x n)
  // untransposed or (n x m) for a tall block
  auto* prm = STAGE == NS_PX_APPLY ? reinterpret_cast<typename TP::storage*>(a.blocks[b].param) : nullptr;
  const int m = a.m, n = a.n;
  // 16-B vector access: aligned blocks and a row length that keeps chunks aligned
  const bool vec = a.vec && ((TRANS ? m : n) % 8 == 0);
  // bf16 parameters, tile inside the block: every parameter chunk of this
  // thread is loaded in batches ahead of its use (the first batch before the
  // tile is staged), then combined and stored
  constexpr bool BF16P = sizeof(typename TP::storage) == 2;
  const bool fast = STAGE == NS_PX_APPLY && BF16P && vec && r0 + BM <= m && c0 + BN <= n;
  constexpr int CH = BN * BM / 8 / NT;  // 16-B chunks per thread
  constexpr int BATCH = 8;
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
  // chunk q of this thread: parameter offset, staged row r and column c of
  // its first element (TRANS: 8 consecutive staged columns; else 8 staged rows)
  auto chunk = [&](int q, int& r, int& c) -> int64_t {
    if (TRANS) {
      r = q * (NT / 32) + (tid >> 5);
      c = (tid & 31) * 8;
      return int64_t(c0 + r) * m + r0 + c;
    }
    const int task = wave + NWAVES * q;  // the stage_cols mapping
    c = (task & 15) * 16;                // i0
    r = (task >> 4) * 32 + grp * 8;
    return int64_t(r0 + c + l16) * n + c0 + r;
  };
  uint4 pv[BATCH];
  if constexpr (STAGE == NS_PX_APPLY && BF16P) {
    if (fast) {
#pragma unroll
      for (int q = 0; q < BATCH; ++q) {
        int r, c;
        pv[q] = *reinterpret_cast<const uint4*>(prm + chunk(q, r, c));
      }
    }
  }
  barrier();  // every wave is done with the ring
  stage_tile(stage, acc, s, mv);
  barrier_after_lds_writes();
  if (STAGE == NS_PX) {
    // X'[r0 + i][c0 + r] = T[r][i]
    uint16_t* dst = static_cast<uint16_t*>(a.out) + int64_t(b) * a.mp * a.np + (c0 / PANEL) * pstride +
                    int64_t(r0) * PANEL;
    stage_cols(stage, [&](int i, int r, const uint4& u) {
      if (!PART || (i < rows && r < cols)) *reinterpret_cast<uint4*>(dst + (r >> 5) * pstride + i * PANEL + (r & 31)) = u;
    });
    return;
  }
  const float alpha = a.alpha;
  if constexpr (BF16P) {
    if (fast) {
#pragma unroll
      for (int q0 = 0; q0 < CH; q0 += BATCH) {
        if (q0 > 0) {
#pragma unroll
          for (int q = 0; q < BATCH; ++q) {
            int r, c;
            pv[q] = *reinterpret_cast<const uint4*>(prm + chunk(q0 + q, r, c));
          }
        }
#pragma unroll
        for (int q = 0; q < BATCH; ++q) {
          int r, c;
          const int64_t o = chunk(q0 + q, r, c);
          uint4 u;
          if (TRANS) {
            u = *reinterpret_cast<const uint4*>(stage + tile_off(r, c));
          } else {
            const int tr = r + (l16 >> 2), tc = c + ((l16 & 3) << 2);
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr, tc)));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + tile_off(tr + 4, tc)));
            u.x = uint32_t(uint16_t(lo[0])) | (uint32_t(uint16_t(lo[1])) << 16);
            u.y = uint32_t(uint16_t(lo[2])) | (uint32_t(uint16_t(lo[3])) << 16);
            u.z = uint32_t(uint16_t(hi[0])) | (uint32_t(uint16_t(hi[1])) << 16);
            u.w = uint32_t(uint16_t(hi[2])) | (uint32_t(uint16_t(hi[3])) << 16);
          }
          const uint32_t w[4] = {u.x, u.y, u.z, u.w};
          uint32_t pw[4] = {pv[q].x, pv[q].y, pv[q].z, pv[q].w};
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            const float u0 = __uint_as_float(w[h] << 16), u1 = __uint_as_float(w[h] & 0xffff0000u);
            const float p0 = __uint_as_float(pw[h] << 16), p1 = __uint_as_float(pw[h] & 0xffff0000u);
            pw[h] = f2bf2(fmaf(alpha, u0, p0), fmaf(alpha, u1, p1));
          }
          *reinterpret_cast<uint4*>(prm + o) = make_uint4(pw[0], pw[1], pw[2], pw[3]);
        }
      }
      return;
    }
  }
  if (TRANS) {
    const int c = (tid & 31) * 8;
    for (int q = 0; q < BN / (NT / 32); ++q) {
      const int r = q * (NT / 32) + (tid >> 5);  // staged row = X' column = parameter row
      const int pr = c0 + r, pc = r0 + c;
      if (pr >= n || pc >= m) continue;
      const uint4 u8 = *reinterpret_cast<const uint4*>(stage + tile_off(r, c));
      apply_chunk<TP>(prm, int64_t(pr) * m + pc, u8, alpha, min(8, m - pc), vec);
    }
  } else {
    stage_cols(stage, [&](int i, int r, const uint4& u) {
      const int pr = r0 + i, pc = c0 + r;
      if (pr < m && pc < n) apply_chunk<TP>(prm, int64_t(pr) * n + pc, u, alpha, min(8, n - pc), vec);
    });
  }
}

template <int STAGE, bool TRANS, class TP>
__global__ __launch_bounds__(NT, WG_PER_CU) void ns_px_bf16(NsArgs a, int total) {
  __shared__ __attribute__((aligned(1024))) uint16_t lds[LDS_ELEMS];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    px_work<STAGE, false, TRANS, TP>(a, lds, v);
    barrier();  // the staging area is read before the next tile's loads refill the ring
  }
}
template <int STAGE, bool TRANS, class TP>
__global__ __launch_bounds__(NT, WG_PER_CU) void ns_px_edge_bf16(NsArgs a, int total) {
  __shared__ __attribute__((aligned(1024))) uint16_t lds[LDS_ELEMS];
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    px_work<STAGE, true, TRANS, TP>(a, lds, v);
    barrier();
  }
}

// ---------------------------------------------------------------------------
// fp32 Newton-Schulz (the pretrain copy keeps the buffer dtype) on the bf16
// matrix cores.  An fp32 value is the exact sum of three bf16 values
// (h = bf16(x), m = bf16(x - h), l = x - h - m: 8 + 8 + 8 significant bits, signs
// included), and a product of two of them is taken as the six terms
//   hh + hm + mh + hl + lh + mm
// (Henry, Tang, Heinecke: Leveraging the bfloat16 artificial intelligence datatype
// for higher-precision computations, 2019), accumulated in fp32 by
// v_mfma_f32_32x32x16_bf16.  The dropped ml, lm and ll are below 2^-23 of the
// product's leading term and of random sign, and the accumulators are rounded once
// per 16 terms instead of once per two (v_mfma_f32_32x32x2_f32): against fp64 the
// five iterations are off by 0.6-1.2e-6 on Gaussian blocks from 96 x 136 to
// 1024 x 2752, where the fp32 MFMA gave 1.4-3.4e-6, and by 3.0-5.0e-6 against
// 6.9-13.6e-6 on singular values spread over four decades.
//
// Why: six such MFMAs take 192 cycles for 16 k against 512 of the fp32 MFMA, which
// bound these kernels (71% busy at the 1.3B shapes).  Measured there, 176 blocks of
// 512 x 512: SYRK 297 -> 168 us, POLY 302 -> 181, PX 407 -> 265, PX + apply 469 ->
// 322; 48 of 512 x 1376: SYRK 198 -> 118.  Now no unit is full: the MFMAs are busy
// 46-53% of the cycles at 1.8-1.9 GHz (the package-power limit), the LDS reads and
// writes of a step take 0.75 of its MFMA time and the split's VALU work 0.55.
// Measured without gain: the split's subtractions as v_dot2_f32_bf16 (slower),
// raised wave priority during the MFMAs, the lower-left wave of a diagonal tile
// left idle, one accumulator and three waves per SIMD (SYRK 190 us, and see lo).
//
// Tiles of FT x FT (FT = 64 TW) per 256-thread workgroup, 2 x 2 waves of TW x TW
// MFMA tiles; K advances 16 per step, double-buffered in LDS: the next step's
// global loads (fp32, into registers) are in flight during the current step's
// MFMAs, are split after them and stored to the other buffer as three bf16 planes.
// Operands reach LDS in one of two forms, 16 k x FT x 2 B per plane:
//   K: operand rows, [row][16 k] (rows of X for SYRK; rows of A / P, and by
//      symmetry A's columns).  A row is two 16-B chunks; chunk c of row r sits at
//      c ^ ((r >> 3) & 1), so the 16 rows of a quarter-wave's ds_read_b128 cover
//      all 64 banks;
//   T: [k][FT columns] (PX's X operand, k = rows of X), read with
//      ds_read_b64_tr_b16; the 64-B chunk of columns 32 p .. 32 p + 31 of row k sits
//      at p ^ (k & 3) (FT = 128) or p ^ ((k >> 1) & 1) (FT = 64), so the four rows
//      of a transposed read lie in different banks.
// SYRK and POLY produce symmetric matrices: only the tiles on and above the
// diagonal are computed, each stored with its mirror (staged in LDS so both
// stores are row-contiguous), so the stored matrix is exactly symmetric.  A tile
// that lies in the zero padding is stored as zeros without running its products.
// ---------------------------------------------------------------------------
constexpr int F_NT = 256;              // 4 waves, 2 x 2
constexpr int FK = 16;                 // K per step
constexpr int F_PAD = 128;             // padding granularity of the fp32 stacks
// Tiles of 128 x 128 from which a launch uses them, about one per CU; with fewer,
// 64 x 64 tiles spread the work over more CUs (measured: 48 blocks of 512 x 1376,
// 480 tiles: SYRK 139 us with 64 x 64 tiles, 118 with 128 x 128; 44 blocks of 256 x
// 256, 132 tiles: 12.4 against 16.3; 12 blocks of 256 x 688, 36 tiles: 16.1 against 29.7).
constexpr int F32_FILL = 256;
// Blocks go to XCDs whole, which keeps a block's operands, and what the stage before
// wrote, in one L2 (48 blocks of 512 x 512: SYRK 48.9 us, 50.8 when every block is spread
// over all XCDs; 64: 69.8 / 73.8), unless that fills some XCDs' 32 CUs more than once
// while others idle: with one 2048 x 2048 block on one XCD SYRK takes 306 us, spread over
// all 86; two 1024 x 1024 blocks 70 / 32, twelve (two on half of the XCDs, one on the
// others) 123 / 87, twenty 162 / 142.  With a quarter of the slots idle spreading is as
// fast or faster at every such size; from 512 on also with 15% (twenty 384 x 384: 15.9 /
// 17.5, twenty 512 x 1376: 68.8 / 65.5; 9%, 44 blocks of 512 x 512: 48.3 / 50.6).  A step of
// twelve 256 x 256 blocks, 20 tiles on the fullest XCD: 136 / 152.
// The same for every stage of a chain, from its SYRK's 64-wide tiles (PX of the twelve
// 256 x 688 blocks spread between stages that are not: the toy model's step 797 / 804 us).
bool f32_spread(int blocks, int side) {
  const int slots = (blocks + 7) / 8 * 8, nt = side / 64;
  return slots / 8 * int64_t(nt * (nt + 1) / 2) > 32 &&
         (4 * slots >= 5 * blocks || (side >= 512 && 20 * slots >= 23 * blocks));
}

template <int TW>
struct F32Geo {
  static constexpr int FT = 64 * TW;              // output tile
  static constexpr int WT = 32 * TW;              // wave sub-tile
  static constexpr int PLANE = FT * FK * 2;       // bytes of one bf16 plane of an operand's K step
  static constexpr int OPER = 3 * PLANE;          // bytes of an operand's K step
  static constexpr int QPT = FT * FK / 4 / F_NT;  // float4 per thread and operand K step
  static constexpr int LDS = 4 * OPER;            // [buffer 0: A, B][buffer 1: A, B]
  static_assert(64 * FT * 4 <= LDS, "64 rows of the staged tile fit in the operand buffers");
  static_assert(QPT == TW, "whole float4 loads per thread");
};

// This thread's float4 j of an operand's K step: rows r0 .. r0+FT-1, k0 .. k0+FK-1 of
// a row-major matrix (leading dimension ld) ...
template <int TW>
__device__ __forceinline__ const float* f32_src_rows(const float* src, int64_t ld, int r0, int j) {
  const int idx = threadIdx.x + F_NT * j;
  return src + int64_t(r0 + (idx >> 2)) * ld + 4 * (idx & 3);
}
// ... or rows k0 .. k0+FK-1 of X (leading dimension ld), columns c0 .. c0+FT-1
template <int TW>
__device__ __forceinline__ const float* f32_src_cols(const float* X, int64_t ld, int c0, int j) {
  constexpr int Q = F32Geo<TW>::FT / 4;
  const int idx = threadIdx.x + F_NT * j;
  return X + int64_t(idx / Q) * ld + c0 + 4 * (idx % Q);
}

// Splitting four values into three planes of four bf16 values each, PLANE bytes
// apart from d, in six parts of two to six VALU instructions, so that the main
// loop can put one part behind each of its MFMAs.
struct F32Split {
  uint32_t h0, h1, m0, m1;
  float a0, a1, a2, a3;
  static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
  template <int PLANE>
  __device__ __forceinline__ void part(int n, const float4& v, char* d) {
    switch (n) {
      case 0:
        h0 = f2bf2(v.x, v.y);
        h1 = f2bf2(v.z, v.w);
        break;
      case 1:
        a0 = v.x - lo(h0);
        a1 = v.y - hi(h0);
        break;
      case 2:
        a2 = v.z - lo(h1);
        a3 = v.w - hi(h1);
        *reinterpret_cast<uint2*>(d) = make_uint2(h0, h1);
        break;
      case 3:
        m0 = f2bf2(a0, a1);
        m1 = f2bf2(a2, a3);
        *reinterpret_cast<uint2*>(d + PLANE) = make_uint2(m0, m1);
        break;
      case 4:
        a0 -= lo(m0);
        a1 -= hi(m0);
        a2 -= lo(m1);
        break;
      default:
        a3 -= hi(m1);
        *reinterpret_cast<uint2*>(d + 2 * PLANE) = make_uint2(f2bf2(a0, a1), f2bf2(a2, a3));
    }
  }
};
// LDS offset, within an operand's buffer, of this thread's float4 j
template <int TW>
__device__ __forceinline__ uint32_t f32_off_k(int j) {
  const int idx = threadIdx.x + F_NT * j, r = idx >> 2, q = idx & 3;
  return uint32_t(r * 32 + (((q >> 1) ^ ((r >> 3) & 1)) << 4) + ((q & 1) << 3));
}
template <int TW>
__device__ __forceinline__ int f32_tswz(int k) { return TW == 2 ? (k & 3) : ((k >> 1) & 1); }
template <int TW>
__device__ __forceinline__ uint32_t f32_off_t(int j) {
  constexpr int FT = F32Geo<TW>::FT, Q = FT / 4;
  const int idx = threadIdx.x + F_NT * j, k = idx / Q, n = 4 * (idx % Q);
  return uint32_t(k * FT * 2 + (((n >> 5) ^ f32_tswz<TW>(k)) << 6) + ((n & 31) << 1));
}

// Upper tile t of an nt x nt grid of tiles (ti <= tj), row-major over the
// upper triangle.
__device__ __forceinline__ void f32_sym_tile(int t, int nt, int& ti, int& tj) {
  int i = 0;
  while (t >= nt - i) {
    t -= nt - i;
    ++i;
  }
  ti = i;
  tj = i + t;
}

// Swizzle of the staged output tile's 16-B chunks within a column: distinct for 16
// consecutive columns (the accumulator writes) and for 16 columns four apart (the
// 4 x 4 block reads).
__device__ __forceinline__ int f32_tile_swz(int c) { return ((c >> 2) & 15) ^ ((c & 3) << 2); }

// param[pr][pc .. pc+3] += alpha s v[k] over this thread's N chunks (at(k, pr, pc)
// gives chunk k's place), one rounding to the parameter dtype per element, as
// torch's foreach add with alpha.  All loads are issued before the first store.
// rows, cols: the parameter block's sides.
template <class TP, int N, class At>
__device__ __forceinline__ void f32_update(typename TP::storage* prm, const NsArgs& a, float s, const float4 (&v)[N],
                                           At&& at, int rows, int cols) {
  const bool vec = a.vec && cols % 4 == 0;  // 16-B (bf16: 8-B) accesses
  float p[N][4];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    int pr, pc;
    at(k, pr, pc);
    const int64_t o = int64_t(pr) * cols + pc;
    if (vec && pr < rows && pc < cols) {
      if constexpr (sizeof(typename TP::storage) == 2) {
        const uint2 w = *reinterpret_cast<const uint2*>(prm + o);
        p[k][0] = __uint_as_float(w.x << 16);
        p[k][1] = __uint_as_float(w.x & 0xffff0000u);
        p[k][2] = __uint_as_float(w.y << 16);
        p[k][3] = __uint_as_float(w.y & 0xffff0000u);
      } else {
        const float4 w = *reinterpret_cast<const float4*>(prm + o);
        p[k][0] = w.x;
        p[k][1] = w.y;
        p[k][2] = w.z;
        p[k][3] = w.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) p[k][e] = pr < rows && pc + e < cols ? TP::load(prm, o + e) : 0.f;
    }
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    int pr, pc;
    at(k, pr, pc);
    const int64_t o = int64_t(pr) * cols + pc;
    const float u[4] = {s * v[k].x, s * v[k].y, s * v[k].z, s * v[k].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) p[k][e] = fmaf(a.alpha, u[e], p[k][e]);
    if (vec && pr < rows && pc < cols) {
      if constexpr (sizeof(typename TP::storage) == 2)
        *reinterpret_cast<uint2*>(prm + o) = make_uint2(f2bf2(p[k][0], p[k][1]), f2bf2(p[k][2], p[k][3]));
      else
        *reinterpret_cast<float4*>(prm + o) = make_float4(p[k][0], p[k][1], p[k][2], p[k][3]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (pr < rows && pc + e < cols) TP::store(prm, o + e, p[k][e]);
    }
  }
}

template <int STAGE, class TP, int TW>
__global__ __launch_bounds__(F_NT) __attribute__((amdgpu_waves_per_eu(2))) void ns_f32(NsArgs a, int spread) {
  using G = F32Geo<TW>;
  constexpr int FT = G::FT, WT = G::WT;
  __shared__ __attribute__((aligned(1024))) char lds[G::LDS];
  constexpr bool PX = STAGE == NS_PX || STAGE == NS_PX_APPLY;
  constexpr bool SYM = STAGE == NS_SYRK || STAGE == NS_POLY;
  const int nt = a.mp / FT, nc = a.np / FT;
  const int tiles = SYM ? nt * (nt + 1) / 2 : nt * nc;
  int b, t0;
  if (!decode_tile(blockIdx.x, tiles, a.N, b, t0, spread)) return;
  int ti, tj;
  if (SYM) {
    f32_sym_tile(t0, nt, ti, tj);
  } else {
    ti = t0 % nt;  // the tiles that read one column band of X are neighbours
    tj = t0 / nt;
  }
  const int r0 = ti * FT, c0 = tj * FT;
  const float* X = static_cast<const float*>(a.x_in) + int64_t(b) * a.mp * a.np;
  const float* A = static_cast<const float*>(a.a_in) + int64_t(b) * a.mp * a.mp;
  const float* rsrc = STAGE == NS_SYRK ? X : A;  // rows of the row operand (and of SYRK / POLY's column operand)
  const int64_t rld = STAGE == NS_SYRK ? a.np : a.mp;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const bool diag = SYM && tj == ti;
  // K steps over the valid extent; none where the tile holds only padding
  const int K = STAGE == NS_SYRK ? a.kx : (a.m + FK - 1) / FK * FK;
  const int KT = r0 >= a.m || c0 >= (PX ? a.n : a.m) ? 0 : K / FK;
  f32x16 acc[TW][TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < TW; ++j) acc[i][j] = f32x16{};
  // float4 q of this thread's share of a K step: q < TW the row operand, else the
  // column operand; dst: its LDS offset within a buffer
  constexpr int NQ = 2 * TW;
  const float* src[NQ];
  uint32_t dst[NQ];
  float4 g[2][NQ];  // K steps t + 1 and t + 2
  const int64_t kstep_a = FK, kstep_b = PX ? int64_t(FK) * a.np : FK;
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    src[j] = f32_src_rows<TW>(rsrc, rld, r0, j);
    src[TW + j] = PX ? f32_src_cols<TW>(X, a.np, c0, j) : f32_src_rows<TW>(rsrc, rld, c0, j);
    dst[j] = f32_off_k<TW>(j);
    dst[TW + j] = G::OPER + (PX ? f32_off_t<TW>(j) : f32_off_k<TW>(j));
  }
  auto fetch = [&](float4 (&v)[NQ]) {  // the next K step
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      v[q] = *reinterpret_cast<const float4*>(src[q]);
      src[q] += q < TW ? kstep_a : kstep_b;
    }
  };
  // per-lane fragment offsets: K form, row lane%32, k 8 (lane/32) .. +7; T form,
  // column lane%32, the same k (two transposed reads, four k apart)
  const int l16 = lane & 15;
  const uint32_t kf = uint32_t((lane & 31) * 32 + (((lane >> 5) ^ ((lane >> 3) & 1)) << 4));
  const int tk = ((lane >> 5) << 3) + (l16 >> 2);
  const uint32_t tf = uint32_t(tk * FT * 2 + ((((lane >> 4) & 1) << 4) + ((l16 & 3) << 2)) * 2);
  const int tz = f32_tswz<TW>(tk);
  auto frag_k = [&](const char* s, int row, int p) {
    return *reinterpret_cast<const bf16x8*>(s + p * G::PLANE + row * 32 + kf);
  };
  auto frag_t = [&](const char* s, int panel, int p) {
    const char* q = s + p * G::PLANE + tf + ((panel ^ tz) << 6);
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(q));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(q + 4 * FT * 2));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    const i16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, v);
  };
  F32Split sp;
  if (KT > 0) {
    fetch(g[0]);
    if (KT > 1) fetch(g[1]);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int n = 0; n < 6; ++n) sp.part<G::PLANE>(n, g[0][q], lds + dst[q]);
  }
  __syncthreads();
  // lo: the five small terms in an accumulator of their own.  The MFMA aligns its
  // products to the accumulator and cuts what falls below it, so small terms added
  // to the large sum lean to one side (2752 k: the Gram diagonal off by -1.6e-6
  // relative with one accumulator); beside sums of their own size they do not.
  f32x16 lo[TW][TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < TW; ++j) lo[i][j] = f32x16{};
  // K step t: the loads of step t + 2 go out first, then behind each MFMA (32
  // cycles) goes a part of splitting step t + 1.  Past the last step the split goes
  // to a buffer nobody reads and the loads are left out.
  constexpr int PA[6] = {0, 0, 1, 1, 0, 2}, PB[6] = {0, 1, 0, 1, 2, 0};
  auto step = [&](int t, float4 (&next)[NQ], float4 (&after)[NQ]) {
    const char* sa = lds + (t & 1) * 2 * G::OPER;
    const char* sb = sa + G::OPER;
    char* nx = lds + ((t + 1) & 1) * 2 * G::OPER;
    if (t + 2 < KT) fetch(after);
    bf16x8 av[TW][3], bv[TW][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TW; ++i) av[i][p] = frag_k(sa, wr * WT + i * 32, p);
#pragma unroll
      for (int j = 0; j < TW; ++j) bv[j][p] = PX ? frag_t(sb, wc * TW + j, p) : frag_k(sb, wc * WT + j * 32, p);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 6 * TW * TW; ++n) {
      const int q = n / (TW * TW), i = n / TW % TW, j = n % TW;
      f32x16& d = q == 0 ? acc[i][j] : lo[i][j];
      d = mfma(av[i][PA[q]], bv[j][PB[q]], d);
#pragma unroll
      for (int u = 0; u < 2 / TW; ++u) {
        const int x = n * (2 / TW) + u;
        sp.part<G::PLANE>(x % 6, next[x / 6], nx + dst[x / 6]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  for (int t = 0; t < KT; t += 2) {
    step(t, g[1], g[0]);
    if (t + 1 < KT) step(t + 1, g[0], g[1]);
  }
  if (STAGE == NS_POLY && KT > 0) {
    // + (b/c) A, A symmetric: the lane's four consecutive rows of one column are
    // four consecutive columns of a row
    const float bc = a.cb / a.cc;
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = r0 + wr * WT + i * 32 + 8 * q + 4 * (lane >> 5), c = c0 + wc * WT + j * 32 + (lane & 31);
          const float4 v = *reinterpret_cast<const float4*>(A + int64_t(c) * a.mp + r);
          lo[i][j][4 * q] = fmaf(bc, v.x, lo[i][j][4 * q]);
          lo[i][j][4 * q + 1] = fmaf(bc, v.y, lo[i][j][4 * q + 1]);
          lo[i][j][4 * q + 2] = fmaf(bc, v.z, lo[i][j][4 * q + 2]);
          lo[i][j][4 * q + 3] = fmaf(bc, v.w, lo[i][j][4 * q + 3]);
        }
  }
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < TW; ++j) acc[i][j] += lo[i][j];
  const float s = a.scale != nullptr ? a.scale[b] : 1.f;
  // Output: 64 rows of the tile per pass go through LDS as T[column][row], 16-B
  // chunks of four rows, chunk q of column c at q ^ f32_tile_swz(c).  They are read
  // back as 4 x 4 blocks (four chunks: rows r .. r+3 of columns c .. c+3, stored as
  // four rows of a row-major matrix, 512 B of consecutive columns per 32 lanes) or
  // as single chunks (four rows of one column, stored along a row of the transpose);
  // none of the accesses has a bank conflict.
  constexpr int PASSES = FT / 64;
  constexpr int BPT = 64 * FT / 16 / F_NT;  // 4 x 4 blocks per thread and pass
  constexpr int CPT = 64 * FT / 4 / F_NT;   // chunks per thread and pass
  auto chunk = [&](int c, int q) { return reinterpret_cast<float4*>(lds + c * 256 + ((q ^ f32_tile_swz(c)) << 4)); };
  // block k of this thread: columns 4 x .. 4 x + 3, rows 4 y .. 4 y + 3 of the pass
  auto blk = [&](int k, int& x, int& y) {
    const int idx = threadIdx.x + F_NT * k;
    x = idx % (FT / 4);
    y = idx / (FT / 4);
  };
  // chunk k of this thread: column c, rows 4 y .. 4 y + 3 of the pass
  auto col = [&](int k, int& c, int& y) {
    const int idx = threadIdx.x + F_NT * k;
    c = idx >> 4;
    y = idx & 15;
  };
  auto read_blk = [&](int x, int y, float (&v)[4][4]) {  // v[row][column]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 w = *chunk(4 * x + i, y);
      v[0][i] = w.x;
      v[1][i] = w.y;
      v[2][i] = w.z;
      v[3][i] = w.w;
    }
  };
  [[maybe_unused]] auto* prm =
      STAGE == NS_PX_APPLY ? reinterpret_cast<typename TP::storage*>(a.blocks[b].param) : nullptr;
#pragma unroll 1
  for (int h = 0; h < PASSES; ++h) {
    if (h) __syncthreads();  // every wave is done reading the previous pass
    // accumulator value 4 q + e of MFMA tile (i, j) holds row WT wr + 32 i + 8 q +
    // 4 (lane/32) + e, column WT wc + 32 j + lane%32
    if (TW == 1 || wr == h) {
#pragma unroll
      for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x16& v = acc[i][j];
            const int r4 = (TW == 1 ? wr * 8 : 0) + i * 8 + 2 * q + (lane >> 5), c = wc * WT + j * 32 + (lane & 31);
            *chunk(c, r4) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
          }
    }
    __syncthreads();
    const int rh = r0 + 64 * h;  // first row of the pass
    if constexpr (SYM) {
      // SYRK: A = s^2 acc; POLY: P = c (A A + (b/c) A) + a I.  Each tile is stored
      // with its mirror; a diagonal tile stores its 4 x 4 blocks above the diagonal
      // and their mirrors, and those on it from their upper triangles.
      float* out = static_cast<float*>(a.out) + int64_t(b) * a.mp * a.mp;
      const float f = STAGE == NS_SYRK ? s * s : a.cc;
#pragma unroll
      for (int k = 0; k < BPT; ++k) {
        int x, y;
        blk(k, x, y);
        const int r = rh + 4 * y, c = c0 + 4 * x;
        if (diag && r > c) continue;
        float v[4][4];
        read_blk(x, y, v);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[e][i] *= f;
        if (diag && r == c) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int i = 0; i < e; ++i) v[e][i] = v[i][e];
            if (STAGE == NS_POLY && r + e < a.m) v[e][e] += a.ca;  // the quintic's a X: P's diagonal
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float4*>(out + int64_t(r + e) * a.mp + c) = make_float4(v[e][0], v[e][1], v[e][2], v[e][3]);
      }
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        int c, y;
        col(k, c, y);
        const int r = rh + 4 * y;
        if (diag && r >= ((c0 + c) & ~3)) continue;
        float4 v = *chunk(c, y);
        v.x *= f;
        v.y *= f;
        v.z *= f;
        v.w *= f;
        *reinterpret_cast<float4*>(out + int64_t(c0 + c) * a.mp + r) = v;  // the mirror
      }
    } else if constexpr (STAGE == NS_PX) {  // X' = s P X
      float* out = static_cast<float*>(a.out) + int64_t(b) * a.mp * a.np;
#pragma unroll
      for (int k = 0; k < BPT; ++k) {
        int x, y;
        blk(k, x, y);
        float v[4][4];
        read_blk(x, y, v);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float4*>(out + int64_t(rh + 4 * y + e) * a.np + c0 + 4 * x) =
              make_float4(s * v[e][0], s * v[e][1], s * v[e][2], s * v[e][3]);
      }
    } else if (a.transposed) {
      // PX_APPLY of a tall block: param (n x m) [column][row] += alpha X'
      float4 v[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        int c, y;
        col(k, c, y);
        v[k] = *chunk(c, y);
      }
      f32_update<TP, CPT>(prm, a, s, v, [&](int k, int& pr, int& pc) {
        int c, y;
        col(k, c, y);
        pr = c0 + c;
        pc = rh + 4 * y;
      }, a.n, a.m);
    } else {
      // ... of a wide or square block: param (m x n) [row][column]
#pragma unroll
      for (int k = 0; k < BPT; ++k) {
        int x, y;
        blk(k, x, y);
        float w[4][4];
        read_blk(x, y, w);
        float4 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = make_float4(w[e][0], w[e][1], w[e][2], w[e][3]);
        f32_update<TP, 4>(prm, a, s, v, [&](int e, int& pr, int& pc) {
          pr = rh + 4 * y + e;
          pc = c0 + 4 * x;
        }, a.m, a.n);
      }
    }
  }
}

// The kernels with partial tiles where the stacks' extents ask for them.
template <int STAGE, class TP>
void launch_bf16(const NsArgs& a, hipStream_t s) {
  const int nb8 = 8 * ((a.N + 7) / 8);
  const bool edge_m = a.mp % BM != 0;
  if constexpr (STAGE == NS_SYRK || STAGE == NS_POLY || STAGE == NS_SYMM) {
    const int nt = tiles_of(a.mp), nc = nt;
    const int total = nb8 * (nt * nc - R_SYM * nt * (nt - 1) / 2);
    const dim3 grid(resident_grid(total));
    if (edge_m) hipLaunchKernelGGL((ns_sym_edge_bf16<STAGE>), grid, dim3(NT), 0, s, a, total);
    else hipLaunchKernelGGL((ns_sym_bf16<STAGE>), grid, dim3(NT), 0, s, a, total);
  } else {
    const int total = nb8 * tiles_of(a.mp) * tiles_of(a.np);
    const dim3 grid(resident_grid(total));
    const bool edge = edge_m || a.np % BN != 0;
    if (STAGE == NS_PX || !a.transposed) {
      if (edge) hipLaunchKernelGGL((ns_px_edge_bf16<STAGE, false, TP>), grid, dim3(NT), 0, s, a, total);
      else hipLaunchKernelGGL((ns_px_bf16<STAGE, false, TP>), grid, dim3(NT), 0, s, a, total);
    } else if constexpr (STAGE == NS_PX_APPLY) {
      if (edge) hipLaunchKernelGGL((ns_px_edge_bf16<STAGE, true, TP>), grid, dim3(NT), 0, s, a, total);
      else hipLaunchKernelGGL((ns_px_bf16<STAGE, true, TP>), grid, dim3(NT), 0, s, a, total);
    }
  }
}

template <int STAGE, class TP, int TW>
void launch_f32_t(const NsArgs& a, hipStream_t s) {
  constexpr int FT = F32Geo<TW>::FT;
  constexpr bool SYM = STAGE == NS_SYRK || STAGE == NS_POLY;
  const int nt = a.mp / FT;
  const int64_t tiles = SYM ? int64_t(nt) * (nt + 1) / 2 : int64_t(nt) * (a.np / FT);
  const int64_t per_x = int64_t(a.mp) * a.np, per_a = int64_t(a.mp) * a.mp;
  const int64_t per_out = SYM ? per_a : per_x;
  // at most 2^30 workgroups per launch: larger stacks in chunks of blocks
  const int chunk = int(std::max<int64_t>(8, (int64_t(1) << 30) / tiles / 8 * 8));
  for (int b0 = 0; b0 < a.N; b0 += chunk) {
    NsArgs c = a;
    c.N = std::min(a.N - b0, chunk);
    if (a.x_in) c.x_in = static_cast<const float*>(a.x_in) + b0 * per_x;
    if (a.a_in) c.a_in = static_cast<const float*>(a.a_in) + b0 * per_a;
    if (a.out) c.out = static_cast<float*>(a.out) + b0 * per_out;
    if (a.scale) c.scale = a.scale + b0;
    if (a.blocks) c.blocks = a.blocks + b0;
    const bool spread = f32_spread(c.N, a.mp);
    const int slots = spread ? c.N : (c.N + 7) / 8 * 8;
    hipLaunchKernelGGL((ns_f32<STAGE, TP, TW>), dim3(unsigned(slots * tiles)), dim3(F_NT), 0, s, c, int(spread));
  }
}
template <int STAGE, class TP>
void launch_f32(const NsArgs& a, hipStream_t s) {
  constexpr bool SYM = STAGE == NS_SYRK || STAGE == NS_POLY;
  const int nt = a.mp / 128;
  const int64_t tiles = int64_t(a.N) * (SYM ? nt * (nt + 1) / 2 : int64_t(nt) * (a.np / 128));
  if (tiles >= F32_FILL) launch_f32_t<STAGE, TP, 2>(a, s);
  else launch_f32_t<STAGE, TP, 1>(a, s);
}

}  // namespace

// bf16: 64, two K slices, so that the stacks' traffic, the K extents and the waves'
// work follow the block's sides (264 blocks of 384 x 384 padded to 384 instead of 512:
// PX 88 -> 60 us, 4.9 TB/s; SYRK 57 -> 48, POLY 70 -> 50, pack 120 -> 95); beyond 2048
// whole tiles, which the kernels without partial ones take (at most an eighth of padding).
int ns_pad(int ns_dtype, int side) { return ns_dtype != MMUON_BF16 ? F_PAD : side <= 2048 ? 64 : 256; }
int ns_tile_k(int ns_dtype) { return ns_dtype == MMUON_BF16 ? BK : FK; }

int launch_ns_stage(const NsArgs& a, int stage, int ns_dtype, int param_dtype, hipStream_t s) {
  if (ns_dtype == MMUON_BF16) {
    switch (stage) {
      case NS_SYRK: launch_bf16<NS_SYRK, BF16T>(a, s); return 0;
      case NS_POLY: launch_bf16<NS_POLY, BF16T>(a, s); return 0;
      case NS_SYMM: launch_bf16<NS_SYMM, BF16T>(a, s); return 0;
      case NS_PX: launch_bf16<NS_PX, BF16T>(a, s); return 0;
      case NS_PX_APPLY:
        if (param_dtype == MMUON_BF16) launch_bf16<NS_PX_APPLY, BF16T>(a, s);
        else launch_bf16<NS_PX_APPLY, F32T>(a, s);
        return 0;
    }
  } else if (ns_dtype == MMUON_F32) {
    switch (stage) {
      case NS_SYRK: launch_f32<NS_SYRK, F32T>(a, s); return 0;
      case NS_POLY: launch_f32<NS_POLY, F32T>(a, s); return 0;
      case NS_PX: launch_f32<NS_PX, F32T>(a, s); return 0;
      case NS_PX_APPLY:
        if (param_dtype == MMUON_BF16) launch_f32<NS_PX_APPLY, BF16T>(a, s);
        else launch_f32<NS_PX_APPLY, F32T>(a, s);
        return 0;
    }
  }
  return -1;
}

}  // namespace mmuon
