// Monarch butterfly multiply (MonarchLinear.forward_matmul) and its backward
// as batched gfx950 MFMA GEMMs.
//
// x (B, k p), w1 (k, q, p), w2 (l, s, r), k = l blocks, q = r:
//   forward   out1[kk][b][jq] = x[b][kk p : (kk+1) p] . w1[kk][jq]          (F1)
//             t[ll][b][i]     = out1 flat (b, i l + ll)   (the riffle)
//             out[b][ll][j]   = t[ll][b] . w2[ll][j]                         (F2)
//   backward  dw2[ll]  = dout[:, ll]^T t[ll]                                (B1)
//             dt[ll]   = dout[:, ll] w2[ll]                                 (B2)
//             dout1    = unriffle(dt);  dx[kk] = dout1[kk] w1[kk]           (B3)
//             dw1[kk]  = dout1[kk]^T x[kk]                                  (B4)
// (pretrain/src/models/monarch/monarch_ops.py:23-36, 57-82; the riffle and its
// inverse: monarch_riffle.py:13-57, 60-107.)
//
// The permutations cost no pass of their own: F1's epilogue writes t in riffled
// order (the staged tile is read back with the columns permuted), B3 reads dt
// with its K index permuted (K runs over (ll, j) and its w1 rows are j l + ll),
// B4 computes dw1 with its rows permuted and the split-K reduction writes them
// back in place.  bf16 operands, fp32 accumulation, bf16 results (the rounding
// points of the reference's bf16 bmms: out1, out, dt, dx, dw1, dw2).
//
// One GEMM kernel serves the six products (a second one the forward's two for a few
// tokens), in 256-, 128- and 64-wide tiles (gemm_plan
// picks by the shapes): the MFMA pipeline and LDS slice forms of mfma_tile.hpp,
// operands K-major (K form) or MN-major (T form, read transposed with
// ds_read_b64_tr_b16), staged by buffer loads straight into LDS.  A buffer load
// whose lane offset is beyond the resource's range returns zeros, which pads
// partial tiles (token counts and block sides that are not multiples of the tile)
// without branches in the loop.  The weight-gradient products contract over the
// tokens and have few output tiles; they split K and reduce the fp32 partials
// in a fixed order (deterministic).  The layer's own output is in feature order,
// (B, s l) with feature j l + ll = out[b][ll][j]: F2 can store it so directly, and the
// backward splits dout's blocks in one pass (to_blocks_kernel).
//
// What bounds it, one 6.89B up-projection (4 x 1024 x 1024, 4 x 2752 x 1024) at 4096
// tokens, forward + backward 567 -> 457 us with the output stored in feature order
// (two strided copies of 63-72 us before; now a pass of 33 over the gradient, and F2 takes
// 118 us where the blocked store takes 96): the 256-wide products spend 8 us of a 45 us
// round filling and draining the pipeline, and read and write LDS as long as their MFMAs
// run.  At 4096 tokens of 4 x 512 x 512 the 128-wide tiles took the six products from 157
// to 121 us, at 1000 tokens of 2 x 256 x 256 the 64-wide ones from 125 to 52.  Up to 64
// tokens the forward's two products have a kernel of their own (butterfly_few).
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "kernels.hpp"
#include "mfma_tile.hpp"

namespace mmuon {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Lane offset that reads zeros: the resource covers [0, OOB) bytes.
constexpr uint32_t OOB = 0x80000000u;

// Raw buffer resource over [base, base + OOB): base address, stride 0,
// num_records OOB, the gfx9 data-format word.
__device__ __forceinline__ i32x4 buffer_rsrc(const char* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane(int(low_word(a)));
  r[1] = __builtin_amdgcn_readfirstlane(int(high_word(a) & 0xffffu));
  r[2] = int(OOB);
  r[3] = 0x00020000;
  return r;
}

// 16-B buffer load straight into LDS: lane l lands at lds + 16 l (M0 holds the
// wave-uniform LDS address).  Inline assembly for the same reason as dma16: the
// pipeline waits for exactly the slice it reads.
// m0 is listed as clobbered (the asm writes it); clang warns that m0 is a
// register it reserves for its own uses, which it sets right before each.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void bdma16(i32x4 rsrc, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(lds))
               : "memory", "m0");
}
#pragma clang diagnostic pop

// floor(n / d) for 0 <= n < 2^24, 1 <= d < 2^16, with magic = ceil(2^40 / d)
// (exact because n d < 2^40).
__host__ __device__ __forceinline__ int64_t seg_div(int64_t n, uint64_t magic) {
  return int64_t((uint64_t(n) * magic) >> 40);
}
uint64_t seg_magic(int64_t d) { return ((uint64_t(1) << 40) + uint64_t(d) - 1) / uint64_t(d); }

// GEMM operand: element (mn, k) of batch g sits at
//   base + g bstride + seg(mn) + seg(k),
//   seg(x) = (x / xseg) xseg_stride + (x % xseg) xstride.
// Segments express the riffle permutations; an unsegmented index has
// xseg > its extent.  K form: kstride == 2 (rows of K contiguous); T form:
// mstride == 2 (MN contiguous).  Indices mn >= extent read as zeros.
struct GOp {
  const char* base;
  int64_t bstride;
  int64_t mstride, mseg_stride;
  int64_t kstride, kseg_stride;
  uint64_t mmagic, kmagic;
  int32_t mseg, kseg;
  int32_t extent;
  int32_t pad;
};

__device__ __forceinline__ int64_t mn_off(const GOp& o, int64_t m) {
  const int64_t s = seg_div(m, o.mmagic);
  return s * o.mseg_stride + (m - s * o.mseg) * o.mstride;
}
// An operand's walk over K, one slice of BK at a time.  Segments are whole slices
// (multiples of 32), so a slice lies in one.  (Forming each slice's address from its
// index, a 64-bit division and three products, and testing every load for the end of K
// paced the small tiles: 8 tokens of 4 x 1024 x 1024 11.5 -> 10.4 us, 500 tokens of 4 x
// 512 x 1376 12.7 -> 11.4.  Rings of 8 or 16 slots, and reading a whole slice's fragments
// behind the barrier, did not help them.)
struct KWalk {
  const char* p;       // the slice's first element (tile row 0)
  int64_t step, wrap;  // bytes to the next slice, and beyond that into the next segment
  int pos, seg;        // the slice's place in its segment, the segment's length
  __device__ __forceinline__ void start(const GOp& o, const char* base, int k) {
    const int64_t s = seg_div(k, o.kmagic);
    pos = k - int(s) * o.kseg;
    seg = o.kseg;
    p = base + s * o.kseg_stride + int64_t(pos) * o.kstride;
    step = int64_t(BK) * o.kstride;
    wrap = o.kseg_stride - int64_t(o.kseg) * o.kstride;
  }
  __device__ __forceinline__ void next() {
    p += step;
    pos += BK;
    if (pos == seg) {
      p += wrap;
      pos = 0;
    }
  }
};

// bf16 result: row m of batch g at base + g bstride + seg(m), column n at
// 2 n; riffle (log2 l > 0): column jq of the tile's columns goes to plane
// jq % l, column jq / l (plane stride cplane).
struct GOut {
  char* base;
  int64_t bstride;
  int64_t rstride, rseg_stride;
  int64_t cplane;
  uint64_t rmagic;
  int32_t rseg;
  int32_t log2l;
};

// What the epilogue writes: bf16 rows (c), fp32 partials, or bf16 in feature order
// (column j of batch g at base + row rstride + (j G + g) 2).
enum { OUT_TILE = 0, OUT_PARTIAL = 1, OUT_FEATURES = 2 };
struct GemmArgs {
  GOp a, b;        // row operand (M x K), column operand (N x K)
  GOut c;          // bf16 result (partial == null)
  float* partial;  // split-K: fp32 partials [S][G][M][N]
  int M, N, K, G, S;
  int kchunk;      // K per split, a multiple of BK
  int tile;        // tile geometry
  int tiles_m, tiles_n;
  int vtiles;      // virtual tiles: 8 XCDs x ceil(G * S * tiles_m / 8) groups x tiles_n
};

// ---------------------------------------------------------------------------
// Tile geometries: GM x GN waves, each WI x WJ MFMA tiles of 32 x 32; RING slices
// of 32 k in LDS.
// ---------------------------------------------------------------------------
template <int GM_, int GN_, int WI_, int WJ_, int RING_>
struct Geo {
  static constexpr int GM = GM_, GN = GN_, WI = WI_, WJ = WJ_, RING = RING_;
  static constexpr int NW = GM * GN, NTH = 64 * NW;
  static constexpr int BM = 32 * WI * GM, BN = 32 * WJ * GN;
  static constexpr int RSLB = BM * BK * 2, SLOTB = (BM + BN) * BK * 2;  // bytes of a row slice, of a slot
  static constexpr int RL = BM / 16 / NW, CL = BN / 16 / NW;            // 1 KiB loads per wave and operand slice
  static constexpr int DMA = RL + CL;
  static constexpr int LDS = RING * SLOTB;
  static constexpr int PER_CU = 160 * 1024 / LDS < 4 ? 160 * 1024 / LDS : 4;  // workgroups resident per CU
  static_assert(RL * NW * 16 == BM && CL * NW * 16 == BN, "whole loads per wave");
  static_assert(BM * BN * 2 <= LDS && LDS <= 160 * 1024, "the staged tile fits in the ring");
  // Staged tile T[j][i] = D[i][j]: rows of BM bf16, 16-B chunk c of row r at c ^ g(r),
  // g distinct over the rows that one access touches (mfma_tile.hpp, tile_off; rows of
  // 128 B take two per pass over the banks)
  static __device__ __forceinline__ uint32_t tile_at(int r, int c) {
    const int g = BM >= 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (r >> 1) & 7;
    return uint32_t(r * BM * 2 + (((c >> 3) ^ g) << 4) + ((c & 7) << 1));
  }
};

// ---------------------------------------------------------------------------
// The pipelined main loop (the NS kernels' schedule with both operand forms
// fixed per launch): slice kt in ring slot kt % RING, RING - 2 slices in flight
// behind the one being read, fragment reads and buffer loads interleaved with the
// MFMAs.  (256 x 256 tiles: a fifth slot, the whole LDS, measured slightly slower.)
// ---------------------------------------------------------------------------
template <class GE, bool AT, bool BT>
struct GPipe {
  static constexpr int RING = GE::RING, WI = GE::WI, WJ = GE::WJ, NM = WI * WJ, NR = WI + WJ;
  struct Fr {
    bf16x8 r[WI];
    bf16x8 c[WJ];
  };
  typedef f32x16 Acc[WI][WJ];
  KWalk ak, bk;            // the slice to load next, of the two operands
  int nxt;                 // its index (the last slice stays: it refills consumed slots)
  uint32_t loff[GE::DMA];  // per-lane byte offsets of the loads (OOB: beyond the extent)
  uint32_t tail[GE::DMA];  // OOB where the load's element lies beyond the last slice's K
  int KT;
  int wave, lane, wm, wn;
  char* lds;
  uint32_t lds0;
  uint32_t kfrag[BK / 16];
  uint32_t tfrag_r, tfrag_c;

  __device__ __forceinline__ const uint16_t* slot(int kt) const {
    return reinterpret_cast<const uint16_t*>(lds + (uint32_t(kt) % RING) * GE::SLOTB);
  }

  // Load Q (row operand first) of the next slice into the slot of slice slot_kt.
  // Load u = RL wave + Q (CL wave + Q - RL) of the operand's BM / 16 (BN / 16).
  // K form: operand rows 16 u + lane/4, chunk (lane%4) ^ ((lane>>4)&3); T form: k rows
  // 16 (u%2) + lane/4 of the slice, MN 32 (u/2) + 8 (lane%4).  Either way the load
  // lands at byte 1024 u of the operand's slice.
  template <int Q>
  __device__ __forceinline__ void issue_one(int slot_kt) const {
    constexpr bool ROW = Q < GE::RL;
    const int u = ROW ? GE::RL * wave + Q : GE::CL * wave + Q - GE::RL;
    const uint32_t dst = lds0 + (uint32_t(slot_kt) % RING) * GE::SLOTB + (ROW ? 0 : GE::RSLB) + u * 1024;
    const uint32_t last = nxt == KT - 1 ? OOB : 0;
    bdma16(buffer_rsrc(ROW ? ak.p : bk.p), loff[Q] | (tail[Q] & last), dst);
  }
  template <int Q0, int Q1>
  __device__ __forceinline__ void issue(int slot_kt) const {
    if constexpr (Q0 < Q1) {
      issue_one<Q0>(slot_kt);
      issue<Q0 + 1, Q1>(slot_kt);
    }
  }
  __device__ __forceinline__ void advance() {
    if (nxt + 1 < KT) {
      ak.next();
      bk.next();
      ++nxt;
    }
  }

  template <int KK, int G>
  __device__ __forceinline__ void load_one(int kt, Fr& f) const {
    const uint16_t* sr = slot(kt);
    const uint16_t* sc = sr + GE::RSLB / 2;
    if constexpr (G < WJ)
      f.c[G] = BT ? frag_rowmajor_tr(sc, tfrag_c + G * 2048, KK) : frag_kmajor(sc, kfrag[KK], (wn * WJ + G) * 32);
    else
      f.r[G - WJ] = AT ? frag_rowmajor_tr(sr, tfrag_r + (G - WJ) * 2048, KK)
                       : frag_kmajor(sr, kfrag[KK], (wm * WI + G - WJ) * 32);
  }
  template <int KK, int G0, int G1>
  __device__ __forceinline__ void load(int kt, Fr& f) const {
    if constexpr (G0 < G1) {
      load_one<KK, G0>(kt, f);
      load<KK, G0 + 1, G1>(kt, f);
    }
  }

  // MFMA g of a k step, with its share of the fragment reads of the next step and,
  // in the second k step, of the direct loads
  template <int KK, int g>
  __device__ __forceinline__ void half(int kt, const Fr& f, Fr& n, Acc& acc) const {
    if constexpr (g < NM) {
      acc[g / WJ][g % WJ] = mfma(f.r[g / WJ], f.c[g % WJ], acc[g / WJ][g % WJ]);
      if constexpr (KK == 0) {
        load<1, g * NR / NM, (g + 1) * NR / NM>(kt, n);
      } else {
        load<0, g * NR / NM, (g + 1) * NR / NM>(kt + 1, n);
        issue<g * GE::DMA / NM, (g + 1) * GE::DMA / NM>(kt + RING - 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      half<KK, g + 1>(kt, f, n, acc);
    }
  }

  __device__ __forceinline__ void body(int kt, Fr& fa, Fr& fb, Acc& acc) {
    half<0, 0>(kt, fa, fb, acc);
    wait_vm<(RING - 3) * GE::DMA>();  // slice kt+1 landed
    barrier();
    // raised wave priority from the barrier to the end of k step 1, so the
    // SIMD's wave still in this phase wins issue over one already in the next
    // step and catches up before the next barrier
    __builtin_amdgcn_s_setprio(1);
    half<1, 0>(kt, fb, fa, acc);
    __builtin_amdgcn_s_setprio(0);
    advance();
  }

  __device__ __forceinline__ void run(Acc& acc) {
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j) acc[i][j] = f32x16{};
#pragma unroll
    for (int q = 0; q < RING - 1; ++q) {
      issue<0, GE::DMA>(q);
      advance();
    }
    wait_vm<(RING - 2) * GE::DMA>();  // slice 0 landed
    barrier();
    Fr fa, fb;
    load<0, 0, NR>(0, fa);
    for (int kt = 0; kt < KT; ++kt) body(kt, fa, fb, acc);
    wait_vm<0>();  // the refills of the last steps land before the ring is reused
  }
};

// Per-lane byte offset of load u of an operand (tile origin mn0), OOB beyond
// its extent.
template <bool T>
__device__ __forceinline__ uint32_t lane_offset(const GOp& o, int mn0, int u, int lane) {
  int mn;
  int64_t off;
  if (T) {
    mn = mn0 + 32 * (u >> 1) + 8 * (lane & 3);
    off = int64_t(16 * (u & 1) + (lane >> 2)) * o.kstride;
  } else {
    mn = mn0 + 16 * u + (lane >> 2);
    off = int64_t((lane & 3) ^ ((lane >> 4) & 3)) * 16;
  }
  if (mn >= o.extent) return OOB;
  return uint32_t(off + mn_off(o, mn) - mn_off(o, mn0));
}

// Accumulators -> the staging area as T[j][i] = D[i][j], bf16.
template <class GE>
__device__ __forceinline__ void stage_acc(char* stage, const f32x16 (&acc)[GE::WI][GE::WJ]) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / GE::GN, wn = wave % GE::GN;
#pragma unroll
  for (int i = 0; i < GE::WI; ++i)
#pragma unroll
    for (int j = 0; j < GE::WJ; ++j)
#pragma unroll
      for (int qg = 0; qg < 4; ++qg) {
        const f32x16& v = acc[i][j];
        const int row = (wn * GE::WJ + j) * 32 + (lane & 31);
        const int col = (wm * GE::WI + i) * 32 + qg * 8 + (lane >> 5) * 4;
        *reinterpret_cast<uint2*>(stage + GE::tile_at(row, col)) =
            make_uint2(f2bf2(v[qg * 4], v[qg * 4 + 1]), f2bf2(v[qg * 4 + 2], v[qg * 4 + 3]));
      }
}

// Staged tile -> destination rows.  Tile column order is permuted by the
// riffle: destination position dc (plane dc / (BN/l), column dc % (BN/l))
// holds tile column (dc % (BN/l)) l + dc / (BN/l).  ds_read_b64_tr_b16 on
// 16-lane groups: lanes 4e..4e+3 address staged row (tile column) R(e), four
// consecutive tile rows each, and lane i receives D[i0 + i][R(0..3)].  A wave
// task covers 16 tile rows x 64 destination columns; a lane writes two 16-B
// chunks.  fn(row, dc, uint4) stores destination columns dc .. dc+7 of a row
// (BN / l is a multiple of 8, so they lie in one plane).
constexpr int log2i(int n) { return n <= 1 ? 0 : 1 + log2i(n / 2); }
template <class GE, class Fn>
__device__ __forceinline__ void write_tile(const char* stage, int log2l, Fn&& fn) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, grp = lane >> 4;
  const int wshift = log2i(GE::BN) - log2l, wmask = (1 << wshift) - 1;  // plane width BN / l
  auto trow = [&](int dc) { return ((dc & wmask) << log2l) | (dc >> wshift); };
  constexpr int RB = GE::BM / 16;  // row blocks
#pragma unroll 2
  for (int it = 0; it < RB * (GE::BN / 64) / GE::NW; ++it) {
    const int task = wave + GE::NW * it;
    const int i0 = (task % RB) * 16;
    const int tc = i0 + ((l16 & 3) << 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int dc = (task / RB) * 64 + grp * 16 + h * 8;
      const i16x4 lo =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + GE::tile_at(trow(dc + (l16 >> 2)), tc)));
      const i16x4 hi =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stage + GE::tile_at(trow(dc + 4 + (l16 >> 2)), tc)));
      uint4 v;
      v.x = uint32_t(uint16_t(lo[0])) | (uint32_t(uint16_t(lo[1])) << 16);
      v.y = uint32_t(uint16_t(lo[2])) | (uint32_t(uint16_t(lo[3])) << 16);
      v.z = uint32_t(uint16_t(hi[0])) | (uint32_t(uint16_t(hi[1])) << 16);
      v.w = uint32_t(uint16_t(hi[2])) | (uint32_t(uint16_t(hi[3])) << 16);
      fn(i0 + l16, dc, v);
    }
  }
}

// Virtual tile v -> (batch g, split sp, tile row tm, tile column tn).  A group
// (g, sp, tm) is the tiles_n tiles that share a row-operand band; groups are
// numbered tm fastest and dealt to the XCDs in contiguous runs (virtual tile v
// runs on XCD v % 8), so the tiles of one XCD share one batch's column operand
// and few row bands, and each operand block is fetched from HBM by one or two
// XCDs rather than by all eight.
// Feature-order output: a group is the G tiles (one per batch) of one (tm, tn), which
// write the same lines; groups are numbered tn fastest.
template <bool FEATURES>
__device__ __forceinline__ bool decode_gemm_tile(const GemmArgs& a, int v, int& g, int& sp, int& tm, int& tn) {
  const int xcd = v & 7, local = v >> 3;
  const int per = FEATURES ? a.G : a.tiles_n;  // tiles of a group
  const int ngroups = FEATURES ? a.tiles_m * a.tiles_n : a.G * a.S * a.tiles_m;
  const int gpx = (ngroups + 7) / 8;  // groups per XCD
  const int lg = local / per;
  const int grp = xcd * gpx + lg;
  const int in = local % per;
  if (lg >= gpx || grp >= ngroups) return false;
  if constexpr (FEATURES) {
    g = in;
    sp = 0;
    tn = grp % a.tiles_n;
    tm = grp / a.tiles_n;
  } else {
    tn = in;
    tm = grp % a.tiles_m;
    sp = (grp / a.tiles_m) % a.S;
    g = grp / (a.tiles_m * a.S);
  }
  return true;
}

template <class GE, bool AT, bool BT, int OUT>
__device__ __forceinline__ void gemm_work(const GemmArgs& a, char* lds, int v) {
  int g, sp, tm, tn;
  if (!decode_gemm_tile<OUT == OUT_FEATURES>(a, v, g, sp, tm, tn)) return;
  const int m0 = tm * GE::BM, n0 = tn * GE::BN;
  GPipe<GE, AT, BT> p;
  p.lane = threadIdx.x & 63;
  p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  p.wm = p.wave / GE::GN;
  p.wn = p.wave % GE::GN;
  const int kbeg = sp * a.kchunk, kend = min(a.K, kbeg + a.kchunk);
  p.ak.start(a.a, a.a.base + int64_t(g) * a.a.bstride + mn_off(a.a, m0), kbeg);
  p.bk.start(a.b, a.b.base + int64_t(g) * a.b.bstride + mn_off(a.b, n0), kbeg);
  p.nxt = 0;
  p.KT = (kend - kbeg + BK - 1) / BK;
  const int rem = kend - kbeg - (p.KT - 1) * BK;  // K of the last slice
#pragma unroll
  for (int q = 0; q < GE::DMA; ++q) {
    const bool row = q < GE::RL;
    const int u = row ? GE::RL * p.wave + q : GE::CL * p.wave + q - GE::RL;
    p.loff[q] = row ? lane_offset<AT>(a.a, m0, u, p.lane) : lane_offset<BT>(a.b, n0, u, p.lane);
    // K delta of this lane's load within a slice: K form, its 8-element chunk; T form, its k row
    const int kd = (row ? AT : BT) ? 16 * (u & 1) + (p.lane >> 2) : 8 * ((p.lane & 3) ^ ((p.lane >> 4) & 3));
    p.tail[q] = kd >= rem ? OOB : 0;
  }
  p.lds = lds;
  p.lds0 = lds_addr(lds);
#pragma unroll
  for (int kk = 0; kk < BK / 16; ++kk) p.kfrag[kk] = kmajor_frag_base(kk, p.lane);
  p.tfrag_r = rowmajor_frag_base(p.wm * GE::WI, p.lane);
  p.tfrag_c = rowmajor_frag_base(p.wn * GE::WJ, p.lane);
  f32x16 acc[GE::WI][GE::WJ];
  p.run(acc);

  if constexpr (OUT == OUT_FEATURES) {
    // bf16 straight from the accumulators: column j of batch g is feature j G + g of
    // the row, so a wave store puts 2 B at 32 places 2 G B apart in two rows; the
    // other batches' tiles fill the rest of the lines in the same L2: HBM writes are
    // the output's bytes at 4 x 1024 columns, 2-12% more at 4 x 2752.  Slower than the
    // staged stores of the blocked output (4096 tokens, us): 4 x 1024 x 1024 48.4
    // against 42.9, 4 x 2752 x 1024 118 against 96, 4 x 512 x 512 18.3 against 16.6;
    // for the same order the blocked output needs a copy, 63-72 for the second.  Part of
    // the difference is reading: a group's G tiles share no operand, so 4 x 1024 x 1024
    // fetches 101 MB where F1 of the same size fetches 50
    const GOut& c = a.c;
    const int lane = p.lane;
#pragma unroll
    for (int j = 0; j < GE::WJ; ++j) {
      const int col = n0 + (p.wn * GE::WJ + j) * 32 + (lane & 31);
      if (col >= a.N) continue;
      char* cb = c.base + int64_t(g) * 2 + int64_t(col) * a.G * 2;
#pragma unroll
      for (int i = 0; i < GE::WI; ++i)
#pragma unroll
        for (int qg = 0; qg < 4; ++qg)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = m0 + (p.wm * GE::WI + i) * 32 + qg * 8 + (lane >> 5) * 4 + e;
            if (row < a.M) *reinterpret_cast<uint16_t*>(cb + int64_t(row) * c.rstride) = f2bf(acc[i][j][qg * 4 + e]);
          }
    }
  } else if constexpr (OUT == OUT_PARTIAL) {
    // fp32 partial tile, straight from the accumulators: lane = one column,
    // 16 rows per MFMA tile; a wave store covers two 128-B row segments
    float* P = a.partial + (int64_t(sp) * a.G + g) * int64_t(a.M) * a.N;
    const int lane = p.lane;
#pragma unroll
    for (int i = 0; i < GE::WI; ++i)
#pragma unroll
      for (int j = 0; j < GE::WJ; ++j) {
        const int col = n0 + (p.wn * GE::WJ + j) * 32 + (lane & 31);
        if (col >= a.N) continue;
#pragma unroll
        for (int qg = 0; qg < 4; ++qg)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = m0 + (p.wm * GE::WI + i) * 32 + qg * 8 + (lane >> 5) * 4 + e;
            if (row < a.M) P[int64_t(row) * a.N + col] = acc[i][j][qg * 4 + e];
          }
      }
  } else {
    barrier();  // every wave is done with the ring
    stage_acc<GE>(lds, acc);
    barrier_after_lds_writes();
    const GOut& c = a.c;
    char* cb = c.base + int64_t(g) * c.bstride;
    const int wshift = log2i(GE::BN) - c.log2l;
    const int ncol = (a.N - n0) >> c.log2l;  // valid destination columns per plane
    write_tile<GE>(lds, c.log2l, [&](int r, int dc, const uint4& u) {
      const int row = m0 + r;
      const int plane = dc >> wshift, col = dc & ((1 << wshift) - 1);
      if (row >= a.M || col >= ncol) return;
      const int64_t s = seg_div(row, c.rmagic);
      char* dst = cb + s * c.rseg_stride + (row - s * c.rseg) * c.rstride + plane * c.cplane +
                  int64_t((n0 >> c.log2l) + col) * 2;
      *reinterpret_cast<uint4*>(dst) = u;
    });
  }
}

template <class GE, bool AT, bool BT, int OUT>
__global__ __launch_bounds__(GE::NTH, GE::PER_CU * GE::NW / 4) void butterfly_gemm(GemmArgs a) {
  __shared__ __attribute__((aligned(1024))) char lds[GE::LDS];
  for (int v = blockIdx.x; v < a.vtiles; v += gridDim.x) {
    gemm_work<GE, AT, BT, OUT>(a, lds, v);
    barrier();  // the staging area is read before the next tile's loads refill the ring
  }
}

// ---------------------------------------------------------------------------
// The forward products for a few tokens (generation): 16 features x 16 NT tokens per
// workgroup, all of K.  LW waves load: they keep RING groups of U steps of 32 k in LDS;
// NT waves multiply, one per token tile.
//
// Each output is one chain of MFMAs over K in the order of the tiles above
// (v_mfma_f32_16x16x32_bf16 gives the bits of two v_mfma_f32_32x32x16_bf16 in a row:
// measured on 8192 sums of 1024 products), so a row does not depend on the number of
// tokens that share its call.  Eight waves with an eighth of K each, their partials added
// at the end, were no faster (below, in brackets) and gave other bits.
//
// A 64-wide tile leaves most of the chip idle here (4 x 1024 features are 64 workgroups),
// and a wave issues a 1 KiB load in about 100 cycles, so the loads are spread over four
// waves that do nothing else; the multiplying waves read a group while the products of
// the one before run.  Forward in us at 1 / 8 / 32 / 64 tokens, tiles -> now [split K]:
//   6.89B up     53 / 55 / 55 / 56 -> 7.5 / 8.0 / 11.3 / 16.2  [8.1 / 8.7 / 12.5 / 19.1]
//   6.89B down   83 / 84 / 85 / 85 -> 7.7 / 8.1 / 10.3 / 14.7  [7.3 / 8.2 / 12.2 / 18.0]
//   1.3B query   35 / 36 / 36 / 36 -> 5.1 / 5.5 /  6.2 /  7.6  [5.4 / 5.5 /  6.5 /  8.6]
// (tiles: the 256-wide ones and the interleaving copy; the 64-wide tiles take 22.6, 30.9
// and 12.6 us at 65 tokens).  With weights that come from HBM (a rotation through 512 MB)
// the first takes 11.1 / 11.5 / 16.3 / 20.5 us, the second 11.8 / 12.2 / 14.6 / 18.9.
// What bounds it: of the 8.0 us at 8 tokens, two dependent launches that fill and drain
// take 4.9 (the toy up-projection, 1 MB of weights); the rest reads 31 MB of weights, at
// 10 TB/s from the Infinity Cache or 4.7 from HBM.  Each workgroup reads all tokens again,
// which is what grows with them.  A single wave that loads and multiplies took 9.1 and
// 12.1 us (first and second at 8 tokens); groups of eight steps in three slots 9.8 and
// 8.5; six slots 8.5 and 8.2, five with NT > 1 12.2 us at 32 tokens and 18.4 at 64 (fewer
// workgroups per CU); eight loading waves 8.7 and 8.5.
// ---------------------------------------------------------------------------
constexpr int FEW_TOKENS = 64;  // largest number of tokens
constexpr int FEW_K = 32;       // k of a step

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int NT, int LW, int U, int RING, bool FEATURES>
__global__ __launch_bounds__(64 * (LW + NT)) void butterfly_few(GemmArgs a) {
  constexpr int TILES = 1 + NT;             // 1 KiB loads of a step: the features, the token tiles
  constexpr int PW = U * TILES / LW;        // loads per loading wave and group
  constexpr int GROUPB = U * TILES * 1024;  // LDS bytes of a group
  static_assert(PW * LW == U * TILES && RING >= 2 && PW * RING <= 63, "whole loads per wave, counted by vmcnt");
  __shared__ __attribute__((aligned(1024))) char lds[RING * GROUPB];
  const int g = blockIdx.x / a.tiles_n, n0 = (blockIdx.x % a.tiles_n) * 16;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave < LW) {
    // load q of this wave in a group: load u = wave + LW q, tile u % TILES of step u / TILES.
    // A lane loads row lane/4, 16-B chunk of the step's 64 B at (lane%4) ^ (row/4)%4.
    const int lrow = lane >> 2, lk = ((lane & 3) ^ ((lane >> 4) & 3)) * 8;
    const i32x4 wr = buffer_rsrc(a.b.base + int64_t(g) * a.b.bstride + n0 * a.b.mstride);
    const i32x4 xr = buffer_rsrc(a.a.base + int64_t(g) * a.a.bstride);
    uint32_t off[PW];  // lane offset in the group that starts at k = 0; OOB beyond M and N
    int kq[PW];        // this lane's k within the group
#pragma unroll
    for (int q = 0; q < PW; ++q) {
      const int u = wave + LW * q, tile = u % TILES, row = (tile == 0 ? 0 : (tile - 1) * 16) + lrow;
      kq[q] = (u / TILES) * FEW_K + lk;
      const bool in = tile == 0 ? n0 + lrow < a.N : row < a.M;
      off[q] = in ? uint32_t(row * (tile == 0 ? a.b.mstride : a.a.mstride)) + kq[q] * 2 : OOB;
    }
    const uint32_t lds0 = lds_addr(lds) + wave * 1024;
    // the group that starts at k; beyond K it loads zeros
    auto issue = [&](int k, int slot) {
#pragma unroll
      for (int q = 0; q < PW; ++q) {
        const int u = wave + LW * q;
        const bool in = off[q] != OOB && k + kq[q] < a.K;
        bdma16(u % TILES == 0 ? wr : xr, in ? off[q] + uint32_t(k) * 2 : OOB, lds0 + slot * GROUPB + LW * q * 1024);
      }
    };
#pragma unroll
    for (int r = 0; r < RING - 1; ++r) issue(FEW_K * U * r, r);
    int slot = RING - 1;
    for (int k = 0; k < a.K; k += FEW_K * U) {
      wait_vm<(RING - 2) * PW>();  // this wave's loads of the group landed
      barrier();                   // every wave's, and the group before is read
      issue(k + FEW_K * U * (RING - 1), slot);
      slot = slot + 1 == RING ? 0 : slot + 1;
    }
    wait_vm<0>();  // no load is left in flight to LDS that another workgroup may own next
    return;
  }
  const int tile = wave - LW, l16 = lane & 15;
  // fragments: row lane%16, k 8 (lane/16) .. +7
  const char* const frag = lds + l16 * 64 + (((lane >> 4) ^ (l16 >> 2)) << 4);
  struct Fr {
    bf16x8 w[U], x[U];
  };
  f32x4 acc = {};
  int k = 0, slot = 0;
  auto read = [&](Fr& f) {  // the group that the barrier just completed
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const char* s = frag + slot * GROUPB + u * TILES * 1024;
      f.w[u] = *reinterpret_cast<const bf16x8*>(s);
      f.x[u] = *reinterpret_cast<const bf16x8*>(s + (1 + tile) * 1024);
    }
    slot = slot + 1 == RING ? 0 : slot + 1;
    k += FEW_K * U;
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mul = [&](const Fr& f) {
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.x[u], f.w[u], acc, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto next_group = [&] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this group is read: its slot may be loaded again
    barrier();
  };
  Fr fa, fb;
  barrier();
  read(fa);
  while (k < a.K) {
    next_group();
    read(fb);
    mul(fa);
    if (k >= a.K) {
      fa = fb;
      break;
    }
    next_group();
    read(fa);
    mul(fb);
  }
  mul(fa);
  // lane: feature l16, tokens 4 (lane/16) .. +3 of the wave's token tile
  const int col = n0 + l16;
  if (col >= a.N) return;
  char* dst = a.c.base;
  if (FEATURES)
    dst += (int64_t(col) * a.G + g) * 2;
  else
    dst += int64_t(g) * a.c.bstride + (col & ((1 << a.c.log2l) - 1)) * a.c.cplane + int64_t(col >> a.c.log2l) * 2;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int tok = tile * 16 + (lane >> 4) * 4 + e;
    if (tok < a.M) *reinterpret_cast<uint16_t*>(dst + int64_t(tok) * a.c.rstride) = f2bf(acc[e]);
  }
}

// Split-K reduction: out row seg(m) of batch g, columns n..n+7 =
// bf16(sum over splits, in split order, of the fp32 partials).  S = 0 writes zeros.
__global__ __launch_bounds__(256) void splitk_reduce(const float* partial, int S, int G, int M, int N, GOut c) {
  const int n8 = N / 8;
  const int64_t total = int64_t(G) * M * n8;
  for (int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x; t < total; t += int64_t(gridDim.x) * 256) {
    const int n = int(t % n8) * 8;
    const int64_t gm = t / n8;
    const int m = int(gm % M), g = int(gm / M);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < S; ++s) {
      const float* p = partial + ((int64_t(s) * G + g) * M + m) * int64_t(N) + n;
      const float4 x = reinterpret_cast<const float4*>(p)[0];
      const float4 y = reinterpret_cast<const float4*>(p)[1];
      v[0] += x.x; v[1] += x.y; v[2] += x.z; v[3] += x.w;
      v[4] += y.x; v[5] += y.y; v[6] += y.z; v[7] += y.w;
    }
    const int64_t sg = seg_div(m, c.rmagic);
    uint16_t* dst = reinterpret_cast<uint16_t*>(c.base + int64_t(g) * c.bstride + sg * c.rseg_stride +
                                                (m - sg * c.rseg) * c.rstride) + n;
    uint4 r;
    r.x = f2bf2(v[0], v[1]);
    r.y = f2bf2(v[2], v[3]);
    r.z = f2bf2(v[4], v[5]);
    r.w = f2bf2(v[6], v[7]);
    *reinterpret_cast<uint4*>(dst) = r;
  }
}

// Feature order (B, s l) -> blocked rows (B, l, s): feature j l + b of a row is column j
// of block b.  A thread reads 8 consecutive features (16 B) and writes 8 / l columns of
// each block (one column of 8 of the 16 blocks), so a wave reads 1 KiB runs and writes
// runs of 1 KiB / l per block.  Bound by the copy rate: 4096 rows of 4 x 2752 are read
// and written (90 MB each way, both counted at the L2) in 33 us, 5.4 TB/s, which is what a
// large copy reaches; 4 x 1024 in 14.8 us, 4.5 TB/s.  A strided copy by torch took 61.
template <int L>
__global__ __launch_bounds__(256) void to_blocks_kernel(const uint16_t* src, uint16_t* dst, int64_t chunks, int s) {
  constexpr int U = 4;                        // chunks per thread
  constexpr int C = L >= 8 ? 1 : 8 / L;       // columns per chunk and block
  typedef uint16_t ColV __attribute__((ext_vector_type(C)));
  const int cpr = s * L / 8;                  // chunks per row
  const int64_t base = int64_t(blockIdx.x) * (256 * U) + threadIdx.x;
  uint4 w[U];
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (base + u * 256 < chunks) w[u] = *reinterpret_cast<const uint4*>(src + (base + u * 256) * 8);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * 256;
    if (i >= chunks) continue;
    const int64_t row = i / cpr;
    const int f = int(i - row * cpr) * 8;     // first feature of the chunk
    uint16_t* d = dst + row * (int64_t(s) * L) + int64_t(f % L) * s + f / L;
    const uint32_t q[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
    for (int b = 0; b < 8 / C; ++b) {
      ColV v;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int k = c * (8 / C) + b;
        v[c] = uint16_t(q[k >> 1] >> (16 * (k & 1)));
      }
      *reinterpret_cast<ColV*>(d + int64_t(b) * s) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Host side: the six products as GemmArgs.
// ---------------------------------------------------------------------------
constexpr int64_t UNSEG = int64_t(1) << 24;  // segment length of an unsegmented index

GOp make_op(const void* base, int64_t bstride, int64_t mstride, int64_t kstride, int extent,
            int64_t mseg = UNSEG, int64_t mseg_stride = 0, int64_t kseg = UNSEG, int64_t kseg_stride = 0) {
  GOp o{};
  o.base = static_cast<const char*>(base);
  o.bstride = bstride;
  o.mstride = mstride;
  o.kstride = kstride;
  o.mseg = int32_t(mseg);
  o.mseg_stride = mseg_stride;
  o.kseg = int32_t(kseg);
  o.kseg_stride = kseg_stride;
  o.mmagic = seg_magic(mseg);
  o.kmagic = seg_magic(kseg);
  o.extent = extent;
  return o;
}

GOut make_out(void* base, int64_t bstride, int64_t rstride, int64_t rseg = UNSEG, int64_t rseg_stride = 0,
              int log2l = 0, int64_t cplane = 0) {
  GOut c{};
  c.base = static_cast<char*>(base);
  c.bstride = bstride;
  c.rstride = rstride;
  c.rseg = int32_t(rseg);
  c.rseg_stride = rseg_stride;
  c.rmagic = seg_magic(rseg);
  c.log2l = log2l;
  c.cplane = cplane;
  return c;
}

int cdiv(int64_t a, int64_t b) { return int((a + b - 1) / b); }

typedef Geo<2, 4, 4, 2, 4> G256;  // 256 x 256 tiles, one workgroup per CU
typedef Geo<2, 2, 2, 2, 4> G128;  // 128 x 128, two per CU
typedef Geo<2, 2, 1, 1, 4> G64;   // 64 x 64, four per CU
enum { T256 = 0, T128 = 1, T64 = 2 };

// Tile size and number of K splits of a product, by a model of its time in ns on a
// 256-CU part (a function of the shapes only, so the summation order, and with it the
// result, does not depend on the device).  Large tiles read least per FLOP, small ones
// fill the chip and have shorter prologues and epilogues.  Fitted to kernel times
// (4096 tokens unless noted, us at 256 / 128 / 64-wide tiles): 4 x 512 x 512 products
// 21.8 / 18.2 / 29.8, their weight gradients in 4 splits 29.8 / 18.6 / 29.8; 4 x 1024 x
// 1024 44 / 58 / 96; 1000 tokens of 2 x 256 x 256 14.4 / 8.8 / 7.1; 8 tokens of 4 x 1024
// x 1024 26 / 14 / 12.  (256 x 128 tiles, two workgroups per CU, were slower than 256 x
// 256 wherever those fill the chip: 54 against 46 us on 16384 tokens of 2 x 512 x 1368.)
// A last round of few 256-wide tiles runs at their unloaded rate: 288 of them (2049 tokens
// of 4 x 2048 x 2048) 100 us a product against 109 in 128-wide ones, with K = 2464 (8 x 1024)
// 173 / 194 both products, 576 (9000 tokens of 8 x 512 x 512) 65 / 68.  Counted for the
// products whose sums do not depend on the choice; a weight gradient's splits stay.
struct GemmPlan {
  int tile, S;
};
int64_t gemm_cost(int tile, int64_t M, int64_t N, int64_t G, int64_t K, int64_t S, bool wgrad) {
  const int64_t side = tile == T256 ? 256 : tile == T128 ? 128 : 64;
  const int64_t tiles = G * S * ((M + side - 1) / side) * ((N + side - 1) / side);
  const int64_t rounds = (tiles + 255) / 256, k = (K + S - 1) / S;
  const auto one_round = [k](int64_t n) { return n > 0 ? 8000 + k * (22 + 14 * n / 256) : 0; };
  int64_t t;
  if (tile == T256 && !wgrad) t = tiles / 256 * one_round(256) + one_round(tiles % 256);
  else if (tile == T256) t = rounds * (8000 + k * (22 + 14 * std::min<int64_t>(tiles, 256) / 256));
  else if (tile == T128) t = 4000 + rounds * (1000 + k * (wgrad ? 14 : rounds == 1 ? 9 : rounds == 2 ? 11 : 14));
  else t = 4700 + std::max<int64_t>(tiles, 256) * (300 + k * 13 / 2) / 256;
  // splits: the partials' write and read, and the reduction's launch
  return S > 1 ? t + 4000 + S * G * M * N / 1400 : t;
}
// wgrad: a weight gradient, contracted over the tokens, whose K may be split (at least
// 256 tokens per split).  no64: without the 64-wide tile.
GemmPlan gemm_plan(int64_t M, int64_t N, int64_t G, int64_t K, bool wgrad, bool no64 = false) {
  GemmPlan best{T256, 1};
  int64_t best_cost = gemm_cost(T256, M, N, G, K, 1, wgrad);
  for (int S = 1; S <= 64 && (S == 1 || (wgrad && K >= int64_t(S) * 256)); S *= 2)
    for (int tile = T256; tile <= (no64 ? T128 : T64); ++tile) {
      const int64_t c = gemm_cost(tile, M, N, G, K, S, wgrad);
      if (c < best_cost) best = GemmPlan{tile, S}, best_cost = c;
    }
  return best;
}

void set_geometry(GemmArgs& a, int M, int N, int K, int G, GemmPlan plan) {
  a.M = M;
  a.N = N;
  a.K = K;
  a.G = G;
  a.tile = plan.tile;
  if (plan.S > 1) {
    a.kchunk = cdiv(cdiv(K, plan.S), BK) * BK;
    a.S = cdiv(K, a.kchunk);
  } else {
    a.kchunk = cdiv(std::max(K, 1), BK) * BK;
    a.S = 1;
  }
}

template <class GE, bool AT, bool BT, int OUT>
void launch_gemm_g(GemmArgs a, hipStream_t s) {
  a.tiles_m = cdiv(a.M, GE::BM);
  a.tiles_n = cdiv(a.N, GE::BN);
  a.vtiles = OUT == OUT_FEATURES ? 8 * cdiv(int64_t(a.tiles_m) * a.tiles_n, 8) * a.G
                                 : 8 * cdiv(int64_t(a.G) * a.S * a.tiles_m, 8) * a.tiles_n;
  const int grid = std::min(a.vtiles, resident_grid(1 << 30) * GE::PER_CU);
  hipLaunchKernelGGL((butterfly_gemm<GE, AT, BT, OUT>), dim3(grid), dim3(GE::NTH), 0, s, a);
}
template <bool AT, bool BT, int OUT>
void launch_gemm_t(const GemmArgs& a, hipStream_t s) {
  if (a.tile == T256) launch_gemm_g<G256, AT, BT, OUT>(a, s);
  else if (a.tile == T128) launch_gemm_g<G128, AT, BT, OUT>(a, s);
  else launch_gemm_g<G64, AT, BT, OUT>(a, s);
}

// Products that take butterfly_few.  It reads all tokens once per 16 features, so with
// many features the 64-wide tiles, once they fill the chip, overtake it: at 512 of them from
// 17 tokens on (16 x 2048 x 2048, forward us, few / tiles: 16 tokens 58 / 60, 17 68 / 61, 64
// 124 / 65), at 256 between 33 and 64 (16 x 1024 x 1024: 32 tokens 22.7 / 25.0, 33 25.7 /
// 24.9, 64 33 / 27; 8 x 2048 x 2048 35.9 / 35.3, 36.4 / 35.5, 46 / 37; 4 x 4096 x 4096 70 /
// 94, 78 / 93, 103 / 100), below not up to 64 (8 x 1024 x 1024, 128 tiles: 19.0 / 22.0).
bool few_tokens(const GemmArgs& a) {
  if (a.M > FEW_TOKENS) return false;
  const int64_t tiles = int64_t(a.G) * cdiv(a.N, 64);
  return a.M <= 16 || tiles < 256 || tiles * cdiv(a.M, 16) <= 512;
}

template <int NT, int RING, bool FEATURES>
void launch_few_t(const GemmArgs& a, hipStream_t s) {
  constexpr int LW = 4, U = 4;
  const dim3 grid(unsigned(a.G * a.tiles_n)), block(64 * (LW + NT));
  hipLaunchKernelGGL((butterfly_few<NT, LW, U, RING, FEATURES>), grid, block, 0, s, a);
}
template <bool FEATURES>
void launch_few(GemmArgs a, hipStream_t s) {
  a.tiles_n = cdiv(a.N, 16);
  if (a.M <= 16) launch_few_t<1, 5, FEATURES>(a, s);
  else if (a.M <= 32) launch_few_t<2, 4, FEATURES>(a, s);
  else launch_few_t<4, 4, FEATURES>(a, s);
}

void launch_reduce(const GemmArgs& a, const GOut& c, hipStream_t s) {
  const int64_t total = int64_t(a.G) * a.M * (a.N / 8);
  const int blocks = int(std::min<int64_t>(std::max<int64_t>(1, (total + 255) / 256), 8192));
  hipLaunchKernelGGL(splitk_reduce, dim3(blocks), dim3(256), 0, s, a.partial, a.K > 0 ? a.S : 0, a.G, a.M, a.N, c);
}

void launch_to_blocks(const void* src, void* dst, int64_t rows, int l, int s, hipStream_t st) {
  const int64_t chunks = rows * l * s / 8;
  const dim3 grid(unsigned((chunks + 1023) / 1024)), block(256);
  const auto* a = static_cast<const uint16_t*>(src);
  auto* b = static_cast<uint16_t*>(dst);
  switch (l) {
    case 2: hipLaunchKernelGGL(to_blocks_kernel<2>, grid, block, 0, st, a, b, chunks, s); break;
    case 4: hipLaunchKernelGGL(to_blocks_kernel<4>, grid, block, 0, st, a, b, chunks, s); break;
    case 8: hipLaunchKernelGGL(to_blocks_kernel<8>, grid, block, 0, st, a, b, chunks, s); break;
    default: hipLaunchKernelGGL(to_blocks_kernel<16>, grid, block, 0, st, a, b, chunks, s); break;
  }
}

struct Dims {
  int64_t B;
  int nb, q, p, s, log2l;
};

Dims dims(const mmuon_butterfly_args& x) {
  Dims d{x.tokens, x.nblocks, x.q, x.p, x.s, 0};
  while ((1 << d.log2l) < d.nb) ++d.log2l;
  return d;
}

}  // namespace

// Weight gradients: dw2 (s x q per block) and dw1 (q x p), contracted over the tokens.
GemmPlan dw2_plan(const Dims& d) { return gemm_plan(d.s, d.q, d.nb, d.B, true); }
GemmPlan dw1_plan(const Dims& d) { return gemm_plan(d.q, d.p, d.nb, d.B, true); }

size_t round256(size_t n) { return (n + 255) / 256 * 256; }

size_t butterfly_workspace(const mmuon_butterfly_args& x) {
  const Dims d = dims(x);
  const size_t dt = size_t(d.nb) * d.B * d.q * 2;
  const int s1 = dw2_plan(d).S, s4 = dw1_plan(d).S;
  const size_t part = std::max(size_t(s1) * d.nb * d.s * d.q, size_t(s4) * d.nb * d.q * d.p) * 4;
  return round256(dt) + part;
}
size_t butterfly_linear_workspace(const mmuon_butterfly_args& x) {
  return butterfly_workspace(x) + (x.nblocks > 1 ? round256(size_t(x.nblocks) * x.tokens * x.s * 2) : 0);
}

// features: out in feature order (B, s l) instead of (B, l, s)
int launch_butterfly_fwd(const mmuon_butterfly_args& x, bool features, hipStream_t st) {
  const Dims d = dims(x);
  if (d.B == 0) return 0;
  const int64_t n = int64_t(d.nb) * d.p, ql = d.q / d.nb;
  GemmArgs f1{};  // out1 (riffled into t) = x . w1^T per block kk
  f1.a = make_op(x.x, d.p * 2, n * 2, 2, int(d.B));
  f1.b = make_op(x.w1, int64_t(d.q) * d.p * 2, int64_t(d.p) * 2, 2, d.q);
  f1.c = make_out(x.out1, ql * 2, int64_t(d.q) * 2, UNSEG, 0, d.log2l, d.B * d.q * 2);
  // (a 64-wide tile of 16 planes would write runs shorter than 16 B)
  set_geometry(f1, int(d.B), d.q, d.p, d.nb, gemm_plan(d.B, d.q, d.nb, d.p, false, d.nb > 8));
  if (few_tokens(f1)) launch_few<false>(f1, st);
  else launch_gemm_t<false, false, OUT_TILE>(f1, st);
  GemmArgs f2{};  // out[:, ll] = t[ll] . w2[ll]^T
  f2.a = make_op(x.out1, d.B * d.q * 2, int64_t(d.q) * 2, 2, int(d.B));
  f2.b = make_op(x.w2, int64_t(d.s) * d.q * 2, int64_t(d.q) * 2, 2, d.s);
  f2.c = make_out(x.out, int64_t(d.s) * 2, int64_t(d.nb) * d.s * 2);
  set_geometry(f2, int(d.B), d.s, d.q, d.nb, gemm_plan(d.B, d.s, d.nb, d.q, false));
  const bool few = few_tokens(f2);
  if (few && features && d.nb > 1) launch_few<true>(f2, st);
  else if (few) launch_few<false>(f2, st);
  else if (features && d.nb > 1) launch_gemm_t<false, false, OUT_FEATURES>(f2, st);
  else launch_gemm_t<false, false, OUT_TILE>(f2, st);
  return 0;
}

// features: dout in feature order (B, s l) instead of (B, l, s)
int launch_butterfly_bwd(const mmuon_butterfly_args& xa, bool features, hipStream_t st) {
  mmuon_butterfly_args x = xa;
  const Dims d = dims(x);
  const int64_t n = int64_t(d.nb) * d.p, ql = d.q / d.nb;
  char* ws = static_cast<char*>(x.workspace);
  if (features && d.nb > 1 && d.B > 0) {
    launch_to_blocks(x.dout, ws, d.B, d.nb, d.s, st);
    x.dout = ws;
    ws += round256(size_t(d.nb) * d.B * d.s * 2);
  }
  void* dt = ws;
  float* part = reinterpret_cast<float*>(ws + round256(size_t(d.nb) * d.B * d.q * 2));

  // dw2[ll] = dout[:, ll]^T t[ll]  (K = tokens, split; unsplit: bf16 straight
  // from the tile)
  GemmArgs b1{};
  b1.a = make_op(x.dout, int64_t(d.s) * 2, 2, int64_t(d.nb) * d.s * 2, d.s);
  b1.b = make_op(x.out1, d.B * d.q * 2, 2, int64_t(d.q) * 2, d.q);
  b1.partial = part;
  b1.c = make_out(x.dw2, int64_t(d.s) * d.q * 2, int64_t(d.q) * 2);
  set_geometry(b1, d.s, d.q, int(d.B), d.nb, dw2_plan(d));
  if (d.B > 0 && b1.S == 1) {
    launch_gemm_t<true, true, OUT_TILE>(b1, st);
  } else {
    if (d.B > 0) launch_gemm_t<true, true, OUT_PARTIAL>(b1, st);
    launch_reduce(b1, b1.c, st);
  }
  if (d.B == 0) {
    GemmArgs b4{};
    b4.partial = part;
    set_geometry(b4, d.q, d.p, 0, d.nb, GemmPlan{T256, 1});
    launch_reduce(b4, make_out(x.dw1, int64_t(d.q) * d.p * 2, int64_t(d.p) * 2), st);
    return 0;
  }

  GemmArgs b2{};  // dt[ll] = dout[:, ll] w2[ll]
  b2.a = make_op(x.dout, int64_t(d.s) * 2, int64_t(d.nb) * d.s * 2, 2, int(d.B));
  b2.b = make_op(x.w2, int64_t(d.s) * d.q * 2, 2, int64_t(d.q) * 2, d.q);
  b2.c = make_out(dt, d.B * d.q * 2, int64_t(d.q) * 2);
  set_geometry(b2, int(d.B), d.q, d.s, d.nb, gemm_plan(d.B, d.q, d.nb, d.s, false));
  launch_gemm_t<false, true, OUT_TILE>(b2, st);

  // dx[:, kk] = sum over (ll, j) of dt[ll][:, kk q/l + j] w1[kk][j l + ll]: K in
  // segments of q/l, one per plane ll (the unriffle folded into the addressing)
  GemmArgs b3{};
  b3.a = make_op(dt, ql * 2, int64_t(d.q) * 2, 2, int(d.B), UNSEG, 0, ql, d.B * d.q * 2);
  b3.b = make_op(x.w1, int64_t(d.q) * d.p * 2, 2, int64_t(d.nb) * d.p * 2, d.p, UNSEG, 0, ql, int64_t(d.p) * 2);
  b3.c = make_out(x.dx, int64_t(d.p) * 2, n * 2);
  set_geometry(b3, int(d.B), d.p, d.q, d.nb, gemm_plan(d.B, d.p, d.nb, d.q, false));
  launch_gemm_t<false, true, OUT_TILE>(b3, st);

  // dw1[kk] with rows in (ll, j) order: row ll q/l + j of the product is
  // dw1 row j l + ll (the reduction writes it there)
  GemmArgs b4{};
  b4.a = make_op(dt, ql * 2, 2, int64_t(d.q) * 2, d.q, ql, d.B * d.q * 2);
  b4.b = make_op(x.x, int64_t(d.p) * 2, 2, n * 2, d.p);
  b4.partial = part;
  b4.c = make_out(x.dw1, int64_t(d.q) * d.p * 2, int64_t(d.nb) * d.p * 2, ql, int64_t(d.p) * 2);
  set_geometry(b4, d.q, d.p, int(d.B), d.nb, dw1_plan(d));
  if (b4.S == 1) {
    launch_gemm_t<true, true, OUT_TILE>(b4, st);
  } else {
    launch_gemm_t<true, true, OUT_PARTIAL>(b4, st);
    launch_reduce(b4, b4.c, st);
  }
  return 0;
}

}  // namespace mmuon
