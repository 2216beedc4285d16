// Wave-tile GEMMs C[M, N] = A[M, K] W[N, K]^T for few bf16 rows (M <= WT_MAX_M): a decode step's
// projection, refine, W_O and MLP products, the steps of the exact scan, and the sweep GEMMs of
// cells with few rows (small batches, long layers).
//
// With so few rows neither the matrix cores nor HBM bound a product but how the loads are spread
// over the chip: 64-wide block tiles leave most of the 256 CUs without work, and a block's waves
// walk K in step, each 64-wide step a round trip behind a barrier. Here one wave is the whole block:
// it owns 8 NA rows x 16 CT columns over all of K, fills a private ring of S LDS stages straight from
// global memory (S - 1 of the 64-wide k steps in flight, no register held by a load) and waits for
// its own loads only; there is no barrier. A load instruction moves eight whole 128-byte lines
// (fragments loaded straight into registers, half a line per row, moved half as many bytes per clock
// of a CU). The tile is chosen (with_wt) so that the waves spread over the CUs.
// Measured on MI355X (K = 1024, weights from HBM, plain store; launch alone 2.3 us):
//   M =   8, N = 4096: 3.9 us, N = 6144: 4.3     (64 x 64 block tiles in place: 12.1, 9.5 with their epilogues)
//   M =  64, N = 4096: 5.8;  M = 128: 6.7;  M = 256: 9.0
// With more rows or wider operands sharing them between a block's waves wins; each product's rule says where.
// The order of an output's sum over k is fixed by the product, not by the tile that computes it (WtSum): the
// products that larger calls run on the tiled GEMMs sum as those do, one chain over ascending 32-wide MFMA
// steps; a step's W_O and MLP products, of 1 to ROWS_MAX rows, sum partial chains (a W_O of more rows one
// chain). So a row's result is the same in every batch of either kind.
//
// An epilogue chooses the 16 CT weight rows of a tile (wrow), so that its items are complete inside
// the tile (a RoPE pair, a key's candidate and gate halves), gathers its inputs ahead of the k-loop
// (prefetch) and sees the tile staged in LDS (apply).
#pragma once

#include <utility>

#include "dm_kernels.h"

namespace dm {

constexpr int WT_MAX_M = 256;
constexpr int ROWS_MAX = 64;   // rows of a decode-style call (dm_swiglu_rows)

template <int NA_, int CT_, int S_ = 0> struct WTile {
  static constexpr int NA = NA_, CT = CT_;              // 8-row groups of A, 16-column tiles of W
  static constexpr int RT = (NA + 1) / 2;               // 16-row MFMA tiles
  static constexpr int ROWS = 8 * NA, COLS = 16 * CT;
  static constexpr int L = 2 * CT + NA;                 // load instructions per stage
  static constexpr int S = S_ > 0 ? S_ : (L <= 4 ? 8 : (L <= 6 ? 10 : (L <= 8 ? 7 : 5)));   // stages (measured)
  static constexpr int STAGE = (16 * CT + 8 * NA) * 128;
  static constexpr int LDT = COLS + 4;                  // floats per row of the staged output tile
  static constexpr int LDS = S * STAGE;
  static_assert((S - 1) * L < 64, "vmcnt range");
  static_assert(16 * RT * LDT * 4 + ROWS * 4 <= LDS, "the output tile and its row scales fit the stages");
};

template <int... I, class F> DM_DEV void static_steps(std::integer_sequence<int, I...>, const F& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// The order of the sum over k: one chain of ascending 32-wide MFMA steps; four chains over K's quarters
// (K a multiple of 128), added in order; or eight chains, the j-th over the steps j, j + 8, ..., added in
// order. One wave walks the quarters one after the other, the eighths as four pairs (steps j, j + 1 share
// a 64-wide load; eight accumulators per output over an ascending walk: W_O at d = 1024 6.1 us against
// 4.7); four waves (k_wt_ksplit) take a quarter or a pair each: the same sums.
enum WtSum { WT_CHAIN = 0, WT_QUARTERS = 1, WT_EIGHTHS = 2 };
constexpr int WT_PARTS = 4;   // quarters, or pairs of eighths
template <int SUM, bool PART> struct WtWalk {   // over the 64-wide loads of one part, or of all
  int K, k, end, part;
  static constexpr bool PARTS = SUM != WT_CHAIN && !PART;
  static constexpr int STRIDE = SUM == WT_EIGHTHS ? 64 * WT_PARTS : 64;
  DM_DEV WtWalk(int K_, int part_) : K(K_), k(0), end(K_), part(part_) { set(); }
  DM_DEV void set() {
    if (SUM == WT_EIGHTHS) k = 64 * part;
    if (SUM == WT_QUARTERS) {
      k = part * (K / 4);
      end = k + K / 4;
    }
  }
  DM_DEV bool last() const { return k + STRIDE >= end; }   // of its part
  DM_DEV void next() {
    k += STRIDE;
    if (PARTS && k >= end) {
      ++part;
      set();
    }
  }
  DM_DEV int steps() const {
    if (SUM == WT_QUARTERS) return (PARTS ? WT_PARTS : 1) * ((K / 4 + 63) / 64);
    return SUM == WT_EIGHTHS && PART ? max(0, (K - 64 * part + STRIDE - 1) / STRIDE) : (K + 63) / 64;
  }
};

template <typename T> struct WtOp {   // the A operand: row m at A + m lda; K a multiple of 32
  const T* A;
  long lda;
  int M, K, nx;   // nx column tiles
};

// The sums of one tile (column tile bx, row tile by) by one wave: every part of E's sum into acc[0], or
// with PART only part `part` (its two chains of eighths apart in acc[0] and acc[1]); leaves the stages free.
template <typename T, class WT, bool PART, class E>
DM_DEV void wt_kloop(const E& e, const WtOp<T>& op, int bx, int by, int part, char* smem,
                     floatx4 (&acc)[E::SUM == WT_EIGHTHS ? 2 : 1][WT::RT][WT::CT]) {
  using MF = Mfma<T>;
  constexpr int NA = WT::NA, CT = WT::CT, RT = WT::RT, S = WT::S, L = WT::L, SUM = E::SUM;
  constexpr bool FLUSH = SUM != WT_CHAIN && !PART;   // chains added up on the way
  constexpr int NC = SUM == WT_EIGHTHS ? 2 : 1;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;   // the lane's row of an 8-row load; its 16-byte chunk, swizzled
  const int m0 = by * WT::ROWS, K = op.K;
  const T* pw[2 * CT];
  const T* pa[NA];
#pragma unroll
  for (int i = 0; i < 2 * CT; ++i) pw[i] = e.wrow(bx, WT{}, 8 * i + lr);
#pragma unroll
  for (int i = 0; i < NA; ++i) pa[i] = op.A + (long)min(m0 + 8 * i + lr, op.M - 1) * op.lda;   // past M: row M - 1 again
  WtWalk<SUM, PART> wi(K, PART ? part : 0), wc = wi;   // of the loads issued, of the steps computed
  auto issue = [&](int kt, int st) {
    char* b = smem + st * WT::STAGE;
    const int k = min((SUM == WT_CHAIN ? 64 * kt : wi.k) + 8 * lc, K - 8);   // a half last step: chunks past K read K's last, unused
#pragma unroll
    for (int i = 0; i < 2 * CT; ++i)
      __builtin_amdgcn_global_load_lds((const void*)(pw[i] + k), (lds_void_t*)(b + i * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < NA; ++i)
      __builtin_amdgcn_global_load_lds((const void*)(pa[i] + k), (lds_void_t*)(b + (2 * CT + i) * 1024), 16, 0, 0);
    wi.next();
  };
  floatx4 chain[NC][RT][CT];   // without FLUSH: unused, the chains are acc
  auto& run = [&]() -> auto& { if constexpr (FLUSH) return chain; else return acc; }();
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int q = 0; q < CT; ++q) {
        acc[c][t][q] = zero4();
        if constexpr (FLUSH) chain[c][t][q] = zero4();
      }
  auto compute = [&](int kt, int st) {
    const char* b = smem + st * WT::STAGE;
    const int kc = SUM == WT_CHAIN ? 64 * kt : wc.k, kend = SUM == WT_CHAIN ? K : wc.end;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      if (kc + 32 * hf >= kend) break;   // uniform
      const int sw = ((4 * hf + g) ^ (r & 7)) << 4;
      typename MF::frag w[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) w[c] = *reinterpret_cast<const typename MF::frag*>(b + (16 * c + r) * 128 + sw);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        // NA odd: the last row tile's upper half reads the lower half's rows again (never stored)
        const int ar = 16 * t + ((NA & 1) && t == RT - 1 ? (r & 7) : r);
        const typename MF::frag a = *reinterpret_cast<const typename MF::frag*>(b + (WT::COLS + ar) * 128 + sw);
#pragma unroll
        for (int c = 0; c < CT; ++c) run[NC == 2 ? hf : 0][t][c] = MF::mma(a, w[c], run[NC == 2 ? hf : 0][t][c]);
      }
    }
    if constexpr (FLUSH) {
      if (wc.last()) {   // uniform
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int q = 0; q < CT; ++q) {
              acc[0][t][q] += chain[c][t][q];
              chain[c][t][q] = zero4();
            }
      }
    }
    wc.next();
  };
  const int nk = wi.steps();
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue(s, s);
  int kt = 0;
  for (; kt + S < nk; ++kt) {
    wait_vm_lgkm0<(S - 1) * L>();   // stage kt has landed
    compute(kt, kt % S);
    wait_vm_lgkm0<63>();            // its fragment reads are done: the stage is free
    issue(kt + S, kt % S);
  }
  static_steps(std::make_integer_sequence<int, S>{}, [&](auto ic) {
    constexpr int j = S - 1 - decltype(ic)::value;   // stages issued after this one
    if (j < nk - kt) {   // uniform
      wait_vm_lgkm0<j * L>();
      compute(nk - 1 - j, (nk - 1 - j) % S);
    }
  });
  // every load has landed and one wave's LDS operations complete in order: the stages are free
}

// the accumulators staged as the output tile
template <class WT> DM_DEV void wt_stage(const floatx4 (&acc)[WT::RT][WT::CT], float* tile) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int t = 0; t < WT::RT; ++t)
#pragma unroll
    for (int c = 0; c < WT::CT; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) tile[(16 * t + 4 * g + q) * WT::LDT + 16 * c + r] = acc[t][c][q];
}

// one tile by one wave: a block's waves each call it with LDS of their own
template <typename T, class WT, class E>
DM_DEV void wt_tile(const E& e, const WtOp<T>& op, int bx, int by, char* smem) {
  typename E::template Pre<WT> pre;
  e.prefetch(bx, by * WT::ROWS, pre);
  floatx4 acc[E::SUM == WT_EIGHTHS ? 2 : 1][WT::RT][WT::CT];
  wt_kloop<T, WT, false>(e, op, bx, by, 0, smem, acc);
  float* tile = reinterpret_cast<float*>(smem);
  wt_stage<WT>(acc[0], tile);
  __syncthreads();
  e.apply(bx, by * WT::ROWS, tile, pre);
}

template <typename T, class WT, class E>
static __global__ __launch_bounds__(64) void k_wt(WtOp<T> op, E e) {
  __shared__ __attribute__((aligned(1024))) char smem[WT::LDS];
  wt_tile<T, WT>(e, op, blockIdx.x, blockIdx.y, smem);
}
// two independent products of the same rows in one launch: the first's column tiles, then the second's
template <typename T, class WT, class E1, class E2>
static __global__ __launch_bounds__(64) void k_wt2(WtOp<T> op1, E1 e1, WtOp<T> op2, E2 e2) {
  __shared__ __attribute__((aligned(1024))) char smem[WT::LDS];
  const int b = blockIdx.x;
  if (b < op1.nx) wt_tile<T, WT>(e1, op1, b, blockIdx.y, smem);
  else wt_tile<T, WT>(e2, op2, b - op1.nx, blockIdx.y, smem);
}

// A product summed in parts by four waves per tile, each a part of E's sum with its own ring, their partial
// tiles added in the sum's order: a tile's chain of k steps is a quarter as long, and four times the
// bytes are in flight (launch_wt_parts, with what both measured).
template <typename T, class WT, class E>
static __global__ __launch_bounds__(64 * WT_PARTS) void k_wt_ksplit(WtOp<T> op, E e) {
  static_assert(E::SUM != WT_CHAIN, "a sum of parts");
  constexpr int NC = E::SUM == WT_EIGHTHS ? 2 : 1, TILE = 16 * WT::RT * WT::LDT;
  static_assert(NC * TILE * 4 <= WT::LDS, "a wave's partial tiles fit its stages");
  __shared__ __attribute__((aligned(1024))) char smem[WT_PARTS * WT::LDS];
  const int wave = threadIdx.x >> 6;
  typename E::template Pre<WT> pre;
  e.prefetch(blockIdx.x, blockIdx.y * WT::ROWS, pre);
  floatx4 acc[NC][WT::RT][WT::CT];
  char* mine = smem + wave * WT::LDS;
  wt_kloop<T, WT, true>(e, op, blockIdx.x, blockIdx.y, wave, mine, acc);
#pragma unroll
  for (int c = 0; c < NC; ++c) wt_stage<WT>(acc[c], reinterpret_cast<float*>(mine) + c * TILE);
  __syncthreads();
  if (wave > 0) return;
  float* tile = reinterpret_cast<float*>(smem);
  constexpr int NE = WT::ROWS * WT::LDT;
  for (int i = threadIdx.x; i < NE; i += 64) {
    float v = tile[i];
#pragma unroll
    for (int p = 1; p < WT_PARTS * NC; ++p)
      v += reinterpret_cast<const float*>(smem + p / NC * WT::LDS)[p % NC * TILE + i];
    tile[i] = v;
  }
  __builtin_amdgcn_wave_barrier();   // one wave's LDS operations complete in order
  e.apply(blockIdx.x, blockIdx.y * WT::ROWS, tile, pre);
}

// ---- epilogues ----------------------------------------------------------------------------------
// out[M, N] = the product
template <typename T, int SUM_> struct WtStore {
  static constexpr int SUM = SUM_;
  static constexpr int TILES = 5;   // forms with_wt may choose
  const T* W;
  long ldw;
  T* out;
  int M, N;
  template <class WT> struct Pre {};
  template <class WT> DM_DEV const T* wrow(int bx, WT, int r) const { return W + (long)(WT::COLS * bx + r) * ldw; }
  template <class WT> DM_DEV void prefetch(int, int, Pre<WT>&) const {}
  template <class WT> DM_DEV void apply(int bx, int m0, const float* tile, const Pre<WT>&) const {
    constexpr int IPR = WT::COLS / 4, NI = WT::ROWS * IPR;   // items of 4 columns
    const bool vec = (reinterpret_cast<uintptr_t>(out) & 7) == 0;   // uniform; any caller's pointer is taken
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 64) {
      const int i = i0 + (int)(threadIdx.x & 63), row = i / IPR, c = 4 * (i % IPR), m = m0 + row;
      if (i >= NI || m >= M) continue;
      const floatx4 v = *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + c);
      const float o[4] = {v.x, v.y, v.z, v.w};
      T* p = out + (long)m * N + WT::COLS * bx + c;
      if (vec) {
        st4<T>(p, o);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = from_f<T>(o[k]);
      }
    }
  }
};

// act[M, H] = silu(x W1^T) (x W3^T): a tile's first half of columns from W1, the second the same from W3
template <typename T> struct WtSwiGLU {
  static constexpr int SUM = WT_QUARTERS;
  static constexpr int TILES = 6;
  const T* W1;
  const T* W3;
  long ldw;
  T* out;
  int M, H;
  template <class WT> struct Pre {};
  template <class WT> DM_DEV const T* wrow(int bx, WT, int r) const {
    constexpr int HC = WT::COLS / 2;
    return (r < HC ? W1 : W3) + (long)(HC * bx + r % HC) * ldw;
  }
  template <class WT> DM_DEV void prefetch(int, int, Pre<WT>&) const {}
  template <class WT> DM_DEV void apply(int bx, int m0, const float* tile, const Pre<WT>&) const {
    constexpr int HC = WT::COLS / 2, IPR = HC / 4, NI = WT::ROWS * IPR;
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 64) {
      const int i = i0 + (int)(threadIdx.x & 63), row = i / IPR, c = 4 * (i % IPR), m = m0 + row;
      if (i >= NI || m >= M) continue;
      const floatx4 g = *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + c);
      const floatx4 u = *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + HC + c);
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = g[k] * sigmoidf_(g[k]) * u[k];
      st4<T>(out + (long)m * H + HC * bx + c, o);
    }
  }
};

// the projection (EpiProj without the value norm): q / k / v tiles hold 8 CT RoPE pairs of one head
template <typename T, int DH, bool DEVPOS> struct WtProj {
  static constexpr int SUM = WT_CHAIN;
  static constexpr int TILES = 4;
  const T* W;   // [nseg d, d]
  EpiProj<T, DH, DEVPOS> e;
  template <class WT> struct Pre {
    static constexpr int IPR = WT::COLS / 8, NP = (WT::ROWS * IPR + 63) / 64;   // q / k items of 4 pairs
    floatx4 x[NP], y[NP];   // cos, sin of the lane's q / k items; x[0] the bias of its gate columns
  };
  template <class WT> DM_DEV const T* wrow(int bx, WT, int r) const {
    static_assert(DH % WT::COLS == 0, "a tile lies inside one head");
    const int c0 = WT::COLS * bx, sg = c0 / e.d;
    long row = c0 + r;
    if (sg <= 2) {
      constexpr int HC = WT::COLS / 2;
      const int c = c0 - sg * e.d, hh = c / DH, jj = (c - hh * DH) / 2;
      row = (long)sg * e.d + hh * DH + jj + (r < HC ? r : DH / 2 + r - HC);
    }
    return W + row * e.d;
  }
  template <class WT> DM_DEV void prefetch(int bx, int m0, Pre<WT>& pre) const {
    using P = Pre<WT>;
    const int c0 = WT::COLS * bx, sg = c0 / e.d, lane = threadIdx.x & 63;
    if (sg <= 1) {
      const int jj = ((c0 - sg * e.d) % DH) / 2;
      const int r0 = DEVPOS ? dev_position(e.pos_dev, e.pos_cap) : e.rope_t0;
#pragma unroll
      for (int p = 0; p < P::NP; ++p) {
        const int i = lane + 64 * p, m = min(m0 + i / P::IPR, e.M - 1);
        const long rr = (long)(r0 + m % e.Tl) * (DH / 2) + jj + 4 * (i % P::IPR);
        pre.x[p] = ld_global<floatx4>(e.cos + rr);
        pre.y[p] = ld_global<floatx4>(e.sin + rr);
      }
    } else {
      pre.x[0] = zero4();
      if (sg >= 3 && !(sg == 5 && e.fusion))
        pre.x[0] = ld_global<floatx4>(e.bias + (c0 - 3 * e.d) + 4 * (lane % (WT::COLS / 4)));
    }
  }
  template <class WT> DM_DEV void apply(int bx, int m0, const float* tile, const Pre<WT>& pre) const {
    using P = Pre<WT>;
    const int c0 = WT::COLS * bx, sg = c0 / e.d, c = c0 - sg * e.d, lane = threadIdx.x & 63;
    if (sg <= 2) {
      const int hh = c / DH, jj0 = (c - hh * DH) / 2;
#pragma unroll
      for (int p = 0; p < P::NP; ++p) {
        const int i = lane + 64 * p, row = i / P::IPR, q = 4 * (i % P::IPR), m = m0 + row;
        if (row >= WT::ROWS || m >= e.M) continue;
        const floatx4 av = *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + q);
        const floatx4 bv = *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + WT::COLS / 2 + q);
        const float a[4] = {av.x, av.y, av.z, av.w}, b[4] = {bv.x, bv.y, bv.z, bv.w};
        const int bb = m / e.Tl, t = m - bb * e.Tl;
        const long hrow = (((long)bb * e.h + hh) * e.Tbuf + e.buf_t0 + t) * DH + jj0 + q;
        if (sg <= 1) {
          float cs[4], sn[4];
          unpackf4(pre.x[p], cs);
          unpackf4(pre.y[p], sn);
          e.rope_item(sg, hrow, a, b, cs, sn);
        } else {
          st4<T>(e.vraw + hrow, a);
          st4<T>(e.vraw + hrow + DH / 2, b);
        }
      }
    } else {
      constexpr int IPR = WT::COLS / 4, NI = WT::ROWS * IPR;
      float bs[4];
      unpackf4(pre.x[0], bs);
#pragma unroll
      for (int i0 = 0; i0 < NI; i0 += 64) {
        const int i = i0 + lane, row = i / IPR, q = 4 * (i % IPR), m = m0 + row;
        if (i >= NI || m >= e.M) continue;
        e.gate_item(sg, m, c + q, *reinterpret_cast<const floatx4*>(tile + row * WT::LDT + q), bs);
      }
    }
  }
};

// sweep GEMM 1 (EpiSweep1 without head norms). A tile of a sectioned group (K, linear V) holds the
// same 4 CT columns of each of its four sections, a v_map / g_v tile 16 CT plain columns; an item is
// V columns (of each section) of one row, V so that the wave's lanes are used.
template <typename T, int DH, bool DEVPOS> struct WtSweep1 {
  static constexpr int SUM = WT_CHAIN;
  static constexpr int TILES = 4;
  typedef EpiSweep1<T, DH, 1, DEVPOS> Epi;
  const T* W;   // [4d, d], packed
  Epi e;
  const float* ssq;   // [M, nparts]
  int nparts;
  float inv_d, eps;
  static constexpr int Q = MAX_HEADS / 4;
  template <class WT> struct Shape {
    static constexpr int SEC = 4 * WT::CT;                                             // columns per section
    static constexpr int V = WT::NA * WT::CT >= 8 ? 4 : (WT::NA * WT::CT >= 4 ? 2 : 1);
    static constexpr int IPR = SEC / V, NP = (WT::ROWS * IPR + 63) / 64;
    static constexpr int VP = 2 * V, IPP = WT::COLS / VP, NPP = (WT::ROWS * IPP + 63) / 64;   // plain columns
    static constexpr int RP = (WT::ROWS + 15) / 16;                                    // row-scale passes
  };
  template <class WT> struct Pre {
    typename Epi::template KPre<Shape<WT>::V> k[Shape<WT>::NP];
    typename Epi::template LPre<Shape<WT>::V> l[Shape<WT>::NP];
    typename Epi::template MPre<Shape<WT>::VP> m[Shape<WT>::NPP];
    float v[Shape<WT>::RP][Q];   // the lane's partial sums of squares (added in apply: no wait here)
  };
  template <class WT> DM_DEV static int group0(int bx) { return bx / (4 / WT::CT) * 64; }
  template <class WT> DM_DEV static int sub0(int bx) { return bx % (4 / WT::CT) * Shape<WT>::SEC; }   // first column of a section
  template <class WT> DM_DEV const T* wrow(int bx, WT, int r) const {
    constexpr int SEC = Shape<WT>::SEC;
    const bool plain = e.kind(WT::COLS * bx) >= Epi::V_MAP;
    const int row = plain ? WT::COLS * bx + r : group0<WT>(bx) + 16 * (r / SEC) + sub0<WT>(bx) + r % SEC;
    return W + (long)row * e.g.d;
  }
  template <class WT> DM_DEV void prefetch(int bx, int m0, Pre<WT>& pre) const {
    using Sh = Shape<WT>;
    const int lane = threadIdx.x & 63, kd = e.kind(WT::COLS * bx);   // uniform
    if (kd <= Epi::LIN_V) {
#pragma unroll
      for (int p = 0; p < Sh::NP; ++p) {
        const int i = lane + 64 * p, row = m0 + i / Sh::IPR, lc0 = sub0<WT>(bx) + Sh::V * (i % Sh::IPR);
        if (kd == Epi::K_ROWS) pre.k[p] = e.template k_prefetch<Sh::V>(row, group0<WT>(bx), lc0);
        else pre.l[p] = e.template l_prefetch<Sh::V>(row, group0<WT>(bx), lc0);
      }
    } else if (kd == Epi::V_MAP) {
#pragma unroll
      for (int p = 0; p < Sh::NPP; ++p) {
        const int i = lane + 64 * p;
        pre.m[p] = e.template m_prefetch<Sh::VP>(m0 + i / Sh::IPP, WT::COLS * bx - 2 * e.g.d + Sh::VP * (i % Sh::IPP));
      }
    }
    // row scales, four lanes per row (SrcRowsRs's order of the sum)
#pragma unroll
    for (int p = 0; p < Sh::RP; ++p) {
      const float* row = ssq + (long)min(m0 + 16 * p + (lane >> 2), e.M - 1) * nparts;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        pre.v[p][i] = 0.f;
        if (4 * i < nparts) pre.v[p][i] = row[min((lane & 3) + 4 * i, nparts - 1)];   // uniform
      }
    }
  }
  template <class WT> DM_DEV void apply(int bx, int m0, float* tile, const Pre<WT>& pre) const {
    using Sh = Shape<WT>;
    const int lane = threadIdx.x & 63, kd = e.kind(WT::COLS * bx), d = e.g.d;
    float* rs = tile + 16 * WT::RT * WT::LDT;   // [ROWS]
#pragma unroll
    for (int p = 0; p < Sh::RP; ++p) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < Q; ++i) s += (lane & 3) + 4 * i < nparts ? pre.v[p][i] : 0.f;
      s = lanes_sum<1, 2>(s);
      const int row = 16 * p + (lane >> 2);
      if ((lane & 3) == 0 && row < WT::ROWS) rs[row] = rsqrtf(s * inv_d + eps);
    }
    __syncthreads();
    if (kd <= Epi::LIN_V) {
      const int n0 = group0<WT>(bx);
#pragma unroll
      for (int p = 0; p < Sh::NP; ++p) {
        const int i = lane + 64 * p, row = i / Sh::IPR, cg = Sh::V * (i % Sh::IPR), m = m0 + row;
        if (row >= WT::ROWS) continue;
        const int lc0 = sub0<WT>(bx) + cg;
        float a[4][Sh::V];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int j = 0; j < Sh::V; ++j) a[k][j] = tile[row * WT::LDT + Sh::SEC * k + cg + j] * rs[row];
        auto save_raw = [&]() {
          if (e.save == nullptr) return;   // uniform
#pragma unroll
          for (int k = 0; k < 4; ++k) stv_nt<T, Sh::V>(e.save + (long)m * 4 * d + n0 + 16 * k + lc0, a[k]);
        };
        if (kd == Epi::K_ROWS) e.template k_apply<Sh::V>(a, m, n0, lc0, pre.k[p], save_raw);
        else e.template l_apply<Sh::V>(a, m, n0, lc0, pre.l[p], save_raw);
      }
    } else {
#pragma unroll
      for (int p = 0; p < Sh::NPP; ++p) {
        const int i = lane + 64 * p, row = i / Sh::IPP, c = Sh::VP * (i % Sh::IPP), m = m0 + row, n = WT::COLS * bx + c;
        if (row >= WT::ROWS || m >= e.M) continue;
        float a[Sh::VP];
#pragma unroll
        for (int j = 0; j < Sh::VP; ++j) a[j] = tile[row * WT::LDT + c + j] * rs[row];
        if (e.save != nullptr) stv_nt<T, Sh::VP>(e.save + (long)m * 4 * d + n, a);
        if (kd == Epi::V_MAP) e.template m_apply<Sh::VP>(a, rs[row], m, n - 2 * d, pre.m[p]);
        else stv<T, Sh::VP>(e.gvu + (long)m * d + n - 3 * d, a);
      }
    }
  }
};

// sweep GEMM 2 (EpiSweep2): items of V columns of one row
template <typename T, int DH, bool DEVPOS> struct WtSweep2 {
  static constexpr int SUM = WT_CHAIN;
  static constexpr int TILES = 3;
  typedef EpiSweep2<T, DH, DEVPOS> Epi;
  const T* W;   // [d, d]
  Epi e;
  template <class WT> struct Shape {
    static constexpr int V = WT::NA * WT::CT >= 4 ? 8 : 2 * WT::NA * WT::CT;
    static constexpr int IPR = WT::COLS / V, NI = WT::ROWS * IPR, NP = (NI + 63) / 64;
  };
  template <class WT> struct Pre {
    typename Epi::template ItemPre<Shape<WT>::V> g[Shape<WT>::NP];
  };
  template <class WT> DM_DEV const T* wrow(int bx, WT, int r) const { return W + (long)(WT::COLS * bx + r) * e.g.d; }
  template <class WT> DM_DEV void prefetch(int bx, int m0, Pre<WT>& pre) const {
    using Sh = Shape<WT>;
#pragma unroll
    for (int p = 0; p < Sh::NP; ++p) {
      const int i = (int)(threadIdx.x & 63) + 64 * p;
      pre.g[p] = e.template item_prefetch<Sh::V>(m0 + i / Sh::IPR, WT::COLS * bx + Sh::V * (i % Sh::IPR));
    }
  }
  template <class WT> DM_DEV void apply(int bx, int m0, const float* tile, const Pre<WT>& pre) const {
    using Sh = Shape<WT>;
#pragma unroll
    for (int p = 0; p < Sh::NP; ++p) {
      const int i = (int)(threadIdx.x & 63) + 64 * p, row = i / Sh::IPR, c = Sh::V * (i % Sh::IPR);
      if (row < WT::ROWS)
        e.template item_apply<Sh::V>(tile + row * WT::LDT + c, m0 + row, WT::COLS * bx + c, pre.g[p]);
    }
  }
};

}  // namespace dm
