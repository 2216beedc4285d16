// Host-side launch sequences of the forward: layer projections and one chunk
// cell (committed accumulator + n_sweeps Jacobi sweeps). Shared by the forward
// entry points and by the backward's exact recompute (which keeps every sweep's
// state in a CellSave instead of overwriting it in place).
#pragma once

#include <vector>

#include "dm_decode.h"
#include "dm_host.h"
#include "dm_rows.h"

namespace dm {

// cell workspace (forward): per-sweep scratch reused across sweeps
struct CellWs {
  void* o; float* ssq;
  float* Ap; float* Zp; float* Mp;   // committed split partials
  float* A; float* Z; float* M;      // merged committed accumulator
  void* vin; void* gvu;              // v_in, g_v(u) [N, d] (storage dtype)
  size_t bytes;
};

inline CellWs carve_cell(const dm_config* c, int cache_T, void* base) {
  CellWs w{};
  const size_t N = (size_t)c->B * CMAX, BH = (size_t)c->B * c->h;
  const size_t ns = comm_splits_max(cache_T);
  Carver cv(base);
  w.o = cv.take<void>(N * c->d * esz(c->dtype));
  w.ssq = cv.take<float>(N * c->h * 4);
  w.Ap = cv.take<float>(ns * BH * CMAX * c->dh * 4);
  w.Zp = cv.take<float>(ns * BH * CMAX * 4);
  w.Mp = cv.take<float>(ns * BH * CMAX * 4);
  w.A = cv.take<float>(BH * CMAX * c->dh * 4);
  w.Z = cv.take<float>(BH * CMAX * 4);
  w.M = cv.take<float>(BH * CMAX * 4);
  w.vin = cv.take<void>(N * c->d * esz(c->dtype));
  w.gvu = cv.take<void>(N * c->d * esz(c->dtype));
  w.bytes = cv.off;
  return w;
}

// Every sweep's state of one cell, kept for the backward. Per-sweep arrays are
// stacked with the cell's own row count N = B*c (so the K sweeps of a [N, x]
// array form one [K*N, x] matrix); attention rows use B*h*CMAX slots.
template <typename T> struct CellSave {
  T* o;              // [K][N, d]      o of sweep s (storage dtype, as stored by the attention)
  float* ssq;        // [K][N, h]      per-head sums of squares of o
  float* stat_m;     // [K][BH, CMAX]  final row max of sweep s
  float* stat_z;     // [K][BH, CMAX]  final row sum of sweep s
  T* save1;          // [K][N, 4d]     raw sweep GEMM 1 outputs (rounded to the storage dtype,
  T* save2;          // [K][N, d]      raw v_ctx (mult family)    as the reference's GEMM outputs)
  T* vin;            // [K][N, d]      v_in (mult family): rows of the layer's stacked v_in
                     //   (the backward's cell order), assigned by the caller
  T* Kin; T* Vin;    // [K+1][BH, CMAX, DH]  intra rows read by sweep s (slot 0 unused: raw rows);
                     //   with last_to_cache only [K] slots: the last sweep writes the cache rows
  float* Mx;         // [BH, CMAX] committed row max (tape cells with pos0 > 0), else nullptr
  bool last_to_cache;
};

// Layout of one cell's saved state for N = B*cc rows and K sweeps. `tape` cells
// (forward-saved) drop the last K/V slot and add the committed row max.
template <typename T>
CellSave<T> carve_save(const dm_config* c, size_t N, int K, bool tape, bool has_comm, Carver& cv) {
  CellSave<T> w{};
  const size_t d = c->d, h = c->h, dh = c->dh, e = sizeof(T), BH = (size_t)c->B * c->h, k = K;
  const bool mult = c->ctx_mod != DM_CTX_LINEAR;
  w.o = cv.take<T>(k * N * d * e);
  w.ssq = cv.take<float>(k * N * h * 4);
  w.stat_m = cv.take<float>(k * BH * CMAX * 4);
  w.stat_z = cv.take<float>(k * BH * CMAX * 4);
  w.save1 = cv.take<T>(k * N * 4 * d * e);
  w.save2 = mult ? cv.take<T>(k * N * d * e) : nullptr;
  w.vin = nullptr;
  const size_t slots = tape ? k : k + 1;
  w.Kin = cv.take<T>(slots * BH * CMAX * dh * e);
  w.Vin = cv.take<T>(slots * BH * CMAX * dh * e);
  w.Mx = (tape && has_comm) ? cv.take<float>(BH * CMAX * 4) : nullptr;
  w.last_to_cache = tape;
  return w;
}

// Row of cell i's first v_in row in the layer's stacked v_in: the backward takes the
// cells last first, so the rows of cells i+1.. precede cell i's.
inline long vin_row(const dm_config* c, const int32_t* sched, int n_cells, int i) {
  long r = 0;
  for (int j = i + 1; j < n_cells; ++j) r += (long)sched[3 * j + 2] * c->B * sched[3 * j + 1];
  return r;
}

// Layout of a layer tape (n_cells + 2 entries): off[i] = cell i's saved state,
// off[n_cells] = the stacked v_in of every cell (mult family; rows in the backward's
// cell order, rounded up to a whole 64-row k-tile), off[n_cells + 1] = total bytes.
template <typename T>
std::vector<size_t> tape_offsets(const dm_config* c, const int32_t* sched, int n_cells) {
  std::vector<size_t> off(n_cells + 2, 0);
  for (int i = 0; i < n_cells; ++i) {
    Carver cv(nullptr);
    carve_save<T>(c, (size_t)c->B * sched[3 * i + 1], sched[3 * i + 2], true, sched[3 * i] > 0, cv);
    off[i + 1] = off[i] + cv.off;
  }
  const long rows = vin_row(c, sched, n_cells, -1);
  const size_t vin_bytes = c->ctx_mod != DM_CTX_LINEAR ? (size_t)((rows + 63) / 64 * 64) * c->d * sizeof(T) : 0;
  off[n_cells + 1] = off[n_cells] + align256(vin_bytes);
  return off;
}

// per-head norm gains of the packed weights (nullptr: that norm is off)
inline const float* kctx_gain(const dm_config* c, const dm_packed* w) {
  return (c->norms & DM_NORM_K_CTX) ? w->gains : nullptr;
}
inline const float* vctx_gain(const dm_config* c, const dm_packed* w) {
  return (c->norms & DM_NORM_V_CTX) ? w->gains + c->h : nullptr;
}
inline const float* v_gain(const dm_config* c, const dm_packed* w) {
  return (c->norms & DM_NORM_V) ? w->gains + 2 * c->h : nullptr;
}

// ---- wave-tile products (dm_rows.h) -----------------------------------------------------------
// Where they are taken: bf16, M <= WT_MAX_M rows, 16-byte aligned operands, the launch issued directly
// (not recorded for a grouped launch). Per-head norms need a whole head per block and stay on the
// tiled GEMMs.
template <typename T> bool wt_ok(int M, const void* A, const void* W) {
  return sizeof(T) == 2 && M <= WT_MAX_M && launch_log() == nullptr && aligned16(A) && aligned16(W);
}
// f(WTile) with the tile of least expected time for M x N outputs (N a multiple of 64): a wave's
// own time goes with its operand rows (8 NA + 16 CT; 57 ns each per 1024 of k), a CU's with the sum
// over its waves (35 ns per row); fitted to 30 measured (M, N, tile) times, K = 512 .. 2048, within 15% of
// the best tile where the products take wave tiles. Of the first TILES forms, the ones a product's sizes can
// reach: GEMM 2 (M N <= 262144) three, the projection and GEMM 1 alone (M d <= 65536) four, a store or GEMM 1
// with W_O five; the MLP's up products all: 64 rows x 32 columns read the weights once where shorter tiles
// read them twice (a tie goes to it: M = 33, N = 11008, K = 2048 17.0 us against 18.5 and 21.8; N = 21888, K =
// 4096 55.4 against 63.9). 32 rows x 16 columns is never the least: 16 x 32 has as many rows and no more waves.
template <int TILES, class F> void with_wt(int M, int N, const F& f) {
  struct C { int na, ct; };
  constexpr C cand[] = {{1, 1}, {2, 1}, {2, 2}, {4, 2}, {4, 4}, {8, 2}};
  int best = 0;
  long bt = -1;
  for (int i = 0; i < TILES; ++i) {
    if (i > 0 && M <= 8 * cand[i - 1].na && cand[i].na > cand[i - 1].na) continue;
    const long rows = 8 * cand[i].na + 16 * cand[i].ct, waves = (long)cdiv(M, 8 * cand[i].na) * (N / (16 * cand[i].ct));
    const long t = std::max<long>(57 * rows, 35 * rows * cdiv(waves, 256));
    if (bt < 0 || t < bt || (i == 5 && t == bt)) {
      bt = t;
      best = i;
    }
  }
  switch (best) {
    case 0: f(WTile<1, 1>{}); break;
    case 1: f(WTile<2, 1>{}); break;
    case 2: f(WTile<2, 2>{}); break;
    case 3:
      if constexpr (TILES > 3) f(WTile<4, 2>{});
      break;
    case 4:
      if constexpr (TILES > 4) f(WTile<4, 4>{});
      break;
    default:
      if constexpr (TILES > 5) f(WTile<8, 2>{});
      break;
  }
}
// N weight rows (WtSwiGLU: both matrices')
template <typename T, class E>
void launch_wt(WtOp<T> op, int N, const E& e, hipStream_t s, int prof_cls = PROF_NONE) {
  with_wt<E::TILES>(op.M, N, [&](auto wt) {
    using WT = decltype(wt);
    op.nx = N / WT::COLS;
    launch_k(prof_cls, k_wt<T, WT, E>, dim3(op.nx, cdiv(op.M, WT::ROWS)), dim3(64), 0, s, op, e);
  });
}
// a product summed in parts (a step's W_O and MLP products, M <= ROWS_MAX): four waves per 16-column tile
// while that gives the CUs at most two such blocks each, of short rings (two to a CU); eighths always, in
// taller and wider tiles beyond. Measured at weights from HBM, four waves against one per tile (which for
// the down products summed one chain): M = 1, d x H = 512 x 1376: up 3.1 against 3.7 us, down 3.5 / 4.9;
// 1024 x 2752: 5.1 / 5.8, 4.9 / 7.9; M = 64: up 9.6 / 8.0, down 5.6 / 8.2; 2048 x 5504, M = 32: up
// 17.7 / 13.5, down 8.5 / 14.6; W_O, M = 16, d = 1024: 3.5 / 4.4. Rings of 6 to 8 stages, one block to a
// CU: down 5.1 against 4.9 at M = 1, 9.5 against 8.5 at M = 32.
template <typename T, class E>
void launch_wt_parts(WtOp<T> op, int N, const E& e, hipStream_t s, int prof_cls = PROF_NONE) {
  auto run = [&](auto wt) {
    using WT = decltype(wt);
    op.nx = N / WT::COLS;
    launch_k(prof_cls, k_wt_ksplit<T, WT, E>, dim3(op.nx, cdiv(op.M, WT::ROWS)), dim3(64 * WT_PARTS), 0, s, op, e);
  };
  if (op.M <= 8) return run(WTile<1, 1, 4>{});
  if ((long)cdiv(op.M, 16) * (N / 16) < 512) return run(WTile<2, 1, 4>{});
  if constexpr (E::SUM == WT_EIGHTHS) {
    if ((long)cdiv(op.M, 32) * (N / 16) < 512) run(WTile<4, 1, 3>{});
    else run(WTile<4, 2, 3>{});
  } else {
    launch_wt(op, N, e, s, prof_cls);
  }
}
template <typename T, class E1, class E2>
void launch_wt2(WtOp<T> op1, int N1, const E1& e1, WtOp<T> op2, int N2, const E2& e2, hipStream_t s,
                int prof_cls = PROF_NONE) {
  with_wt<5>(op1.M, N1 + N2, [&](auto wt) {
    using WT = decltype(wt);
    op1.nx = N1 / WT::COLS;
    op2.nx = N2 / WT::COLS;
    launch_k(prof_cls, k_wt2<T, WT, E1, E2>, dim3(op1.nx + op2.nx, cdiv(op1.M, WT::ROWS)), dim3(64), 0, s, op1, e1, op2,
             e2);
  });
}
// What rides in a decode step's refine: the W_O product in its first launch (both read o_cat), and the
// residual add and norm after it (x += y, h = rmsnorm(x) norm_w) in its second, which they do not depend on
template <typename T> struct WtWo {
  const T* W;
  T* y;
  float* x = nullptr;
  const float* norm_w = nullptr;
  T* h = nullptr;
  float eps = 0.f;
};
// blocks [0, M): one row of the residual norm each; then four column tiles of GEMM 2 per block
template <typename T, class WT, class E>
static __global__ __launch_bounds__(256) void k_norm_wt(WtWo<T> n, int M, int d, WtOp<T> op, E e) {
  __shared__ __attribute__((aligned(1024))) char smem[4 * WT::LDS];
  const int b = blockIdx.x;
  if (b < M) {
    residual_rmsnorm_row<T, 16>(b, n.x, n.y, n.norm_w, n.h, d, n.eps, reinterpret_cast<float*>(smem));
    return;
  }
  const int t = 4 * (b - M) + (threadIdx.x >> 6);   // the grid holds whole fours of tiles
  wt_tile<T, WT>(e, op, t % op.nx, t / op.nx, smem + (threadIdx.x >> 6) * WT::LDS);
}

// vpre: v_raw before the v_norm (nullptr: not kept); sa: the M input rows (x-hat);
// small_tiles: 128 x 128 blocks even where 256 x 256 ones fit (more blocks for a short M; the
// k-order of every output element, and so the result, is the same)
template <typename T, int DH, class SA>
void run_proj_src(const dm_config* c, const dm_packed* w, const SA& sa, int M, int Tl, int Tbuf, int buf_t0,
                  int rope_t0, const float* cos, const float* sin, T* qr, T* kraw, T* kself, T* vraw, T* vpre,
                  T* glogx, T* sig, hipStream_t s, bool small_tiles = false, const int* pos_dev = nullptr,
                  int pos_cap = 0) {
  const int nseg = (c->ctx_mod == DM_CTX_LINEAR) ? 5 : 6;
  SrcRows<T> sb{(const T*)w->w_proj, c->d, nseg * c->d};
  // Few rows, issued directly. Wave tiles while a wave's operands (M d of them) are few: with more, the waves
  // of a block tile share what each of them would load; then 64-row blocks up to d = 2048, 128-row ones
  // beyond. Measured at weights from HBM, head_dim 64, wave tiles / 64-row / 128-row blocks, us: d = 1024,
  // M = 32 6.8 / 9.3 / -, 64 10.2 / 10.2 / 16.6, 96 15.7 / 10.1 / 18.5, 256 21.3 / 11.4 / 20.3 (256 x 256
  // blocks 40); d = 2048, M = 32 15.7 / 16.6 / -, 48 25.9 / 17.0 / 24.9, 256 48.5 / 31.1 / 30.6; d = 4096,
  // M = 8 42.4 / 46.6 / -, 16 49.8 / 44.4 / -, 96 104 / 65 / 55; d = 256, M = 256 5.1 / 4.8 / 13.0.
  const bool few = sizeof(T) == 2 && M <= WT_MAX_M && launch_log() == nullptr;
  if constexpr (std::is_same<SA, SrcRows<bf16>>::value) {
    if (wt_ok<T>(M, sa.p, w->w_proj) && v_gain(c, w) == nullptr && (long)M * c->d <= 65536 && (M <= 8 || c->d <= 2048)) {
      const WtOp<T> op{sa.p, sa.ld, M, c->d};
      if (pos_dev != nullptr)
        launch_wt(op, nseg * c->d, WtProj<T, DH, true>{(const T*)w->w_proj,
                                              EpiProj<T, DH, true>{M, c->d, c->h, Tl, Tbuf, buf_t0, 0, cos, sin, w->b_proj,
                                                                   qr, kraw, kself, vraw, glogx, sig,
                                                                   c->ctx_mod == DM_CTX_FUSION, nullptr, nullptr, pos_dev,
                                                                   pos_cap}},
                    s, PROF_PROJ);
      else
        launch_wt(op, nseg * c->d, WtProj<T, DH, false>{(const T*)w->w_proj,
                                               EpiProj<T, DH>{M, c->d, c->h, Tl, Tbuf, buf_t0, rope_t0, cos, sin,
                                                              w->b_proj, qr, kraw, kself, vraw, glogx, sig,
                                                              c->ctx_mod == DM_CTX_FUSION}},
                    s, PROF_PROJ);
      return;
    }
  }
  if (pos_dev != nullptr) {
    // a decode step at a device position (M <= 64 rows): the RoPE row read from device memory
    EpiProj<T, DH, true> epi{M, c->d, c->h, Tl, Tbuf, buf_t0, 0, cos, sin, w->b_proj, qr, kraw, kself, vraw,
                             glogx, sig, c->ctx_mod == DM_CTX_FUSION, v_gain(c, w), vpre, pos_dev, pos_cap};
    if constexpr (DH == 64)
      launch_gemm_auto<T, 64, 64, 2, 2, 3, 4>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
    else
      launch_gemm_auto<T, 64, 128, 2, 2, 3, 4>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
    return;
  }
  EpiProj<T, DH> epi{M, c->d, c->h, Tl, Tbuf, buf_t0, rope_t0, cos, sin, w->b_proj,
                     qr, kraw, kself, vraw, glogx, sig, c->ctx_mod == DM_CTX_FUSION, v_gain(c, w), vpre};
  // bf16, whole 256-row / 256-column tiles: 256 x 256 blocks (eight 64 x 128 wave tiles,
  // two direct-to-LDS stages); otherwise 128 x 128 with wave tiles spanning whole heads
  if constexpr (sizeof(T) == 2) {
    if (!small_tiles && !few && M % 256 == 0 && (nseg * c->d) % 256 == 0 && c->d % 64 == 0) {
      launch_gemm<T, 256, 256, 4, 2, -2>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
      return;
    }
  }
  if (M <= 64 || (few && c->d <= 2048)) {
    // 64-row blocks, one head wide (twice the blocks of 128 x 128)
    if constexpr (DH == 64)
      launch_gemm_auto<T, 64, 64, 2, 2, 3, 4>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
    else
      launch_gemm_auto<T, 64, 128, 2, 2, 3, 4>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
    return;
  }
  if constexpr (DH == 64)
    launch_gemm_128<T, 2, 2>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
  else
    launch_gemm_128<T, 4, 1>(sa, sb, M, nseg * c->d, c->d, epi, s, PROF_PROJ);
}

template <typename T, int DH>
void run_proj(const dm_config* c, const dm_packed* w, const T* xhat, int M, int Tl, int Tbuf, int buf_t0,
              int rope_t0, const float* cos, const float* sin, T* qr, T* kraw, T* kself, T* vraw, T* vpre,
              T* glogx, T* sig, hipStream_t s, const int* pos_dev = nullptr, int pos_cap = 0) {
  run_proj_src<T, DH>(c, w, SrcRows<T>{xhat, c->d, M}, M, Tl, Tbuf, buf_t0, rope_t0, cos, sin, qr, kraw, kself, vraw,
                      vpre, glogx, sig, s, false, pos_dev, pos_cap);
}

template <typename T>
void run_proj_dispatch(const dm_config* c, const dm_packed* w, const T* xhat, int M, int Tl, int Tbuf,
                       int buf_t0, int rope_t0, const float* cos, const float* sin, T* qr, T* kraw, T* kself,
                       T* vraw, T* vpre, T* glogx, T* sig, hipStream_t s) {
  if (c->dh == 64)
    run_proj<T, 64>(c, w, xhat, M, Tl, Tbuf, buf_t0, rope_t0, cos, sin, qr, kraw, kself, vraw, vpre, glogx, sig, s);
  else
    run_proj<T, 128>(c, w, xhat, M, Tl, Tbuf, buf_t0, rope_t0, cos, sin, qr, kraw, kself, vraw, vpre, glogx, sig,
                     s);
}

// Split partials of the next cell's committed prefix that one fused GEMM 2 + attention launch
// computes as extra blocks (splits s0 .. s0 + ns - 1 of ca)
template <typename T> struct AheadComm {
  CommArgs<T> ca;
  int s0 = 0, ns = 0;
};

// One sweep's refine: sweep GEMM 1 (+ GEMM 2 for the mult family) with the blend
// epilogues, writing the refined rows to (Kout, Vout).
template <typename T, int DH, bool DEVPOS>
void launch_gemm2_wt(const dm_config* c, const dm_packed* w, const CellGeom& g, int N, const T* vraw, const T* glogx,
                     T* Vout, long out_stride, int out_row0, const T* vin, const T* gvu, T* save2, hipStream_t s) {
  launch_wt(WtOp<T>{vin, c->d, N, c->d}, c->d,
            WtSweep2<T, DH, DEVPOS>{(const T*)w->w_vctx, EpiSweep2<T, DH, DEVPOS>{g, N, vraw, glogx, gvu, Vout,
                                                                                 out_stride, out_row0, save2}},
            s, PROF_SWEEP2);
}

template <typename T, int DH, bool DEVPOS>
void run_refine_wt(const dm_config* c, const dm_packed* w, const CellGeom& g, int N, const T* o, const float* ssq,
                     const T* kraw, const T* vraw, const T* glogx, const T* sig, const float* cos, const float* sin,
                     T* Kout, T* Vout, long out_stride, int out_row0, T* vin, T* gvu, T* save1, T* save2,
                   hipStream_t s, const WtWo<T>* wo) {
  const int d = c->d;
  const WtSweep1<T, DH, DEVPOS> e1{
      (const T*)w->w_sweep,
      EpiSweep1<T, DH, 1, DEVPOS>{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o,
                                  (const T*)w->norm_ctx_w, Kout, Vout, out_stride, out_row0, vin, gvu, save1},
      ssq, c->h, 1.0f / (float)d, c->rms_eps};
  const WtOp<T> op1{o, d, N, d};
  if (wo != nullptr)
    launch_wt2(op1, 4 * d, e1, op1, d, WtStore<T, WT_EIGHTHS>{wo->W, d, wo->y, N, d}, s, PROF_SWEEP1);
  else
    launch_wt(op1, 4 * d, e1, s, PROF_SWEEP1);
  if (c->ctx_mod == DM_CTX_LINEAR) return;
  if (wo == nullptr || wo->x == nullptr) {
    launch_gemm2_wt<T, DH, DEVPOS>(c, w, g, N, vraw, glogx, Vout, out_stride, out_row0, vin, gvu, save2, s);
    return;
  }
  const WtSweep2<T, DH, DEVPOS> e2{(const T*)w->w_vctx, EpiSweep2<T, DH, DEVPOS>{g, N, vraw, glogx, gvu, Vout, out_stride,
                                                                                out_row0, save2}};
  auto run = [&](auto wt) {
    using WT = decltype(wt);
    const WtOp<T> op2{vin, d, N, d, d / WT::COLS};   // d a multiple of 128: whole fours of tiles per row tile
    launch_k(PROF_SWEEP2, k_norm_wt<T, WT, WtSweep2<T, DH, DEVPOS>>, dim3(N + op2.nx * cdiv(N, WT::ROWS) / 4), dim3(256),
             0, s, *wo, N, d, op2, e2);
  };
  if (N <= 8) run(WTile<1, 1>{});
  else if (N <= 16) run(WTile<2, 1>{});
  else run(WTile<4, 1, 6>{});
}

// The wave-tile forms apply: no per-head norm.
template <typename T> bool refine_wt_ok(const dm_config* c, const dm_packed* w, int N, const T* o, const T* vin) {
  return wt_ok<T>(N, o, w->w_sweep) && kctx_gain(c, w) == nullptr && vctx_gain(c, w) == nullptr &&
         (c->ctx_mod == DM_CTX_LINEAR || (aligned16(vin) && aligned16(w->w_vctx)));
}
// Both GEMMs in wave tiles, at most 64 rows. With more rows sweep GEMM 1's 64-wide block tiles are the faster
// ones: their epilogue touches each row of its inputs in longer runs (d = 1024, M = 96: 11.0 against 10.3 us,
// 192: 18.8 / 10.5).
template <typename T> bool refine_few_rows(const dm_config* c, const dm_packed* w, int N, const T* o, const T* vin) {
  return N <= ROWS_MAX && refine_wt_ok<T>(c, w, N, o, vin);
}

// Without a W_O product riding along, sweep GEMM 1 pays in wave tiles while a wave's operands are few (as the
// projection's): measured at weights from HBM, against 64 x 64 blocks, d = 1024, M = 64: 8.4 / 10.5 us; 2048,
// 32: 12.6 / 15.9, 48: 17.0 / 16.2 (weights in cache 16.3 / 13.9); 3072, 16: 18.0 / 25.8, 48: 38.4 / 23.8;
// 4096, 16: 33.3 / 35.8 (in cache 31.1 / 24.5)
inline bool sweep1_wt_pays(int N, int d) { return (long)N * d <= 65536 && (N <= 8 || d <= 3072); }

template <typename T, int DH>
void run_refine(const dm_config* c, const dm_packed* w, const CellGeom& g, int N, const T* o, const float* ssq,
                const T* kraw, const T* vraw, const T* glogx, const T* sig, const float* cos,
                const float* sin, T* Kout, T* Vout, long out_stride, int out_row0, T* vin, T* gvu,
                T* save1, T* save2, hipStream_t s, const AttendArgs<T>* next_attend = nullptr,
                bool wide = false, const AheadComm<T>* ahead = nullptr, const WtWo<T>* wo = nullptr) {
  if constexpr (sizeof(T) == 2) {
    // wo: only given where refine_few_rows holds
    if (next_attend == nullptr && !wide && refine_few_rows<T>(c, w, N, o, vin) &&
        (wo != nullptr || sweep1_wt_pays(N, c->d))) {
      if (g.pos_dev != nullptr)
        run_refine_wt<T, DH, true>(c, w, g, N, o, ssq, kraw, vraw, glogx, sig, cos, sin, Kout, Vout, out_stride,
                                     out_row0, vin, gvu, save1, save2, s, wo);
      else
        run_refine_wt<T, DH, false>(c, w, g, N, o, ssq, kraw, vraw, glogx, sig, cos, sin, Kout, Vout, out_stride,
                                      out_row0, vin, gvu, save1, save2, s, wo);
      if (g.v_clamp_tau > 0.f)
        hipLaunchKernelGGL((k_clamp_v<T, DH>), dim3(cdiv((long)N * c->h, 4)), dim3(256), 0, s, g, Vout, out_stride,
                           out_row0, N, g.v_clamp_tau);
      return;
    }
  }
  const T* normw = (const T*)w->norm_ctx_w;
  SrcRowsRs<T> sa{o, c->d, N, ssq, c->h, 1.0f / (float)c->d, c->rms_eps};
  SrcRows<T> sb{(const T*)w->w_sweep, c->d, 4 * c->d};
  const bool linear = c->ctx_mod == DM_CTX_LINEAR;
  const float* kgain = kctx_gain(c, w);
  const float* vgain = vctx_gain(c, w);
  if (kgain != nullptr || (linear && vgain != nullptr)) {
    // a norm of GEMM 1's k_ctx or (linear) v_ctx columns: blocks of one head's 2 DH packed columns
    constexpr int NG = DH / 32;
    EpiSweep1<T, DH, NG> e1{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o, normw,
                            Kout, Vout, out_stride, out_row0, vin, gvu, save1, kgain, linear ? vgain : nullptr};
    if constexpr (DH == 64)
      launch_gemm_auto<T, 64, 2 * DH, 2, 2, SW1_STAGES, 4>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
    else
      launch_gemm_auto<T, 64, 2 * DH, 1, 4, SW1_STAGES, 2>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
  } else if (wide && DM_GROUPED_WIDE_SW1) {
    // 64 x 128 blocks (two column groups each): a quarter less LDS traffic per MFMA and half the
    // o re-reads, for launches that have blocks to spare (the layer-batched forward)
    EpiSweep1<T, DH, 2> e1{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o, normw,
                           Kout, Vout, out_stride, out_row0, vin, gvu, save1};
    launch_gemm_auto<T, 64, 128, 2, 2, SW1_STAGES, 4>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
  } else if (g.pos_dev != nullptr) {
    // a decode step at a device position: RoPE row and output row read from device memory
    EpiSweep1<T, DH, 1, true> e1{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o, normw,
                                 Kout, Vout, out_stride, out_row0, vin, gvu, save1};
    launch_gemm_auto<T, 64, 64, 2, 2, SW1_STAGES, 4>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
  } else if (sizeof(T) == 2 && DM_SW1_EIGHT_WAVES && launch_log() == nullptr &&
             cdiv(N, 64) * (4 * c->d / 128) >= 192) {
    // bf16: 64 x 128 blocks of eight waves (each 256-thread half one 64-column group; d is a
    // multiple of 128, so the direct-to-LDS k-loop always applies) where they give most CUs one (fewer:
    // 64 x 64 blocks. 128 blocks, d = 1024, 256 rows: 12.1 against 10.5 us; 192 blocks, d = 1024, 384
    // rows: 12.2 / 12.3, d = 3072, 128 rows: 29.1 / 33.2): the two column groups share
    // the block's o rows, so a k-step moves 24 KB into a CU's LDS instead of the 32 KB of two
    // 64 x 64 blocks, still with eight waves per CU; the same per-element k order
    if constexpr (sizeof(T) == 2) {
      EpiSweep1<T, DH, 2, false, true> e1{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o,
                                          normw, Kout, Vout, out_stride, out_row0, vin, gvu, save1};
      launch_gemm<T, 64, 128, 2, 4, -SW1_STAGES>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
    }
  } else {
    EpiSweep1<T, DH> e1{g, N, c->ctx_mod, c->mult_res_lambda, kraw, vraw, glogx, sig, cos, sin, o, normw,
                        Kout, Vout, out_stride, out_row0, vin, gvu, save1};
    launch_gemm_auto<T, 64, 64, 2, 2, SW1_STAGES, 4>(sa, sb, N, 4 * c->d, c->d, e1, s, PROF_SWEEP1);
  }
  if (!linear && next_attend != nullptr) {
    // GEMM 2 fused with the next sweep's attention (64-row cells; the clamp and the v_ctx norm
    // are in its epilogue)
    SrcRows<T> av{vin, c->d, N};
    SrcRows<T> bv{(const T*)w->w_vctx, c->d, c->d};
    EpiSweep2Head<T, DH> e2{g, N, vraw, glogx, gvu, Vout, out_stride, out_row0, save2, vgain};
    if (launch_log() != nullptr) {
      record_launch<Sweep2AttendBody<T, DH>>(dim3(c->h, N / CMAX), dim3(256),
                                             typename Sweep2AttendBody<T, DH>::Args{av, bv, c->d, e2, *next_attend});
      return;
    }
    uint64_t* ts;
    const int idx = prof_launch_begin(PROF_SWEEP2, true, ts);
    if (ahead != nullptr && ahead->ns > 0) {
      const int nfused = c->h * (N / CMAX);
      launch_timed(idx, k_sweep2_attend_comm<T, DH>, dim3(nfused + ahead->ns * c->B * c->h), dim3(256), 0, s, av,
                   bv, c->d, e2, *next_attend, ahead->ca, nfused, ahead->s0, ts);
    } else {
      launch_timed(idx, k_sweep2_attend<T, DH>, dim3(c->h, N / CMAX), dim3(256), 0, s, av, bv, c->d, e2,
                   *next_attend, ts);
    }
    return;
  }
  if (!linear && vgain != nullptr) {
    // v_ctx norm: 64 x DH blocks hold whole heads (the clamp runs in the same epilogue)
    SrcRows<T> av{vin, c->d, N};
    SrcRows<T> bv{(const T*)w->w_vctx, c->d, c->d};
    EpiSweep2Head<T, DH> e2{g, N, vraw, glogx, gvu, Vout, out_stride, out_row0, save2, vgain};
    constexpr int S2 = SW2_STAGES > 0 ? SW2_STAGES : 3;
    launch_gemm_auto<T, 64, DH, 4, 1, S2, 4>(av, bv, N, c->d, c->d, e2, s, PROF_SWEEP2);
    return;
  }
  // GEMM 2 in wave tiles while their operands are few; measured against 64 x 32 blocks: d = 1024, 192 rows
  // 5.3 / 6.4 us, 256 6.5 / 6.4; d = 2048, 96 rows 8.1 / 10.0, 128 10.3 / 10.0; d = 3072, 64 rows 11.0 / 13.4, 96
  // 19.0 / 13.6
  bool gemm2_done = false;
  if constexpr (sizeof(T) == 2) {
    if (!linear && (long)N * c->d <= 196608 && refine_wt_ok<T>(c, w, N, o, vin)) {
      if (g.pos_dev != nullptr)
        launch_gemm2_wt<T, DH, true>(c, w, g, N, vraw, glogx, Vout, out_stride, out_row0, vin, gvu, save2, s);
      else
        launch_gemm2_wt<T, DH, false>(c, w, g, N, vraw, glogx, Vout, out_stride, out_row0, vin, gvu, save2, s);
      gemm2_done = true;
    }
  }
  if (!linear && !gemm2_done) {
    SrcRows<T> av{vin, c->d, N};
    SrcRows<T> bv{(const T*)w->w_vctx, c->d, c->d};
    if (g.pos_dev != nullptr) {   // device position (see GEMM 1)
      EpiSweep2<T, DH, true> e2{g, N, vraw, glogx, gvu, Vout, out_stride, out_row0, save2};
      if constexpr (SW2_STAGES > 0)
        launch_gemm_auto<T, 64, 32, 4, 1, SW2_STAGES, 8>(av, bv, N, c->d, c->d, e2, s, PROF_SWEEP2);
      else
        launch_gemm<T, 64, 32, 4, 1, 8>(av, bv, N, c->d, c->d, e2, s, PROF_SWEEP2);
    } else {
      EpiSweep2<T, DH> e2{g, N, vraw, glogx, gvu, Vout, out_stride, out_row0, save2};
      if constexpr (SW2_STAGES > 0)
        launch_gemm_auto<T, 64, 32, 4, 1, SW2_STAGES, 8>(av, bv, N, c->d, c->d, e2, s, PROF_SWEEP2);
      else
        launch_gemm<T, 64, 32, 4, 1, 8>(av, bv, N, c->d, c->d, e2, s, PROF_SWEEP2);
    }
  }
  // v'' entry-norm clamp of the refined value rows (v_clamp_tau > 0 only)
  if (g.v_clamp_tau > 0.f) {
    const dim3 grid(cdiv((long)N * c->h, 4));
    if (launch_log() != nullptr)
      record_launch<ClampBody<T, DH>>(grid, dim3(256),
                                      typename ClampBody<T, DH>::Args{g, Vout, out_stride, out_row0, N, g.v_clamp_tau});
    else
      hipLaunchKernelGGL((k_clamp_v<T, DH>), grid, dim3(256), 0, s, g, Vout, out_stride, out_row0, N, g.v_clamp_tau);
  }
}

// Committed accumulator of a cell: split partials over its committed keys but the last ones
// (comm_prev_lo), merged by the first sweep's attention, which adds those last keys itself.
template <typename T, int DH>
int run_comm(const CellGeom& g, const T* qr, const T* Kc, const T* Vc, float scale, const CellWs& ws,
             hipStream_t s) {
  const int kstart = comm_kstart(g.pos0, g.window);
  const int prev_lo = comm_prev_lo(g.pos0, kstart);
  const CommPlan cp = comm_plan(prev_lo - kstart, g.B * g.h);
  const int BH = g.B * g.h;
  CommArgs<T> ca{g, qr, Kc, Vc, cp.split_len, scale, ws.Ap, ws.Zp, ws.Mp};
  ca.nsplit = cp.nsplit;
  ca.kstart = kstart;
  ca.kend = prev_lo;
  if (launch_log() != nullptr) {
    // recorded even without a committed prefix (grid x 0), so that every chunk of a layer
    // records the same launch sequence
    record_launch<CommBody<T, DH>>(dim3(cp.nsplit, BH), dim3(256), ca);
    return cp.nsplit;
  }
  if (cp.nsplit == 0) return 0;
  launch_k(PROF_COMM, k_comm_partial<T, DH>, dim3(cp.nsplit, BH), dim3(256), 0, s, ca);
  return cp.nsplit;
}

// Where a cell without saved state keeps its intra rows: by default the chunk's own cache rows
// [pos0, pos0 + cc) (refined in place, the last sweep leaving the final rows there); a caller
// that holds the committed prefix apart from the new rows (chunk_cell_forward's K_comm / V_comm)
// gives a separate row buffer.
template <typename T> struct CellRows {
  T* K = nullptr; T* V = nullptr;   // nullptr: the cache rows
  long stride = 0;                  // elements between (b, h) row blocks
  int row0 = 0;                     // row of chunk row 0
  int rope_t0 = -1;                 // RoPE table row of chunk row 0 (-1: pos0)
};

// k_attend over a cell's rows: 16-row waves; the (b, h) blocks split by query rows until there are
// >= 256 blocks
template <typename T, int DH> void launch_attend(const AttendArgs<T>& aa, int BH, hipStream_t s) {
  if (launch_log() != nullptr) {
    if (BH >= 256) record_launch<AttendBody<T, DH, 4>>(dim3(BH, 1), dim3(256), aa);
    else if (BH >= 128) record_launch<AttendBody<T, DH, 2>>(dim3(BH, 2), dim3(128), aa);
    else record_launch<AttendBody<T, DH, 1>>(dim3(BH, 4), dim3(64), aa);
  } else if (BH >= 256) launch_k(PROF_ATTEND, k_attend<T, DH, 4>, dim3(BH, 1), dim3(256), 0, s, aa);
  else if (BH >= 128) launch_k(PROF_ATTEND, k_attend<T, DH, 2>, dim3(BH, 2), dim3(128), 0, s, aa);
  else launch_k(PROF_ATTEND, k_attend<T, DH, 1>, dim3(BH, 4), dim3(64), 0, s, aa);
}

// One chunk cell [pos0, pos0+cc) of the layer: n_sweeps Jacobi sweeps against the
// committed rows [0, pos0) of the cache. Without `sv` the sweeps refine the
// chunk's rows in place (the cache rows, or `rows`) and the last sweep leaves the final rows
// there; with `sv` every sweep's rows and state are kept in sv (cache rows untouched).
// Layer loops hand committed-prefix work from one cell to the next: own_nsplit >= 0 says the
// previous cell's launches already computed this cell's split partials (that many); next_pos0 >= 0
// names the next cell (next_cc rows), whose split partials this cell computes inside its fused
// GEMM 2 + attention launches where it has them. Returns how many it computed (-1: none, the next
// cell runs its own). The partials are the same either way: same plan, same kernel body.
template <typename T, int DH>
int run_cell(const dm_config* c, const dm_packed* w, const dm_layer_bufs* L, const float* cos,
             const float* sin, int pos0, int cc, int n_sweeps, int buf_t0, int Tbuf, T* Kc, T* Vc,
             int cache_T, T* ocat, float* o_last, const CellWs& ws, const CellSave<T>* sv, hipStream_t s,
             const CellRows<T>& rows = CellRows<T>{}, bool wide = false, int own_nsplit = -1, int next_pos0 = -1,
             int next_cc = 0) {
  CellGeom g{c->B, cc, c->d, c->h, DH, pos0, buf_t0, Tbuf, cache_T};
  g.kmod_cols = c->kmod_vraw_heads * DH;
  g.kmod_mode = c->kmod_mode;
  g.v_clamp_tau = c->v_clamp_tau;
  g.rope_t0 = rows.rope_t0;
  g.window = window_of(c);
  T* Kr = rows.K ? rows.K : Kc;
  T* Vr = rows.K ? rows.V : Vc;
  const long rows_stride = rows.K ? rows.stride : (long)cache_T * DH;
  const int rows_row0 = rows.K ? rows.row0 : pos0;
  const int BH = c->B * c->h;
  const int N = c->B * cc;
  const size_t NS = (size_t)N, d = c->d;   // per-sweep row stride of the saved arrays
  const float scale = 1.0f / sqrtf((float)DH);
  const T* qr = (const T*)L->qr;
  const T* kself = (const T*)L->kself;
  const T* vraw = (const T*)L->vraw;
  const T* kraw = (const T*)L->kraw;
  const int nsplit = own_nsplit >= 0 ? own_nsplit : run_comm<T, DH>(g, qr, Kc, Vc, scale, ws, s);
  const int prev_lo = comm_prev_lo(pos0, comm_kstart(pos0, g.window));
  const bool committed = pos0 > comm_kstart(pos0, g.window);
  const long cache_stride = (long)cache_T * DH, ws_stride = (long)CMAX * DH;
  const size_t slot = (size_t)BH * CMAX * DH;

  // Exact cells (K >= c) whose sweeps nobody reads back: row q is final after sweep q and a sweep's
  // rows do not depend on each other, so step q computes row q alone, from the refined rows before
  // it: c steps of B rows instead of c sweeps of B c, every row's arithmetic the same (the same
  // results, bit for bit). A step is three few-row launches: measured on MI355X at B = 2, d = 512,
  // T = 300 (DualModAttention.forward) 13 us against 21 us for a sweep of 128 rows.
  if constexpr (sizeof(T) == 2) {
    if (sv == nullptr && n_sweeps >= cc && cc > 1 && refine_few_rows<T>(c, w, c->B, (const T*)ws.o, (const T*)ws.vin)) {
      AttendArgs<T> aa{g, qr, kself, vraw, Kr, Vr, rows_stride, rows_row0, 0, ws.Ap, ws.Zp, ws.Mp, ws.A, ws.Z, ws.M,
                       scale, (T*)ws.o, ws.ssq, nullptr, nullptr, nullptr, nullptr, 0, Kc, Vc, pos0};
      if (committed) {   // the first sweep's attention merges the committed state of every row
        AttendArgs<T> am = aa;
        am.Kin = kself; am.Vin = vraw; am.in_stride = (long)Tbuf * DH; am.in_row0 = buf_t0;
        am.nsplit = nsplit;
        am.prev_lo = prev_lo;
        launch_attend<T, DH>(am, BH, s);
        aa.merged_in = 1;
      }
      aa.ocat = ocat;
      aa.o_last = o_last;
      for (int q = 0; q < cc; ++q) {
        launch_k(PROF_ATTEND, k_attend_row<T, DH>, dim3(BH), dim3(64), 0, s, aa, q);
        CellGeom gq = g;
        gq.c = 1;
        gq.pos0 = pos0 + q;
        gq.buf_t0 = buf_t0 + q;
        if (g.rope_t0 >= 0) gq.rope_t0 = g.rope_t0 + q;
        run_refine<T, DH>(c, w, gq, c->B, (const T*)ws.o, ws.ssq, kraw, vraw, (const T*)L->glogx, (const T*)L->sig, cos,
                          sin, Kr, Vr, rows_stride, rows_row0 + q, (T*)ws.vin, (T*)ws.gvu, nullptr, nullptr, s);
      }
      return -1;
    }
  }

  // sweep s + 1's attention runs inside sweep s's GEMM 2 launch (mult family, whole 64-row
  // chunks) when B*h gives that kernel enough blocks, or when forced by the flags
  const bool fuse = c->ctx_mod != DM_CTX_LINEAR && cc == CMAX && !(c->flags & DM_FLAG_UNFUSED_ATTEND) &&
                    ((c->flags & DM_FLAG_FUSED_ATTEND) || BH >= 128);
  // the next cell's split partials, spread over this cell's fused GEMM 2 + attention launches
  // (sweeps 0 .. K-2: one block per (b, h), CUs to spare; as extra blocks of the plain 64 x 32 GEMM 2
  // launches, which fill the chip, they cost more than their own launch); they read only keys
  // before this cell (the next cell's last 64 committed keys are its own attention's)
  auto hosts = [&](int sw) { return fuse && sw < n_sweeps - 1; };
  int n_hosts = 0;
  for (int sw = 0; sw < n_sweeps; ++sw) n_hosts += hosts(sw) ? 1 : 0;
  AheadComm<T> ahead;
  int handed = -1;
  if (next_pos0 >= 0 && n_hosts > 0 && launch_log() == nullptr) {
    CellGeom gn = g;
    gn.pos0 = next_pos0;
    gn.c = next_cc;
    gn.buf_t0 = buf_t0 + (next_pos0 - pos0);
    const int kst = comm_kstart(next_pos0, g.window), plo = comm_prev_lo(next_pos0, kst);
    const CommPlan cp = comm_plan(plo - kst, BH);
    if (plo <= pos0) {
      ahead.ca = CommArgs<T>{gn, qr, Kc, Vc, cp.split_len, scale, ws.Ap, ws.Zp, ws.Mp};
      ahead.ca.nsplit = cp.nsplit;
      ahead.ca.kstart = kst;
      ahead.ca.kend = plo;
      handed = cp.nsplit;
    }
  }
  auto ahead_for = [&](int sw) -> const AheadComm<T>* {
    if (handed <= 0 || !hosts(sw)) return nullptr;
    int j = 0;   // this launch's index among the hosting ones
    for (int u = 0; u < sw; ++u) j += hosts(u) ? 1 : 0;
    ahead.s0 = handed * j / n_hosts;
    ahead.ns = handed * (j + 1) / n_hosts - ahead.s0;
    return &ahead;
  };
  // intra rows read by sweep sw (= the rows written by sweep sw - 1)
  auto rows_in = [&](int sw, const T*& Kin, const T*& Vin, long& in_stride, int& in_row0) {
    if (sw == 0) { Kin = kself; Vin = vraw; in_stride = (long)Tbuf * DH; in_row0 = buf_t0; }
    else if (sv) { Kin = sv->Kin + sw * slot; Vin = sv->Vin + sw * slot; in_stride = ws_stride; in_row0 = 0; }
    else { Kin = Kr; Vin = Vr; in_stride = rows_stride; in_row0 = rows_row0; }
  };
  auto attend_args = [&](int sw) {
    const bool last = sw == n_sweeps - 1;
    const T* Kin; const T* Vin; long in_stride; int in_row0;
    rows_in(sw, Kin, Vin, in_stride, in_row0);
    T* o = sv ? sv->o + sw * NS * d : (T*)ws.o;
    float* ssq = sv ? sv->ssq + sw * NS * c->h : ws.ssq;
    return AttendArgs<T>{g, qr, kself, vraw, Kin, Vin, in_stride, in_row0,
                         sw == 0 ? nsplit : 0, ws.Ap, ws.Zp, ws.Mp, ws.A, ws.Z, ws.M,
                         scale, o, ssq, last ? ocat : nullptr, last ? o_last : nullptr,
                         sv ? sv->stat_m + sw * (size_t)BH * CMAX : nullptr,
                         sv ? sv->stat_z + sw * (size_t)BH * CMAX : nullptr,
                         sw > 0 && committed ? 1 : 0, Kc, Vc, sw == 0 ? prev_lo : pos0};
  };

  for (int sw = 0; sw < n_sweeps; ++sw) {
    const bool last = sw == n_sweeps - 1;
    // rows written by this sweep's refine
    T* Kout; T* Vout; long out_stride; int out_row0;
    if (sv && !(last && sv->last_to_cache)) { Kout = sv->Kin + (sw + 1) * slot; Vout = sv->Vin + (sw + 1) * slot; out_stride = ws_stride; out_row0 = 0; }
    else if (sv) { Kout = Kc; Vout = Vc; out_stride = cache_stride; out_row0 = pos0; }
    else { Kout = Kr; Vout = Vr; out_stride = rows_stride; out_row0 = rows_row0; }

    T* o = sv ? sv->o + sw * NS * d : (T*)ws.o;
    float* ssq = sv ? sv->ssq + sw * NS * c->h : ws.ssq;
    if (sw == 0 || !fuse) {   // else the previous sweep's GEMM 2 launch ran it
      const AttendArgs<T> aa = attend_args(sw);
      launch_attend<T, DH>(aa, BH, s);
    }
    T* vin = sv ? sv->vin + sw * NS * d : (T*)ws.vin;
    const AttendArgs<T> next = attend_args(last ? sw : sw + 1);
    run_refine<T, DH>(c, w, g, N, o, ssq, kraw, vraw, (const T*)L->glogx, (const T*)L->sig, cos, sin, Kout, Vout,
                      out_stride, out_row0, vin, (T*)ws.gvu, sv ? sv->save1 + sw * NS * 4 * d : nullptr,
                      sv ? sv->save2 + sw * NS * d : nullptr, s, (fuse && !last) ? &next : nullptr, wide,
                      ahead_for(sw));
  }
  return handed;
}

template <typename T>
int run_cell_dispatch(const dm_config* c, const dm_packed* w, const dm_layer_bufs* L, const float* cos,
                      const float* sin, int pos0, int cc, int n_sweeps, int buf_t0, int Tbuf, void* Kc,
                      void* Vc, int cache_T, void* ocat, float* o_last, const CellWs& ws,
                      const CellSave<T>* sv, hipStream_t s, const CellRows<T>& rows = CellRows<T>{},
                      int own_nsplit = -1, int next_pos0 = -1, int next_cc = 0) {
  if (c->dh == 64)
    return run_cell<T, 64>(c, w, L, cos, sin, pos0, cc, n_sweeps, buf_t0, Tbuf, (T*)Kc, (T*)Vc, cache_T, (T*)ocat,
                           o_last, ws, sv, s, rows, false, own_nsplit, next_pos0, next_cc);
  return run_cell<T, 128>(c, w, L, cos, sin, pos0, cc, n_sweeps, buf_t0, Tbuf, (T*)Kc, (T*)Vc, cache_T, (T*)ocat,
                          o_last, ws, sv, s, rows, false, own_nsplit, next_pos0, next_cc);
}

inline int check_bufs(const dm_config* c, const dm_layer_bufs* L) {
  DM_REQUIRE(L != nullptr, DM_ERR_INVALID, "null layer buffers");
  DM_REQUIRE(L->T > 0, DM_ERR_INVALID, "layer buffer T=%d", L->T);
  DM_REQUIRE(L->qr && L->kraw && L->kself && L->vraw && L->glogx, DM_ERR_INVALID, "null layer buffer");
  DM_REQUIRE(aligned16(L->qr) && aligned16(L->kraw) && aligned16(L->kself) && aligned16(L->vraw),
             DM_ERR_INVALID, "layer buffers must be 16-byte aligned");
  DM_REQUIRE(c->ctx_mod == DM_CTX_LINEAR || L->sig != nullptr, DM_ERR_INVALID,
             "ctx_mod mult/mult_res needs the sig buffer");
  return DM_OK;
}

inline int check_packed(const dm_config* c, const dm_packed* w) {
  DM_REQUIRE(w != nullptr, DM_ERR_INVALID, "null packed weights");
  DM_REQUIRE(w->w_proj && w->b_proj && w->w_sweep && w->norm_ctx_w, DM_ERR_INVALID, "null packed weight");
  DM_REQUIRE(c->ctx_mod == DM_CTX_LINEAR || w->w_vctx, DM_ERR_INVALID, "mult family needs w_vctx");
  DM_REQUIRE(c->norms == 0 || w->gains, DM_ERR_INVALID, "the head norms need the packed gains");
  DM_REQUIRE(aligned16(w->w_proj) && aligned16(w->w_sweep) && aligned16(w->norm_ctx_w) &&
                 (w->w_vctx == nullptr || aligned16(w->w_vctx)),
             DM_ERR_INVALID, "packed weights must be 16-byte aligned");
  return DM_OK;
}

}  // namespace dm
