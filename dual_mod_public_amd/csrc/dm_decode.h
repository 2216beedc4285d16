// Decode kernels: split-P streaming read of the static tape + LSE merge.
#pragma once

#include "dm_attn.h"

namespace dm {

// ---------------------------------------------------------------------------
// decode: split-P read of the tape (attention.py:283-312 over a static tape)
// grid (nsplit, B*h); keys [lo + s*L, min(lo + (s+1)*L, pos))
// With pos_dev set, the position is read from device memory at run time (one launch
// shape serves every position, as a captured graph needs): the grid covers the whole
// tape, blocks past the position return, and (pos, lo, nsplit) follow from *pos_dev.
// ---------------------------------------------------------------------------
template <typename T> struct DecodeArgs {
  int B, h, d, tape_T, pos, lo, split_len, nsplit;
  float scale;
  const T* q;        // [B, h, 1, dh] rotated query of this step
  const T* kself;    // [B, h, 1, dh]
  const T* vself;    // [B, h, 1, dh]
  const T* Kt; const T* Vt;   // tape [B, h, tape_T, dh]
  float* part;       // [nsplit, B*h, dh + 2]: A[dh], Z, m
  float* o;          // [B, d] fp32
  float* ssq;        // [B, h]
  T* o_cat;          // [B, d] storage dtype
  uint64_t* prof_ts; // per-dispatch timing slots (nullptr: untimed)
  const int* pos_dev = nullptr;   // device position (nullptr: pos / lo / nsplit above)
  int window = 0;                 // local_window (W tokens incl. self, 0 = full) for pos_dev
};

// a device position clamped into the tape (a caller's position past the tape reads and
// writes inside it instead of out of bounds)
DM_DEV int clamp_pos(int p, int tape_T) { return p < 0 ? 0 : (p >= tape_T ? tape_T - 1 : p); }
DM_DEV int window_lo(int pos, int W) { return (W > 0 && pos > W - 1) ? pos - (W - 1) : 0; }
template <typename T>
DM_DEV void dec_geometry(const DecodeArgs<T>& a, int& pos, int& lo, int& nsplit) {
  if (a.pos_dev == nullptr) {
    pos = a.pos; lo = a.lo; nsplit = a.nsplit;
    return;
  }
  pos = clamp_pos(*a.pos_dev, a.tape_T);
  lo = window_lo(pos, a.window);
  nsplit = pos > lo ? (pos - lo + a.split_len - 1) / a.split_len : 0;
}

// Threads per split: 16 passes of whole key rows over a split of 512 keys in bf16. Bound by the read of
// the tape; at head_dim 128 256 threads held 32 passes = 128 registers of loads, three blocks per CU,
// and 512 threads read faster (a step of B = 16, h = 16, 3001 keys: 121 us against 99).
template <typename T, int DH> constexpr int dec_threads() { return sizeof(T) == 2 ? 4 * DH : 256; }

// The unnormalised state of one split's keys [k_begin, k_end) by NT threads (tid 0 .. NT - 1): A[DH], Z, m
// into out[0 .. DH + 2). red is the group's LDS; block-wide barriers, so every group of a block calls it.
// EARLY: the V rows are loaded with the K rows (short reads, whose time is their round trips) instead of
// in K's registers after the scores (long ones, where more blocks per CU hide them). L: the keys whose
// passes are made, at least the split's (a pass past its keys adds probabilities 0: the same results).
// No pass is made conditional: with branches between the loads each use would wait for all of them
// (measured at B*h = 1024, P = 32769: 1360 us against 1302).
template <typename T, int DH, int L, bool EARLY>
DM_DEV void decode_split(const DecodeArgs<T>& a, int bh, int k_begin, int k_end, int tid, float (*red)[DH + 2],
                         float* out) {
  constexpr int NT = dec_threads<T, DH>(), NW = NT / 64;
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int LPK = DH / VEC;          // lanes per key row
  constexpr int KPP = NT / LPK;          // keys per pass
  constexpr int NP = L / KPP;            // passes
  constexpr bool V_FOLLOWS = !EARLY && regs_full<T, DH>();
  static_assert(L % KPP == 0, "split length");
  const int lane = tid & 63, wave = tid >> 6;
  const int kslot = tid / LPK, part = tid - kslot * LPK;

  float qv[VEC];
  unpack16<T>(*reinterpret_cast<const uint4*>(a.q + (long)bh * DH + part * VEC), qv);
  const T* Kb = a.Kt + (long)bh * a.tape_T * DH + part * VEC;
  const T* Vb = a.Vt + (long)bh * a.tape_T * DH + part * VEC;

  uint4 raw[NP], rv[EARLY ? NP : 1];
  auto load = [&](const T* base, int i) {
    const int key = k_begin + i * KPP + kslot;
    return keep_if(ld_nt(base + (long)(key < k_end ? key : k_begin) * DH), key < k_end);
  };
#pragma unroll
  for (int i = 0; i < NP; ++i) raw[i] = load(Kb, i);
  if constexpr (EARLY) {
#pragma unroll
    for (int i = 0; i < NP; ++i) rv[i] = load(Vb, i);
  }
  float sc[NP];
  float mx = NEG_INF;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const bool ok = k_begin + i * KPP + kslot < k_end;
    float kv[VEC];
    unpack16<T>(raw[i], kv);
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) dot += qv[j] * kv[j];
    dot = lanes_sum<1, LPK / 2>(dot);
    sc[i] = ok ? dot * a.scale : NEG_INF;
    mx = fmaxf(mx, sc[i]);
    // 256 registers of K rows: a V row is loaded as soon as its K row's are free (B*h = 512, 1600 keys: 322 us with
    // V's loads behind all scores, 242 so)
    if constexpr (V_FOLLOWS) raw[i] = load(Vb, i);
  }
  if constexpr (!EARLY && !V_FOLLOWS) {
#pragma unroll
    for (int i = 0; i < NP; ++i) raw[i] = load(Vb, i);
  }
  // group max
  mx = lanes_max<LPK, 32>(mx);
  if (lane == 0) red[wave][0] = mx;
  __syncthreads();
  float M = red[0][0];
#pragma unroll
  for (int w = 1; w < NW; ++w) M = fmaxf(M, red[w][0]);
  __syncthreads();
  float acc[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) acc[j] = 0.f;
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const float p = (sc[i] == NEG_INF) ? 0.f : __expf(sc[i] - M);
    z += p;
    float vv[VEC];
    unpack16<T>(EARLY ? rv[EARLY ? i : 0] : raw[i], vv);
#pragma unroll
    for (int j = 0; j < VEC; ++j) acc[j] += p * vv[j];
  }
  // reduce over key slots: lanes with equal `part` inside the wave, then waves
#pragma unroll
  for (int j = 0; j < VEC; ++j) acc[j] = lanes_sum<LPK, 32>(acc[j]);
  // z counted once per key (all LPK lanes of a key hold the same p): use part 0
  float zz = (part == 0) ? z : 0.f;
  zz = wave_sum(zz);
  if (lane < LPK) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) red[wave][lane * VEC + j] = acc[j];
  }
  if (lane == 0) red[wave][DH] = zz;
  __syncthreads();
  for (int i = tid; i < DH + 1; i += NT) {
    float v = red[0][i];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][i];
    out[i] = v;
  }
  if (tid == 0) out[DH + 1] = M;
}

template <typename T, int DH, int L>
__global__ __launch_bounds__((dec_threads<T, DH>())) void k_decode_partial(DecodeArgs<T> a) {
  const uint64_t t0 = prof_begin(a.prof_ts);
  __shared__ float red[dec_threads<T, DH>() / 64][DH + 2];
  const int s = blockIdx.x, bh = blockIdx.y;
  int pos, lo, nsplit;
  dec_geometry(a, pos, lo, nsplit);
  if (s >= nsplit) return;   // whole block: past the position (device-position grids only)
  const int k_begin = lo + s * a.split_len;
  decode_split<T, DH, L, false>(a, bh, k_begin, min(k_begin + a.split_len, pos), threadIdx.x, red,
                         a.part + ((long)s * (a.B * a.h) + bh) * (DH + 2));
  prof_end(a.prof_ts, t0);
}

// The step's own inputs of one (b, h) for the merge, per lane of one wave
template <int DH> struct DecodeSelf {
  float qk, v[DH / 64];
};
template <typename T, int DH> DM_DEV DecodeSelf<DH> decode_self(const DecodeArgs<T>& a, int bh, int lane) {
  constexpr int PER = DH / 64;
  DecodeSelf<DH> sf;
  sf.qk = 0.f;
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    sf.qk += to_f(a.q[(long)bh * DH + lane * PER + e]) * to_f(a.kself[(long)bh * DH + lane * PER + e]);
    sf.v[e] = to_f(a.vself[(long)bh * DH + lane * PER + e]);
  }
  return sf;
}

// merge of nsplit split states (split s at part + s pstride) and the raw self column -> o, ssq, o_cat,
// by the 64 lanes of one wave
template <typename T, int DH>
DM_DEV void decode_merge(const DecodeArgs<T>& a, const DecodeSelf<DH>& sf, const float* part, long pstride, int nsplit,
                         int bh, int lane) {
  constexpr int PER = DH / 64;
  const int b = bh / a.h, hh = bh - b * a.h;
  const float ss = wave_sum(sf.qk) * a.scale;
  float M = ss;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, part[s * pstride + DH + 1]);
  const float es = __expf(ss - M);
  float z = es;
  float acc[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) acc[e] = es * sf.v[e];
  for (int s = 0; s < nsplit; ++s) {
    const float* pp = part + s * pstride;
    const float w = (pp[DH + 1] == NEG_INF) ? 0.f : __expf(pp[DH + 1] - M);
    z += w * pp[DH];
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] += w * pp[lane * PER + e];
  }
  const float inv = 1.0f / z;
  float sq = 0.f;
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const float v = acc[e] * inv;
    sq += v * v;
    a.o[(long)b * a.d + hh * DH + lane * PER + e] = v;
    a.o_cat[(long)b * a.d + hh * DH + lane * PER + e] = from_f<T>(v);
  }
  sq = wave_sum(sq);
  if (lane == 0) a.ssq[(long)b * a.h + hh] = sq;
}

// merge split partials + raw self column -> o, ssq, o_cat (one wave per (b, h))
template <typename T, int DH>
__global__ __launch_bounds__(64) void k_decode_merge(DecodeArgs<T> a) {
  const int bh = blockIdx.x, lane = threadIdx.x;
  int pos, lo, nsplit;
  dec_geometry(a, pos, lo, nsplit);
  const DecodeSelf<DH> sf = decode_self<T, DH>(a, bh, lane);
  decode_merge<T, DH>(a, sf, a.part + (long)bh * (DH + 2), (long)(a.B * a.h) * (DH + 2), nsplit, bh, lane);
}

// The whole read of a short tape in one launch: block = one (b, h), NS groups of threads each one
// split of L keys (the split kernel's arithmetic), their states in LDS, merged by the first wave (the
// merge kernel's arithmetic: the same results as the two launches). A launch and a round trip of the
// partials less; the grid is B*h blocks whatever the tape's length, so it pays while NS groups cover
// the read and B*h blocks of them are resident together (run_decode_read).
template <typename T, int DH, int L, int NS>
__global__ __launch_bounds__((dec_threads<T, DH>() * NS)) void k_decode_direct(DecodeArgs<T> a) {
  constexpr int NT = dec_threads<T, DH>();
  __shared__ float red[NS][NT / 64][DH + 2];
  __shared__ float part[NS][DH + 2];
  const int bh = blockIdx.x, grp = threadIdx.x / NT, tid = threadIdx.x % NT;
  int pos, lo, nsplit;
  dec_geometry(a, pos, lo, nsplit);
  DecodeSelf<DH> sf{};
  if (threadIdx.x < 64) sf = decode_self<T, DH>(a, bh, threadIdx.x);
  // a group past the position reads no key (k_end = k_begin, clamped into the tape) and its state is not merged
  const int kb = min(lo + grp * L, max(pos - 1, 0));
  const int ke = grp < nsplit ? min(lo + (grp + 1) * L, pos) : kb;
  // EARLY in blocks of 256 threads only: with 512 (two splits, 777 keys) a step took 24.0 us against 23.4.
  // The first split's keys bound every group's passes (uniform over the block): up to a quarter of a
  // split makes a quarter of the passes.
  constexpr bool EARLY = NT * NS <= 256;
  if (pos - lo <= L / 4) decode_split<T, DH, L / 4, EARLY>(a, bh, kb, ke, tid, red[grp], part[grp]);
  else decode_split<T, DH, L, EARLY>(a, bh, kb, ke, tid, red[grp], part[grp]);
  __syncthreads();
  if (threadIdx.x < 64) decode_merge<T, DH>(a, sf, &part[0][0], DH + 2, min(nsplit, NS), bh, threadIdx.x);
}

// device position: the RoPE rows of position *pos_dev -> rope[0, half) cos, rope[half, 2 half) sin
static __global__ __launch_bounds__(64) void k_decode_pos_rope(const int* pos_dev, int tape_T, const float* cos,
                                                        const float* sin, int half, float* rope) {
  const int pos = clamp_pos(*pos_dev, tape_T);
  for (int i = threadIdx.x; i < half; i += 64) {
    rope[i] = cos[(long)pos * half + i];
    rope[half + i] = sin[(long)pos * half + i];
  }
}

// device position: the refined rows [B*h, DH] staged by the refine -> tape slot *pos_dev
template <typename T, int DH>
__global__ __launch_bounds__(DH) void k_decode_commit(const int* pos_dev, int tape_T, const T* Kst, const T* Vst,
                                                      T* Kt, T* Vt) {
  const int pos = clamp_pos(*pos_dev, tape_T);
  const long bh = blockIdx.x;
  const long dst = (bh * tape_T + pos) * DH + threadIdx.x;
  Kt[dst] = Kst[bh * DH + threadIdx.x];
  Vt[dst] = Vst[bh * DH + threadIdx.x];
}

// the trunk's fp32 residual stream around a decode step (models/dualmod/model.py:127-130,
// attention.py:74-83): x[r] += delta[r] (when delta), then y[r] = x[r] * rsqrt(mean(x[r]^2) + eps)
// * w (when w), in the storage dtype. One block per row; each thread re-reads only the
// elements it wrote itself.
template <typename T>
__global__ __launch_bounds__(256) void k_residual_rmsnorm(float* x, const T* delta, const float* w, T* y, int d,
                                                         float eps) {
  __shared__ float red[4];
  float* xr = x + (long)blockIdx.x * d;
  float ss = 0.f;
  for (int j = threadIdx.x; j < d; j += 256) {
    float v = xr[j];
    if (delta != nullptr) {
      v += to_f(delta[(long)blockIdx.x * d + j]);
      xr[j] = v;
    }
    ss += v * v;
  }
  if (w == nullptr) return;
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rs = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)d + eps);
  T* yr = y + (long)blockIdx.x * d;
  for (int j = threadIdx.x; j < d; j += 256) yr[j] = from_f<T>(xr[j] * rs * w[j]);
}

// torch.argmax's order: NaN is greater than every number (the first NaN wins), otherwise the
// larger value, the smaller index on ties. argmax_takes: a lane's scan in increasing column
// order replaces its pick only by a strictly greater value or by a first NaN.
DM_DEV bool argmax_takes(float f, float v) { return f > v || (f != f && v == v); }
DM_DEV bool argmax_better(float ov, int oi, float v, int idx) {
  const bool on = ov != ov, vn = v != v;
  if (on != vn) return on;
  if (on) return oi < idx;
  return ov > v || (ov == v && oi < idx);
}

// row argmax of x [rows, cols] (first index of the maximum; one block per row)
template <typename T>
__global__ __launch_bounds__(256) void k_argmax_rows(const T* x, long ld, int cols, int64_t* out) {
  __shared__ float bv[4];
  __shared__ int bi[4];
  const T* r = x + blockIdx.x * ld;
  float v = NEG_INF;
  int idx = 0x7fffffff;
  for (int j = threadIdx.x; j < cols; j += 256) {
    const float f = to_f(r[j]);
    if (argmax_takes(f, v)) { v = f; idx = j; }   // strided scan: this lane's first maximum
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(v, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (argmax_better(ov, oi, v, idx)) { v = ov; idx = oi; }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { bv[wave] = v; bi[wave] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w)
      if (argmax_better(bv[w], bi[w], v, idx)) { v = bv[w]; idx = bi[w]; }
    out[blockIdx.x] = idx == 0x7fffffff ? 0 : idx;
  }
}

// k_residual_rmsnorm with the row held in registers (d <= 256 NPT): every load (x, delta, w) is
// issued before the reduction and nothing is re-read; the same per-element arithmetic and the same
// order of the sums, so the same results. Row `row` by a 256-thread block.
template <typename T, int NPT>
DM_DEV void residual_rmsnorm_row(int row, float* x, const T* delta, const float* w, T* y, int d, float eps, float* red) {
  float* xr = x + (long)row * d;
  float v[NPT], wv[NPT];
#pragma unroll
  for (int i = 0; i < NPT; ++i) {
    if (256 * i >= d) break;   // uniform
    const int j = threadIdx.x + 256 * i;
    const int jc = j < d ? j : 0;
    v[i] = xr[jc];
    if (delta != nullptr) v[i] += to_f(delta[(long)row * d + jc]);
    wv[i] = w != nullptr ? w[jc] : 0.f;
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NPT; ++i) {
    if (256 * i >= d) break;
    const int j = threadIdx.x + 256 * i;
    if (j < d) {
      if (delta != nullptr) xr[j] = v[i];
      ss += v[i] * v[i];
    }
  }
  if (w == nullptr) return;
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rs = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)d + eps);
  T* yr = y + (long)row * d;
#pragma unroll
  for (int i = 0; i < NPT; ++i) {
    if (256 * i >= d) break;
    const int j = threadIdx.x + 256 * i;
    if (j < d) yr[j] = from_f<T>(v[i] * rs * wv[i]);
  }
}
template <typename T, int NPT>
__global__ __launch_bounds__(256) void k_residual_rmsnorm_reg(float* x, const T* delta, const float* w, T* y, int d,
                                                             float eps) {
  __shared__ float red[4];
  residual_rmsnorm_row<T, NPT>(blockIdx.x, x, delta, w, y, d, eps, red);
}

// ---- embedding backward --------------------------------------------------------------------------
// g[idx[m]] += the sum of the rows dx[m'] with idx[m'] = idx[m], in ascending order in fp32, added up by
// chains of EMB_CHAIN rows (a frequent id's error is that of two short chains, not of one over thousands of
// rows). No sort and nothing cleared by a memset node, so it may be captured. An id outside [0, n) is left out.
constexpr int EMB_CHAIN = 64;   // rows per chain
constexpr int EMB_VEC = 4;      // columns per thread and pass of 256 threads

// acc[e] += the chained sum of the rows rows[0 .. count) (ascending; LDS) at the thread's columns of the pass
// from c0. VEC: four adjacent columns by vector loads (d a multiple of 4, aligned rows), else every 256th.
// Eight rows in flight: the loads are unconditional (the last column again past d), so that they are hoisted
// over the sums (16 rows took more registers, fewer blocks: 4096 distinct rows 26 us against 20).
template <typename T, bool VEC>
DM_DEV void emb_sum_rows(const T* dx, const int* rows, int count, int d, int c0, float (&acc)[EMB_VEC]) {
  const int cv = min(c0 + EMB_VEC * (int)threadIdx.x, d - EMB_VEC);
  for (int q0 = 0; q0 < count; q0 += EMB_CHAIN) {
    const int q1 = min(q0 + EMB_CHAIN, count);
    float ch[EMB_VEC];
#pragma unroll
    for (int e = 0; e < EMB_VEC; ++e) ch[e] = 0.f;
#pragma unroll 8
    for (int q = q0; q < q1; ++q) {
      const T* row = dx + (long)rows[q] * d;
      if constexpr (VEC) {
        float v[EMB_VEC];
        unpackv<T, EMB_VEC>(*reinterpret_cast<const typename RawV<T, EMB_VEC>::type*>(row + cv), v);
#pragma unroll
        for (int e = 0; e < EMB_VEC; ++e) ch[e] += v[e];
      } else {
#pragma unroll
        for (int e = 0; e < EMB_VEC; ++e) ch[e] += to_f(row[min(c0 + (int)threadIdx.x + 256 * e, d - 1)]);
      }
    }
#pragma unroll
    for (int e = 0; e < EMB_VEC; ++e) acc[e] += ch[e];
  }
}
// dst[columns] (+)= acc
template <bool VEC, bool ADD>
DM_DEV void emb_store(float* dst, int d, int c0, const float (&acc)[EMB_VEC]) {
  if constexpr (VEC) {
    const int c = c0 + EMB_VEC * threadIdx.x;
    if (c >= d) return;
    floatx4* p = reinterpret_cast<floatx4*>(dst + c);
    const floatx4 v = {acc[0], acc[1], acc[2], acc[3]};
    *p = ADD ? *p + v : v;
  } else {
#pragma unroll
    for (int e = 0; e < EMB_VEC; ++e) {
      const int c = c0 + threadIdx.x + 256 * e;
      if (c < d) dst[c] = ADD ? dst[c] + acc[e] : acc[e];
    }
  }
}
// The tokens of ids[j0, j0 + 256) with this id, ascending, into hits; returns their number (block-wide)
template <typename I> DM_DEV int emb_hits(const I* ids, int j0, int M, I id, int* hits, int* wcount) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = j0 + threadIdx.x;
  const bool hit = j < M && ids[j] == id;
  const unsigned long long mask = __ballot(hit);
  if (lane == 0) wcount[wave] = __popcll(mask);
  __syncthreads();
  int base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w < wave) base += wcount[w];
    total += wcount[w];
  }
  if (hit) hits[base + __popcll(mask & ((1ull << lane) - 1))] = j;
  __syncthreads();
  return total;
}

// Few tokens (EMB_ONE): one launch, the block of an id's first token sums its rows; the blocks of its later
// tokens find that one and end. Every block reads the ids (M^2 of them, from L2), and one block sums a frequent
// id's rows. bf16, us, distinct ids / half of them one padding id: 2048 x 1024 9.7 / 63 (lists: 22 / 56), 4096
// 16 / 158 (24 / 77), 6144 30 / 236 (28 / 95).
constexpr int EMB_ONE = 4096;
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void k_embed_bwd(const T* dx, const int64_t* idx, float* g, int M, int d, int n) {
  __shared__ int hits[256];
  __shared__ int wcount[4];
  __shared__ int seen;
  const int m = blockIdx.x;
  const int64_t id = idx[m];
  if (id < 0 || id >= n) return;   // uniform
  if (threadIdx.x == 0) seen = 0;
  __syncthreads();
  int any = 0;
  for (int j = threadIdx.x; j < m; j += 256) any |= idx[j] == id;
  if (any) seen = 1;
  __syncthreads();
  if (seen) return;   // uniform
  for (int c0 = 0; c0 < d; c0 += 256 * EMB_VEC) {
    float acc[EMB_VEC] = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = m; j0 < M; j0 += 256) {
      const int total = emb_hits<int64_t>(idx, j0, M, id, hits, wcount);
      emb_sum_rows<T, VEC>(dx, hits, total, d, c0, acc);
      __syncthreads();
    }
    emb_store<VEC, true>(g + id * (long)d, d, c0, acc);
  }
}

// Many tokens: the ids' row lists are found once. An id of at most EMB_LIST tokens gets a list (filled in any
// order, sorted by the block that sums it); a more frequent one is summed in pieces of `plen` tokens by the
// blocks of its first token in each, the pieces added up in order by a last launch. Bound by reading dx and
// updating g; a frequent id by its pieces' chains. bf16, us, against the library's sort and sums with their add
// into g: 16384 x 1024 distinct 42 / 268, half one padding id 174 / 442; 16384 x 2048 Zipf 80 / 451; 65536 x
// 1024 Zipf 151 / 615.
constexpr int EMB_LIST = 256, EMB_PASS = 1024, EMB_PIECES = 64, EMB_NONE = 0x7fffffff;
struct EmbWs {
  int* cnt;     // [n] tokens of an id
  int* start;   // [n] its list, or -1 - its number among the frequent ids
  int* slot;    // [M] a token's place among its id's tokens
  int* list;    // [M]
  int* fid;     // [frequent] the id
  int* first;   // [frequent, pieces] its first token in the piece, EMB_NONE without
  int* cursor;  // list entries and frequent ids handed out
  float* part;  // [frequent, pieces, d]
  int pieces, plen, frequent;
  size_t bytes;
};
static __global__ __launch_bounds__(256) void k_emb_clear(EmbWs w, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) w.cnt[i] = 0;
  if (i < w.frequent * w.pieces) w.first[i] = EMB_NONE;
  if (i < 2) w.cursor[i] = 0;
}
// one atomic per wave and id: a wave of one padding id would queue 64 at one address
static __global__ __launch_bounds__(256) void k_emb_count(EmbWs w, const int64_t* idx, int M, int n) {
  const int m = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
  const int64_t id64 = m < M ? idx[m] : -1;
  const bool ok = id64 >= 0 && id64 < n;
  const int id = ok ? (int)id64 : -1;
  unsigned long long left = __ballot(ok), mine = 0;
  while (left != 0) {   // uniform
    const int lead = __ffsll((long long)left) - 1;
    const unsigned long long same = __ballot(id == __shfl(id, lead, 64)) & left;
    if ((same >> lane) & 1) mine = same;
    left &= ~same;
  }
  const int lead = ok ? __ffsll((long long)mine) - 1 : lane;
  int base = 0;
  if (ok && lead == lane) base = atomicAdd(w.cnt + id, (int)__popcll(mine));
  base = __shfl(base, lead, 64);
  if (ok) w.slot[m] = base + (int)__popcll(mine & ((1ull << lane) - 1));
}
static __global__ __launch_bounds__(256) void k_emb_start(EmbWs w, const int64_t* idx, int M, int n) {
  const int m = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
  const int64_t id = m < M ? idx[m] : -1;
  const bool own = id >= 0 && id < n && w.slot[m] == 0;
  const int c = own ? w.cnt[id] : 0;
  const int need = c > 1 && c <= EMB_LIST ? c : 0;
  int sum = need;   // inclusive over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(sum, o, 64);
    if (lane >= o) sum += v;
  }
  const int total = __shfl(sum, 63, 64);
  int base = 0;
  if (lane == 0 && total > 0) base = atomicAdd(w.cursor, total);
  base = __shfl(base, 0, 64);
  if (need > 0) w.start[id] = base + sum - need;
  if (c > EMB_LIST) {
    const int f = atomicAdd(w.cursor + 1, 1);
    w.fid[f] = (int)id;
    w.start[id] = -1 - f;
  }
}
static __global__ __launch_bounds__(256) void k_emb_place(EmbWs w, const int64_t* idx, int M, int n) {
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m >= M) return;
  const int64_t id = idx[m];
  if (id < 0 || id >= n) return;
  const int c = w.cnt[id];
  if (c > EMB_LIST) atomicMin(w.first + (-1 - w.start[id]) * w.pieces + m / w.plen, m);
  else if (c > 1) w.list[w.start[id] + w.slot[m]] = m;
}
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void k_emb_sum(EmbWs w, const T* dx, const int64_t* idx, float* g, int M, int d, int n) {
  __shared__ int raw[EMB_LIST], rows[EMB_PASS];
  __shared__ int wcount[4];
  const int m = blockIdx.x;
  const int64_t id = idx[m];
  if (id < 0 || id >= n) return;   // uniform, as every branch below
  const int c = w.cnt[id];
  if (c > EMB_LIST) {
    const int p = m / w.plen, slot = (-1 - w.start[id]) * w.pieces + p;
    if (w.first[slot] != m) return;
    const int j1 = min((p + 1) * w.plen, M);
    for (int c0 = 0; c0 < d; c0 += 256 * EMB_VEC) {
      float acc[EMB_VEC] = {0.f, 0.f, 0.f, 0.f};
      for (int j0 = m; j0 < j1; j0 += EMB_PASS) {
        int count = 0;
        for (int j = j0; j < min(j0 + EMB_PASS, j1); j += 256)
          count += emb_hits<int64_t>(idx, j, j1, id, rows + count, wcount);
        emb_sum_rows<T, VEC>(dx, rows, count, d, c0, acc);
        __syncthreads();
      }
      emb_store<VEC, false>(w.part + (long)slot * d, d, c0, acc);
    }
    return;
  }
  if (c == 1) {
    if (threadIdx.x == 0) rows[0] = m;
    __syncthreads();
  } else {
    static_assert(EMB_LIST == 256, "an entry per thread");
    const int e = (int)threadIdx.x < c ? w.list[w.start[id] + threadIdx.x] : EMB_NONE;
    raw[threadIdx.x] = e;
    __syncthreads();
    int rank = 0;
    for (int i = 0; i < c; ++i) rank += raw[i] < e;
    if ((int)threadIdx.x < c) rows[rank] = e;
    __syncthreads();
    if (rows[0] != m) return;
  }
  for (int c0 = 0; c0 < d; c0 += 256 * EMB_VEC) {
    float acc[EMB_VEC] = {0.f, 0.f, 0.f, 0.f};
    emb_sum_rows<T, VEC>(dx, rows, c, d, c0, acc);
    emb_store<VEC, true>(g + id * (long)d, d, c0, acc);
  }
}
// block (f, x): the pieces of frequent id f in order, columns [256 x, 256 (x + 1))
static __global__ __launch_bounds__(256) void k_emb_pieces(EmbWs w, float* g, int d) {
  const int f = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (f >= w.cursor[1] || c >= d) return;
  float acc = 0.f;
  for (int p = 0; p < w.pieces; ++p)
    if (w.first[f * w.pieces + p] != EMB_NONE) acc += w.part[((long)f * w.pieces + p) * d + c];
  g[w.fid[f] * (long)d + c] += acc;
}

// Cross entropy of one row of logits per block, with its gradient in place: loss[row] = lse - x[t] and
// x <- (softmax(x) - onehot(t)) / nvalid (both 0 for t < 0, the ignored target; a t >= n gives a NaN loss).
// Statistics in fp32. Bound by reading the logits and writing the gradient: one pass over the row for the
// maximum and the sum together (rescaled once per vector), a second for the gradient. 4096 x 32000 in
// bf16: 171 us, against about 1.5 ms of elementwise passes over fp32 copies. V: elements per load (1 where the
// rows are not 16-byte aligned).
template <typename T, int V>
__global__ __launch_bounds__(256) void k_ce_rows(T* x, const int64_t* target, const float* nvalid, float* loss, int n) {
  __shared__ float red[8];
  T* xr = x + (long)blockIdx.x * n;
  const long t = target[blockIdx.x];
  const bool valid = t >= 0;
  const float xt = valid ? (t < n ? to_f(xr[t]) : __builtin_nanf("")) : to_f(xr[0]);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto load = [&](int i, float (&v)[V]) {
    if constexpr (V > 1) {
      unpack16<T>(*reinterpret_cast<const uint4*>(xr + i), v);
    } else {
      v[0] = to_f(xr[i]);
    }
  };
  float m = -3.402823466e38f, z = 0.f;
#pragma unroll 4
  for (int i = V * threadIdx.x; i < n; i += V * 256) {
    float v[V];
    load(i, v);
    float vm = m;
#pragma unroll
    for (int j = 0; j < V; ++j) vm = fmaxf(vm, v[j]);
    z *= expf(m - vm);
#pragma unroll
    for (int j = 0; j < V; ++j) z += expf(v[j] - vm);
    m = vm;
  }
  const float wm = lanes_max<1, 32>(m);
  const float wz = wave_sum(z * expf(m - wm));
  if (lane == 0) {
    red[wave] = wm;
    red[4 + wave] = wz;
  }
  __syncthreads();   // also: every thread has read x[t]
  const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float Z = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) Z += red[4 + w] * expf(red[w] - M);
  float lse = M + logf(Z);
  if (M == __builtin_inff()) {   // uniform: Z is NaN (inf - inf) whether or not the row holds one
    int bad = 0;
    for (int i = threadIdx.x; i < n; i += 256) {
      const float v = to_f(xr[i]);
      bad |= v != v;
    }
    lse = __syncthreads_or(bad) ? __builtin_nanf("") : M;
  }
  if (threadIdx.x == 0) loss[blockIdx.x] = valid ? lse - xt : 0.f;
  const float sc = valid ? 1.f / *nvalid : 0.f;
#pragma unroll 4
  for (int i = V * threadIdx.x; i < n; i += V * 256) {
    float v[V];
    load(i, v);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = (expf(v[j] - lse) - (i + j == t ? 1.f : 0.f)) * sc;
    if constexpr (V > 1) {
      store_vec<T, V>(xr + i, v);
    } else {
      xr[i] = from_f<T>(v[0]);
    }
  }
}

// The sums around k_ce_rows by one block each, in a fixed order and without state to clear: the library's sums
// split such a column over blocks and clear their counters by a memset, which a captured step would hold as
// a node. 16384 tokens: 8 us each (the library's passes 24 and 15).
// nvalid = max(number of targets >= 0, 1)
static __global__ __launch_bounds__(1024) void k_ce_count(const int64_t* target, int M, float* nvalid) {
  __shared__ int red[16];
  int c = 0;
#pragma unroll 8
  for (int m = threadIdx.x; m < M; m += 1024) c += target[m] >= 0;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x > 0) return;
  for (int w = 1; w < 16; ++w) c += red[w];
  *nvalid = (float)max(c, 1);
}
// out = (sum of x[0 .. M)) / nvalid
static __global__ __launch_bounds__(1024) void k_ce_mean(const float* x, int M, const float* nvalid, float* out) {
  __shared__ float red[16];
  float v = 0.f;
#pragma unroll 8
  for (int m = threadIdx.x; m < M; m += 1024) v += x[m];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x > 0) return;
  for (int w = 1; w < 16; ++w) v += red[w];
  *out = v / *nvalid;
}

// k_argmax_rows for 16-byte aligned rows (ld a multiple of the vector width): 1024 threads per row,
// 16-byte loads. A lane visits its columns in increasing order (its vectors, then the tail columns,
// which come last in the row), so a strict > keeps its first maximum; lanes and waves then merge
// by value, the smaller index on ties; a NaN is the maximum (the first NaN wins), as torch.argmax.
template <typename T>
__global__ __launch_bounds__(1024) void k_argmax_rows_vec(const T* x, long ld, int cols, int64_t* out) {
  constexpr int VEC = 16 / (int)sizeof(T);
  __shared__ float bv[16];
  __shared__ int bi[16];
  const T* r = x + blockIdx.x * ld;
  const int nv = cols / VEC;
  float v = NEG_INF;
  int idx = 0x7fffffff;
  for (int q = threadIdx.x; q < nv; q += 1024) {
    float f[VEC];
    unpack16<T>(*reinterpret_cast<const uint4*>(r + (long)q * VEC), f);
#pragma unroll
    for (int e = 0; e < VEC; ++e)
      if (argmax_takes(f[e], v)) { v = f[e]; idx = q * VEC + e; }
  }
  for (int j = nv * VEC + threadIdx.x; j < cols; j += 1024) {
    const float f = to_f(r[j]);
    if (argmax_takes(f, v)) { v = f; idx = j; }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(v, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (argmax_better(ov, oi, v, idx)) { v = ov; idx = oi; }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { bv[wave] = v; bi[wave] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w)
      if (argmax_better(bv[w], bi[w], v, idx)) { v = bv[w]; idx = bi[w]; }
    out[blockIdx.x] = idx == 0x7fffffff ? 0 : idx;
  }
}

}  // namespace dm
