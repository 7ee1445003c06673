// Decode-shape expert GEMVs for several rows per weight, on the fp32 matrix
// instruction v_mfma_f32_4x4x1_16b_f32.
//
// The arithmetic is gemv.hip's, bit for bit: per output and 128-element chunk
// one fma chain in ascending k from 0, the chunks folded in order.  One
// 4x4x1 instruction is 16 blocks of 4 x 4 outputs, D = A B + C with K = 1:
// each output takes one fused multiply-add, rounded as fmaf rounds it
// (denormals kept; the tests compare bits with the oracle's fmaf chains, with
// denormal, infinite and NaN rows, weights and scales among them), so a series
// of them over k is the chain.  Block b's 4 columns are lanes 4b .. 4b + 3 of
// the B operand, so B is "lane = output column" and D's register r is row r:
// the layout of the VALU kernel.  The A operand broadcasts one block (cbsz
// 4, abid = the block) to all 16: lane 4b + r holds row r's activation of the
// k that block b stands for, so one register feeds 16 k steps and no scalar
// loads are left.
//
// Why: with R rows per weight the VALU chain issues R fmas of 4 cycles and
// waits for R scalar loads per weight (a wave's chunk of 8 rows: 1 024 scalar
// values); the matrix instruction takes 8 cycles for 4 rows (measured 67-72 T
// fma/s against 35-37 on the VALU), beside one conversion a weight (a step of
// k takes 7 ns for up to 4 rows, 9 for 8, 13 for 12, 16 for 16; the waves of a
// SIMD take turns).  Against the VALU kernel: 37 int8 decode rows, gate/up 224
// -> 47 us (156 MB; 33 us with the chains left out, 45 with the loads left
// out) and down 157 -> 26 us; lm_head (331 MB) at 2 / 8 / 64 rows 69 / 84 /
// 662 -> 58 / 58 / 207 us; q/k/v at 1 / 8 / 64 rows 6.5 / 13.5 / 88 -> 5.2 /
// 6.8 / 14 us; the 6848-wide down at 8 rows 59 -> 11 us.  A layer's pair of
// launches at any number of rows, also 1: hidden 4096, ffn 1408, 64 experts, 1
// / 8 int8 rows 145 / 565 -> 90 / 176 us.
#include "uocr_device.h"
#include "uocr_kernels.h"

#include <utility>

namespace uocr {

// The byte offset, from a wave's first column, of 16-byte piece `piece` of the
// wave's column `col` (0 .. 63), or of the last of the `cols` columns from the
// first one on (rows rowb bytes apart, at most 2^17).  The column is clamped
// before it is multiplied: a matrix may hold more bytes than an int counts, the
// wave's 64 columns do not.
__host__ __device__ int rows_offset(int col, int cols, int rowb, int piece) {
  return (col < cols ? col : cols - 1) * rowb + 16 * piece;
}

namespace {

// A stage is 64 x 128 bytes of weights: 128 k of int8, 64 k of bf16.
constexpr int kStageBytes = kWave * 128;
template <WKind W>
constexpr int kStageK = W == kInt8Rows ? 128 : 64;
// C, the output columns of a wave: 64 (lane = column), or 16 for narrow
// outputs, whose few columns would leave most CUs idle: then lane = (one of 4
// chunks, column), and the A operand broadcasts inside each 16-lane quarter
// (cbsz 2).  Floats of one row's activations a lane holds per stage (its
// block's k):
template <WKind W, int C>
constexpr int kLaneX = kStageK<W> / (C / 4);

// The four weights of k = 4 q .. 4 q + 3 of a lane's column.  Plain conversions
// (the compiler folds the byte select into them), not inline asm: a matrix
// instruction may not read a VALU result in the two slots after it, and the
// compiler keeps that distance only for instructions it knows.
template <WKind W, int q>
__device__ __forceinline__ void quad(const i32x4 (&wv)[8], float (&w)[4]) {
  if constexpr (W == kInt8Rows) {
    const int v = wv[q >> 2][q & 3];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (float)(int8_t)(v >> (8 * j));
  } else {
    const uint32_t lo = (uint32_t)wv[q >> 1][(q & 1) * 2], hi = (uint32_t)wv[q >> 1][(q & 1) * 2 + 1];
    w[0] = bf16_lo(lo);
    w[1] = bf16_hi(lo);
    w[2] = bf16_lo(hi);
    w[3] = bf16_hi(hi);
  }
}
// k = 4 q .. 4 q + 3 of a stage for every row tile, from w; wn becomes the next
// four weights, converted ahead of this quad's matrix instructions (one weight
// at a time, each conversion is followed by two wait slots).  fetch(i) makes
// 16-byte piece i of the column's weights available, two pieces ahead.
template <WKind W, int C, int NT, int q, typename Fetch>
__device__ __forceinline__ void quad_chain(const i32x4 (&wv)[8], const f32x4 (&x)[NT][kLaneX<W, C> / 4],
                                           f32x4 (&part)[NT], const float (&w)[4], float (&wn)[4], Fetch&& fetch) {
  constexpr int NB = C / 4;  // blocks that share the A operand's broadcast
  constexpr int QP = kStageK<W> / 32;  // quads per piece
  if constexpr (q % QP == 0 && q / QP + 2 < 8) fetch(std::integral_constant<int, q / QP + 2>{});
  if constexpr (4 * q + 4 < kStageK<W>) quad<W, q + 1>(wv, wn);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      part[t] =
          __builtin_amdgcn_mfma_f32_4x4x1f32(x[t][q / NB][j], w[j], part[t], C == kWave ? 4 : 2, q % NB, 0);
  __builtin_amdgcn_sched_barrier(0);
}
template <WKind W, int C, int NT, typename Fetch, int... h>
__device__ __forceinline__ void quad_chains(const i32x4 (&wv)[8], const f32x4 (&x)[NT][kLaneX<W, C> / 4],
                                            f32x4 (&part)[NT], Fetch&& fetch, std::integer_sequence<int, h...>) {
  float w0[4], w1[4];
  quad<W, 0>(wv, w0);
  ((quad_chain<W, C, NT, 2 * h>(wv, x, part, w0, w1, fetch),
    quad_chain<W, C, NT, 2 * h + 1>(wv, x, part, w1, w0, fetch)),
   ...);
}
template <WKind W, int C, int NT, typename Fetch>
__device__ __forceinline__ void stage_chain(const i32x4 (&wv)[8], const f32x4 (&x)[NT][kLaneX<W, C> / 4],
                                            f32x4 (&part)[NT], Fetch&& fetch) {
  quad_chains<W, C, NT>(wv, x, part, fetch, std::make_integer_sequence<int, kStageK<W> / 8>{});
}
struct NoFetch {
  template <typename I>
  __device__ __forceinline__ void operator()(I) const {}
};

// A lane's activations of stage `stage`: block b (of C / 4) holds k = 4 b ..
// 4 b + 3 of every C consecutive k, so the blocks of a row load contiguous
// bytes.
template <WKind W, int C, int NT>
__device__ __forceinline__ void load_x(const float* const (&xp)[NT], int stage, f32x4 (&x)[NT][kLaneX<W, C> / 4]) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < kLaneX<W, C> / 4; ++v) x[t][v] = *(const UOCR_GLOBAL f32x4*)(xp[t] + stage * kStageK<W> + C * v);
}

template <int NT>
__device__ __forceinline__ void zero(f32x4 (&v)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t) v[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}

// Row-major weights of expert e, projection p: every chunk of columns n0 ..
// n0 + 63 (lane = column) for the rows at xp (lane l: its row's activations,
// from k 4 (l / 4)), folded into acc in chunk order.
//
// The weights pass through the wave's LDS stage: a lane that loaded its own
// column's 16 bytes would touch 64 cache lines per instruction, so the loads
// run 8 lanes to a column's 128 bytes (lane l of load i: column 8 i + l / 8,
// piece l % 8), the pieces are stored at piece ^ column % 8 (8 neighbouring
// columns cover all banks) and a lane reads its column's back.  The next
// stage's loads are in flight while one is computed; every load is issued in
// every iteration, so that the waits the compiler derives stay exact counts,
// and one past the last stage re-reads 16 bytes (weights) or the last stage
// (activations).
template <WKind W, int NT>
__device__ __forceinline__ void rows_chain(const GemvArgs& a, int p, int e, int n0, const float* const (&xp)[NT],
                                           char* stage, f32x4 (&acc)[NT]) {
  constexpr int C = kWave;
  constexpr int SK = kStageK<W>;
  constexpr int SPC = kChunk / SK;  // stages per chunk
  constexpr int XV = kLaneX<W, C> / 4;
  const int l = lane_id();
  const int n = min(n0 + l, a.N - 1);
  const int S = a.K / SK;
  const int64_t rowb = (int64_t)a.K * (W == kInt8Rows ? 1 : 2);
  const char* base = (const char*)a.p[p].w + ((int64_t)e * a.N + n0) * rowb;
  // load i's lane offset: column n0 + 8 i + l / 8 (past N: the last column)
  const int off0 = (l >> 3) * (int)rowb + 16 * (l & 7);
  const int off_last = rows_offset(kWave - 1, a.N - n0, (int)rowb, l & 7);
  const float* sp = W == kInt8Rows ? a.p[p].s + ((int64_t)e * a.N + n) * a.nchunks : nullptr;
  i32x4 wn[8], wv[8];
  f32x4 xn[NT][XV], x[NT][XV], part[NT];
  float scale_n = 1.0f, scale = 1.0f;
  auto load = [&](int s) {
    const bool live = s < S;
    const int sc = live ? s : S - 1;
    load_x<W, C, NT>(xp, sc, xn);
    if constexpr (W == kInt8Rows) scale_n = ldg(sp + sc);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      wn[i] = *(const UOCR_GLOBAL i32x4*)(base + (int64_t)sc * 128 + (live ? min(off0 + 8 * i * (int)rowb, off_last) : 0));
  };
  char* put = stage + 128 * (l >> 3) + 16 * ((l & 7) ^ (l >> 3));
  const char* get = stage + 128 * l;
  zero(part);
  load(0);
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *(i32x4*)(put + 1024 * i) = wn[i];
    auto fetch = [&](auto i) { wv[i] = *(const i32x4*)(get + 16 * (i ^ (l & 7))); };
    fetch(std::integral_constant<int, 0>{});
    fetch(std::integral_constant<int, 1>{});
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < XV; ++v) x[t][v] = xn[t][v];
    scale = scale_n;
    load(s + 1);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before the chain
    stage_chain<W, C, NT>(wv, x, part, fetch);
    if ((s + 1) % SPC == 0 || s + 1 == S) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t][r] = W == kInt8Rows ? __builtin_fmaf(scale, part[t][r], acc[t][r]) : acc[t][r] + part[t][r];
      zero(part);
    }
  }
}

// K-blocked weights: chunks c0 .. c1 - 1 of C columns from n0.  Lane = column,
// or, C = 16, lane = (chunk c0 + 4 j + l / 16, column n0 + l % 16) in step j
// (then always SPLIT).  SPLIT: each chunk's sums go to part_out[chunk][4 NT
// rows][C] (LDS); else into acc in chunk order.
template <int C, int NT, bool SPLIT>
__device__ __forceinline__ void kblocked_chain(const GemvArgs& a, int p, int n0, const float* const (&xp)[NT], int c0,
                                               int c1, f32x4 (&acc)[NT], float* part_out) {
  constexpr WKind W = kBf16KBlocked;
  static_assert(C == kWave || SPLIT, "a quarter's chunks are folded through LDS");
  constexpr int XV = kLaneX<W, C> / 4;
  constexpr int Q = kWave / C;  // chunks side by side
  const int l = lane_id();
  const int lc = l % C;
  const int n = min(n0 + lc, a.N - 1);
  const int S = a.K / 64;  // K may end half a chunk short
  if (c0 >= c1) return;
  const char* base = (const char*)a.p[p].w + (int64_t)n * 32;
  const int64_t kb = (int64_t)a.N * 32;
  i32x4 w0[8], w1[8];
  f32x4 x0[NT][XV], x1[NT][XV], part[NT];
  // half h (0, 1) of the lane's chunk of step j, c = c0 + Q j the step's first chunk
  auto load = [&](int c, int h, i32x4(&w)[8], f32x4(&x)[NT][XV]) {
    int s = 2 * (c + (C == kWave ? 0 : l / C)) + h;
    const bool live = C == kWave ? c < c1 && s < S : s < S && s < 2 * c1;
    s = live ? s : S - 1;
    const char* src = live || C != kWave ? base + 4 * s * kb : (const char*)a.p[p].w;
    const int64_t step = live || C != kWave ? kb : 0;
    load_x<W, C, NT>(xp, s, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = *(const UOCR_GLOBAL i32x4*)(src + (j >> 1) * step + 16 * (j & 1));
  };
  zero(part);
  load(c0, 0, w0, x0);
  for (int c = c0; c < c1; c += Q) {
    load(c, 1, w1, x1);
    __builtin_amdgcn_sched_barrier(0);
    stage_chain<W, C, NT>(w0, x0, part, NoFetch{});
    __builtin_amdgcn_sched_barrier(0);
    load(c + Q, 0, w0, x0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C == kWave) {
      if (2 * c + 1 < S) stage_chain<W, C, NT>(w1, x1, part, NoFetch{});
    } else {
      // a half past K adds 0 x 0, which leaves the sum
      if (2 * (c + Q) > S && 2 * (c + l / C) + 1 >= S) {
#pragma unroll
        for (int j = 0; j < 8; ++j) w1[j] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < NT; ++t) zero(x1[t]);
      }
      stage_chain<W, C, NT>(w1, x1, part, NoFetch{});
    }
    const int lchunk = c + (C == kWave ? 0 : l / C);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (!SPLIT)
          acc[t][r] = acc[t][r] + part[t][r];
        else if (C == kWave || lchunk < c1)
          part_out[(lchunk * 4 * NT + 4 * t + r) * C + lc] = part[t][r];
      }
    zero(part);
  }
}

// The rows of a tile: lane l's row of each 4-row tile (padded rows repeat the
// last real one and are not stored) and its activation pointer.  ROUTED: lane
// i's `row` is row i of up to 64, else the rows are their own numbers.
template <WKind W, int C, int NT, bool ROUTED>
__device__ __forceinline__ void tile_rows(const GemvArgs& a, int row, int t0, int cnt, int (&rowv)[NT],
                                          const float* (&xp)[NT]) {
  const int l = lane_id();
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int rr = t0 + min(4 * t + (l & 3), cnt - 1);
    rowv[t] = ROUTED ? __builtin_amdgcn_ds_bpermute(rr << 2, row) : rr;
    xp[t] = a.x + (int64_t)(rowv[t] / a.x_div) * a.ldx + 4 * (l % C >> 2);
  }
}

template <int NT>
__device__ __forceinline__ void store_rows(const GemvArgs& a, int n0, int cnt, const int (&rowv)[NT],
                                           const f32x4 (&acc)[NT]) {
  const int n = n0 + lane_id();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = __builtin_amdgcn_readlane(rowv[t], r);
      if (4 * t + r < cnt && n < a.N) stg(a.out + (int64_t)row * a.ldo + n, acc[t][r]);
    }
}

// A workgroup's waves on one row tile (cnt <= 4 NT rows from t0 of the 64 that
// the lanes' `row` hold) of a routed expert: wave w takes projection w % NPROJ of column block cb0 + w / NPROJ,
// all chunks.
template <WKind W, int NPROJ, int NT>
__device__ __forceinline__ void routed_tile(const GemvArgs& a, int e, int rows, int t0, int cnt, int cb0, char* lds) {
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int l = lane_id();
  const int p = w % NPROJ;
  const int n0 = (cb0 + w / NPROJ) * kWave;
  int rowv[NT];
  const float* xp[NT];
  tile_rows<W, kWave, NT, true>(a, rows, t0, cnt, rowv, xp);
  f32x4 acc[NT];
  zero(acc);
  char* stage = lds + w * kStageBytes;
  if (n0 < a.N) rows_chain<W, NT>(a, p, e, n0, xp, stage, acc);
  if constexpr (NPROJ == 2) {
    float* own = (float*)stage;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) own[(4 * t + r) * kWave + l] = acc[t][r];
    __syncthreads();
    const float* g = (const float*)(lds + (w & ~1) * kStageBytes);
    const float* u = (const float*)(lds + (w | 1) * kStageBytes);
    // the pair's waves take the even and the odd rows
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j) {
      const int r = 2 * j + p;
      const int row = __builtin_amdgcn_readlane(rowv[(2 * j) / 4], (2 * j) % 4 + p);
      if (r < cnt && n0 + l < a.N)
        stg(a.out + (int64_t)row * a.ldo + n0 + l, silu(g[r * kWave + l]) * u[r * kWave + l]);
    }
    __syncthreads();  // the stages are rewritten by the next tile
  } else {
    store_rows<NT>(a, n0, cnt, rowv, acc);
  }
}

// A dense K-blocked weight's tile (cnt <= 4 NT rows from t0) of C columns from
// n0, its chunks split over the workgroup's waves: wave w takes projection w %
// NPROJ and an equal run of chunks (of 4-chunk steps, C = 16).  The sums meet
// in LDS ([projection][chunk][row][C]) and are folded in chunk order, a thread
// per (row, column).
template <int C, int NPROJ, int NT>
__device__ __forceinline__ void dense_tile(const GemvArgs& a, int t0, int cnt, int n0, float* parts) {
  const int tid = (int)threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = w % NPROJ, q = w / NPROJ, Q = (int)(blockDim.x >> 6) / NPROJ;
  int rowv[NT];
  const float* xp[NT];
  tile_rows<kBf16KBlocked, C, NT, false>(a, 0, t0, cnt, rowv, xp);
  f32x4 unused[NT];
  constexpr int U = kWave / C;
  const int units = (a.nchunks + U - 1) / U;
  const int c0 = units * q / Q * U, c1 = min(units * (q + 1) / Q * U, a.nchunks);
  kblocked_chain<C, NT, true>(a, p, n0, xp, c0, c1, unused, parts + p * a.nchunks * 4 * NT * C);
  __syncthreads();
  const int n = n0 + tid % C;
  for (int r = tid / C; r < cnt; r += (int)blockDim.x / C) {
    float v[NPROJ];
#pragma unroll
    for (int j = 0; j < NPROJ; ++j) {
      const float* src = parts + (j * a.nchunks * 4 * NT + r) * C + tid % C;
      float s = 0.0f;
      for (int c = 0; c < a.nchunks; ++c) s = s + src[c * 4 * NT * C];
      v[j] = s;
    }
    float o = v[0];
    if constexpr (NPROJ == 2) o = silu(v[0]) * v[1];
    if (n < a.N) stg(a.out + (int64_t)(t0 + r) * a.ldo + n, o);
  }
}

// Group g of a decode step's routed rows: the g-th expert that has rows, and
// those, ascending.  Row i's expert is ids[i], each token's ids differ, so an
// expert has at most one row a token (64).  Lane i's `row` becomes row i; the
// return value is their number, 0 past the last group.  list: 64 words of the
// wave's LDS (its stage, idle until its first tile).
__device__ __forceinline__ int group_of_ids(const int32_t* ids, int nr, int g, int* list, int& e, int& row) {
  constexpr int kBatch = 8;  // loads in flight
  const int l = lane_id();
  int id[kBatch];
  auto load = [&](int i0) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) id[j] = ldg(ids + min(i0 + j * kWave + l, nr - 1));
  };
  uint32_t lo = 0u, hi = 0u;
  for (int i0 = 0; i0 < nr; i0 += kBatch * kWave) {
    load(i0);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {  // (past the last row: a repeat of it)
      lo |= id[j] < 32 ? 1u << (id[j] & 31) : 0u;
      hi |= id[j] < 32 ? 0u : 1u << (id[j] & 31);
    }
  }
  const uint64_t used = ((uint64_t)tree_or(hi) << 32) | tree_or(lo);
  const uint64_t nth = __ballot(((used >> l) & 1ull) != 0ull && lanes_below(used) == g);
  if (nth == 0ull) return 0;
  e = (int)__builtin_ctzll(nth);
  int cnt = 0;
  for (int i0 = 0; i0 < nr; i0 += kBatch * kWave) {
    if (nr > kBatch * kWave) load(i0);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int i = i0 + j * kWave + l;
      const bool mine = i < nr && id[j] == e;
      const uint64_t m = __ballot(mine);
      const int at = cnt + lanes_below(m);
      if (mine && at < kWave) list[at] = i;
      cnt += __builtin_popcountll(m);
    }
  }
  cnt = min(cnt, kWave);
  __builtin_amdgcn_wave_barrier();
  row = list[min(l, cnt - 1)];
  return cnt;
}

// The routed part of a launch: workgroup wg takes group wg / per and the
// kMfmaWaves / NPROJ column blocks from (wg % per) * that many on.  With
// rows.ids a workgroup finds its group among the ids itself: one round trip to
// memory instead of the three dependent ones of the group tables, and no
// grouping launch before.
template <WKind W, int NPROJ>
__device__ __forceinline__ void routed_part(const GemvArgs& a, int wg, char* lds) {
  constexpr int CB = kMfmaWaves / NPROJ;
  const int l = lane_id();
  const int per = ((a.N + kWave - 1) / kWave + CB - 1) / CB;
  const int g = wg / per;
  const int cb0 = (wg - g * per) * CB;
  int e = 0, r0 = 0, n = 0, row = 0;
  if (a.rows.ids != nullptr) {
    n = group_of_ids(a.rows.ids, a.rows.nids, g, (int*)(lds + (threadIdx.x >> 6) * kStageBytes), e, row);
  } else {
    if (g >= ldc(a.rows.n_groups)) return;
    e = ldc(a.rows.group_expert + g);
    r0 = ldc(a.rows.group_start + g);
    n = ldc(a.rows.group_start + g + 1) - r0;
  }
  for (int c0 = 0; c0 < n; c0 += kWave) {
    if (a.rows.ids == nullptr) row = ldg(a.rows.group_rows + r0 + min(c0 + l, n - 1));
    const int nc = min(n - c0, kWave);
    for (int t = 0; t < nc; t += 16) {
      const int cnt = min(16, nc - t);
      if (cnt <= 4)
        routed_tile<W, NPROJ, 1>(a, e, row, t, cnt, cb0, lds);
      else if (cnt <= 8)
        routed_tile<W, NPROJ, 2>(a, e, row, t, cnt, cb0, lds);
      else if (cnt <= 12)
        routed_tile<W, NPROJ, 3>(a, e, row, t, cnt, cb0, lds);
      else
        routed_tile<W, NPROJ, 4>(a, e, row, t, cnt, cb0, lds);
    }
  }
}

// The (column block, row group) of workgroup wg of a dense weight: the row
// groups of a column block run side by side on one XCD (workgroup b on XCD
// b % 8), whose L2 then fetches the block's weights once.  Workgroups come in
// runs of 8 column blocks, each run group by group.
struct DenseRef {
  int block, t0;
};
__device__ __forceinline__ DenseRef dense_ref(int wg, int blocks, int M, int rows) {
  const int G = (M + rows - 1) / rows;
  const int q = wg / (8 * G), rem = wg - q * 8 * G;
  const int run = min(8, blocks - 8 * q);
  const int g = rem / run;
  return DenseRef{8 * q + rem - g * run, g * rows};
}
template <int C, int NPROJ, int NT>
__device__ __forceinline__ void dense_part(const GemvArgs& a, int wg, char* lds) {
  const DenseRef d = dense_ref(wg, (a.N + C - 1) / C, a.rows.identity, 4 * NT);
  dense_tile<C, NPROJ, NT>(a, d.t0, min(4 * NT, a.rows.identity - d.t0), d.block * C, (float*)lds);
}

// Routed experts and the shared ones in one launch, the shared workgroups
// (the longest) first.
template <WKind W, int NPROJ>
__global__ void __launch_bounds__(kMfmaWaves* kWave) k_rows_pair(GemvArgs routed, GemvArgs shared, int nt, int split) {
  extern __shared__ __align__(16) char mlds[];
  const int wg = (int)blockIdx.x;
  if (wg >= split)
    routed_part<W, NPROJ>(routed, wg - split, mlds);
  else if (nt == 1)
    dense_part<kWave, NPROJ, 1>(shared, wg, mlds);
  else
    dense_part<kWave, NPROJ, 2>(shared, wg, mlds);
}

// The standalone routed ops.
template <WKind W>
__global__ void __launch_bounds__(kMfmaWaves* kWave) k_rows_routed(GemvArgs a) {
  extern __shared__ __align__(16) char mlds[];
  routed_part<W, 1>(a, (int)blockIdx.x, mlds);
}

// Split over chunks (dense_tile): up to 10 waves.
template <int C, int NT>
__global__ void __launch_bounds__(10 * kWave) k_dense_split(GemvArgs a) {
  extern __shared__ __align__(16) char mlds[];
  dense_part<C, 1, NT>(a, (int)blockIdx.x, mlds);
}

// Wide outputs: a wave per column block, all chunks, no meeting in LDS.
template <int NT>
__global__ void __launch_bounds__(kMfmaWaves* kWave) k_dense_whole(GemvArgs a) {
  const int blocks = (a.N + kWave - 1) / kWave;
  const DenseRef d = dense_ref((int)blockIdx.x, (blocks + kMfmaWaves - 1) / kMfmaWaves, a.rows.identity, 4 * NT);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int n0 = (d.block * kMfmaWaves + w) * kWave;
  if (n0 >= a.N) return;
  const int cnt = min(4 * NT, a.rows.identity - d.t0);
  int rowv[NT];
  const float* xp[NT];
  tile_rows<kBf16KBlocked, kWave, NT, false>(a, 0, d.t0, cnt, rowv, xp);
  f32x4 acc[NT];
  zero(acc);
  kblocked_chain<kWave, NT, false>(a, 0, n0, xp, 0, a.nchunks, acc, nullptr);
  store_rows<NT>(a, n0, cnt, rowv, acc);
}

int blocks_of(const GemvArgs& a, int c = kWave) { return (a.N + c - 1) / c; }
int routed_wgs(const GemvArgs& a, int max_groups, int nproj) {
  const int cb = kMfmaWaves / nproj;
  return max_groups * ((blocks_of(a) + cb - 1) / cb);
}
size_t split_lds(const GemvArgs& a, int nproj, int nt, int c = kWave) {
  return (size_t)nproj * a.nchunks * 4 * nt * c * sizeof(float);
}

}  // namespace

static bool rows_mfma_ok(const GemvArgs& a) {
  if (a.K <= 0) return false;  // no stage to load; the VALU kernels store the empty sums
  if (!a.vec || (reinterpret_cast<uintptr_t>(a.x) & 15u) != 0 || a.ldx % 4 || a.K > (1 << 16)) return false;
  if (a.kind == kInt8Rows) return a.gsize == kChunk && a.K % kChunk == 0;
  return a.K % 64 == 0;
}

// LDS a launch may take on gfx950.
static constexpr size_t kMaxLds = 160 * 1024;

// Row tiles of the shared experts in a pair launch: 8 rows, or 4 where that is all there is.
static int shared_tiles(const GemvArgs& shared) { return shared.rows.identity <= 4 ? 1 : 2; }

bool rows_pair_ok(const GemvArgs& routed, const GemvArgs& shared, int nproj) {
  return rows_mfma_ok(routed) && rows_mfma_ok(shared) && split_lds(shared, nproj, shared_tiles(shared)) <= kMaxLds;
}

template <WKind W, int NPROJ>
static hipError_t launch_pair(const char* name, const GemvArgs& routed, int max_groups, const GemvArgs& shared,
                              hipStream_t s) {
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)k_rows_pair<W, NPROJ>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
  if (attr != hipSuccess) return attr;
  const int nt = shared_tiles(shared);
  const int split = blocks_of(shared) * ((shared.rows.identity + 4 * nt - 1) / (4 * nt));
  size_t lds = (size_t)kMfmaWaves * kStageBytes;
  if (split_lds(shared, NPROJ, nt) > lds) lds = split_lds(shared, NPROJ, nt);
  UOCR_LAUNCH(name, (k_rows_pair<W, NPROJ>), dim3(split + routed_wgs(routed, max_groups, NPROJ)),
              dim3(kMfmaWaves * kWave), lds, s, routed, shared, nt, split);
  return hipGetLastError();
}

hipError_t launch_rows_pair(const GemvArgs& routed, int max_groups, const GemvArgs& shared, int nproj, hipStream_t s) {
  if (routed.kind == kInt8Rows)
    return nproj == 2 ? launch_pair<kInt8Rows, 2>("rows_gateup", routed, max_groups, shared, s)
                      : launch_pair<kInt8Rows, 1>("rows_down", routed, max_groups, shared, s);
  return nproj == 2 ? launch_pair<kBf16Rows, 2>("rows_gateup", routed, max_groups, shared, s)
                    : launch_pair<kBf16Rows, 1>("rows_down", routed, max_groups, shared, s);
}

bool rows_routed_ok(const GemvArgs& a) { return a.rows.n_groups != nullptr && rows_mfma_ok(a); }

hipError_t launch_rows_routed(const GemvArgs& a, int max_groups, hipStream_t s) {
  const dim3 grid(routed_wgs(a, max_groups, 1)), block(kMfmaWaves * kWave);
  const size_t lds = (size_t)kMfmaWaves * kStageBytes;
  if (a.kind == kInt8Rows)
    UOCR_LAUNCH("rows_op", k_rows_routed<kInt8Rows>, grid, block, lds, s, a);
  else
    UOCR_LAUNCH("rows_op", k_rows_routed<kBf16Rows>, grid, block, lds, s, a);
  return hipGetLastError();
}

// A launch has a workgroup per row group, and a grid at most 2^32 threads (of narrow outputs, 256 for 32 rows:
// beyond kMaxDenseRows the VALU kernel's workgroups go over all rows).
static constexpr int kMaxDenseRows = 1 << 28;

bool rows_dense_ok(const GemvArgs& a) {
  return a.kind == kBf16KBlocked && a.rows.n_groups == nullptr && a.rows.identity <= kMaxDenseRows &&
         rows_mfma_ok(a) && split_lds(a, 1, 1) <= kMaxLds;
}

// How a dense launch is cut: C columns a wave, `waves` of a workgroup on one
// column block's chunks (0: a wave has all of them, 4 column blocks a
// workgroup), nt row tiles.
struct DensePlan {
  int c, waves, nt;
};

static DensePlan dense_plan(const GemvArgs& a) {
  const int tiles = (a.rows.identity + 3) / 4;
  DensePlan best{};
  double cost = 0;
  // Estimated time in ns, fitted to a sweep of the projections at 3 to 64 rows.
  // The waves of a SIMD do not overlap: a k step takes `step` ns a wave (a
  // conversion and 8 cycles per row tile; a lone 4-row chain waits for its
  // sums).  A split launch also meets in LDS, and several of its workgroups on
  // a CU cost more than their sum.
  auto consider = [&](int c, int waves, int nt) {
    if (waves > 0 && split_lds(a, 1, nt, c) > kMaxLds) return;
    const double step = nt == 1 ? 8 : nt == 2 ? 11 : nt == 3 ? 15.5 : nt == 4 ? 21 : nt == 6 ? 29 : 40;
    const int groups = (tiles + nt - 1) / nt;
    const int units = (a.nchunks + kWave / c - 1) / (kWave / c);
    const int wgs = (waves == 0 ? (blocks_of(a) + kMfmaWaves - 1) / kMfmaWaves : blocks_of(a, c)) * groups;
    const int rounds = (wgs + 255) / 256;
    const double steps = 128.0 * (waves == 0 ? units : (units + waves - 1) / waves);
    double t;
    if (waves == 0)
      t = 3500 + steps * step * rounds;
    else if (c == kWave)
      t = 4500 + steps * step * (rounds * waves < 4 ? 1.0 : rounds * waves / 4.0) * (rounds > 1 ? 1.3 : 1.0);
    else
      t = 3600 + steps * step * ((waves < 4 ? 1.0 : waves / 4.0) + 0.63 * waves * (rounds - 1));
    if (cost == 0 || t < cost) {
      cost = t;
      best = DensePlan{c, waves, nt};
    }
  };
  for (int nt : {1, 2, 3, 4, 6, 8}) {
    if (nt > 1 && nt > tiles && !(nt == 6 && tiles == 5) && !(nt == 8 && tiles == 7)) break;
    consider(kWave, 0, nt);
    if (nt <= 4) {
      for (int r = (a.nchunks + 9) / 10, i = 0; i < 2; ++i, r *= 2) consider(kWave, (a.nchunks + r - 1) / r, nt);
    }
    if (nt <= 2) {
      const int units = (a.nchunks + 3) / 4, r = (units + 9) / 10;
      consider(16, (units + r - 1) / r, nt);
    }
  }
  return best;
}

template <int C, int NT>
static hipError_t launch_split(const GemvArgs& a, int waves, hipStream_t s) {
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)k_dense_split<C, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
  if (attr != hipSuccess) return attr;
  const int groups = (a.rows.identity + 4 * NT - 1) / (4 * NT);
  UOCR_LAUNCH("rows_dense", (k_dense_split<C, NT>), dim3((unsigned)(blocks_of(a, C) * groups)), dim3(waves * kWave),
              split_lds(a, 1, NT, C), s, a);
  return hipGetLastError();
}

template <int NT>
static hipError_t launch_whole(const GemvArgs& a, hipStream_t s) {
  const int groups = (a.rows.identity + 4 * NT - 1) / (4 * NT);
  UOCR_LAUNCH("rows_dense", k_dense_whole<NT>,
              dim3((unsigned)((blocks_of(a) + kMfmaWaves - 1) / kMfmaWaves * groups)), dim3(kMfmaWaves * kWave), 0, s,
              a);
  return hipGetLastError();
}

hipError_t launch_rows_dense(const GemvArgs& a, hipStream_t s) {
  if (a.rows.identity == 0 || a.N == 0) return hipSuccess;
  const DensePlan p = dense_plan(a);
  if (p.waves == 0) {
    switch (p.nt) {
      case 1: return launch_whole<1>(a, s);
      case 2: return launch_whole<2>(a, s);
      case 3: return launch_whole<3>(a, s);
      case 4: return launch_whole<4>(a, s);
      case 6: return launch_whole<6>(a, s);
      default: return launch_whole<8>(a, s);
    }
  }
  if (p.c == 16) return p.nt == 1 ? launch_split<16, 1>(a, p.waves, s) : launch_split<16, 2>(a, p.waves, s);
  switch (p.nt) {
    case 1: return launch_split<kWave, 1>(a, p.waves, s);
    case 2: return launch_split<kWave, 2>(a, p.waves, s);
    case 3: return launch_split<kWave, 3>(a, p.waves, s);
    default: return launch_split<kWave, 4>(a, p.waves, s);
  }
}

}  // namespace uocr
