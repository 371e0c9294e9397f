// Projections of a neighborhood attention layer for gfx950 (MI355X): y = x w^T + b, and its backward.
//
// The products around the attention of a layer (reference src/natten/modules.py:83-132: one linear map to queries, keys
// and values, one behind the attention) have many rows (tokens) and few columns (64 .. some hundred).  One kernel template
// forms all three of them, with v_mfma_f32_32x32x16 and both operands staged through LDS, 64 steps of the
// contraction at a time, by asynchronous copies into alternating stages:
//   forward  y[m, n]  = sum_k x[m, k] w[n, k] + b[n]     both operands as they lie
//   input    dx[m, k] = sum_n dy[m, n] w[n, k]           w by transpose reads
//   weight   dw[n, k] = sum_m dy[m, n] x[m, k]           both by transpose reads, and db[n] = sum_m dy[m, n]
// A lane owns a row of the result (the "row side": m, m, n), its registers hold columns of it (the "column side": n, k,
// k), so that results are stored sixteen bytes per lane.  The columns of y and dy may be up to three tensors of
// `part` columns each: queries, keys and values as the attention takes and returns them.
//
// The weight gradient is the long contraction of the three (all tokens) with a result of some ten tiles: it is cut into
// `slices` runs of tokens, each a workgroup per tile that stores float32 sums, and linear_reduce_kernel adds the slices
// up in order, so that results do not differ from run to run.
//
// What bounds them: memory (12544 tokens, 256 -> 768 columns: 26 MB and 4.9 GFLOP) and the first tiles' way to LDS, with
// four steps of the contraction in a forward tile.
#pragma once

#include "fna_fwd.hpp"

namespace natten_amd {

enum LinearMode : int { kLinearForward = 0, kLinearInput = 1, kLinearWeight = 2 };

struct LinearParams {
  const void* row[3];  // x (forward) or the tensors of dy
  const void* col;     // w, w, x
  void* out[3];        // the tensors of y, dx
  const void* bias;    // forward: null for none
  float* partial;      // weight: [slices, n, k], and the sums of dy's columns [slices, n] behind them if `want_bias`
  float* partial_bias;
  int m, n, k;         // tokens, output columns and input columns of the linear map
  int part;            // columns of each tensor of y / dy
  int slices, slice_rows;  // weight: runs of tokens (slice_rows a multiple of 64)
  int row_tiles, col_tiles;
  NaDiv d_row_tiles, d_col_tiles, d_part;
};

// A tile of LDS: rows of `E` 16-bit elements, read along its rows (b128) or transposed
template <int ROWS, int E>
struct LinearTile {
  using L = FnaSmem<E, ROWS>;
  static constexpr int BYTES = ROWS * E * 2;
  static constexpr int CHUNKS = ROWS * E / 8;
};

// Two stages: a third keeps workgroups out of the compute unit (36864 tokens, 512 -> 1536: forward 80 us, 106 with three).
constexpr int kLinearStep = 64;  // of the contraction
constexpr int kLinearStages = 2;
constexpr int linear_lds_bytes(int rt, int ct) { return kLinearStages * (rt + ct) * kLinearStep * 2; }

// One tile of a result, RT rows by CT columns, four waves in a square; `block`: the workgroup's number in this part of a
// launch (which has a multiple of the XCD count of them), `lds`: linear_lds_bytes(RT, CT).
template <typename T, int MODE, int RT, int CT>
static __device__ __forceinline__ void linear_tile(const LinearParams& p, const int block, char* lds) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  constexpr int STEP = kLinearStep;
  constexpr bool ROW_TR = MODE == kLinearWeight, COL_TR = MODE != kLinearForward;
  using RowTile = LinearTile<ROW_TR ? STEP : RT, ROW_TR ? RT : STEP>;
  using ColTile = LinearTile<COL_TR ? STEP : CT, COL_TR ? CT : STEP>;
  constexpr int MI = RT / 64, NI = CT / 64;  // 32 x 32 blocks of a wave
  constexpr int PER_R = RowTile::CHUNKS / 256, PER_C = ColTile::CHUNKS / 256;
  static_assert(PER_R * 256 == RowTile::CHUNKS && PER_C * 256 == ColTile::CHUNKS, "a tile is a whole number of copies");
  char *const sR = lds, *const sC = lds + kLinearStages * RowTile::BYTES;

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;

  // tile of the workgroup: each XCD takes one contiguous eighth of (slice, row tile, column tile), columns fastest, so that
  // the tiles that read the same rows meet in its L2
  const int total = p.row_tiles * p.col_tiles * p.slices;
  const int chunk = (total + kNumXcd - 1) / kNumXcd;
  const int lin = (block % kNumXcd) * chunk + block / kNumXcd;
  if (block / kNumXcd >= chunk || lin >= total) return;
  const int rt = na_div(lin, p.d_col_tiles);
  const int col0 = (lin - rt * p.col_tiles) * CT;
  const int slice = MODE == kLinearWeight ? na_div(rt, p.d_row_tiles) : 0;
  const int row0 = (rt - slice * p.row_tiles) * RT;
  const int step0 = MODE == kLinearWeight ? slice * p.slice_rows : 0;  // first position of the contraction
  const int extent = MODE == kLinearForward ? p.k : MODE == kLinearInput ? p.n : na_min(p.slice_rows, p.m - step0);
  const int steps = (extent + STEP - 1) / STEP;

  // elements of a row of the two operands as they lie in memory
  const int row_len = MODE == kLinearForward ? p.k : p.part;
  const int col_len = p.k;  // (w's and x's rows hold k elements)
  // Copy i of a thread fills LDS chunk i * 256 + tid; its place in memory is a base that moves with the step and
  // an offset that does not: row side by rows of the result (forward, input; rows past the last are copies of it) or by
  // rows of the step (weight), the column side likewise.
  uint32_t off_r[PER_R], off_c[PER_C];
#pragma unroll
  for (int i = 0; i < PER_R; ++i) {
    constexpr int CPR = RowTile::L::CPR;
    const int P = i * 256 + tid, r = P / CPR;
    const int c = ROW_TR ? RowTile::L::v_slot(r, P % CPR) : RowTile::L::k_slot(r, P % CPR);
    off_r[i] = uint32_t(ROW_TR ? r : na_min(r, p.m - 1 - row0)) * uint32_t(row_len * 2) + uint32_t(c * 16);
  }
#pragma unroll
  for (int i = 0; i < PER_C; ++i) {
    constexpr int CPR = ColTile::L::CPR;
    const int P = i * 256 + tid, r = P / CPR;
    const int c = COL_TR ? ColTile::L::v_slot(r, P % CPR) : ColTile::L::k_slot(r, P % CPR);
    off_c[i] = uint32_t(r) * uint32_t(col_len * 2) + uint32_t(c * 16);
  }
  const uint32_t lds_r = uint32_t(__builtin_amdgcn_readfirstlane(int(lds_address(sR)))) + uint32_t(wave * 1024);
  const uint32_t lds_c = uint32_t(__builtin_amdgcn_readfirstlane(int(lds_address(sC)))) + uint32_t(wave * 1024);
  auto issue = [&](int s, int stage) __attribute__((always_inline)) {
    const int at = step0 + s * STEP;
    const char *r, *c;
    if constexpr (MODE == kLinearForward) {
      r = static_cast<const char*>(p.row[0]) + (int64_t(row0) * row_len + at) * 2;
      c = static_cast<const char*>(p.col) + (int64_t(col0) * col_len + at) * 2;
    } else if constexpr (MODE == kLinearInput) {
      const int t = na_div(at, p.d_part);
      r = static_cast<const char*>(t == 0 ? p.row[0] : t == 1 ? p.row[1] : p.row[2]) + (int64_t(row0) * row_len + at - t * p.part) * 2;
      c = static_cast<const char*>(p.col) + (int64_t(at) * col_len + col0) * 2;
    } else {
      const int t = na_div(row0, p.d_part);
      r = static_cast<const char*>(t == 0 ? p.row[0] : t == 1 ? p.row[1] : p.row[2]) + (int64_t(at) * row_len + row0 - t * p.part) * 2;
      c = static_cast<const char*>(p.col) + (int64_t(at) * col_len + col0) * 2;
    }
    const uint64_t rb = uniform64(r), cb = uniform64(c);
    // weight: rows past the last token are copies of it (their places in the fragments are cleared)
    const int last = MODE == kLinearWeight ? p.m - 1 - at : STEP;
    const bool partial = MODE == kLinearWeight && last < STEP - 1;
#pragma unroll
    for (int i = 0; i < PER_R; ++i) {
      uint32_t off = off_r[i];
      if (partial) off -= uint32_t(na_max((i * 256 + tid) / RowTile::L::CPR - last, 0)) * uint32_t(row_len * 2);
      async_copy16_uniform(rb, off, lds_r + uint32_t(stage * RowTile::BYTES + i * 4096));
    }
#pragma unroll
    for (int i = 0; i < PER_C; ++i) {
      uint32_t off = off_c[i];
      if (partial) off -= uint32_t(na_max((i * 256 + tid) / ColTile::L::CPR - last, 0)) * uint32_t(col_len * 2);
      async_copy16_uniform(cb, off, lds_c + uint32_t(stage * ColTile::BYTES + i * 4096));
    }
  };

  // Fragments: element e of a lane is position 8 g + e of the sixteen of a step, in either way of reading: row l32 of a
  // block (chunk 2 ks + g), or transposed rows 8 g + 0 .. 7 of the sixteen, four at a time, column l32 of the block.
  const int l16 = lane & 15, t_row = 8 * g + (l16 >> 2), t_chunk = (l32 >> 4) * 2 + ((l16 & 3) >> 1), t_sub = (l16 & 1) * 8;
  auto fragment = [&](auto tile_tag, auto tr_tag, const char* s, int block, int ks) __attribute__((always_inline)) {
    using Tile = typename decltype(tile_tag)::type;
    using L = typename Tile::L;
    if constexpr (decltype(tr_tag)::value) {
      const int r = ks * 16 + t_row;
      const char* at = s + r * L::ROWB + L::v_slot(t_row, block * 4 + t_chunk) * 16 + t_sub;
      const s16x4_t lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * L::ROWB);
      return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      return *reinterpret_cast<const vec8*>(s + (block * 32 + l32) * L::ROWB + L::k_slot(l32, ks * 2 + g) * 16);
    }
  };
  struct RowTag { using type = RowTile; };
  struct ColTag { using type = ColTile; };

  f32x16_t acc[MI][NI], acc_bias[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc_bias[i][r] = 0.f;
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j][r] = 0.f;
    }
  const bool sums = MODE == kLinearWeight && p.partial_bias != nullptr && col0 == 0 && wc == 0;
  vec8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = static_cast<T>(1.f);

  issue(0, 0);
  for (int s = 0; s < steps; ++s) {
    const int stage = s & 1;
    wait_vmcnt<0>();
    workgroup_sync();  // step s is in LDS; everyone is done with the stage of step s - 1
    if (s + 1 < steps) issue(s + 1, stage ^ 1);
    const char *r = sR + stage * RowTile::BYTES, *c = sC + stage * ColTile::BYTES;
    const int valid = MODE == kLinearWeight ? na_min(extent - s * STEP, STEP) : STEP;
#pragma unroll
    for (int ks = 0; ks < STEP / 16; ++ks) {
      vec8 fr[MI], fc[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) fr[i] = fragment(RowTag{}, std::integral_constant<bool, ROW_TR>{}, r, wr * MI + i, ks);
#pragma unroll
      for (int j = 0; j < NI; ++j) fc[j] = fragment(ColTag{}, std::integral_constant<bool, COL_TR>{}, c, wc * NI + j, ks);
      if (MODE == kLinearWeight && valid < STEP) {
        // tokens past the slice's last: nothing, whatever the copies in their places hold
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (ks * 16 + 8 * g + e < valid) continue;
#pragma unroll
          for (int i = 0; i < MI; ++i) fr[i][e] = static_cast<T>(0.f);
#pragma unroll
          for (int j = 0; j < NI; ++j) fc[j][e] = static_cast<T>(0.f);
        }
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = M::run(fc[j], fr[i], acc[i][j]);
      if (sums) {
#pragma unroll
        for (int i = 0; i < MI; ++i) acc_bias[i] = M::run(ones, fr[i], acc_bias[i]);
      }
    }
  }

  const int cw = col0 + wc * (CT / 2);  // first column of the wave
  if constexpr (MODE == kLinearForward) {
    if (p.bias != nullptr) {
      typedef T tx4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const tx4 v = *reinterpret_cast<const tx4*>(static_cast<const T*>(p.bias) + cw + j * 32 + 8 * b + 4 * g);
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][4 * b + e] += float(v[e]);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = row0 + wr * (RT / 2) + i * 32 + l32;
    if constexpr (MODE == kLinearWeight) {
      const int64_t at = int64_t(slice) * p.n + row;
      float* out = p.partial + at * p.k + cw + 4 * g;
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * b + e];
          *reinterpret_cast<f32x4_t*>(out + j * 32 + 8 * b) = v;
        }
      if (sums && g == 0) p.partial_bias[at] = acc_bias[i][0];
    } else {
      const int t = MODE == kLinearForward ? na_div(cw, p.d_part) : 0;
      const int len = MODE == kLinearForward ? p.part : p.k;
      T* out = static_cast<T*>(t == 0 ? p.out[0] : t == 1 ? p.out[1] : p.out[2]) + int64_t(row) * len + cw - t * p.part;
      store_row_blocks<T, NI>(out, acc[i], 1.f, g, row < p.m, CT / 2);
    }
  }
}

template <typename T, int RT, int CT>
__global__ void __launch_bounds__(256) linear_forward_kernel(const LinearParams p) {
  __shared__ __attribute__((aligned(1024))) char lds[linear_lds_bytes(RT, CT)];
  linear_tile<T, kLinearForward, RT, CT>(p, int(blockIdx.x), lds);
}

// Both products of the backward read dy, and at the sizes of layers neither fills the chip by itself: one launch, the
// workgroups of the weight gradient (the longer ones) first.  In two launches / in one, tokens x in -> out: 12544, 256 -> 768
// 31.0 / 28.1 us, 256 -> 256 23.0 / 19.0; 784, 64 -> 192 15.5 / 9.8; 36864, 512 -> 1536 177 / 134, the end of one product
// filled by the other.  W: extents of its tiles; C: columns of the input gradient's.
struct LinearBackwardParams {
  LinearParams weight, input;
  int weight_blocks, input_blocks;  // multiples of the XCD count, or 0
};
template <typename T, int W, int C>
__global__ void __launch_bounds__(256) linear_backward_kernel(const LinearBackwardParams p) {
  constexpr int BYTES = linear_lds_bytes(W, W) > linear_lds_bytes(128, C) ? linear_lds_bytes(W, W) : linear_lds_bytes(128, C);
  __shared__ __attribute__((aligned(1024))) char lds[BYTES];
  if (int(blockIdx.x) < p.weight_blocks) linear_tile<T, kLinearWeight, W, W>(p.weight, int(blockIdx.x), lds);
  else linear_tile<T, kLinearInput, 128, C>(p.input, int(blockIdx.x) - p.weight_blocks, lds);
}

// dw and db: the float32 sums of the slices, added up in order and rounded once.  Four elements a thread; `elements` of dw
// first (a multiple of 4), then the n of db.
template <typename T>
__global__ void __launch_bounds__(256) linear_reduce_kernel(const float* __restrict__ partial, const float* __restrict__ partial_bias,
                                                            T* __restrict__ dw, T* __restrict__ db, int elements, int n, int slices) {
  typedef T tx4 __attribute__((ext_vector_type(4)));
  int at = (int(blockIdx.x) * 256 + int(threadIdx.x)) * 4;
  const bool bias = at >= elements;
  if (bias) at -= elements;
  const int count = bias ? n : elements;
  if (at >= count || (bias && db == nullptr)) return;
  const float* src = (bias ? partial_bias : partial) + at;
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < slices; ++s) sum += *reinterpret_cast<const f32x4_t*>(src + int64_t(s) * count);
  tx4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = static_cast<T>(sum[e]);
  *reinterpret_cast<tx4*>((bias ? db : dw) + at) = v;
}

}  // namespace natten_amd
