// Neighborhood attention forward for float32 operands on gfx950, two kernels: fna_fwd_f32_direct_kernel on the
// original tensors (the default; described where it stands), and fna_fwd_f32_kernel on token-permuted
// sequences, for callers that fix tile shapes or ask for that route.
// The reference runs float32 through its CUTLASS 2.x kernels and, on CPU, through flex attention
// (SHI-Labs/NATTEN tests/test_fna.py:107-131 states the tolerance: 1e-4 on the output).  Both kernels keep
// products, sums and softmax in IEEE float32, P unrounded.  The permuted one: S^T = K Q^T and O^T += V^T P^T on
// v_mfma_f32_32x32x2_f32, exact online softmax (its maximum is followed at once, the direct kernel's lags),
// every logit tested against its query's window (no whole-tile classification), one workgroup per Q tile of
// 128 rows, 64-key tiles staged through LDS with ordinary loads.
#pragma once

#include "fna_fwd.hpp"

namespace natten_amd {

// Same matrix layouts as the 16-bit kernel: the lane (l32 = lane % 32, g = lane / 32) owns query
// column l32 of the wave's 32-row block; of a 32 x 32 result block it holds rows
// 8 * (r / 4) + 4 * g + r % 4, r = 0..15.  A 32x32x2 instruction multiplies two k-indices, one per
// g; which head-dim element (QK) or key (PV) a k-index stands for is free as long as both operands
// agree: QK uses element g * D/2 + step, PV key 8 * (r / 4) + 4 * g + r % 4 (so a P register is the
// B operand as it stands).
template <int D>
__global__ void __launch_bounds__(256) fna_fwd_f32_kernel(const FnaParams p) {
  constexpr int KVT = 64, QT = 128, NT = 256;
  constexpr int LDW = D + 4;   // floats per LDS row: 16-byte aligned rows, 4 banks apart
  constexpr int HALF = D / 2;  // head-dim elements per k-index half
  constexpr int DB = D / 32;
  __shared__ __attribute__((aligned(16))) float sK[KVT * LDW];
  __shared__ __attribute__((aligned(16))) float sV[KVT * LDW];
  __shared__ int sCrd[KVT][4];  // in-tile coordinates of every KV position (dimension 0 fastest)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int l32 = lane & 31;
  const int g = lane >> 5;

  // ---- workgroup -> (batch * dilation group, head, Q tile) ---------------------------------------
  const int pid = blockIdx.x;
  const int qtile = pid % p.num_q_tiles;
  const int bh = pid / p.num_q_tiles;
  const int head = bh % p.heads_q;
  const int bg = bh / p.heads_q;
  const int head_kv = head / (p.heads_q / p.heads_kv);

  int extent[3], q_first[3], t_lo[3], t_hi[3];
  {
    int gl = bg % p.num_groups;
    int tq = qtile;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int gi = gl % p.dil[a];
      gl /= p.dil[a];
      extent[a] = na_group_extent(p.qkv_shape[a], p.dil[a], gi);
      const int tc = tq % p.q_tiled[a];  // Q tiles are enumerated with dimension 0 fastest
      tq /= p.q_tiled[a];
      q_first[a] = tc * p.q_tile[a];
      // KV tiles that the windows of the tile's queries reach (padding queries act as the last real one)
      const bool c = p.causal[a] != 0;
      const int qf = na_min(q_first[a], extent[a] - 1);
      const int ql = na_min(q_first[a] + p.q_tile[a] - 1, extent[a] - 1);
      const int st_f = na_window_start(qf, p.ksize[a], p.stride[a], extent[a], c);
      const int st_l = na_window_start(ql, p.ksize[a], p.stride[a], extent[a], c);
      const int en_l = na_window_end(ql, st_l, p.ksize[a], extent[a], c);
      t_lo[a] = st_f / p.kv_tile[a];
      t_hi[a] = (en_l - 1) / p.kv_tile[a];
    }
  }
  if (tid < KVT) {
    int i = tid;
    sCrd[tid][0] = i % p.kv_tile[0];
    i /= p.kv_tile[0];
    sCrd[tid][1] = i % p.kv_tile[1];
    sCrd[tid][2] = i / p.kv_tile[1];
    sCrd[tid][3] = 0;
  }

  // ---- this lane's query: row of the tile (dimension 0 fastest), window, fragment ----------------
  const int row = wave * 32 + l32;
  int ws[3], we[3];
  {
    int r = row;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int off = r % p.q_tile[a];
      r /= p.q_tile[a];
      const int c = na_min(q_first[a] + off, extent[a] - 1);
      const bool cz = p.causal[a] != 0;
      ws[a] = na_window_start(c, p.ksize[a], p.stride[a], extent[a], cz);
      we[a] = na_window_end(c, ws[a], p.ksize[a], extent[a], cz);
    }
  }
  const int64_t q_row = int64_t(bg) * p.seqlen_q + int64_t(qtile) * QT + row;
  const float c_log2 = p.scale * 1.4426950408889634f;
  float qf[HALF];
  {
    const float* qrow = static_cast<const float*>(p.q) + (q_row * p.heads_q + head) * D + g * HALF;
#pragma unroll
    for (int i = 0; i < HALF; i += 4) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(qrow + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[i + e] = x[e] * c_log2;
    }
  }

  f32x16_t acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int64_t kv_row_stride = int64_t(p.heads_kv) * D;
  const float* kbase = static_cast<const float*>(p.k) + (int64_t(bg) * p.seqlen_kv * p.heads_kv + head_kv) * D;
  const float* vbase = static_cast<const float*>(p.v) + (int64_t(bg) * p.seqlen_kv * p.heads_kv + head_kv) * D;

  for (int t2 = t_lo[2]; t2 <= t_hi[2]; ++t2)
    for (int t1 = t_lo[1]; t1 <= t_hi[1]; ++t1)
      for (int t0 = t_lo[0]; t0 <= t_hi[0]; ++t0) {
        const int64_t row0 = int64_t(t0 + p.kv_tiled[0] * (t1 + p.kv_tiled[1] * t2)) * KVT;
        const int org[3] = {t0 * p.kv_tile[0], t1 * p.kv_tile[1], t2 * p.kv_tile[2]};
        workgroup_sync();  // everyone is done with the previous tile (and sCrd is written)
#pragma unroll
        for (int c = tid; c < KVT * (D / 4); c += NT) {
          const int r = c / (D / 4), c4 = c % (D / 4);
          const int64_t off = (row0 + r) * kv_row_stride + c4 * 4;
          *reinterpret_cast<f32x4_t*>(&sK[r * LDW + c4 * 4]) = *reinterpret_cast<const f32x4_t*>(kbase + off);
          *reinterpret_cast<f32x4_t*>(&sV[r * LDW + c4 * 4]) = *reinterpret_cast<const f32x4_t*>(vbase + off);
        }
        workgroup_sync();

        // S^T = K Q^T (already in the exp2 domain), two blocks of 32 keys
        f32x16_t S[2];
#pragma unroll
        for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
          for (int r = 0; r < 16; ++r) S[sb][r] = 0.f;
          const float* krow = &sK[(sb * 32 + l32) * LDW + g * HALF];
#pragma unroll
          for (int i = 0; i < HALF; i += 4) {
            const f32x4_t k4 = *reinterpret_cast<const f32x4_t*>(krow + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) S[sb] = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[e], qf[i + e], S[sb], 0, 0, 0);
          }
        }
        // window test of every (key, query) pair, row maximum
        float mx = -INFINITY;
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = sb * 32 + 8 * (r / 4) + 4 * g + (r % 4);
            bool in = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              const int kc = org[a] + sCrd[key][a];
              in = in && (kc >= ws[a]) && (kc < we[a]);
            }
            S[sb][r] = in ? S[sb][r] : -INFINITY;
            mx = fmaxf(mx, S[sb][r]);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 32));  // the two halves of a query's keys
        const float m_new = fmaxf(m_run, mx);
        // (a query none of whose keys lie in this tile keeps m_new = m_run, possibly -inf: all p are 0)
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = exp2f(m_run - m_use);  // 0 while m_run is -inf
        float psum = 0.f;
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            S[sb][r] = exp2f(S[sb][r] - m_use);
            psum += S[sb][r];
          }
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
        // O^T += V^T P^T: k-index g of step (sb, r) is key sb * 32 + 8 * (r / 4) + 4 * g + r % 4
#pragma unroll
        for (int sb = 0; sb < 2; ++sb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = sb * 32 + 8 * (r / 4) + 4 * g + (r % 4);
#pragma unroll
            for (int db = 0; db < DB; ++db)
              acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(sV[key * LDW + db * 32 + l32], S[sb][r], acc[db], 0, 0, 0);
          }
      }

  // ---- epilogue: O = acc / rowsum, LSE = ln(rowsum) + ln2 * rowmax --------------------------------
  const float l = l_run + __shfl_xor(l_run, 32);
  const float inv = (l > 0.f) ? 1.f / l : 0.f;
  float* orow = static_cast<float*>(p.o) + (q_row * p.heads_q + head) * D;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4_t o4;
#pragma unroll
      for (int i = 0; i < 4; ++i) o4[i] = acc[db][4 * j + i] * inv;
      *reinterpret_cast<f32x4_t*>(orow + db * 32 + 8 * j + 4 * g) = o4;
    }
  if (g == 0) p.lse[q_row * p.heads_q + head] = (l > 0.f) ? (m_run * 0.6931471805599453f + logf(l)) : -INFINITY;
}

// ---- on the original tensors ----------------------------------------------------------------------
struct FnaF32Params {
  const float *q, *k, *v;
  float *o, *lse;
  int heads_q, heads_kv, head_dim;  // head_dim: elements of a row, a multiple of 4, at most the instance's D
  int dims;                         // dimensions that can mask anything: 1, 2 or 3 (the rest have extent 1)
  int ksize[3], stride[3], dil[3], causal[3];
  int ext_base[3], ext_rem[3];      // extent of dilation group g along a dimension = base + (g < rem)
  int tok_stride[3], tokens;
  int q_lg[3], kv_lg[3];            // log2 extents of a wave's box of 16 queries / of a block of 16 keys (sums 4)
  int q_boxes[3];                   // boxes per dimension
  NaDiv d_stride[3], d_dil[3], d_q_boxes[3], d_boxes, d_heads_q, d_q_per_kv, d_num_groups;
  int num_boxes, num_groups;
  int waves, wgs_per_xcd;           // one wave per (batch, dilation group, head, box)
  float scale;
};

// Boxes of 16 queries and blocks of 16 keys that let the fewest (query, key) pairs be multiplied: along a
// dimension a box of tq queries spans the window plus the distance its stride groups' leaders cover,
// rounded up to whole blocks.  Ties go to boxes that are long in the last dimension.
inline void choose_f32_boxes(FnaF32Params& p) {
  long long cost[3][5][5];
  for (int a = 0; a < 3; ++a) {
    const int ext = p.ext_base[a] + (p.ext_rem[a] > 0);
    for (int lq = 0; lq < 5; ++lq)
      for (int lk = 0; lk < 5; ++lk) {
        const int tq = 1 << lq, s = p.stride[a];
        const int reach = s % tq == 0 ? 0 : ((tq - 1 + s - 1) / s) * s;
        const int span = na_min(ext, p.ksize[a] + (p.causal[a] ? tq - 1 : reach));
        cost[a][lq][lk] = (long long)(((ext + tq - 1) >> lq) << lq) * (((span + (1 << lk) - 1) >> lk) << lk);
      }
  }
  // (dimensions from p.dims on have extent 1: boxes and blocks stay inside it, the element mask skips them)
  double best = -1;
  for (int q0 = 0; q0 <= 4; ++q0)
    for (int q1 = 0; q0 + q1 <= 4; ++q1)
      for (int k0 = 0; k0 <= 4; ++k0)
        for (int k1 = 0; k0 + k1 <= 4; ++k1) {
          const int q2 = 4 - q0 - q1, k2 = 4 - k0 - k1;
          if ((p.dims < 2 && (q1 | k1)) || (p.dims < 3 && (q2 | k2))) continue;
          const double c = double(cost[0][q0][k0]) * double(cost[1][q1][k1]) * double(cost[2][q2][k2]);
          if (best >= 0 && c >= best) continue;
          best = c;
          p.q_lg[0] = q0, p.q_lg[1] = q1, p.q_lg[2] = q2;
          p.kv_lg[0] = k0, p.kv_lg[1] = k1, p.kv_lg[2] = k2;
        }
}

// One wave per box of 16 queries; no LDS and no barriers.  What bounds the float32 path is the matrix rate
// (1/16 of bf16's), so what counts is how few pairs outside the windows are multiplied: with boxes of
// 16 queries and blocks of 16 keys laid out from the first key of the wave's own windows a 13 x 13
// window costs 256 keys a query, where a 128-query tile over 64-key tiles at multiples of their extent
// costs 1024.  Each 16 x D block of K and of V goes straight from memory (mostly L1 / L2: neighbouring waves read
// nearly the same keys) to the registers the matrix instruction reads, 8 D bytes per lane group against
// 16 D matrix cycles, half a block ahead of its use or more; the loads add a lane's constant distances to a uniform base.
//
// v_mfma_f32_16x16x4_f32: with i = lane % 16, g = lane / 16 the A operand holds row i, the B operand
// column i, k-index g; the result's register r is row 4 g + r, column i.  S^T = K Q^T: which head-dim
// element k-index g of a step stands for is free as long as both operands agree: step (j, e) uses
// element 16 j + 4 g + e, so that a lane's operands are float4 loads of its row.  The result holds the
// logits of keys 4 g + r of query i, which is the B operand of O^T += V^T P^T step r (k-index g = key
// 4 g + r) as it stands; row i of result block (h, c) is head-dim element VEC (16 h + i) + c, so that
// V operands and results are VEC-wide loads and stores of whole rows.
// Softmax in float32; a row's maximum is followed once it grew by more than 2^8 (exact: the sums are
// normalised by the same maximum).
// 2 x 64 x 64 tokens, H 8, D 64, 13 x 13 windows: 50 us (57 TFLOP/s of window pairs, 83 of pairs
// multiplied), 300 us as permutes, 128-query kernel and unpermutes; 256 tokens, H 2, D 32, window 7: 17 us, all of it the
// call, from 83.  Where the first's time goes (all 4096 waves are resident at once, four a SIMD): the launch keeps the shader
// engines busy for 110000 cycles (SQ_BUSY_CYCLES), of which the matrix pipe of a SIMD works 63000 (SQ_VALU_MFMA_BUSY_CYCLES), the
// fifteen blocks of its four waves, nearly without a gap.  A wave lives 81000 to 85000 (SQ_WAVE_CYCLES), 16000 of them and more
// set-up and the way of the first block; the 25000 others are the begin and end of the launch, when a SIMD does not have its
// waves yet or no longer.  0.57 of the pipe's time, at 2.2 of the 2.35 GHz at which a large product reaches 154
// TFLOP/s, are those 83.
template <int D, bool PAD, bool WIDE = false, int SETS = (D == 32 ? 2 : 1)>
__global__ void __launch_bounds__(256, 2) fna_fwd_f32_direct_kernel(const FnaF32Params p) {
  constexpr int KJ = D / 16;
  constexpr int VEC = KJ < 4 ? KJ : 4;
  constexpr int NH = D / (16 * VEC);
  typedef float fvec __attribute__((ext_vector_type(VEC)));
  touch_launch_params<sizeof(FnaF32Params)>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int i16 = lane & 15, g = lane >> 4;

  // waves are numbered box fastest, then head, then batch entry; every XCD takes a contiguous run of them
  const int w = (int(blockIdx.x % kNumXcd) * p.wgs_per_xcd + int(blockIdx.x / kNumXcd)) * 4 + wave;
  if (w >= p.waves) return;
  const int bh = na_div(w, p.d_boxes);
  int box = w - bh * p.num_boxes;
  const int bg = na_div(bh, p.d_heads_q);
  const int head = bh - bg * p.heads_q;
  const int head_kv = na_div(head, p.d_q_per_kv);
  const int b = na_div(bg, p.d_num_groups);
  int gl = bg - b * p.num_groups;

  int extent[3], step[3], org0[3], nblk[3], full_lo[3], full_hi[3];
  int ws[3], width[3];  // this lane's query: window start and length
  int q_tok = 0, group_tok = 0;
  bool valid = true;
  {
    int q_in = i16;
    int bc[3];
    const int t01 = na_div(box, p.d_q_boxes[2]);
    bc[2] = box - t01 * p.q_boxes[2];
    bc[0] = na_div(t01, p.d_q_boxes[1]);
    bc[1] = t01 - bc[0] * p.q_boxes[1];
    bool empty = false;
#pragma unroll
    for (int a = 2; a >= 0; --a) {
      const int off = q_in & ((1 << p.q_lg[a]) - 1);
      q_in >>= p.q_lg[a];
      bc[a] = (bc[a] << p.q_lg[a]);
      ws[a] = off;
    }
    // One window evaluation per dimension: a lane's own query.  The box's first query is lane 0's, its last one lane 15's (queries
    // past the group act as its last one and are not stored).
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int rest = na_div(gl, p.d_dil[a]);
      const int gi = gl - rest * p.dil[a];
      gl = rest;
      extent[a] = p.ext_base[a] + (gi < p.ext_rem[a] ? 1 : 0);
      step[a] = p.dil[a] * p.tok_stride[a];
      group_tok += gi * p.tok_stride[a];
      empty = empty || bc[a] >= extent[a];  // (groups may be one shorter than the boxes were counted for)
      const bool c = p.causal[a] != 0;
      const int qc = bc[a] + ws[a];
      valid = valid && qc < extent[a];
      const int q = na_min(qc, extent[a] - 1);
      const int start = na_window_start(q, p.ksize[a], p.stride[a], p.d_stride[a], extent[a], c);
      const int end = na_window_end(q, start, p.ksize[a], extent[a], c);
      ws[a] = start;
      width[a] = end - start;
      org0[a] = __builtin_amdgcn_readlane(start, 0);
      full_hi[a] = __builtin_amdgcn_readlane(end, 0);
      full_lo[a] = __builtin_amdgcn_readlane(start, 15);
      nblk[a] = (__builtin_amdgcn_readlane(end, 15) - org0[a] + (1 << p.kv_lg[a]) - 1) >> p.kv_lg[a];
      q_tok += q * step[a];
    }
    if (empty) return;
  }
  const int64_t token0 = int64_t(b) * p.tokens + group_tok;
  const int64_t q_row = (token0 + q_tok) * p.heads_q + head;
  const int kv_row = p.heads_kv * p.head_dim;
  const float* kbase = p.k + (token0 * p.heads_kv + head_kv) * p.head_dim;
  const float* vbase = p.v + (token0 * p.heads_kv + head_kv) * p.head_dim;
  const float c_log2 = p.scale * 1.4426950408889634f;

  f32x4_t qf[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    qf[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (!PAD || 16 * j + 4 * g < p.head_dim)
      qf[j] = *reinterpret_cast<const f32x4_t*>(p.q + q_row * p.head_dim + 16 * j + 4 * g) * c_log2;
  }

  f32x4_t acc[NH][VEC];
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[h][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  // A lane's rows of a block: 32-bit byte distances from the block's first token, which the load instructions add to a uniform
  // base (the launch takes blocks that span less than 2^32 bytes; WIDE: longer ones, with addresses of their own).
  using Offset = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
  const uint32_t row_bytes = uint32_t(kv_row) * 4u;
  // the row with coordinates `c` inside a block that begins at `org` (those past the group are masked: its last ones are
  // read in their place)
  auto row_offset = [&](const int (&c)[3], const int (&org)[3], bool clamp) __attribute__((always_inline)) {
    Offset o = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      o += Offset(uint32_t((clamp ? na_min(c[a], extent[a] - 1 - org[a]) : c[a]) * step[a])) * row_bytes;
    return o;
  };
  // coordinates inside a block of key `k` (dimension 2 fastest)
  auto key_coordinates = [&](int k, int (&c)[3]) __attribute__((always_inline)) {
    c[2] = k & ((1 << p.kv_lg[2]) - 1);
    k >>= p.kv_lg[2];
    c[1] = k & ((1 << p.kv_lg[1]) - 1);
    c[0] = k >> p.kv_lg[1];
  };
  // (at the group's edge formed from the lane number each time: such blocks are few, and fifteen coordinates kept for them are
  // a wave per SIMD less)
  auto lane_number = [&]() __attribute__((always_inline)) {
    uint32_t l = uint32_t(lane);
    pin(l);
    return l;
  };
  auto k_offset = [&](const int (&org)[3], bool clamp = true) __attribute__((always_inline)) {
    const uint32_t l = lane_number();
    int c[3];
    key_coordinates(int(l & 15), c);
    return row_offset(c, org, clamp) + (l >> 4) * 16;
  };
  auto v_offsets = [&](const int (&org)[3], Offset (&vo)[4], bool clamp = true) __attribute__((always_inline)) {
    const uint32_t l = lane_number();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int c[3];
      key_coordinates(int(l >> 4) * 4 + r, c);
      vo[r] = row_offset(c, org, clamp) + (l & 15) * (4 * VEC);
    }
  };
  const Offset k_off = k_offset(org0, false);
  Offset v_off[4];
  v_offsets(org0, v_off, false);
  int v_rel[3][4];  // in-block coordinates of the lane's four keys less its window's start
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    int c[3];
    key_coordinates(4 * g + r, c);
#pragma unroll
    for (int a = 0; a < 3; ++a) v_rel[a][r] = c[a] - ws[a];
  }

  // A block's K rows are read by S = K Q^T, its V rows by O += V^T P^T half a block later, and the rows of the block SETS
  // further on take their registers from then on: one set where the products of half a block are long enough to wait for
  // memory, and the registers saved are a wave more per SIMD at head dim 64 (2 x 64 x 64, H 8, 13 x 13: 54 us as two sets of whole
  // blocks, now 51; at 128, 48 x 80, 21 x 17, stride 2 x 4, H 8: 116 and 95; 2 x 8192, 257, stride 8, H 8: 221 and 188), two at head
  // dim 32 (12 x 24 x 30, 5 x 7 x 9, dilated, H 4: 43.2 us with one set, 41.4 with two; 96 x 96, 25 x 25, H 6: 126 either way, 134 before).
  // The loads are not conditional (past the last block they fetch it again, which nothing reads): behind a branch the
  // wait for rows becomes a wait for everything outstanding.
  // Blocks are described 64 at a time, one per lane, and read back by lane number (a scalar walk with its edge cases took some
  // hundred of a block's 133 scalar instructions, as long as its matrix instructions at head dim 32).
  const int total = nblk[0] * nblk[1] * nblk[2];
  int d_first = 0, d_row0 = 0, d_org[3] = {0, 0, 0};
  uint64_t d_full = 0, d_inside = 0;  // by lane: no key needs a mask; all keys lie inside the group
  auto describe = [&](int first) __attribute__((always_inline)) {
    d_first = first;
    int t[3];
    const int number = na_min(first + lane, total - 1);  // past the last block: that one again, which nothing reads
    if (__builtin_expect(total < (1 << 24), 1)) {
      kv_tile_of_box(number, nblk, t);
    } else {
      t[2] = number % nblk[2];
      t[1] = number / nblk[2] % nblk[1];
      t[0] = number / nblk[2] / nblk[1];
    }
    bool full = true, inside = true;
    d_row0 = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      d_org[a] = org0[a] + (t[a] << p.kv_lg[a]);
      const int end = d_org[a] + (1 << p.kv_lg[a]);
      inside = inside && end <= extent[a];
      full = full && d_org[a] >= full_lo[a] && end <= full_hi[a];
      d_row0 += d_org[a] * step[a];
    }
    d_full = __ballot(full);
    d_inside = __ballot(inside);
  };
  // what the loads of a block need
  struct Place {
    int row0, org[3];
    bool inside;
  };
  auto place = [&](int n) __attribute__((always_inline)) {
    const int l = n - d_first;
    Place t;
    t.row0 = __builtin_amdgcn_readlane(d_row0, l);
    t.inside = (d_inside >> l) & 1;
#pragma unroll
    for (int a = 0; a < 3; ++a) t.org[a] = __builtin_amdgcn_readlane(d_org[a], l);
    return t;
  };
  f32x4_t kf[SETS][KJ];
  fvec vf[SETS][4][NH];
  auto load_k = [&](int set, const Place& t) __attribute__((always_inline)) {
    Offset ko = k_off;
    if (!t.inside) ko = k_offset(t.org);
    const char* kb = reinterpret_cast<const char*>(kbase + int64_t(t.row0) * kv_row);
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      if constexpr (PAD) kf[set][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (!PAD || 16 * j + 4 * g < p.head_dim) kf[set][j] = *reinterpret_cast<const f32x4_t*>(kb + ko + 64 * j);
    }
  };
  auto load_v = [&](int set, const Place& t) __attribute__((always_inline)) {
    Offset vo[4] = {v_off[0], v_off[1], v_off[2], v_off[3]};
    if (!t.inside) v_offsets(t.org, vo);
    const char* vb = reinterpret_cast<const char*>(vbase + int64_t(t.row0) * kv_row);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        if constexpr (PAD) vf[set][r][h] = fvec(0.f);
        if (!PAD || VEC * (16 * h + i16) < p.head_dim) vf[set][r][h] = *reinterpret_cast<const fvec*>(vb + vo[r] + 64 * VEC * h);
      }
  };

  auto block = [&](int n, int set) __attribute__((always_inline)) {
    f32x4_t S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      if (PAD && 16 * j >= p.head_dim) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) S = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[set][j][e], qf[j][e], S, 0, 0, 0);
    }
    if (!((d_full >> (n - d_first)) & 1)) {
      const Place here = place(n);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (a < p.dims) {
#pragma unroll
          for (int r = 0; r < 4; ++r) S[r] = uint32_t(v_rel[a][r] + here.org[a]) < uint32_t(width[a]) ? S[r] : -INFINITY;
        }
      }
    }
    if (n + SETS - d_first >= 64) describe(n + 1);
    const Place next = place(n + SETS);
    load_k(set, next);
    const float mx_own = fmaxf(fmaxf(S[0], S[1]), fmaxf(S[2], S[3]));
    if (__ballot(mx_own > m_run + kLazyRescaleLog2) != 0) {
      float mx = fmaxf(mx_own, __shfl_xor(mx_own, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float m_new = fmaxf(m_run, mx);
      const float alpha = fast_exp2(m_run - (m_new == -INFINITY ? 0.f : m_new));  // 0 while m_run is -inf
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int c = 0; c < VEC; ++c) acc[h][c] *= alpha;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = fast_exp2(S[r] - m_use);
    l_run += (S[0] + S[1]) + (S[2] + S[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int c = 0; c < VEC; ++c) acc[h][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[set][r][h][c], S[r], acc[h][c], 0, 0, 0);
    load_v(set, next);
  };
  describe(0);
#pragma unroll
  for (int i = 0; i < SETS; ++i) {
    load_k(i, place(i));
    load_v(i, place(i));
  }
  for (int n = 0; n < total; n += SETS) {
    block(n, 0);
    if (SETS > 1 && n + 1 < total) block(n + 1, SETS - 1);
  }

  float l = l_run + __shfl_xor(l_run, 16);
  l += __shfl_xor(l, 32);
  const float inv = (l > 0.f) ? 1.f / l : 0.f;
  if (valid) {
    float* orow = p.o + q_row * p.head_dim;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = VEC * (16 * h + 4 * g + r);
        fvec o;
#pragma unroll
        for (int c = 0; c < VEC; ++c) o[c] = acc[h][c][r] * inv;
        if (!PAD || d < p.head_dim) *reinterpret_cast<fvec*>(orow + d) = o;
      }
    // The logarithm of a mantissa, not of the sum: the hardware's is low by up to a unit in the last place of its
    // result, and a sum whose maximum lags is large (windows of 1025 keys: 4.2e-7 rms from float64, 3.2e-7
    // on permuted sequences, where the maximum is followed at once; like this 2.1e-7)
    int e;
    const float log_l = logf(frexpf(l, &e));
    if (g == 0) p.lse[q_row] = (l > 0.f) ? fmaf(m_run, 0.6931471805599453f, fmaf(float(e), 0.6931471805599453f, log_l)) : -INFINITY;
  }
}

}  // namespace natten_amd
