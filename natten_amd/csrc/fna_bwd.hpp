// Fused neighborhood attention backward for gfx950 (MI355X).
//
// One kernel template, several roles.  A workgroup owns a "stationary" tile of 128 rows (one
// row per lane and 32-row block, four waves) and streams 64-row tiles of the other side
// through LDS:
//   dQ role          : stationary = queries (operands Q, dO; result dQ), streamed = keys (K, V)
//   dKV, paired role : stationary = keys    (operands K, V; results dK and dV), streamed = queries (Q, dO)
// Per streamed tile, with Y1/Y2 the streamed and X1/X2 the stationary operands:
//   S^T  = Y1 X1^T,  dP^T = Y2 X2^T                     (32x32x16 MFMA, the lane owns a stationary row)
//   P    = exp2(S - log2e LSE) on unmasked pairs, 0 elsewhere;  dS = P (dP - delta)   (both differences
//          are the products' accumulator inputs)
//   acc1^T += Y1^T dS^T   (dQ = scale * sum_k dS k  /  dK = ln 2 * sum_q dS q')
// The logits are formed from the same operand as in the forward kernel, q' = round(q * scale *
// log2(e)) in the operand type, so that S is the forward's logit to the last bit of its operands
// and P the probability its LSE normalises (the rows of P sum to one); with the unscaled queries
// the two passes' logits differ by the rounding of q', and a probability of a one-key window
// comes out as 1 +- 0.5 % instead of 1.  The dQ role scales its stationary query fragments as it
// loads them; the key-stationary roles stream q' from a copy (qs) that a pass over q writes first.
//   acc2^T += Y2^T P^T    (dV = sum_q P dO)
// In the dKV role one wave forms all of this for its 32 key rows.  At head dim 128 the
// accumulators, stationary fragments and both products of that no longer fit the 256 vector
// registers a matrix instruction can address directly; the paired role then splits the work
// over two waves without recomputing anything: eight waves per workgroup, waves w and w + 4
// share the 32 key rows of block w; wave w ("P wave") forms S^T, the probabilities and dV,
// wave w + 4 ("dS wave") forms dP^T, takes the probabilities from LDS (fp16, one tile later),
// and forms dS and dK.  LSE and delta = rowsum(dO * O) belong to the
// query: per-lane scalars in the dQ role, a small per-tile LDS table in the others.  Nothing
// is accumulated through memory, so the results are deterministic.
//
// What bounds it is the instruction issue of two waves per SIMD next to the matrix pipe: per wave and tile of
// head dim 128 the paired role's P waves issue 49 vector instructions and 32 exponentials beside 32
// matrix instructions (115 under the mask), its dS waves 66.  That took: products that start from
// -log2e LSE and -delta (no subtraction per pair), the mask as one bit per pair (two instructions
// where the comparison of packed coordinates took five), dS from the half-precision probabilities by
// mixed multiply-adds, tile descriptors formed 64 at a time.  Before it the counts were 82 / 244 / 131 and
// the dK / dV launch took 25.2 ms on 29 x 46 x 78 tokens, window 9 x 24 x 24, H 24 (now 20.7), 569 us on
// 128 x 128, window 32 x 32, stride 16, H 16 (433); head dim 32, 4 x 56 x 56, window 7 x 7, H 8: 59 (43).
//
// What it restates (not the code): SHI-Labs/NATTEN
//   csrc/include/natten/cuda/reference/fna_reference_backward.hpp:60-150, :165-265, :282-380
//     (P = exp(scale q.k - LSE), dS = P scale (dO.v - dO.o), dQ / dK / dV as sums over the mask)
//   csrc/include/natten/cuda/fna_blackwell/collective/fna_fusion_bwd.hpp:256-318 (the Q tiles a KV tile meets;
//     here the query interval is inverted from the forward's own window functions)
// Operands are token-permuted sequences whose tiles hold 128 tokens; such a tile splits, along
// its slowest dimension, into two contiguous 64-token tiles, which is what the other role streams.
#pragma once

#include "fna_fwd.hpp"

namespace natten_amd {

struct FnaBwdParams {
  const void* q;      // [batch, seqlen_q, heads_q, D]   (batch counts dilation groups)
  const void* qs;     // like q: round(q * scale * log2(e)), the forward kernel's logit operand (key-stationary roles)
  const void* k;      // [batch, seqlen_kv, heads_kv, D]
  const void* v;
  const void* d_out;  // like q
  // [batch, heads_q, seqlen_q] (head-major: a tile's values are contiguous).  The kernels' accumulators
  // start from lse_mul times `lse` and delta_mul times `delta`, that is from -log2(e) LSE and -rowsum(d_out *
  // out).  prepared != 0: the arrays hold these values already (both factors are 1; bwd_prepare_kernel);
  // 0: the forward's LSE and the row sums themselves, which the RAW instances scale as they read a tile's.
  const float* lse;
  const float* delta;
  int prepared;
  float lse_mul, delta_mul;
  // dQ launches that come first (RAW instances of that role, original layout): the forward's output and its LSE [batch,
  // tokens, heads].  The launch forms both values of its rows itself and leaves them, and its scaled queries, in `lse`, `delta`
  // and `qs` for the launch behind it.
  const void* out;
  const float* lse_rows;
  void* dq;
  void* dk;
  void* dv;
  int batch, heads_q, heads_kv;
  int seqlen_q, seqlen_kv;
  int num_groups;
  int qkv_shape[3];
  int q_extent0;  // > 0: queries along dimension 0 (dense attention with its own query count); 0: as the keys
  int ksize[3], stride[3], dil[3], causal[3];
  int q_tile[3], kv_tile[3];    // 128-token tiles of the two permuted layouts
  int q_tiled[3], kv_tiled[3];  // tiles per dimension
  int kv_shift[3];              // fused == 1, key-stationary launches: key tile t holds the keys from t kv_tile - kv_shift on (choose_kv_shift)
  int q_split, kv_split;        // the dimension along which a 128-token tile of either side halves
                                // (its last dimension of extent > 1, so that the halves are contiguous)
  float scale;
  // Operand layout.  fused == 0: token-permuted sequences as described above.  fused == 1: the
  // original tensors [batch, X0, X1, X2, heads, D] (lse / delta [batch, heads, X0 * X1 * X2]);
  // the kernel gathers and scatters the rows of a tile itself.
  int fused;
  // fused == 1 only: some extent is not a multiple of dilation x tile, so tiles may reach past a
  // dilation group (every group is at least a tile wide in every dimension).  Rows of the stationary
  // tile past the group's end are computed on a clamped copy and not stored; a streamed tile that
  // would reach past it is gathered from one tile extent before the end, and its leading rows,
  // which the tile before it delivered, take no part (as in the forward kernel).
  int edge;
  int tok_stride[3];  // tokens per unit step of an original coordinate: X1*X2, X2, 1
  int tokens;         // X0 * X1 * X2
  // Sequence-packed dense attention (RAGGED instances only; null otherwise): num_seqs sequences lie
  // back to back in one row range (the tensors have batch 1; seqlen_q / seqlen_kv count all their
  // rows), sequence b owns query rows cu_q[b] .. cu_q[b+1]-1 and key rows cu_kv[b] .. cu_kv[b+1]-1;
  // q_tiled[0] / kv_tiled[0] count the tiles that any such batch has at most (see PackedTile).
  const int32_t* cu_q;    // [num_seqs + 1]
  const int32_t* cu_kv;
  const int2* packed_q;   // [num_seqs + 2] (count_packed_tiles)
  const int2* packed_kv;
  int num_seqs;
  // Workgroup order of the key-stationary launch.  0: every XCD takes one contiguous eighth of
  // the (batch, head, tile) space.  > 0: runs of this many consecutive tiles are dealt round-robin
  // to the XCDs (the grid is then a whole number of rounds of 8 runs).
  int kv_wg_run;
  // Host side only: which launches a call makes (bit 0: the dQ role, bit 1: the dK / dV role; 0 = both), and kBwdOverlap.
  int roles;
  // Derived by set_bwd_divisions(): what the per-workgroup set-up would otherwise divide for (tile
  // extents are powers of two, the other divisors get multiply-shift pairs).
  // Dividing and bisecting for the query ranges in the kernel cost every workgroup several
  // thousand instructions: a training step of 128 x 128 tokens, H 16, D 128 (2 048 key tiles, one
  // workgroup per CU at a time) 1046 -> 956 us, 29 x 46 x 78 dilated H 24 50.3 -> 48.4 ms.
  int q_tile_lg[3], kv_tile_lg[3];
  int ext_base[3], ext_rem[3];  // qkv_shape / dil and qkv_shape % dil
  NaDiv d_stride[3], d_dil[3], d_num_groups, d_rep, d_kv_wg_run;
  NaDiv d_q_tiled[3], d_kv_tiled[3], d_num_q, d_num_kv, d_heads_q, d_heads_kv;
};

inline void set_bwd_divisions(FnaBwdParams& p) {
  p.lse_mul = p.prepared ? 1.f : -1.4426950408889634f;
  p.delta_mul = p.prepared ? 1.f : -1.f;
  for (int a = 0; a < 3; ++a) {
    p.q_tile_lg[a] = p.kv_tile_lg[a] = 0;
    while ((1 << p.q_tile_lg[a]) < p.q_tile[a]) ++p.q_tile_lg[a];
    while ((1 << p.kv_tile_lg[a]) < p.kv_tile[a]) ++p.kv_tile_lg[a];
    p.ext_base[a] = p.qkv_shape[a] / p.dil[a];
    p.ext_rem[a] = p.qkv_shape[a] % p.dil[a];
    p.d_stride[a] = na_make_div(p.stride[a]);
    p.d_dil[a] = na_make_div(p.dil[a]);
    p.d_q_tiled[a] = na_make_div(p.q_tiled[a]);
    p.d_kv_tiled[a] = na_make_div(p.kv_tiled[a]);
  }
  p.d_num_groups = na_make_div(p.num_groups);
  p.d_rep = na_make_div(p.heads_q / p.heads_kv);
  p.d_kv_wg_run = na_make_div(p.kv_wg_run > 0 ? p.kv_wg_run : 1);
  p.d_num_q = na_make_div(p.q_tiled[0] * p.q_tiled[1] * p.q_tiled[2]);
  p.d_num_kv = na_make_div(p.kv_tiled[0] * p.kv_tiled[1] * p.kv_tiled[2]);
  p.d_heads_q = na_make_div(p.heads_q);
  p.d_heads_kv = na_make_div(p.heads_kv);
}

// Where the key tiles of the key-stationary launch begin (original layout).  With strided windows the queries that
// attend a key change at the keys where a stride group's window begins or ends; tiles that begin there meet fewer
// query tiles than tiles at multiples of their extent, which cross such a key in the middle (128 x 128 tokens, window
// 32 x 32, stride 16 x 16, H 16, D 128, key tiles of 8 x 16: the launch takes 430 us with tiles at multiples of 16 and 362
// with the first tile beginning 8 keys early).  Per dimension, the choice that meets the fewest among: multiples of
// the extent, the first keys of windows, their ends, the last tile ending with the keys -- and at least a
// twentieth fewer than the first, since other choices may take a tile more.  Tiles are counted from both
// ends where there are many: what lies between repeats.
inline int choose_kv_shift(int L, int k, int s, bool causal, int tile, int q_sub) {
  if (s <= 1 || tile <= 1 || L <= tile) return 0;
  const NaDiv d = na_make_div(s);
  const int begin = causal ? s - k : s / 2 - k / 2;  // windows of whole groups begin at begin + i s
  auto place = [&](int x) { return ((-x) % tile + tile) % tile; };
  const int candidate[4] = {0, place(begin), place(begin + k), place(L)};
  auto met = [&](int shift) {
    const int n = (L + shift + tile - 1) / tile;
    double sum = 0;
    int counted = 0;
    for (int t = 0; t < n; ++t) {
      if (n > 64 && t == 32) t = n - 32;
      const int j0 = na_max(t * tile - shift, 0), j1 = na_min((t + 1) * tile - shift, L) - 1;
      const int lo = na_first_query_attending(j0, k, s, d, L, causal), hi = na_last_query_attending(j1, k, s, d, L, L, causal);
      const int flo = na_first_query_attending(j1, k, s, d, L, causal), fhi = na_last_query_attending(j0, k, s, d, L, L, causal);
      ++counted;
      if (lo > hi) continue;
      const int tiles = hi / q_sub - lo / q_sub + 1;
      const int whole = na_max((fhi + 1) / q_sub - (flo + q_sub - 1) / q_sub, 0);
      sum += tiles + 0.3 * (tiles - whole);
    }
    return sum * n / counted;
  };
  const double plain = met(0);
  double least = plain * 0.95;
  int best = 0;
  for (int i = 1; i < 4; ++i) {
    const double m = candidate[i] ? met(candidate[i]) : plain;
    if (m < least) {
      least = m;
      best = candidate[i];
    }
  }
  return best;
}

// FnaBwdParams::roles: the dQ launch runs beside the dK / dV launch, on a stream of its own (dq is not the workspace that the
// other one reads).  That launch lasts as long as its longest workgroup, and while that walks its query tiles most
// compute units have nothing left to do: both launches of a packed step, 10 sequences of 1 .. 2048, H 16 / 4, D 128, with
// the pass before, 310 us one behind the other and 255 side by side; the callers know where it pays.
constexpr int kBwdOverlap = 16;

enum BwdRole : int { kBwdDQ = 0, kBwdDKV = 1, kBwdPair = 2 };

// Tiles of a sequence-packed batch.  The rows 0 .. total - 1 of one side are the sequences cu[i] ..
// cu[i + 1] - 1 (those whose offsets the rows can hold and that do not reach back over rows of an earlier
// one) and the gaps around them, whose rows belong to no sequence; tiles of 2^tile_lg rows are counted
// through both, a sequence's gap first, the rows behind the last sequence as the gap of sequence num_seqs.
// Every row is in one sequence or gap, whatever the offsets: a launch leaves none unwritten.  There are at
// most num_seqs + 2 of them (where a sequence follows one that counts, it begins where that ends: a gap takes
// a sequence that does not count, or is the first or the last), so a launch of total / tile + num_seqs + 3
// tiles per head covers any lengths, where one sized for the longest sequence starts a workgroup per sequence
// and tile of that one (10 sequences of 1 .. 2048: 160 tiles a head, of which 87 find nothing to do).
// One workgroup of the pass before counts (count_packed_tiles), and a tile finds its sequence in the
// counts (locate_packed_tile): 64 places looked at per step, one step up to 64 sequences, three up to
// 262144.  Counting through the lengths in every workgroup instead is quadratic in their number: 10000
// sequences of 50 rows, H 2, D 32, training step: 10.7 ms like that, 0.65 with the counts; 4000 of 16, H 4, D 64:
// 4.7 and 0.64; 1000 of 64, H 8, D 64: 1.06 and 0.43.
struct PackedSeq {
  int gap0, gap_rows, row0, rows;
  int end;  // rows below it are covered with this entry (0: by the entries before it only)
};
// `covered`: the rows below it lie in a sequence or gap before number i
static __device__ __forceinline__ PackedSeq packed_seq(const int32_t* cu, int i, int num_seqs, int total, int covered) {
  int beg = 0, end = 0;
  if (i < num_seqs) {
    beg = cu[i];
    end = cu[i + 1];
  }
  const bool valid = i < num_seqs && beg >= 0 && end >= beg && end <= total;
  const bool counts = valid && beg >= covered;
  PackedSeq s;
  s.gap0 = covered;
  s.gap_rows = na_max((i == num_seqs ? total : counts ? beg : valid ? end : 0) - covered, 0);
  s.row0 = beg;
  s.rows = counts ? end - beg : 0;
  s.end = valid ? end : 0;
  return s;
}
static __device__ __forceinline__ int packed_tiles_of(int rows, int tile_lg) { return (rows + (1 << tile_lg) - 1) >> tile_lg; }

// Inclusive scan over the 256 threads of a workgroup; `totals`: four words of LDS.
template <typename Op>
static __device__ __forceinline__ int scan256(int x, int tid, int* totals, Op op) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o);
    if ((tid & 63) >= o) x = op(y, x);
  }
  workgroup_sync();  // the totals of the scan before have been read
  if ((tid & 63) == 63) totals[tid >> 6] = x;
  workgroup_sync();
  for (int w = 0; w < (tid >> 6); ++w) x = op(totals[w], x);
  return x;
}

// One workgroup of 256 threads: out[i] = {tiles before sequence i and its gap, rows covered before them} for
// i = 0 .. num_seqs, out[num_seqs + 1] = {all tiles, all rows}.
static __device__ __forceinline__ void count_packed_tiles(const int32_t* __restrict__ cu, int num_seqs, int total, int tile_lg,
                                                          int2* __restrict__ out, int* totals) {
  constexpr int PER = 8;
  const int tid = threadIdx.x;
  __shared__ int s_carry[2];
  int covered0 = 0, first0 = 0;  // of the entries of earlier steps
  for (int s0 = 0; s0 <= num_seqs; s0 += 256 * PER) {
    const int i0 = s0 + tid * PER;
    int top = 0;
    for (int e = 0; e < PER; ++e) {
      if (i0 + e > num_seqs) break;
      top = na_max(top, packed_seq(cu, i0 + e, num_seqs, total, 0).end);
    }
    const int upto = scan256(top, tid, totals, [](int a, int b) { return na_max(a, b); });
    const int before = __shfl_up(upto, 1);
    int wave_before = 0;  // what the waves before this one cover
    for (int w = 0; w < (tid >> 6); ++w) wave_before = na_max(wave_before, totals[w]);
    const int covered_in = na_max(covered0, (tid & 63) ? before : wave_before);
    int covered = covered_in, tiles = 0;
    for (int e = 0; e < PER; ++e) {
      if (i0 + e > num_seqs) break;
      const PackedSeq s = packed_seq(cu, i0 + e, num_seqs, total, covered);
      tiles += packed_tiles_of(s.gap_rows, tile_lg) + packed_tiles_of(s.rows, tile_lg);
      covered = na_max(covered, s.end);
    }
    const int sum = scan256(tiles, tid, totals, [](int a, int b) { return a + b; });
    int first = first0 + sum - tiles;
    covered = covered_in;
    for (int e = 0; e < PER; ++e) {
      if (i0 + e > num_seqs) break;
      const PackedSeq s = packed_seq(cu, i0 + e, num_seqs, total, covered);
      out[i0 + e] = make_int2(first, covered);
      first += packed_tiles_of(s.gap_rows, tile_lg) + packed_tiles_of(s.rows, tile_lg);
      covered = na_max(covered, s.end);
      if (i0 + e == num_seqs) out[num_seqs + 1] = make_int2(first, total);
    }
    if (tid == 255) {
      s_carry[0] = covered;
      s_carry[1] = first;
    }
    workgroup_sync();
    covered0 = s_carry[0];
    first0 = s_carry[1];
    workgroup_sync();
  }
}

struct PackedTile {
  int seq;
  bool gap;        // rows of no sequence
  int row0, rows;  // first row and row count of the sequence (or the gap)
  int tile;        // position of the tile inside it
};
// Tile x of the batch; all 64 lanes of a wave call it together.  false: there are fewer tiles than x.
static __device__ __forceinline__ bool locate_packed_tile(const int2* __restrict__ counts, const int32_t* __restrict__ cu,
                                                          const int num_seqs, const int total, const int tile_lg, const int x,
                                                          const int lane, PackedTile& t) {
  if (x >= counts[num_seqs + 1].x) return false;
  // the last entry whose tiles begin at or before x, among `n` from `lo` on
  int lo = 0, n = num_seqs + 1;
  while (n > 1) {
    const int step = (n + 63) >> 6;
    const int at = lane * step;
    const uint64_t below = __ballot(at < n && counts[lo + na_min(at, n - 1)].x <= x);
    const int l = 63 - __builtin_clzll(below | 1);
    lo += l * step;
    n = na_min(step, n - l * step);
  }
  const int2 c = counts[lo];
  const PackedSeq s = packed_seq(cu, lo, num_seqs, total, c.y);
  const int gap_tiles = packed_tiles_of(s.gap_rows, tile_lg);
  const int local = x - c.x;
  t.seq = lo;
  t.gap = local < gap_tiles;
  t.tile = t.gap ? local : local - gap_tiles;
  t.row0 = t.gap ? s.gap0 : s.row0;
  t.rows = t.gap ? s.gap_rows : s.rows;
  return true;
}

// sum_e a[e] b[e] of eight elements in order, in float.  (One routine for whoever forms delta: the compiler makes pairwise
// products of fp16 of some such loops and not of others, and the routes promise each other's bits.)
template <typename T>
static __device__ __forceinline__ float dot8(typename Mma<T>::vec8 a, typename Mma<T>::vec8 b) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    if constexpr (std::is_same<T, _Float16>::value) {
      s = __builtin_amdgcn_fdot2(typename Mma<T>::vec2{a[e], a[e + 1]}, typename Mma<T>::vec2{b[e], b[e + 1]}, s, false);
    } else {
      s = __builtin_fmaf(float(a[e + 1]), float(b[e + 1]), __builtin_fmaf(float(a[e]), float(b[e]), s));
    }
  }
  return s;
}

// Waves per SIMD the compiler makes room for (and, as the attribute's maximum, limits the kernel to).  Of the
// SIMD's 512 registers a lane, the key-stationary and the dQ instance take 213 to 219 and 248 at head dim 128 (249
// where it comes first and holds the output's fragments as well, 252 where sequences end inside a tile), 213 to 217
// and 198 to 200 at 64, 158 to 162 and 159 or 160 at 32; none spills.  One wave
// more for the dQ role at 64 and 32 needs its LSE and delta in a register each instead of sixteen copies that
// the accumulators start from, and two additions a logit: dQ launch in us, copies / one wave more, D 64: 48 x 48
// tokens, H 6, 11 x 11 18.5 / 20.3; 4 x 56 x 56, H 8, 7 x 7 39.5 / 41.9; 16 x 40 x 40, H 12, 7 x 15 x 15 409 / 424; D 32: 24 x
// 32 x 32, H 8, 9 x 9 x 9 105 / 115; 2 x 40 x 40, H 16, 25 x 25 31.9 / 36.2; 4 x 56 x 56, H 8, 7 x 7 33.3 / 32.1.
// Head dim 32 with two waves instead of three on the last: 52, and dK and dV 82 instead of 59.
constexpr int bwd_waves_per_simd(int head_dim) { return head_dim > 32 ? 2 : 3; }

// RAGGED: dense attention whose sequences end inside a tile, packed ones among them.  Rows past the end
// of a sequence are gathered from its last row; stationary ones store nothing, streamed ones are masked.
// (Padding the sequences into copies first made 67 launches of a packed training step, of index arithmetic
// and copies most of them: 10 sequences of 1 .. 2048, H 16 / 4, D 128 919 us, now 6 launches and 424 us.)
// RAW: in the key-stationary roles LSE and delta as they are, scaled on the way from LDS to the accumulators
// (the dQ role scales its two values per lane in every instance).  In the dQ role the launch that comes first and prepares the other's
// arrays (see FnaBwdParams::out): a pass of its own over q, out and d_out reads two of them once more and is waited for
// (the pass and both launches / both launches, us: 4 x 56 x 56, 7 x 7, H 8, D 32 74.2 / 69.5; 96 x 96, 24 x 24, stride 8, H 8, D 64 91 / 83; 128 x 128,
// 32 x 32, stride 16, H 16, D 128 594 / 573; 29 x 46 x 78, 9 x 24 x 24, dilated, H 8 12340 / 12270).
template <typename T, int D, int ROLE, bool RAGGED = false, bool RAW = false>
__global__ void __launch_bounds__(ROLE == kBwdPair ? 512 : 256)
__attribute__((amdgpu_waves_per_eu(bwd_waves_per_simd(D), bwd_waves_per_simd(D))))
fna_bwd_kernel(const FnaBwdParams p) {
  constexpr bool KV_STATIONARY = ROLE != kBwdDQ;
  constexpr bool PAIR = ROLE == kBwdPair;
  // what one wave's tile body forms (a P wave of the paired role is a dV wave that also hands on
  // its probabilities; the dS waves have a body of their own)
  constexpr bool HAS_DS = !PAIR;                      // dP, dS and acc1 (dQ or dK)
  constexpr bool HAS_PV = ROLE == kBwdDKV || PAIR;  // acc2 (dV; dK in a dS wave)
  constexpr int NT = PAIR ? 512 : 256;
  constexpr int AT = 128;  // stationary rows
  constexpr int BT = 64;   // streamed rows per tile
  constexpr int KSTEPS = D / 16;
  constexpr int DB = D / 32;
  constexpr int NSB = BT / 32;
  using L = FnaSmem<D, BT>;
  constexpr int ROWB = L::ROWB;
  constexpr int CPR = L::CPR;
  constexpr int TILE_BYTES = L::TILE_BYTES;
  constexpr int CHUNKS = BT * CPR;
  constexpr int PER = CHUNKS / NT;
  static_assert(CHUNKS % NT == 0 && PER >= 1, "a streamed tile must be a whole number of workgroup-wide copies");
  static_assert(NSB == 2, "the slot schedule is written for two 32-row sub-blocks");
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using vec2 = typename M::vec2;
  typedef _Float16 h16x2_t __attribute__((ext_vector_type(2)));

  // One copy of Y1 and one of Y2 per stage, in the layout that serves row reads (S, dP) and
  // transpose reads (the accumulations) alike.
  // Stages: tiles are copied NS - 1 ahead.  Two stages at head dim 128 keep a workgroup under
  // half of the CU's LDS, so that two workgroups (two waves per SIMD) share a CU.
  // The paired role copies two tiles ahead, at any point of a step: Y2 (dO) is read in its own
  // step only and has three stages; Y1 (Q) and the tables are read for two steps (the dS waves
  // run one tile behind) and have four.
  constexpr int NS = (D == 128 && !PAIR) ? 2 : 3;
  constexpr int NS1 = PAIR ? 4 : NS;  // stages of Y1 and of the tables
  static_assert(!PAIR || D == 128, "the paired role is for head dim 128 (smaller ones fit the combined role)");
  __shared__ __attribute__((aligned(1024))) char sY1[NS1 * TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) char sY2[NS * TILE_BYTES];
  // sRows[a][g][x]: the rows of a streamed tile whose coordinate along dimension a is >= x, one bit per
  // row: the 32 bits that the lanes of wave half g hold logits for (as sKeys of the forward kernel)
  __shared__ __attribute__((aligned(16))) uint32_t sRows[3][2][BT + 1];
  __shared__ __attribute__((aligned(16))) float sLse[NS1 * BT];
  __shared__ __attribute__((aligned(16))) float sDelta[NS1 * BT];
  __shared__ __attribute__((aligned(16))) float sSpare[BT];
  // paired role: probabilities from the P waves to the dS waves, fp16, [tile parity][row block]
  // [sub-block][half of the 16 values][lane] x 16 bytes
  __shared__ __attribute__((aligned(16))) char sX[PAIR ? 2 * 4 * NSB * 2 * 64 * 16 : 16];

  touch_launch_params<sizeof(FnaBwdParams)>();
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = PAIR ? (wave & 3) : wave;  // 32-row block of the stationary tile
  const int part = PAIR ? (wave >> 2) : 0;  // paired role: 0 = P wave, 1 = dS wave
  const int l32 = lane & 31;
  const int g = lane >> 5;

  const int* a_tile = KV_STATIONARY ? p.kv_tile : p.q_tile;
  const int* a_tiled = KV_STATIONARY ? p.kv_tiled : p.q_tiled;
  const int* a_tile_lg = KV_STATIONARY ? p.kv_tile_lg : p.q_tile_lg;
  const int* b_tile = KV_STATIONARY ? p.q_tile : p.kv_tile;
  const int* b_tile_lg = KV_STATIONARY ? p.q_tile_lg : p.kv_tile_lg;
  const int* b_tiled = KV_STATIONARY ? p.q_tiled : p.kv_tiled;
  const int heads_a = KV_STATIONARY ? p.heads_kv : p.heads_q;
  const int heads_b = KV_STATIONARY ? p.heads_q : p.heads_kv;
  const int seq_a = KV_STATIONARY ? p.seqlen_kv : p.seqlen_q;
  const int seq_b = KV_STATIONARY ? p.seqlen_q : p.seqlen_kv;
  const int rep = na_div(p.heads_q, p.d_heads_kv);
  const int split_dim = KV_STATIONARY ? p.q_split : p.kv_split;  // of the streamed side

  // ---- workgroup -> (batch * group, head, stationary tile) --------------------------------------
  // Workgroup ids go round-robin to the 8 XCDs; each XCD takes one contiguous eighth of the
  // (batch, head, tile) space, so that the workgroups resident on an XCD are neighbouring tiles
  // of one head and find each other's streamed tiles in that XCD's L2.  The paired role, with
  // half as many workgroups resident, does better with short runs dealt round-robin: the XCDs
  // then work on neighbouring runs of one head at a time and meet in the memory-side cache.
  const int num_a = a_tiled[0] * a_tiled[1] * a_tiled[2];
  const int total_wg = p.batch * heads_a * num_a;
  const int wg_run = KV_STATIONARY ? p.kv_wg_run : 0;
  int lin;
  if (wg_run > 0) {
    const int local = int(blockIdx.x) / kNumXcd;
    const int round = na_div(local, p.d_kv_wg_run);
    lin = (round * kNumXcd + int(blockIdx.x) % kNumXcd) * wg_run + local - round * wg_run;
  } else {
    const int chunk = (total_wg + kNumXcd - 1) / kNumXcd;
    lin = (int(blockIdx.x) % kNumXcd) * chunk + int(blockIdx.x) / kNumXcd;
  }
  // Ragged dense attention: heads fastest, so that the long tiles of a head's sequences (the first key
  // tiles and the last query tiles where causal) are spread over all XCDs, and with as many heads
  // as XCDs, or a divisor of them, every XCD still streams one head's tiles.  Runs of 32 tiles put a whole
  // 2048-token sequence of a head on one XCD: packed training step of 10 sequences of 1 .. 2048, H 16 /
  // 4, D 128: dK / dV launch 326 -> 254 us.
  if constexpr (RAGGED) lin = int(blockIdx.x);
  if (lin >= total_wg) return;
  // Within a head the tiles are taken with dimension 0 slowest: the workgroups running side by
  // side are then neighbours in the faster dimensions at the same dimension-0 position and
  // walk the same streamed tiles at about the same time.
  const NaDiv d_num_a = KV_STATIONARY ? p.d_num_kv : p.d_num_q, d_heads_a = KV_STATIONARY ? p.d_heads_kv : p.d_heads_q;
  int bg, head_a, rm;
  if constexpr (RAGGED) {
    const int bt = na_div(lin, d_heads_a);
    head_a = lin - bt * heads_a;
    bg = na_div(bt, d_num_a);
    rm = bt - bg * num_a;
  } else {
    const int bh = na_div(lin, d_num_a);
    rm = lin - bh * num_a;
    bg = na_div(bh, d_heads_a);
    head_a = bh - bg * heads_a;
  }
  int tc[3];
  {
    const int t01 = na_div(rm, KV_STATIONARY ? p.d_kv_tiled[2] : p.d_q_tiled[2]);
    tc[2] = rm - t01 * a_tiled[2];
    tc[0] = na_div(t01, KV_STATIONARY ? p.d_kv_tiled[1] : p.d_q_tiled[1]);
    tc[1] = t01 - tc[0] * a_tiled[1];
    // a causal dimension 0: the query tiles with the longest key ranges are the last ones;
    // they start first (key tiles are already in that order)
    if (!KV_STATIONARY && p.causal[0] && !(RAGGED && p.cu_q)) tc[0] = a_tiled[0] - 1 - tc[0];
  }
  const int at = tc[0] + a_tiled[0] * (tc[1] + a_tiled[1] * tc[2]);  // position in the permuted sequence
  const int b_orig = na_div(bg, p.d_num_groups);  // batch entry before the dilation groups were folded in

  // first rows of this batch entry's sequences, its lse / delta values of head 0, and the
  // parameters a packed sequence overrides
  int64_t seq_row_a = int64_t(bg) * seq_a, seq_row_b = int64_t(bg) * seq_b;
  int64_t stat_row_q = int64_t(bg) * p.heads_q * p.seqlen_q;
  int64_t stat_head_stride = p.seqlen_q;
  int ksz[3] = {p.ksize[0], p.ksize[1], p.ksize[2]};
  int keys0 = p.ext_base[0], queries0 = p.q_extent0;  // (extents of dimension 0 before the uneven dilation groups)
  bool empty = false;
  if constexpr (RAGGED) {
    if (p.cu_q) {
      PackedTile t;
      if (!locate_packed_tile(KV_STATIONARY ? p.packed_kv : p.packed_q, KV_STATIONARY ? p.cu_kv : p.cu_q, p.num_seqs, seq_a, 7,
                              tc[0], lane, t))
        return;
      tc[0] = t.tile;
      seq_row_a = t.row0;
      int other0 = 0, other = 0;  // the sequence's rows on the streamed side
      if (!t.gap) {
        const int32_t* cu = KV_STATIONARY ? p.cu_q : p.cu_kv;
        other0 = cu[t.seq];
        other = cu[t.seq + 1] - other0;
        if (other0 < 0 || other < 0 || other0 > seq_b - other) other0 = other = 0;  // offsets the tensors cannot hold are not followed
        // (the query tiles with the longest key ranges first, as above)
        if (!KV_STATIONARY && p.causal[0]) tc[0] = ((t.rows + AT - 1) / AT) - 1 - tc[0];
      }
      empty = other == 0;  // nothing attends, or attends to nothing: zero gradients
      seq_row_b = other0;
      stat_row_q = KV_STATIONARY ? other0 : t.row0;
      keys0 = ksz[0] = na_max(KV_STATIONARY ? t.rows : other, 1);
      queries0 = na_max(KV_STATIONARY ? other : t.rows, 1);
    }
  }

  int extent[3], q_extent[3], a_first[3], b_sub[3], b_sub_lg[3];
  int tok_step[3];    // original layout: tokens per unit step of a coordinate inside a dilation group
  int group_tok = 0;  // original layout: token of the dilation group's first element
  {
    int gl = bg - b_orig * p.num_groups;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int rest = na_div(gl, p.d_dil[a]);
      const int gi = gl - rest * p.dil[a];
      gl = rest;
      tok_step[a] = p.dil[a] * p.tok_stride[a];
      group_tok += gi * p.tok_stride[a];
      // (as in the forward kernel: the first groups hold one token more when the dilation does not divide the extent)
      extent[a] = (a == 0 ? keys0 : p.ext_base[a]) + (gi < p.ext_rem[a] ? 1 : 0);
      q_extent[a] = (a == 0 && queries0 > 0) ? queries0 : extent[a];
      a_first[a] = (tc[a] << a_tile_lg[a]) - (KV_STATIONARY && !RAGGED ? p.kv_shift[a] : 0);
      b_sub_lg[a] = b_tile_lg[a] - (a == split_dim ? 1 : 0);
      b_sub[a] = 1 << b_sub_lg[a];
      if (a_first[a] >= (KV_STATIONARY ? extent[a] : q_extent[a])) empty = true;
    }
  }

  // ---- this lane's stationary row -----------------------------------------------------------------
  const int r_in = rw * 32 + l32;  // row inside the tile: dimension 0 fastest
  int a_off[3];
  a_off[0] = r_in & (a_tile[0] - 1);
  a_off[1] = (r_in >> a_tile_lg[0]) & (a_tile[1] - 1);
  a_off[2] = r_in >> (a_tile_lg[0] + a_tile_lg[1]);
  // Row of the tensors / index into lse and delta: position in the permuted sequence, or the
  // token of the lane's coordinate in the original layout.
  // (original layout: a row past an end of its dilation group works on the group's first or last row and stores nothing)
  int a_crd[3];
  bool a_valid = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int c = a_first[a] + a_off[a];
    const int e = KV_STATIONARY ? extent[a] : q_extent[a];
    a_valid = a_valid && ((c >= 0 && c < e) || !(RAGGED || p.fused));
    a_crd[a] = (RAGGED || p.fused) ? na_max(na_min(c, e - 1), 0) : c;
  }
  const int a_tok = group_tok + a_crd[0] * tok_step[0] + a_crd[1] * tok_step[1] + a_crd[2] * tok_step[2];
  const int64_t batch_row0 = p.fused ? int64_t(b_orig) * p.tokens : 0;  // first row of the batch entry (original layout)
  const int a_seq_row = RAGGED ? a_crd[0] : at * AT + r_in;  // its row of the permuted / ragged sequence
  const int64_t a_row = p.fused ? batch_row0 + a_tok : seq_row_a + a_seq_row;
  const int64_t a_stride = int64_t(heads_a) * D;
  const int64_t b_stride = int64_t(heads_b) * D;
  const float kLog2e = 1.4426950408889634f;

  // Stationary operand fragments: row r_in, elements 16*ks + 8*g .. +7 (paired role: K for the P waves, V
  // for the dS waves).  On their way from here on, and scaled (dQ role) once everything else is set up.
  const T* x1 = reinterpret_cast<const T*>(KV_STATIONARY ? ((PAIR && part) ? p.v : p.k) : p.q) + a_row * a_stride +
                int64_t(head_a) * D + g * 8;
  const T* x2 = reinterpret_cast<const T*>(KV_STATIONARY ? p.v : p.d_out) + a_row * a_stride + int64_t(head_a) * D + g * 8;
  constexpr bool FIRST = ROLE == kBwdDQ && RAW;
  vec8 x1f[KSTEPS], x2f[HAS_DS ? KSTEPS : 1], of[FIRST ? KSTEPS : 1];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    x1f[ks] = *reinterpret_cast<const vec8*>(x1 + ks * 16);
    if constexpr (HAS_DS) x2f[ks] = *reinterpret_cast<const vec8*>(x2 + ks * 16);
    if constexpr (FIRST)
      of[ks] = *reinterpret_cast<const vec8*>(reinterpret_cast<const T*>(p.out) + a_row * a_stride + int64_t(head_a) * D + g * 8 + ks * 16);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- which streamed rows meet -----------------------------------------------------------------------
  // Along every dimension the streamed rows that pair with a stationary row are an interval (the window of a
  // query; the queries whose windows hold a key), monotone in the row, so that the tile's first and last
  // rows give the box of streamed tiles it meets, and the inner box of those every row of which pairs with
  // every row of the tile (no mask needed).  One evaluation per dimension serves all of it: the lower half of
  // the wave takes its lanes' rows (the lanes of the upper half, which hold the same ones, get the results
  // from there), lane 32 the tile's first row inside the extent, lane 33 its last one inside the extent, lane 34 its last one.
  // A workgroup's first step began after 10000 cycles: the loads of the launch parameters one behind the other, 18
  // evaluations of which 12 on the scalar unit, and the tables before the first copies.  dK / dV and dQ launches,
  // us before / after: 4 x 56 x 56, 7 x 7, H 8, D 32 41.4 / 39.0 and 32.4 / 31.3; 56 x 56, H 32, D 64 56.2 / 53.7 and 43.2 / 42.7;
  // 96 x 96, 24 x 24, stride 8, H 8, D 64 51.0 / 48.8 and 37.4 / 36.6; dense 2 x 1000, H 8, D 128 33.6 / 32.4 and 30.5 / 29.0.  Large
  // launches of head dim 128 run at the card's power limit and take as long as before.
  int win_lo[3], win_hi[3];  // the rows win_lo .. win_hi - 1 pair with the lane's
  int box_tile0[3], box_n[3], full_t0[3], full_t1[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int e = KV_STATIONARY ? extent[a] : q_extent[a];
    const int last = a_first[a] + a_tile[a] - 1, last_in = na_max(na_min(last, e - 1), 0);
    const int c = g == 0 ? a_crd[a] : l32 == 0 ? na_max(a_first[a], 0) : l32 == 1 ? last_in : last;
    const bool cs = p.causal[a] != 0;
    int from, upto;
    if constexpr (!KV_STATIONARY) {
      from = na_window_start(c, ksz[a], p.stride[a], p.d_stride[a], extent[a], cs);
      upto = na_window_end(c, from, ksz[a], extent[a], cs);
    } else {
      from = na_first_query_attending(c, ksz[a], p.stride[a], p.d_stride[a], q_extent[a], cs);
      upto = na_last_query_attending(c, ksz[a], p.stride[a], p.d_stride[a], extent[a], q_extent[a], cs) + 1;
      if (c >= extent[a]) upto = from;  // a padding key of a permuted sequence: nothing attends it
    }
    win_lo[a] = lower_half(from);
    win_hi[a] = lower_half(upto);
    const int first_from = __builtin_amdgcn_readlane(from, 32), first_upto = __builtin_amdgcn_readlane(upto, 32);
    int hi = __builtin_amdgcn_readlane(upto, 33) - 1;
    if (KV_STATIONARY && first_from > hi) empty = true;
    const int lo = na_max(first_from, 0);
    hi = na_max(hi, lo);
    box_tile0[a] = lo >> b_sub_lg[a];
    box_n[a] = (hi >> b_sub_lg[a]) + 1 - box_tile0[a];
    // Whole tiles: streamed coordinates flo .. fhi pair with all stationary ones.  dQ: rows past the extent use the
    // last window.  Key-stationary: rows past the end that are not stored may take part, only zero-padded
    // sequences need their mask.
    int flo = __builtin_amdgcn_readlane(from, (KV_STATIONARY && (RAGGED || p.fused)) ? 33 : 34), fhi = first_upto - 1;
    if (KV_STATIONARY && !(RAGGED || p.fused) && last >= e) {
      flo = 1;  // the tile holds padding keys: never whole
      fhi = 0;
    }
    full_t0[a] = na_max((na_max(flo, 0) + b_sub[a] - 1) >> b_sub_lg[a], box_tile0[a]);
    full_t1[a] = na_min((fhi + 1) >> b_sub_lg[a], box_tile0[a] + box_n[a]);  // one past the last whole tile
    if (fhi < 0 || full_t1[a] < full_t0[a]) full_t1[a] = full_t0[a];
  }

  auto store_rows = [&](void* dst, const f32x16_t (&acc)[DB], float mul) {
    T* orow = reinterpret_cast<T*>(dst) + a_row * a_stride + int64_t(head_a) * D;
    store_row_blocks<T, DB>(orow, acc, mul, g, a_valid, D);
  };
  auto store_results = [&](const f32x16_t (&a1)[DB], const f32x16_t (&a2)[DB], float scale1) {
    if constexpr (ROLE == kBwdDQ) store_rows(p.dq, a1, scale1);
    if constexpr (ROLE == kBwdDKV) store_rows(p.dk, a1, scale1);
    if constexpr (PAIR) {
      if (part) store_rows(p.dk, a2, scale1);  // a dS wave accumulates dK where a P wave accumulates dV
      else store_rows(p.dv, a2, scale1 == 0.f ? 0.f : 1.f);
    } else if constexpr (HAS_PV) {
      store_rows(p.dv, a2, scale1 == 0.f ? 0.f : 1.f);
    }
  };

  f32x16_t acc1[DB], acc2[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc1[db][r] = acc2[db][r] = 0.f;

  if (empty) {
    // padding rows, or rows nothing attends: their gradients are zero
    store_results(acc1, acc2, 0.f);
    return;
  }

  // ---- streamed tiles ---------------------------------------------------------------------------
  const T* y1_all = reinterpret_cast<const T*>(KV_STATIONARY ? p.qs : p.k);
  const T* y2_all = reinterpret_cast<const T*>(KV_STATIONARY ? p.d_out : p.v);

  // row (permuted) or token offset (original layout) of position r (dimension 0 fastest) of a streamed tile
  auto sub_pos = [&](int r) {
    if (!p.fused) return r;
    const int t0 = r & (b_sub[0] - 1);
    r >>= b_sub_lg[0];
    return t0 * tok_step[0] + (r & (b_sub[1] - 1)) * tok_step[1] + (r >> b_sub_lg[1]) * tok_step[2];
  };
  // copy i of a thread moves chunk P = i * NT + tid of the tile (row P / CPR, LDS slot P % CPR)
  uint32_t off_u[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int P = i * NT + tid;
    const int row = P / CPR, slot = P % CPR;
    off_u[i] = uint32_t(sub_pos(row)) * uint32_t(b_stride * 2) + uint32_t(L::u_slot(row, slot) * 16);
  }

  // The streamed tiles in visiting order: the box of tiles the stationary tile meets, dimension 2 fastest,
  // dimension 0 slowest; the key-stationary roles walk it once per query head of the key head's group.
  // First the tiles that need the element mask (the box minus the inner box of whole tiles, see
  // full_t0), then the whole ones: one sequence, but each kind has a loop body of its own.
  // Descriptors are formed 64 box positions at a time, one per lane, and read back by lane number: a
  // tile costs the wave a handful of scalar instructions (a scalar walk of the box with its edge cases
  // took some seventy, every one an issue slot of a wave that also feeds the matrix pipe).
  struct Tile {
    int row0;       // its first row in the streamed side's sequence / its token in the dilation group's batch entry
    int head_b;
    int origin[3];  // coordinate of its first row (a tile moved back from the group's edge: of the first one gathered)
    int lead;       // ... whose first (lead >> 8 a) & 255 positions along dimension a belong to the tile before it
  };
  const int total = box_n[0] * box_n[1] * box_n[2];
  const int heads_walked = KV_STATIONARY ? rep : 1;
  const int n_whole = (full_t1[0] - full_t0[0]) * (full_t1[1] - full_t0[1]) * (full_t1[2] - full_t0[2]);
  const int n_masked = (total - n_whole) * heads_walked;  // the first n_masked of the n_iter tiles need the mask
  const int n_iter = total * heads_walked;
  const int head_b0 = KV_STATIONARY ? head_a * rep : na_div(head_a, p.d_rep);
  const float inv_n1 = 1.f / float(box_n[1]), inv_n2 = 1.f / float(box_n[2]);
  int walk = -64, walk_head = -1;  // first of the 64 positions described, query head of the group
  bool walk_whole = n_masked == 0;
  int r_row0 = 0, r_origin[3] = {0, 0, 0}, r_lead = 0;
  uint64_t whole_bits = 0, todo = 0;  // of the positions described: the whole tiles, the tiles still to visit
  auto load_descriptors = [&]() __attribute__((always_inline)) {
    // quotient by a rounded reciprocal, then put right (positions are far below 2^24)
    auto divide = [](int n, int d, float inv, int& rem) __attribute__((always_inline)) {
      int q = int(float(n) * inv);
      rem = n - q * d;
      if (rem < 0) {
        --q;
        rem += d;
      } else if (rem >= d) {
        ++q;
        rem -= d;
      }
      return q;
    };
    int t[3];
    const int rest = divide(na_min(walk + lane, total - 1), box_n[2], inv_n2, t[2]);
    t[0] = divide(rest, box_n[1], inv_n1, t[1]);
    bool whole = true;
    int cc[3], half = 0;
    r_lead = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      t[a] += box_tile0[a];
      whole = whole && t[a] >= full_t0[a] && t[a] < full_t1[a];
      const int org = t[a] << b_sub_lg[a];
      r_origin[a] = p.edge ? na_min(org, (KV_STATIONARY ? q_extent[a] : extent[a]) - b_sub[a]) : org;
      r_lead |= (org - r_origin[a]) << (8 * a);
      const bool split = (a == split_dim);
      half |= split ? (t[a] & 1) : 0;
      cc[a] = split ? (t[a] >> 1) : t[a];
    }
    r_row0 = p.fused ? group_tok + r_origin[0] * tok_step[0] + r_origin[1] * tok_step[1] + r_origin[2] * tok_step[2]
                     : (cc[0] + b_tiled[0] * (cc[1] + b_tiled[1] * cc[2])) * AT + half * BT;
    whole_bits = __ballot(whole);
  };
  auto next_tile = [&]() __attribute__((always_inline)) {
    while (todo == 0) {  // (called while tiles remain: some position ahead has one)
      walk += 64;
      if (walk_head < 0 || walk >= total) {
        walk = 0;
        if (++walk_head == heads_walked) {
          walk_head = 0;
          walk_whole = true;
        }
        if (total > 64 || whole_bits == 0) load_descriptors();
      } else {
        load_descriptors();
      }
      todo = walk_whole ? whole_bits : ~whole_bits;
      if (total - walk < 64) todo &= (uint64_t(1) << (total - walk)) - 1;
    }
    const int l = __builtin_ctzll(todo);
    todo &= todo - 1;
    Tile t;
    t.row0 = __builtin_amdgcn_readlane(r_row0, l);
    t.head_b = head_b0 + walk_head;
#pragma unroll
    for (int a = 0; a < 3; ++a) t.origin[a] = __builtin_amdgcn_readlane(r_origin[a], l);
    t.lead = __builtin_amdgcn_readlane(r_lead, l);
    return t;
  };
  // bit 16 sb + r: the lane's logit r of sub-block sb belongs to an attended pair
  auto pair_bits = [&](const Tile& t) __attribute__((always_inline)) {
    uint32_t from[3], upto[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int lead = (t.lead >> (8 * a)) & 255;
      from[a] = sRows[a][g][na_min(na_max(win_lo[a] - t.origin[a], lead), b_sub[a])];
      upto[a] = sRows[a][g][na_min(na_max(win_hi[a] - t.origin[a], 0), b_sub[a])];
    }
    return from[0] & ~upto[0] & from[1] & ~upto[1] & from[2] & ~upto[2];
  };

  const uint32_t lds_y1 = uint32_t(__builtin_amdgcn_readfirstlane(int(lds_address(sY1))));
  const uint32_t lds_y2 = uint32_t(__builtin_amdgcn_readfirstlane(int(lds_address(sY2))));
  const uint32_t stat_off = uint32_t(sub_pos(lane)) * 4u;  // byte offset of streamed row `lane` in lse / delta (head-major)
  // the asynchronous copies of a streamed tile (and of its LSE / delta values) into a stage
  auto issue_copies = [&](const Tile& t, int stage, int stage2) {
    const int64_t row = p.fused ? batch_row0 + t.row0 : seq_row_b + t.row0;
    // a tile that ends past its sequence: the rows from `last` on are the sequence's last one
    const int last = (KV_STATIONARY ? q_extent[0] : extent[0]) - 1 - t.origin[0];
    const bool partial = RAGGED && last < BT - 1;
    if constexpr (KV_STATIONARY) {
      // LSE / delta of the tile's 64 queries: one asynchronous 4-byte-per-lane copy each
      // (wave 1, wave 2; the other waves but wave 0 make the same number of copies into a
      // spare row so that every wave counts the same number of outstanding copies per tile)
      const int64_t stat_row0 = p.fused ? (int64_t(b_orig) * p.heads_q + t.head_b) * p.tokens + t.row0
                                        : stat_row_q + t.head_b * stat_head_stride + t.row0;
      const float* src = (wave == 2 ? p.delta : p.lse) + stat_row0;
      float* dst = (wave == 1) ? &sLse[stage * BT] : (wave == 2) ? &sDelta[stage * BT] : &sSpare[0];
      const uint32_t off = partial ? uint32_t(na_min(lane, last)) * 4u : stat_off;
      if (wave != 0) async_copy4_asm(src, off, lds_address(dst));
    }
    const int64_t elem = row * b_stride + int64_t(t.head_b) * D;
    const uint64_t y1 = uniform64(y1_all + elem), y2 = uniform64(y2_all + elem);
    const uint32_t dst = uint32_t(__builtin_amdgcn_readfirstlane(stage * TILE_BYTES + wave * 1024));
    const uint32_t dst2 = uint32_t(__builtin_amdgcn_readfirstlane(stage2 * TILE_BYTES + wave * 1024));
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      uint32_t off = off_u[i];
      if constexpr (RAGGED) {
        if (partial) off -= uint32_t(na_max((i * NT + tid) / CPR - last, 0)) * uint32_t(b_stride * 2);
      }
      async_copy16_uniform(y1, off, lds_y1 + dst + uint32_t(i * NT * 16));
      async_copy16_uniform(y2, off, lds_y2 + dst2 + uint32_t(i * NT * 16));
    }
  };
  // LDS reads of operand fragments (same fragment layouts as the forward kernel): row l32, chunk 2 ks + g, and transposed
  // rows 4 g + e [+ 8], chunk 4 db + v_chunk.  The chunk numbers differ by exclusive or as the swizzle does, and stages begin at
  // multiples of a row of chunks, so that every fragment's address is one lane offset with a few bits turned over: an
  // instruction each where it is used, as an addition to the stage's base would be, and two registers instead of
  // sixteen (head dim 128: the paired role 246 -> 216, the dQ role 256 and 9 spilled -> 244, with three fragments read
  // ahead 248).
  const uint32_t k_lane = uint32_t(l32 * ROWB + L::u_slot(l32, g) * 16);
  const int l16 = lane & 15;
  const int v_e = l16 >> 2, v_j4 = l16 & 3;
  const int v_row = 4 * g + v_e;
  const int v_chunk = (l32 >> 4) * 2 + (v_j4 >> 1);
  const uint32_t v_lane = uint32_t(v_row * ROWB + L::u_slot(v_row, v_chunk) * 16 + (v_j4 & 1) * 8);
  // `s`: LDS address of the stage
  auto row_frag = [&](uint32_t s, int sb, int ks) __attribute__((always_inline)) {
    return *lds_pointer<vec8>(((s + k_lane) ^ uint32_t(ks * 32)) + uint32_t(sb * 32 * ROWB));
  };
  // transposed fragment: sub-block sb, 16-row half h, 32-column block db
  auto tr_frag = [&](uint32_t s, int sb, int h, int db) __attribute__((always_inline)) {
    const uint32_t at = (s + v_lane) ^ uint32_t(db * 64), row0 = uint32_t((sb * 32 + h * 16) * ROWB);
    const s16x4_t lo = lds_read_tr16(at + row0);
    const s16x4_t hi = lds_read_tr16((at ^ 32u) + row0 + 8 * ROWB);
    return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // The first tiles' copies are on their way while the rest is set up: two tiles ahead in the paired role and with
  // three stages, one with two.
  constexpr int CPT = 2 * PER;  // tile copies per thread and tile
  constexpr int AHEAD = NS == 3 ? 2 : 1;
  const Tile tile0 = next_tile();
  issue_copies(tile0, 0, 0);
  Tile tile1 = tile0;
  if (AHEAD > 1 && 1 < n_iter) {
    tile1 = next_tile();
    issue_copies(tile1, 1, 1);
  }
  if (wave < 3) {
    // one row per lane and, by wave, one dimension (the row past the extent holds nothing)
    const int lg_stride = wave == 0 ? 0 : wave == 1 ? b_sub_lg[0] : b_sub_lg[0] + b_sub_lg[1];
    const int lg = wave == 0 ? b_sub_lg[0] : wave == 1 ? b_sub_lg[1] : b_sub_lg[2];
    const uint64_t rows = na_keys_at_or_after(na_min(lane, 1 << lg), lg_stride, lg);
    sRows[wave][0][lane] = na_lane_half_bits(rows, 0);
    sRows[wave][1][lane] = na_lane_half_bits(rows, 1);
    if (lane == 0) sRows[wave][0][BT] = sRows[wave][1][BT] = 0;
  }
  // Accumulator inputs of the first matrix instruction of a logit / dP block: -log2e LSE and -delta of
  // the block's queries, so that P = exp2(S) and dS = P dP are what the matrix pipe returns.  In the
  // key-stationary roles they differ by row and come from the tile's table in LDS; in the dQ role they
  // are the lane's own, sixteen copies of them where the registers allow (head dims below 128).
  constexpr bool INIT_REGS = !KV_STATIONARY && D < 128;
  float lse_l = 0.f, delta_l = 0.f;
  if constexpr (!KV_STATIONARY) {
    const int64_t stat_idx = p.fused ? (int64_t(b_orig) * p.heads_q + head_a) * p.tokens + a_tok
                                     : stat_row_q + head_a * stat_head_stride + a_seq_row;
    if constexpr (FIRST) {
      // (added up as delta_kernel does: eight elements in order, then halves of the row)
      float sum[KSTEPS];
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) sum[ks] = dot8<T>(of[ks], x2f[ks]);
#pragma unroll
      for (int o = KSTEPS / 2; o > 0; o >>= 1)
#pragma unroll
        for (int ks = 0; ks < o; ++ks) sum[ks] += sum[ks + o];
      delta_l = -(sum[0] + __shfl_xor(sum[0], 32));
      lse_l = -kLog2e * p.lse_rows[a_row * heads_a + head_a];
    } else {
      lse_l = p.lse[stat_idx] * p.lse_mul;
      delta_l = p.delta[stat_idx] * p.delta_mul;
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) x1f[ks] = scale_query_fragment<T>(x1f[ks], p.scale * kLog2e);
  }
  f32x16_t lse_init, delta_init;
  if constexpr (INIT_REGS) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      lse_init[r] = lse_l;
      delta_init[r] = delta_l;
    }
  }


  // One streamed tile: its two 32-row sub-blocks one after the other, each as products (S, dP),
  // probabilities, accumulations.  Only one sub-block's products are live at a time, which keeps
  // the kernel within 256 registers: two workgroups share a CU, and the other wave of a SIMD
  // fills the gaps of this one (a measured 1.2-1.3 x over interleaving the sub-blocks inside
  // one wave per SIMD).  The matrix instructions form one sequence of fenced "slots", each with
  // its operand fragment read from LDS a few slots ahead.
  constexpr int WP = HAS_DS ? 2 : 1;                       // products per k-step (S, dP)
  constexpr int W = (HAS_DS ? 1 : 0) + (HAS_PV ? 1 : 0);   // accumulators fed per transposed fragment position
  constexpr int NP = WP * KSTEPS;                          // product slots per sub-block
  constexpr int N1 = 2 * NP;
  constexpr int NC = 2 * DB * W;                           // accumulation slots per sub-block
  constexpr int G = N1 + 2 * NC;
  // fragments read ahead (dQ at head dim 128, two / three: 29 x 46 x 78, 9 x 24 x 24, H 8 4.36 / 4.30 ms; others level)
  constexpr int PF = D == 128 && !KV_STATIONARY ? 3 : 2;
  // P waves of the paired role: the products of both sub-blocks first, then the accumulations of
  // both, and the probabilities of a sub-block two per slot between the matrix instructions that
  // follow its products (sub-block 0: the products of sub-block 1; sub-block 1: the accumulations
  // of sub-block 0), so that the wave's vector work runs while the matrix pipe does.
  constexpr bool SPREAD = PAIR;
  static_assert(!SPREAD || (NP == 8 && NC == 8), "two of a sub-block's 16 probabilities per slot");
  auto tile_body = [&](auto masked_tag, int stage, int stage2, uint32_t bits, int exch, auto&& after_slot) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    (void)exch;  // paired role: which of the two probability buffers this tile writes
    const uint32_t y1 = lds_y1 + uint32_t(stage * TILE_BYTES);
    const uint32_t y2 = lds_y2 + uint32_t(stage2 * TILE_BYTES);  // (stage2 differs from stage in the paired role only)

    // slot x of the tile: a product slot (sub-block, index i < NP) or an accumulation slot (i < NC)
    struct Slot {
      bool prod;
      int sb, i;
    };
    auto slot_of = [](int x) constexpr {
      if constexpr (SPREAD) {
        const bool prod = x < 2 * NP;
        const int z = prod ? x : x - 2 * NP, n = prod ? NP : NC;
        return Slot{prod, z / n, z % n};
      } else {
        const int sb = x / (NP + NC), z = x % (NP + NC);
        return Slot{z < NP, sb, z < NP ? z : z - NP};
      }
    };
    auto frag = [&](auto x_tag) {
      constexpr Slot sl = slot_of(decltype(x_tag)::value);
      if constexpr (sl.prod) {
        constexpr int ks = sl.i / WP, which = sl.i % WP;
        return row_frag(which ? y2 : y1, sl.sb, ks);
      } else {
        constexpr int h = sl.i / (DB * W), db = (sl.i / W) % DB;
        constexpr bool to_acc1 = HAS_DS && (sl.i % W == 0);
        return tr_frag(to_acc1 ? y1 : y2, sl.sb, h, db);
      }
    };

    f32x16_t S[NSB], dP[NSB];
    vec8 pf[NSB][2], dsf[NSB][2];
    // the rows 8*jj + 4*g + i of sub-block sb (logit r = 4 jj + i) of a per-row table
    auto init_from = [&](const float* table, float mul, int sb) __attribute__((always_inline)) {
      f32x16_t c;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&table[stage * BT + sb * 32 + 8 * jj + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) c[4 * jj + i] = RAW ? v[i] * mul : v[i];
      }
      return c;
    };
    auto load_inits = [&](auto sb_tag) __attribute__((always_inline)) {
      constexpr int sb = decltype(sb_tag)::value;
      if constexpr (KV_STATIONARY && sb < NSB) {
        S[sb] = init_from(sLse, -kLog2e, sb);
        if constexpr (HAS_DS) dP[sb] = init_from(sDelta, -1.f, sb);
      }
    };
    float held_p = 0.f, held_ds = 0.f;
    uint32_t px[PAIR ? 8 : 1];  // paired role: the sub-block's probabilities as fp16 pairs
    auto elem = [&](auto sb_tag, auto r_tag) {
      constexpr int sb = decltype(sb_tag)::value, r = decltype(r_tag)::value;
      float x = fast_exp2((KV_STATIONARY || INIT_REGS) ? S[sb][r] : S[sb][r] + lse_l);
      if constexpr (MASKED) {
        // 0 or ~0 (as assembly: from the builtin the compiler forms a test of the bit and a select)
        uint32_t keep;
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(keep) : "v"(bits), "n"(16 * sb + r));
        x = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & keep);
      }
      float ds = 0.f;
      if constexpr (HAS_DS) ds = x * ((KV_STATIONARY || INIT_REGS) ? dP[sb][r] : dP[sb][r] + delta_l);
      if constexpr (r % 2 == 0) {
        pin(x);
        held_p = x;
        if constexpr (HAS_DS) {
          pin(ds);
          held_ds = ds;
        }
      } else {
        if constexpr (PAIR) {
          const h16x2_t h2 = {static_cast<_Float16>(held_p), static_cast<_Float16>(x)};
          px[r / 2] = __builtin_bit_cast(uint32_t, h2);
          if constexpr (r == 15) {
            char* dst = sX + ((((exch * 4 + rw) * NSB + sb) * 2) * 64 + lane) * 16;
            *reinterpret_cast<u32x4_t*>(dst) = u32x4_t{px[0], px[1], px[2], px[3]};
            *reinterpret_cast<u32x4_t*>(dst + 64 * 16) = u32x4_t{px[4], px[5], px[6], px[7]};
          }
        }
        if constexpr (HAS_PV) {
          vec2 p2 = {static_cast<T>(held_p), static_cast<T>(x)};
          uint32_t pb = __builtin_bit_cast(uint32_t, p2);
          pin(pb);
          p2 = __builtin_bit_cast(vec2, pb);
          pf[sb][r / 8][r % 8 - 1] = p2[0];
          pf[sb][r / 8][r % 8] = p2[1];
        }
        if constexpr (HAS_DS) {
          vec2 d2 = {static_cast<T>(held_ds), static_cast<T>(ds)};
          uint32_t db_ = __builtin_bit_cast(uint32_t, d2);
          pin(db_);
          d2 = __builtin_bit_cast(vec2, db_);
          dsf[sb][r / 8][r % 8 - 1] = d2[0];
          dsf[sb][r / 8][r % 8] = d2[1];
        }
      }
    };

    vec8 fr[G];
    load_inits(std::integral_constant<int, 0>{});
    for_range<0, PF>([&](auto x_tag) { fr[decltype(x_tag)::value] = frag(x_tag); });
    for_range<0, G>([&](auto x_tag) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value;
      constexpr Slot sl = slot_of(x);
      constexpr int sb = sl.sb;
      if constexpr (x + PF < G) fr[x + PF] = frag(std::integral_constant<int, x + PF>{});
      if constexpr (sl.prod) {
        constexpr int ks = sl.i / WP, which = sl.i % WP;
        if constexpr (ks == 0 && !KV_STATIONARY) {
          if constexpr (INIT_REGS) {
            if constexpr (which == 0) S[sb] = M::run_from(fr[x], x1f[ks], lse_init);
            else dP[sb] = M::run_from(fr[x], x2f[ks], delta_init);
          } else {
            f32x16_t zero;
#pragma unroll
            for (int r = 0; r < 16; ++r) zero[r] = 0.f;
            if constexpr (which == 0) S[sb] = M::run(fr[x], x1f[ks], zero);
            else dP[sb] = M::run(fr[x], x2f[ks], zero);
          }
        } else {
          if constexpr (which == 0) S[sb] = M::run(fr[x], x1f[ks], S[sb]);
          else dP[sb] = M::run(fr[x], x2f[ks], dP[sb]);
        }
        // the accumulator inputs of the other sub-block's products, a few slots before these begin
        if constexpr (SPREAD && sb == 0 && sl.i == NP - 3) load_inits(std::integral_constant<int, 1>{});
        // all probabilities of the sub-block once its products are complete
        if constexpr (!SPREAD && sl.i == NP - 1) for_range<0, 16>([&](auto r_tag) { elem(std::integral_constant<int, sb>{}, r_tag); });
      } else {
        constexpr int h = sl.i / (DB * W), db = (sl.i / W) % DB;
        constexpr bool to_acc1 = HAS_DS && (sl.i % W == 0);
        if constexpr (to_acc1) acc1[db] = M::run(fr[x], dsf[sb][h], acc1[db]);
        else acc2[db] = M::run(fr[x], pf[sb][h], acc2[db]);
        if constexpr (!SPREAD && sb == 0 && sl.i == NC - 3) load_inits(std::integral_constant<int, 1>{});
      }
      if constexpr (SPREAD && x >= NP && x < 2 * NP + NC) {
        // two probabilities per slot, between the matrix instructions of the other sub-block
        constexpr int esb = x < 2 * NP ? 0 : 1, r0 = 2 * (x < 2 * NP ? x - NP : x - 2 * NP);
        elem(std::integral_constant<int, esb>{}, std::integral_constant<int, r0>{});
        elem(std::integral_constant<int, esb>{}, std::integral_constant<int, r0 + 1>{});
      }
      after_slot(x_tag);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // ---- paired role: the dS waves ----------------------------------------------------------------
  // produce: dP^T of the current tile, kept in registers until the next step;
  // consume: dS of the previous tile from its dP^T, its delta and the P waves' probabilities,
  // then dK += dS^T Q with that tile's Q (still in its stage).
  f32x16_t held_dp[NSB];
  auto pair_produce = [&](int stage1, int stage) __attribute__((always_inline)) {
    const uint32_t y2 = lds_y2 + uint32_t(stage * TILE_BYTES);
    constexpr int N = NSB * KSTEPS;
    vec8 fr[N];
    // the products start from -delta of the tile's queries (tables live in the stages of Y1)
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(&sDelta[stage1 * BT + sb * 32 + 8 * jj + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) held_dp[sb][4 * jj + i] = RAW ? -v[i] : v[i];
      }
    for_range<0, PF>([&](auto x_tag) {
      constexpr int x = decltype(x_tag)::value;
      fr[x] = row_frag(y2, x / KSTEPS, x % KSTEPS);
    });
    for_range<0, N>([&](auto x_tag) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value;
      constexpr int sb = x / KSTEPS, ks = x % KSTEPS;
      if constexpr (x + PF < N) fr[x + PF] = row_frag(y2, (x + PF) / KSTEPS, (x + PF) % KSTEPS);
      held_dp[sb] = M::run(fr[x], x1f[ks], held_dp[sb]);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto pair_consume = [&](int stage, int exch) __attribute__((always_inline)) {
    const uint32_t y1 = lds_y1 + uint32_t(stage * TILE_BYTES);
    vec8 dsf[NSB][2];
    u32x4_t plo[NSB], phi[NSB];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
      const char* src = sX + ((((exch * 4 + rw) * NSB + sb) * 2) * 64 + lane) * 16;
      plo[sb] = *reinterpret_cast<const u32x4_t*>(src);
      phi[sb] = *reinterpret_cast<const u32x4_t*>(src + 64 * 16);
    }
    // dS values 2 k and 2 k + 1 of a sub-block: the probabilities as they lie in the word, times dP
    auto ds_pair = [&](auto sb_tag, auto k_tag) {
      constexpr int sb = decltype(sb_tag)::value, r = 2 * decltype(k_tag)::value;
      const uint32_t pw = (r < 8) ? plo[sb][r / 2] : phi[sb][r / 2 - 4];
      // (as multiply-adds: one mixed-precision instruction each instead of a conversion and a product)
      const h16x2_t h2 = __builtin_bit_cast(h16x2_t, pw);
      const vec2 d2 = {static_cast<T>(__builtin_fmaf(float(h2[0]), held_dp[sb][r], 0.f)),
                       static_cast<T>(__builtin_fmaf(float(h2[1]), held_dp[sb][r + 1], 0.f))};
      dsf[sb][r / 8][r % 8] = d2[0];
      dsf[sb][r / 8][r % 8 + 1] = d2[1];
    };
    constexpr int NCB = 2 * DB;  // accumulation slots per sub-block
    constexpr int N = NSB * NCB;
    static_assert(!PAIR || NCB == 8, "one pair of dS values of sub-block 1 per accumulation slot of sub-block 0");
    vec8 fr[N];
    for_range<0, PF>([&](auto x_tag) {
      constexpr int x = decltype(x_tag)::value;
      fr[x] = tr_frag(y1, x / NCB, (x % NCB) / DB, x % DB);
    });
    for_range<0, 8>([&](auto k_tag) { ds_pair(std::integral_constant<int, 0>{}, k_tag); });
    __builtin_amdgcn_sched_barrier(0);
    for_range<0, N>([&](auto x_tag) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value;
      constexpr int sb = x / NCB, h = (x % NCB) / DB, db = x % DB;
      if constexpr (x + PF < N) {
        constexpr int y = x + PF;
        fr[y] = tr_frag(y1, y / NCB, (y % NCB) / DB, y % DB);
      }
      acc2[db] = M::run(fr[x], dsf[sb][h], acc2[db]);
      if constexpr (PAIR && x < NCB) ds_pair(std::integral_constant<int, 1>{}, x_tag);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // The stationary fragments have landed from here on, as the compiler sees it too: left to the first product of the loop,
  // the wait for them (a countdown to vmcnt(0)) stands in every step, where it also waits for the tile copies just issued.
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    asm volatile("" : "+v"(x1f[ks]));
    if constexpr (HAS_DS) asm volatile("" : "+v"(x2f[ks]));
  }
  workgroup_sync();  // sRows is written
  // The paired role over n_iter tiles: step `it` has the P waves on tile `it` and the dS waves forming
  // dP of tile `it` after finishing tile it - 1; one more step drains the dS waves.  Tiles are copied
  // two steps ahead: tile it + 2 during step `it`, into the Y2 stage of tile it - 1 and the Y1 / table
  // stage of tile it - 2, both last read in step it - 1.  The barrier at the top of a step makes tile
  // `it` and the probabilities of tile it - 1 visible and separates those last reads from the
  // copies that overwrite them.
  auto run_pair = [&](auto ds_wave_tag) __attribute__((always_inline)) {
    constexpr bool DS_WAVE = decltype(ds_wave_tag)::value;
    uint32_t bits0 = 0, bits1 = 0, bits2 = 0;  // P waves: attended pairs of the tiles it, it + 1, it + 2 (while masked)
    if constexpr (!DS_WAVE) {
      bits0 = pair_bits(tile0);
      bits1 = pair_bits(tile1);  // (of tile 0 again, never used, where it is the only one)
    }
    // A wave walks to tile it + 2 and issues its share of the copies where it has vector or
    // scalar work anyway: the dS waves between their two matrix phases, the P waves after the
    // products of their first sub-block; the eight waves then do not queue on the CU's address
    // path together while the matrix pipe idles.
    int s2 = 0;  // it % 3
    auto step = [&](auto masked_tag, int it) __attribute__((always_inline)) {
      constexpr bool MASKED = decltype(masked_tag)::value;
      // this thread's copies of tile `it` have landed once only those of tile it + 1 are
      // outstanding (wave 0 makes one copy less per tile)
      if (it + 1 < n_iter) {
        if (wave != 0) wait_vmcnt<CPT + 1>();
        else wait_vmcnt<CPT>();
      } else {
        wait_vmcnt<0>();
      }
      workgroup_sync();
      const int s2_ahead = s2 == 0 ? 2 : s2 - 1;  // (it + 2) % 3
      auto ahead = [&]() __attribute__((always_inline)) {
        if (it + 2 < n_iter) {
          const Tile t = next_tile();
          issue_copies(t, (it + 2) & 3, s2_ahead);
          if constexpr (MASKED && !DS_WAVE) bits2 = pair_bits(t);
        }
      };
      if constexpr (DS_WAVE) {
        if (it > 0) pair_consume((it - 1) & 3, (it - 1) & 1);
        ahead();
        if (it < n_iter) pair_produce(it & 3, s2);
      } else {
        tile_body(masked_tag, it & 3, s2, bits0, it & 1, [&](auto x_tag) __attribute__((always_inline)) {
          if constexpr (decltype(x_tag)::value == NP - 1) ahead();
        });
        if constexpr (MASKED) {
          bits0 = bits1;
          bits1 = bits2;
        }
      }
      s2 = s2 == 2 ? 0 : s2 + 1;
    };
    if constexpr (DS_WAVE) {
      for (int it = 0; it <= n_iter; ++it) step(std::false_type{}, it);
    } else {
      int it = 0;
      for (; it < n_masked; ++it) step(std::true_type{}, it);
      for (; it < n_iter; ++it) step(std::false_type{}, it);
      workgroup_sync();  // the step in which the dS waves finish the last tile
    }
  };

  // ---- the other roles: tile `it` is multiplied while tiles it+1 .. it+NS-1 are in flight ----------
  auto run_tiles = [&]() __attribute__((always_inline)) {
    uint32_t bits0 = 0, bits1 = 0, bits2 = 0;  // attended pairs of the tiles it, it + 1, it + 2 (while masked)
    auto issue_next = [&](int stage) __attribute__((always_inline)) {
      const Tile t = next_tile();
      issue_copies(t, stage, stage);
      return t;
    };
    bits0 = pair_bits(tile0);
    if (NS > 2) bits1 = pair_bits(tile1);
    int stage = 0;  // it % NS
    auto step = [&](auto masked_tag, int it) __attribute__((always_inline)) {
      constexpr bool MASKED = decltype(masked_tag)::value;
      // this thread's copies of tile `it` have landed once at most those of the later tiles in
      // flight (one tile with three stages, none with two) are outstanding; wave 0 makes one
      // copy less per tile in the key-stationary roles
      if (NS == 3 && it + 1 < n_iter) {
        if (KV_STATIONARY && wave != 0) wait_vmcnt<CPT + 1>();
        else wait_vmcnt<CPT>();
      } else {
        wait_vmcnt<0>();
      }
      workgroup_sync();  // tile `it` and its tables are in LDS; everyone is done with the stage of tile it - 1
      if (it + NS - 1 < n_iter) {
        const Tile t = issue_next(stage == 0 ? NS - 1 : stage - 1);  // stage (it + NS - 1) % NS
        if constexpr (MASKED) (NS == 3 ? bits2 : bits1) = pair_bits(t);
      }
      tile_body(masked_tag, stage, stage, bits0, 0, [](auto) {});
      if constexpr (MASKED) {
        bits0 = bits1;
        bits1 = bits2;
      }
      stage = stage == NS - 1 ? 0 : stage + 1;
    };
    int it = 0;
    for (; it < n_masked; ++it) step(std::true_type{}, it);
    for (; it < n_iter; ++it) step(std::false_type{}, it);
  };
  if constexpr (PAIR) {
    // the two kinds of wave run separate copies of the loop (the same barriers in both), so
    // that neither carries the other's registers
    if (part == 0) run_pair(std::false_type{});
    else run_pair(std::true_type{});
  } else {
    run_tiles();
  }
  wait_vmcnt<0>();

  if constexpr (FIRST) {
    if (a_valid) {
      T* qs = const_cast<T*>(reinterpret_cast<const T*>(p.qs)) + a_row * a_stride + int64_t(head_a) * D + g * 8;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) *reinterpret_cast<vec8*>(qs + ks * 16) = x1f[ks];
      if (g == 0) {
        const int64_t stat_idx = (int64_t(b_orig) * p.heads_q + head_a) * p.tokens + a_tok;
        const_cast<float*>(p.lse)[stat_idx] = lse_l;
        const_cast<float*>(p.delta)[stat_idx] = delta_l;
      }
    }
  }
  // dQ = scale * sum_k dS k;  dK = scale * sum_q dS q = ln 2 * sum_q dS q'
  store_results(acc1, acc2, KV_STATIONARY ? 0.6931471805599453f : p.scale);
}

// qs = round(q * scale * log2(e)) for `chunks` runs of 8 elements: the logit operand of the
// key-stationary roles (see scale_query_fragment).
template <typename T>
__global__ void __launch_bounds__(256) scale_queries_kernel(const T* q, T* qs, int64_t chunks, float c_log2) {
  using vec8 = typename Mma<T>::vec8;
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i < chunks)
    *reinterpret_cast<vec8*>(qs + i * 8) = scale_query_fragment<T>(*reinterpret_cast<const vec8*>(q + i * 8), c_log2);
}

// What the backward launches read besides the operands, in one pass over q, out and d_out
// [batch, tokens, heads, D]: q' (as scale_queries_kernel), and head-major [batch, heads, tokens]
// -rowsum(d_out * out) and -log2(e) lse (lse [batch, tokens, heads]).  HBM-bound (three reads and
// one write of q's size; the reads are non-temporal, 5-10 % faster here).  Against separate launches
// (delta, scaled queries, two transposes): 17.9 -> 6.3 us on 4 x 56 x 56 tokens, H 8, D 32; 52.5 -> 42.8
// on 128 x 128, H 16, D 128 (6.3 TB/s); 450 -> 480 on 29 x 46 x 78, H 24, D 128 (5.3 TB/s).
// A workgroup takes 256 rows: a run of tokens of 2^hb_lg heads (the largest power of two up to 8 that
// divides the head count, so that the reads are runs of heads and the head-major writes runs of 32 or
// more tokens, which meet in LDS).  D / 8 lanes share a row, 16 bytes each.
// A packed batch: the first two workgroups count the tiles of its two sides instead.
struct PackedCounts {
  const int32_t *cu_q, *cu_kv;
  int2 *q, *kv;  // null: not a packed batch
  int num_seqs, rows_q, rows_kv;
};
template <typename T, int D>
__global__ void __launch_bounds__(256) bwd_prepare_kernel(const T* __restrict__ q, const T* __restrict__ out,
                                                          const T* __restrict__ d_out, const float* __restrict__ lse,
                                                          T* __restrict__ qs, float* __restrict__ neg_delta,
                                                          float* __restrict__ neg_lse2, int tokens, int heads, int hb_lg,
                                                          NaDiv d_head_blocks, NaDiv d_token_blocks, float c_log2,
                                                          PackedCounts packed) {
  using vec8 = typename Mma<T>::vec8;
  constexpr int LPI = D / 8;     // lanes per row
  constexpr int RPP = 256 / LPI;  // rows per step
  __shared__ float s_delta[256];
  int block = int(blockIdx.x);
  if (packed.q != nullptr) {
    if (block < 2) {
      count_packed_tiles(block ? packed.cu_kv : packed.cu_q, packed.num_seqs, block ? packed.rows_kv : packed.rows_q, 7,
                         block ? packed.kv : packed.q, reinterpret_cast<int*>(s_delta));
      return;
    }
    block -= 2;
  }
  const int tid = threadIdx.x;
  const int hb = 1 << hb_lg, tb_lg = 8 - hb_lg;  // heads / log2 tokens of the workgroup
  // head blocks fastest: workgroups side by side read side by side
  const int token_blocks = (tokens + (1 << tb_lg) - 1) >> tb_lg;
  const int bt = na_div(block, d_head_blocks), b = na_div(bt, d_token_blocks);
  const int h0 = (block - bt * (heads >> hb_lg)) << hb_lg, t0 = (bt - b * token_blocks) << tb_lg;
  const int part = tid % LPI;
  // row `tid` of the head-major side, read early: token-major LSE
  const int ht = tid >> tb_lg, tt = t0 + (tid & ((1 << tb_lg) - 1));
  const float my_lse = tt < tokens ? lse[(int64_t(b) * tokens + tt) * heads + h0 + ht] : 0.f;
#pragma unroll 4
  for (int i = 0; i < LPI; ++i) {
    const int r = i * RPP + tid / LPI;  // row of the workgroup: head fastest
    const int h = r & (hb - 1), t = r >> hb_lg;
    float s = 0.f;
    if (t0 + t < tokens) {
      const int64_t at = ((int64_t(b) * tokens + t0 + t) * heads + h0 + h) * D + part * 8;
      const vec8 x = __builtin_nontemporal_load(reinterpret_cast<const vec8*>(out + at));
      const vec8 y = __builtin_nontemporal_load(reinterpret_cast<const vec8*>(d_out + at));
      const vec8 z = __builtin_nontemporal_load(reinterpret_cast<const vec8*>(q + at));
      s = dot8<T>(x, y);
      *reinterpret_cast<vec8*>(qs + at) = scale_query_fragment<T>(z, c_log2);
    }
#pragma unroll
    for (int o = LPI / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (part == 0) s_delta[(h << tb_lg) + t] = s;
  }
  workgroup_sync();
  if (tt < tokens) {
    const int64_t at = (int64_t(b) * heads + h0 + ht) * tokens + tt;
    neg_delta[at] = -s_delta[tid];
    neg_lse2[at] = -1.4426950408889634f * my_lse;
  }
}

// delta[item] = sum_d out[item, d] * d_out[item, d] over `items` rows of D contiguous elements
// (the reference's compute_delta, csrc/include/natten/compute_delta.h:33-36,
// csrc/include/natten/cuda/reduction/compute_delta.cuh).  D / 8 lanes
// share a row, 16 bytes each.
template <typename T, int D>
__global__ void __launch_bounds__(256) delta_kernel(const T* out, const T* d_out, float* delta, int64_t items) {
  constexpr int LPI = D / 8;  // lanes per item
  using tx8 = typename Mma<T>::vec8;
  const int64_t gtid = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t item = gtid / LPI;
  const int part = int(gtid % LPI);
  float s = 0.f;
  if (item < items) {
    s = dot8<T>(*reinterpret_cast<const tx8*>(out + item * D + part * 8), *reinterpret_cast<const tx8*>(d_out + item * D + part * 8));
  }
#pragma unroll
  for (int o = LPI / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (item < items && part == 0) delta[item] = s;
}

}  // namespace natten_amd
