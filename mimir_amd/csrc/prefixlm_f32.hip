// float32 prefix-LM attention (forward + backward) for gfx950.
//
// The fp32 path serves the reference's CPU training precision
// (flash_attention_prefixlm_dense.py runs in fp32) and is held to the fp32
// oracle at 1e-5: every product and sum stays in fp32, the products on the fp32
// matrix instruction v_mfma_f32_32x32x2_f32 (64 cycles for 4096 FLOP, 157
// TFLOP/s over the chip; measured 154 in a large matrix product).  Ownership
// follows the Metal kernels of flash_attention_prefixlm_mps.py (forward
// 391-476, dQ 967-1039, dK/dV 1245-1322), extended to GQA.
//
// A workgroup owns 32 rows (queries, or keys for dK / dV) of one head; its four
// waves (fewer for documents of up to two tiles) take the 32-row tiles of the other
// side in turn, each with accumulators of its own that are added through LDS at the end.  Small fp32 batches (a few
// thousand tokens) then still put two waves on every SIMD (one in the backward at
// head_dim 96 and 128, whose operands take more than half of its registers), and
// the tile loop holds no barrier.  With the owned rows on the columns of every product, S^T =
// K Q^T (dK / dV: S = Q K^T) leaves the probabilities in registers exactly as
// the B operand of the next product wants them: register r of lane half hi is
// row 8 (r / 4) + 4 hi + r % 4, and one matrix step sums over the two rows that
// the two halves hold.
//
//  * The owned rows (B operand) sit in LDS, [32][D + 4]: a lane reads 16 bytes
//    per four steps, and the row stride of an odd number of 16-byte units keeps
//    the sixteen rows of a read in distinct banks.
//  * The streamed rows (A operand) come straight from memory into registers, in
//    row form (lane = row, 16 bytes of it per four steps) for S and dP, and in
//    column form (lane = D / 32 neighbouring columns, one row per step) for the
//    second products, so that no transpose is needed.  They are re-read from
//    the caches by every workgroup of a head: 16 KiB per 4096 matrix cycles and
//    wave at head_dim 64, well under what L1 and L2 deliver.  Each operand is
//    requested one product (D / 2 matrix steps, 2048 cycles at head_dim 64)
//    before its use, which covers the latency without double buffers.
//  * S and dP are added up from short chains of matrix steps (kScoreChain), which
//    keeps their rounding at that of a row spread over lanes.
//    Row ranges are enforced by the buffer resource of the tile: rows past the
//    end read as zeros.
//
// Bound by the matrix unit and, on small batches, by the number of workgroups:
// 4 x 512 tokens, 8 heads, head_dim 64 (1.2 GFLOP forward, 5.0 executed in the
// backward): forward 86 -> 27 us (a workgroup's start-up and merge are a third
// of it), dQ + dK / dV 310 -> 78 us against the vector-ALU kernels these
// replace; one sequence of 4096 tokens, same heads, forward + backward 3.20 ->
// 0.75 ms.
#include "prefixlm_common.h"

namespace {
using namespace mimir;

constexpr int kMaxWaves = 4;         // waves of a workgroup: 1, 2 or 4 (waves_for)
constexpr int kThreads = kMaxWaves * 64;
constexpr int kRows = 32;            // rows per workgroup, and per streamed tile
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kDeltaRows = kThreads / 4;  // delta: 64 rows, 4 lanes per row

struct F32Args {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  float* lse;
  const float* olse;  // delta: forward lse
  const float* out;   // bwd: forward output
  const float* dout;
  float* dq;
  float* dk;
  float* dv;
  float* delta;       // [Hq, T], workspace
  float* lse2;        // [Hq, T], lse * log2(e), workspace
  const int32_t* prefix_lens;
  const int32_t* cu_seqlens;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh, do_st, do_sh;
  int64_t dq_st, dq_sh, dk_st, dk_sh, dv_st, dv_sh, lse_sh;
  int T, Hq, Hkv, group, total_seqlen, is_causal, num_tiles, numseqs;
  int longer_than, up_to;  // serves the documents of more than / at most so many tokens
  int z0;  // backward: first role of the grid (0: dK / dV, 1 + g: dQ of q head g of the group)
  float scale, scale_log2;
};

__device__ __forceinline__ bool served(const F32Args& a, int n) { return n > a.longer_than && n <= a.up_to; }

__device__ __forceinline__ float sum4(float x) {
  x += __shfl_xor(x, 1, 64);
  x += __shfl_xor(x, 2, 64);
  return x;
}

// delta = rowsum(O * dO) and lse * log2(e) of every (token, head) row.
template <int D>
__global__ __launch_bounds__(kThreads) void delta_f32_kernel(const F32Args a) {
  const int64_t row = (int64_t)blockIdx.x * kDeltaRows + (threadIdx.x >> 2);
  const int sub = threadIdx.x & 3;
  const bool valid = row < (int64_t)a.T * a.Hq;
  const int t = valid ? (int)(row / a.Hq) : 0;
  const int h = valid ? (int)(row % a.Hq) : 0;
  float acc = 0.f;
  if (valid) {
    const float* orow = a.out + (int64_t)t * a.o_st + (int64_t)h * a.o_sh + 4 * sub;
    const float* drow = a.dout + (int64_t)t * a.do_st + (int64_t)h * a.do_sh + 4 * sub;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      const f32x4 o = *(const f32x4*)&orow[16 * c], d = *(const f32x4*)&drow[16 * c];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_fmaf(o[e], d[e], acc);
    }
  }
  acc = sum4(acc);
  if (valid && sub == 0) {
    a.delta[(int64_t)h * a.T + t] = acc;
    a.lse2[(int64_t)h * a.T + t] = a.olse[(int64_t)h * a.lse_sh + t] * kLog2e;
  }
}

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Keeps the instruction scheduler from moving the loads in front of it behind
// the products (it otherwise sinks them to their use, which then waits for
// memory: forward 26.5 -> 25.3 us), or from moving those behind a product in front
// of it, where they would hold registers that the product needs (backward).
__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(0); }

// Row of accumulator register r in lane half hi.
__device__ __forceinline__ constexpr int acc_row(int r, int hi) { return 8 * (r >> 2) + 4 * hi + (r & 3); }

// LDS of a workgroup of W waves: the owned operands, later the partial sums of the
// waves.
template <int D, int W, int kOwned = 2>
struct Smem {
  static constexpr int kStride = D + 4;
  static constexpr int kTile = kRows * kStride;
  float x[(W > kOwned ? W : kOwned) * kTile];
  float m[W][kRows], l[W][kRows];
};

// One streamed 32-row tile of a [rows, D] fp32 matrix (row stride in elements).
template <int D>
struct Tile {
  static constexpr int kChunks = D / 8;   // 16-byte reads per lane in row form
  static constexpr int kCols = D / 32;    // columns per lane in column form
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Tile(const float* base, int64_t stride, int row0, int nrows) {
    const int left = min(kRows, nrows - row0);
    r = make_rsrc(base + (int64_t)row0 * stride, left > 0 ? (uint32_t)(((left - 1) * stride + D) * 4) : 0u);
  }
  // Row form: lane = row lane % 32, columns 8 c + 4 hi .. + 3 in chunk c.
  __device__ __forceinline__ void rows(f32x4 (&x)[kChunks], uint32_t lane_off) const {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) x[c] = __builtin_bit_cast(f32x4, buf_load16(r, lane_off + 32 * c));
  }
  // Column form: step s holds row acc_row(s, hi), columns kCols * (lane % 32) + 0 .. : one
  // resource per eight rows, so that four lane offsets serve all of them.
  static __device__ __forceinline__ void cols(float (&x)[16][kCols], const float* base, int64_t stride, int row0,
                                              int nrows, uint32_t lane_off, uint32_t row_bytes) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const Tile t(base, stride, row0 + 8 * g, nrows);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int s = 4 * g + e, off = (int)(lane_off + e * row_bytes);
        if constexpr (kCols == 1) {
          x[s][0] = buf_load_f32(t.r, off);
        } else if constexpr (kCols == 2) {
          const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(t.r, off, 0, 0));
          x[s][0] = v[0]; x[s][1] = v[1];
        } else if constexpr (kCols == 3) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b96(t.r, off, 0, 0);
#pragma unroll
          for (int c = 0; c < 3; ++c) x[s][c] = __uint_as_float(v[c]);
        } else {
          const f32x4 v = __builtin_bit_cast(f32x4, buf_load16(t.r, off));
#pragma unroll
          for (int c = 0; c < 4; ++c) x[s][c] = v[c];
        }
      }
    }
  }
};

// The lane's byte offsets into a tile in the two forms.
template <int D>
struct LaneOff {
  uint32_t row, col, row_bytes;
  __device__ __forceinline__ LaneOff(int64_t stride, int l32, int hi) {
    row_bytes = (uint32_t)stride * 4u;
    row = (uint32_t)l32 * row_bytes + 16u * hi;
    col = 4u * hi * row_bytes + (uint32_t)(4 * (D / 32) * l32);
  }
};

// The workgroup's 32 owned rows -> LDS; rows past nrows are zero.
template <int D, int W>
__device__ __forceinline__ void stage_owned(float* dst, const float* base, int64_t stride, int row0, int nrows) {
  constexpr int kThreads = W * 64, N = kRows * (D / 4) / kThreads;  // 16-byte units per thread
  const Tile<D> t(base, stride, row0, nrows);
  i32x4 v[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = threadIdx.x + j * kThreads, row = i / (D / 4), c = i % (D / 4);
    v[j] = buf_load16(t.r, (uint32_t)(row * stride + 4 * c) * 4u);
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = threadIdx.x + j * kThreads, row = i / (D / 4), c = i % (D / 4);
    *(i32x4*)&dst[row * Smem<D, W>::kStride + 4 * c] = v[j];
  }
}

// Matrix steps (two columns each) that S and dP add up in one chain before the chains
// are added to one another.  A chain rounds after every product, so its error grows with
// its length, and one over all of D was up to 1.8 times as far off as the short chains
// and tree of a row spread over lanes (short documents, whose sums over keys are few).
// S is formed alike in the forward and the backward: its error is then in the logsumexp
// too, and the rows of P sum to 1.  The relative error against 64 bits of O, dQ, dK
// (documents of 2 to 12 tokens; one chain / row over lanes / so), x 1e-7:
//   D  32: 0.98 2.5 2.5 / 0.81 2.2 2.2 / 0.76 2.1 2.1    D  64: 1.2 3.0 3.0 / 0.85 2.3 2.5 / 0.80 2.2 2.3
//   D  96: 1.4 3.6 3.6 / 0.91 2.7 2.8 / 0.85 2.7 2.7    D 128: 1.6 4.0 4.0 / 0.91 2.8 3.0 / 0.87 2.7 2.7
// The additions and their waits for the products cost, with one chain / so: forward +
// backward of 8192 tokens in documents of 2048, 8 heads, D 64 0.95 / 0.99 ms, of 4096, 16 / 4
// heads, D 128 2.75 / 2.96 (15.8 on the vector ALUs).
template <int D>
constexpr int kScoreChain = D == 32 ? 2 : D == 128 ? 8 : 4;
template <int D>
constexpr int kDpChain = D == 32 ? 4 : D == 64 ? 8 : 16;

// Steps [S0, S0 + N) of X W^T: chains of kChain steps, added as a tree.
template <int D, int kChain, int S0, int N>
__device__ __forceinline__ f32x16 product_tree(const f32x4 (&x)[D / 8], const float* row) {
  if constexpr (N > kChain) {
    const f32x16 left = product_tree<D, kChain, S0, N / 2>(x, row);
    return left + product_tree<D, kChain, S0 + N / 2, N / 2>(x, row);
  } else {
    f32x16 acc = f32x16{};
#pragma unroll
    for (int s = S0; s < S0 + N; ++s) acc = mfma_f32(x[s / 4][s % 4], row[8 * (s / 4) + s % 4], acc);
    return acc;
  }
}

// X W^T for a streamed tile x in row form and the owned rows w in LDS: 32 x 32, in
// trees of 16 steps added in turn.  Each sum is pinned where it is formed: the compiler
// otherwise moves the additions to their use and holds all chains until then.
template <int D, int kChain>
__device__ __forceinline__ f32x16 product_rows(const f32x4 (&x)[D / 8], const float* w, int l32, int hi) {
  const float* row = w + l32 * Smem<D, 1>::kStride + 4 * hi;
  f32x16 sum = product_tree<D, kChain, 0, 16>(x, row);
  if constexpr (D > 32) {
    sum += product_tree<D, kChain, 16, 16>(x, row);
    __asm__ volatile("" : "+v"(sum));
  }
  if constexpr (D > 64) {
    sum += product_tree<D, kChain, 32, 16>(x, row);
    __asm__ volatile("" : "+v"(sum));
  }
  if constexpr (D > 96) {
    sum += product_tree<D, kChain, 48, 16>(x, row);
    __asm__ volatile("" : "+v"(sum));
  }
  return sum;
}

// acc[dt] += X^T P: X the streamed tile in column form, P [32 x 32] in accumulator
// form.  acc[dt] row i is column D / 32 * i + dt of the result, its lane the owned row.
template <int D>
__device__ __forceinline__ void product_cols(f32x16 (&acc)[D / 32], const float (&x)[16][D / 32], f32x16 p) {
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) acc[dt] = mfma_f32(x[s][dt], p[s], acc[dt]);
}

// This wave's partial result (row = owned row) -> its LDS region.
template <int D>
__device__ __forceinline__ void put_partial(float* dst, const f32x16 (&acc)[D / 32], float scale, int l32, int hi) {
  constexpr int C = D / 32;
  float* row = dst + l32 * Smem<D, 1>::kStride;
#pragma unroll
  for (int g = 0; g < 4; ++g) {  // registers 4 g .. + 3: columns C * (8 g + 4 hi) .. + 4 C
    float v[4 * C];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int dt = 0; dt < C; ++dt) v[e * C + dt] = acc[dt][4 * g + e] * scale;
#pragma unroll
    for (int e = 0; e < C; ++e)
      *(f32x4*)&row[C * (8 * g + 4 * hi) + 4 * e] = f32x4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
  }
}

// finish(row, sum of the waves' partials) -> global rows row0 .. of [rows, D].
template <int D, int W, typename Finish>
__device__ __forceinline__ void store_sum(const float* x, float* base, int64_t stride, int row0, int nrows,
                                          Finish&& finish) {
  using S = Smem<D, W>;
  for (int i = threadIdx.x; i < kRows * (D / 4); i += W * 64) {
    const int row = i / (D / 4), c = i % (D / 4);
    if (row0 + row >= nrows) continue;
    f32x4 t = *(const f32x4*)&x[row * S::kStride + 4 * c];
#pragma unroll
    for (int w = 1; w < W; ++w) t += *(const f32x4*)&x[w * S::kTile + row * S::kStride + 4 * c];
    *(f32x4*)&base[(int64_t)(row0 + row) * stride + 4 * c] = finish(row, t);
  }
}

struct Lanes {
  int wave, l32, hi;
  __device__ __forceinline__ Lanes() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    l32 = threadIdx.x & 31;
    hi = (threadIdx.x >> 5) & 1;
  }
};

template <int D, int W>
__global__ __launch_bounds__(W * 64, 2) void fwd_f32_kernel(const F32Args a) {
  constexpr int C = D / 32;
  __shared__ __attribute__((aligned(16))) Smem<D, W, 1> sm;
  const int h = blockIdx.x % a.Hq;
  const int s = blockIdx.x / a.Hq;
  const int tile = a.num_tiles - 1 - (int)blockIdx.y;  // heaviest first
  const SeqGeom g = load_seq<true>(a.cu_seqlens, a.prefix_lens, s, a.total_seqlen, a.is_causal, a.T);
  const int m0 = tile * kRows;
  if (m0 >= g.nq || !served(a, g.n)) return;
  const int hk = h / a.group;
  const Lanes ln;
  const int kend = kend_of(g.p, m0 + ln.l32);
  const int n_tiles = (max(g.p, min(m0 + kRows, g.nq)) + kRows - 1) / kRows;
  const int kend_min = max(g.p, m0 + 1);  // every row sees the keys before this one
  const float* kb = a.k + (int64_t)g.start * a.k_st + (int64_t)hk * a.k_sh;
  const float* vb = a.v + (int64_t)g.start * a.v_st + (int64_t)hk * a.v_sh;
  const LaneOff<D> ko(a.k_st, ln.l32, ln.hi), vo(a.v_st, ln.l32, ln.hi);

  f32x4 kx[Tile<D>::kChunks];
  float vx[16][C];
  int kt = ln.wave;
  if (kt < n_tiles) Tile<D>(kb, a.k_st, kt * kRows, g.n).rows(kx, ko.row);
  stage_owned<D, W>(sm.x, a.q + (int64_t)g.start * a.q_st + (int64_t)h * a.q_sh, a.q_st, m0, g.nq);
  __syncthreads();

  f32x16 acc[C];
#pragma unroll
  for (int dt = 0; dt < C; ++dt) acc[dt] = f32x16{};
  float m_run = -INFINITY, l_run = 0.f;
  for (; kt < n_tiles; kt += W) {
    const int k0 = kt * kRows;
    Tile<D>::cols(vx, vb, a.v_st, k0, g.n, vo.col, vo.row_bytes);
    pin();
    f32x16 st = product_rows<D, kScoreChain<D>>(kx, sm.x, ln.l32, ln.hi);
    // the next tile's rows (none past the last: an empty range reads zeros)
    Tile<D>(kb, a.k_st, k0 + W * kRows, kt + W < n_tiles ? g.n : 0).rows(kx, ko.row);
    pin();
    if (k0 + kRows > kend_min) {
      __asm__ volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + acc_row(r, ln.hi) >= kend) st[r] = -INFINITY;
    }
    float mx = st[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, st[r]);
    const float m_new = fmaxf(m_run, xor32_max(mx));
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {  // else every factor is 1
      const float alpha = m_run == -INFINITY ? 0.f : fast_exp2((m_run - m_new) * a.scale_log2);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < C; ++dt) acc[dt] *= alpha;
    }
    const float mb = m_new == -INFINITY ? 0.f : m_new * a.scale_log2;  // -inf: no allowed key yet
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      st[r] = fast_exp2(__builtin_fmaf(st[r], a.scale_log2, -mb));
      l_run += st[r];
    }
    m_run = m_new;
    product_cols<D>(acc, vx, st);
  }

  // Merge: every wave scales its sums to the row's largest maximum.
  const float l_tot = xor32_sum(l_run);
  if (ln.hi == 0) {
    sm.m[ln.wave][ln.l32] = m_run;
    sm.l[ln.wave][ln.l32] = l_tot;
  }
  __syncthreads();  // also: every wave is done with the owned rows
  float M = sm.m[0][ln.l32];
#pragma unroll
  for (int w = 1; w < W; ++w) M = fmaxf(M, sm.m[w][ln.l32]);
  const float wt = m_run == -INFINITY ? 0.f : fast_exp2((m_run - M) * a.scale_log2);
  put_partial<D>(sm.x + ln.wave * Smem<D, W>::kTile, acc, wt, ln.l32, ln.hi);
  float l_sum = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float m = sm.m[w][ln.l32];
    l_sum += m == -INFINITY ? 0.f : sm.l[w][ln.l32] * fast_exp2((m - M) * a.scale_log2);
  }
  __syncthreads();
  if (threadIdx.x < kRows) {
    sm.l[0][threadIdx.x] = l_sum;
    if (m0 + (int)threadIdx.x < g.nq && a.lse != nullptr)
      a.lse[(int64_t)h * a.lse_sh + g.start + m0 + threadIdx.x] = M * a.scale + logf(l_sum);
  }
  __syncthreads();
  store_sum<D, W>(sm.x, a.o + (int64_t)g.start * a.o_st + (int64_t)h * a.o_sh, a.o_st, m0, g.nq,
               [&](int row, f32x4 t) { return t / sm.l[0][row]; });  // not times 1 / l: one rounding less
}

// dQ of one (head, sequence, 32-query tile): dQ^T += K^T dS^T over the key tiles.
template <int D, int W>
__device__ __forceinline__ void dq_body(const F32Args& a, Smem<D, W>& sm, int h, int s, int tile) {
  constexpr int C = D / 32;
  const SeqGeom g = load_seq<true>(a.cu_seqlens, a.prefix_lens, s, a.total_seqlen, a.is_causal, a.T);
  const int m0 = tile * kRows;
  if (m0 >= g.nq || !served(a, g.n)) return;
  const int hk = h / a.group;
  const Lanes ln;
  const int qpos = m0 + ln.l32;
  const bool valid = qpos < g.nq;
  const int kend = valid ? kend_of(g.p, qpos) : 0;
  const int n_tiles = (max(g.p, min(m0 + kRows, g.nq)) + kRows - 1) / kRows;
  const int kend_min = m0 + kRows <= g.nq ? max(g.p, m0 + 1) : 0;
  const float* kb = a.k + (int64_t)g.start * a.k_st + (int64_t)hk * a.k_sh;
  const float* vb = a.v + (int64_t)g.start * a.v_st + (int64_t)hk * a.v_sh;
  const LaneOff<D> ko(a.k_st, ln.l32, ln.hi), vo(a.v_st, ln.l32, ln.hi);

  f32x4 kx[Tile<D>::kChunks], vx[Tile<D>::kChunks];
  float kc[16][C];
  int kt = ln.wave;
  {
    const int n = kt < n_tiles ? g.n : 0;
    Tile<D>(kb, a.k_st, kt * kRows, n).rows(kx, ko.row);
    Tile<D>(vb, a.v_st, kt * kRows, n).rows(vx, vo.row);
  }
  const float lse2 = valid ? a.lse2[(int64_t)h * a.T + g.start + qpos] : 0.f;
  const float dlt = valid ? a.delta[(int64_t)h * a.T + g.start + qpos] : 0.f;
  float* const sq = sm.x;
  float* const sdo = sm.x + Smem<D, W>::kTile;
  stage_owned<D, W>(sq, a.q + (int64_t)g.start * a.q_st + (int64_t)h * a.q_sh, a.q_st, m0, g.nq);
  stage_owned<D, W>(sdo, a.dout + (int64_t)g.start * a.do_st + (int64_t)h * a.do_sh, a.do_st, m0, g.nq);
  __syncthreads();

  f32x16 acc[C];
#pragma unroll
  for (int dt = 0; dt < C; ++dt) acc[dt] = f32x16{};
  for (; kt < n_tiles; kt += W) {
    const int k0 = kt * kRows;
    const int n_next = kt + W < n_tiles ? g.n : 0;
    f32x16 st = product_rows<D, kScoreChain<D>>(kx, sq, ln.l32, ln.hi);
    pin();
    Tile<D>::cols(kc, kb, a.k_st, k0, g.n, ko.col, ko.row_bytes);
    Tile<D>(kb, a.k_st, k0 + W * kRows, n_next).rows(kx, ko.row);
    const f32x16 dp = product_rows<D, kDpChain<D>>(vx, sdo, ln.l32, ln.hi);
    pin();
    Tile<D>(vb, a.v_st, k0 + W * kRows, n_next).rows(vx, vo.row);
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] = fast_exp2(__builtin_fmaf(st[r], a.scale_log2, -lse2));
    if (k0 + kRows > kend_min) {
      __asm__ volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + acc_row(r, ln.hi) >= kend) st[r] = 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] *= dp[r] - dlt;
    product_cols<D>(acc, kc, st);
  }
  __syncthreads();  // every wave is done with the owned rows
  put_partial<D>(sm.x + ln.wave * Smem<D, W>::kTile, acc, a.scale, ln.l32, ln.hi);
  __syncthreads();
  store_sum<D, W>(sm.x, a.dq + (int64_t)g.start * a.dq_st + (int64_t)h * a.dq_sh, a.dq_st, m0, g.nq,
               [](int, f32x4 t) { return t; });
}

// dK and dV of one (kv head, sequence, 32-key tile): the waves take the (q head,
// 32-query tile) steps in turn; dV^T += dO^T P, dK^T += Q^T dS.
template <int D, int W>
__device__ __forceinline__ void dkdv_body(const F32Args& a, Smem<D, W>& sm, int hk, int s, int tile) {
  constexpr int C = D / 32;
  const SeqGeom g = load_seq<true>(a.cu_seqlens, a.prefix_lens, s, a.total_seqlen, a.is_causal, a.T);
  const int k0 = tile * kRows;
  if (k0 >= g.n || !served(a, g.n)) return;
  const Lanes ln;
  const int kpos = k0 + ln.l32;
  const bool valid = kpos < g.n;
  const int qs = valid ? qstart_of(g.p, kpos) : 0x7fffffff;
  const int qs_max = k0 + kRows <= g.n ? (k0 + kRows <= g.p ? 0 : k0 + kRows - 1) : 0x7fffffff;
  const int t0 = qstart_of(g.p, k0) / kRows;                      // first query tile with an attended pair
  const int n_q = max((g.nq + kRows - 1) / kRows - t0, 0);        // query tiles per head
  const int steps = n_q * a.group;
  const float* qb = a.q + (int64_t)g.start * a.q_st + (int64_t)hk * a.group * a.q_sh;
  const float* ob = a.dout + (int64_t)g.start * a.do_st + (int64_t)hk * a.group * a.do_sh;
  const LaneOff<D> qo(a.q_st, ln.l32, ln.hi), oo(a.do_st, ln.l32, ln.hi);

  f32x4 qx[Tile<D>::kChunks], ox[Tile<D>::kChunks];
  float qc[16][C], oc[16][C];
  // this wave's step: q head `hh` of the group and query tile t0 + t; advanced by W
  int hh = 0, t = ln.wave;
  auto wrap = [&]() __attribute__((always_inline)) {
    while (hh < a.group && t >= n_q) { t -= n_q; ++hh; }
  };
  auto tile_of = [&](const float* base, int64_t st, int64_t sh) __attribute__((always_inline)) {
    return Tile<D>(base + (int64_t)min(hh, a.group - 1) * sh, st, (t0 + t) * kRows, hh < a.group ? g.nq : 0);
  };
  if (steps > 0) {
    wrap();
    tile_of(qb, a.q_st, a.q_sh).rows(qx, qo.row);
    tile_of(ob, a.do_st, a.do_sh).rows(ox, oo.row);
  }
  float* const sk = sm.x;
  float* const sv = sm.x + Smem<D, W>::kTile;
  stage_owned<D, W>(sk, a.k + (int64_t)g.start * a.k_st + (int64_t)hk * a.k_sh, a.k_st, k0, g.n);
  stage_owned<D, W>(sv, a.v + (int64_t)g.start * a.v_st + (int64_t)hk * a.v_sh, a.v_st, k0, g.n);
  __syncthreads();

  f32x16 dka[C], dva[C];
#pragma unroll
  for (int dt = 0; dt < C; ++dt) dka[dt] = dva[dt] = f32x16{};
  for (int it = ln.wave; it < steps; it += W) {
    const int q0 = (t0 + t) * kRows;
    const int h = hk * a.group + hh;
    const float *const qh = qb + (int64_t)hh * a.q_sh, *const oh = ob + (int64_t)hh * a.do_sh;
    t += W;
    wrap();
    f32x16 p = product_rows<D, kScoreChain<D>>(qx, sk, ln.l32, ln.hi);
    pin();
    Tile<D>::cols(oc, oh, a.do_st, q0, g.nq, oo.col, oo.row_bytes);
    // Rows of the tile past the last query are read too (other rows, or the
    // workspace section behind the array) and masked below.
    const f32x4u* const lp = (const f32x4u*)(a.lse2 + (int64_t)h * a.T + g.start + q0 + 4 * ln.hi);
    const f32x4u* const dp = (const f32x4u*)(a.delta + (int64_t)h * a.T + g.start + q0 + 4 * ln.hi);
    f32x4 lse[4], dlt[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) lse[e] = lp[2 * e];
#pragma unroll
    for (int e = 0; e < 4; ++e) dlt[e] = dp[2 * e];
    f32x16 ds = product_rows<D, kDpChain<D>>(ox, sv, ln.l32, ln.hi);
    pin();
    Tile<D>::cols(qc, qh, a.q_st, q0, g.nq, qo.col, qo.row_bytes);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r] = fast_exp2(__builtin_fmaf(p[r], a.scale_log2, -lse[r >> 2][r & 3]));
      ds[r] = p[r] * (ds[r] - dlt[r >> 2][r & 3]);
    }
    if (q0 < qs_max || q0 + kRows > g.nq) {
      __asm__ volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qp = q0 + acc_row(r, ln.hi);
        if (qp < qs || qp >= g.nq) p[r] = ds[r] = 0.f;
      }
    }
    product_cols<D>(dva, oc, p);
    tile_of(qb, a.q_st, a.q_sh).rows(qx, qo.row);
    product_cols<D>(dka, qc, ds);
    tile_of(ob, a.do_st, a.do_sh).rows(ox, oo.row);
  }
  const float* const base = sm.x;
  float* const mine = sm.x + ln.wave * Smem<D, W>::kTile;
  __syncthreads();  // every wave is done with the owned rows
  put_partial<D>(mine, dva, 1.f, ln.l32, ln.hi);
  __syncthreads();
  store_sum<D, W>(base, a.dv + (int64_t)g.start * a.dv_st + (int64_t)hk * a.dv_sh, a.dv_st, k0, g.n,
               [](int, f32x4 t) { return t; });
  __syncthreads();
  put_partial<D>(mine, dka, a.scale, ln.l32, ln.hi);
  __syncthreads();
  store_sum<D, W>(base, a.dk + (int64_t)g.start * a.dk_st + (int64_t)hk * a.dk_sh, a.dk_st, k0, g.n,
               [](int, f32x4 t) { return t; });
}

// dK / dV units, then dQ units, in one launch: independent work, and the lighter
// dQ units fill the end of the dK / dV ones (4 x 512 tokens, 8 heads, head_dim
// 64: 78 us; the two interleaved tile by tile 85).  blockIdx.x: (sequence, kv
// head); blockIdx.y: the tile, heaviest first (the first key tiles, the last
// query tiles); blockIdx.z + z0: 0 for dK / dV, 1 + q head of the group for dQ.
// Workgroups are dealt round-robin to the XCDs and, inside one, to its shader
// engines, whether or not the next one has room, so the sequences rotate by one
// per row of tiles: a long or prefix-heavy one then does not land on one engine
// while the others idle (78 -> 76.7 us).
template <int D, int W>
__global__ __launch_bounds__(W * 64, D <= 64 ? 2 : 1) void bwd_f32_kernel(const F32Args a) {
  __shared__ __attribute__((aligned(16))) Smem<D, W> sm;
  const int hk = blockIdx.x % a.Hkv, y = blockIdx.y;
  const int s = (int)(blockIdx.x / a.Hkv + y) % a.numseqs;
  const int z = blockIdx.z + a.z0;
  if (z == 0)
    dkdv_body<D, W>(a, sm, hk, s, y);
  else
    dq_body<D, W>(a, sm, hk * a.group + z - 1, s, a.num_tiles - 1 - y);
}

// By name: of several instantiations launched from one place, this toolchain drops host stubs.
#define F32_KERNELS(D, W)                                    \
  template __global__ void fwd_f32_kernel<D, W>(const F32Args); \
  template __global__ void bwd_f32_kernel<D, W>(const F32Args);
#define F32_KERNELS_OF(D) F32_KERNELS(D, 1) F32_KERNELS(D, 2) F32_KERNELS(D, 4)
F32_KERNELS_OF(32)
F32_KERNELS_OF(64)
F32_KERNELS_OF(96)
F32_KERNELS_OF(128)

// Waves of a workgroup whose waves take up to `steps` tiles in turn: no more than find one.
// Idle ones keep other documents from the chip: a SIMD holds two waves, one in the backward at
// head_dim 96 and 128.  Forward and backward, us, on the vector ALUs / four waves always / so:
//   1641 documents of 1 to 4 tokens, 6 heads of 96:  121, 447 / 132, 774 / 58, 227
//   395 documents of 5 to 16, 8 heads of 64:         36, 128 / 41, 111 / 23, 53
//   83 documents of 33 to 64, 6 heads of 96:         37, 96 / 28, 101 / 22, 66
// The results are the same bit for bit: an idle wave adds zeros.
int waves_for(int64_t steps) { return steps <= 1 ? 1 : steps == 2 ? 2 : kMaxWaves; }

// launch(tiles, waves) for the documents of a call, with a's bounds set to those it is to
// serve: all of them, or, where most have one or two tiles but not the longest and they fill
// the chip several times, the short ones in a launch of their own with the waves that they
// need.  On the vector ALUs / one launch / two, us, with one document of 100 tokens among them:
//   1596 of 1 to 4 tokens, 6 heads of 96:    124, 454 / 148, 821 / 80, 328
//   386 of 5 to 16, 8 heads of 64:           39, 141 / 47, 127 / 33, 78
//   498 of 30 to 34, 6 heads of 96:          87, 280 / 89, 415 / 70, 280
// and 164 of 17 to 32, 8 heads of 64, the fewest that this line takes: 29, 104 / 26, 65 / 29, 60.
template <typename Launch>
void launch_documents(F32Args& a, int64_t heads_per_step, Launch&& launch) {
  const int64_t mean = a.numseqs > 0 ? a.total_seqlen / a.numseqs : 0;
  const int short_tiles = mean <= 16 ? 1 : 2;
  const int short_waves = waves_for(short_tiles * heads_per_step), waves = waves_for(a.num_tiles * heads_per_step);
  a.longer_than = 0, a.up_to = 0x7fffffff;
  if (mean <= 40 && short_waves < waves && (int64_t)a.numseqs * a.Hq >= 4 * device_cu_count()) {
    a.up_to = short_tiles * kRows;
    launch(short_tiles, short_waves);
    a.longer_than = a.up_to, a.up_to = 0x7fffffff;
  }
  launch(a.num_tiles, waves);
}

F32Args common_args(int T, int Hq, int Hkv, int total_seqlen, int is_causal, float scale,
                    const int32_t* prefix_lens, const int32_t* cu_seqlens) {
  F32Args a = {};
  a.T = T;
  a.Hq = Hq;
  a.Hkv = Hkv;
  a.group = Hq / Hkv;
  a.total_seqlen = total_seqlen;
  a.is_causal = is_causal;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  a.prefix_lens = prefix_lens;
  a.cu_seqlens = cu_seqlens;
  return a;
}

template <int D>
hipError_t launch_fwd(const MimirPrefixLMFwdParams& p, hipStream_t stream) {
  F32Args a = common_args(p.total_tokens, p.num_q_heads, p.num_kv_heads, p.total_seqlen, p.is_causal,
                          p.softmax_scale, p.prefix_lens, p.cu_seqlens);
  a.q = (const float*)p.q; a.k = (const float*)p.k; a.v = (const float*)p.v;
  a.o = (float*)p.out; a.lse = p.lse;
  a.q_st = p.q_stride_token; a.q_sh = p.q_stride_head;
  a.k_st = p.k_stride_token; a.k_sh = p.k_stride_head;
  a.v_st = p.v_stride_token; a.v_sh = p.v_stride_head;
  a.o_st = p.out_stride_token; a.o_sh = p.out_stride_head;
  a.lse_sh = p.lse_stride_head;
  a.num_tiles = (p.max_seqlen_all + kRows - 1) / kRows;
  a.numseqs = p.numseqs;
  if (a.num_tiles == 0 || p.numseqs == 0) return hipSuccess;
  launch_documents(a, 1, [&](int tiles, int waves) {
    F32Args b = a;
    b.num_tiles = tiles;
    const dim3 grid(p.num_q_heads * p.numseqs, tiles), block(waves * 64);
    if (waves == 1)
      hipLaunchKernelGGL((fwd_f32_kernel<D, 1>), grid, block, 0, stream, b);
    else if (waves == 2)
      hipLaunchKernelGGL((fwd_f32_kernel<D, 2>), grid, block, 0, stream, b);
    else
      hipLaunchKernelGGL((fwd_f32_kernel<D, 4>), grid, block, 0, stream, b);
  });
  return hipGetLastError();
}

template <int D>
hipError_t launch_bwd(const MimirPrefixLMBwdParams& p, hipStream_t stream, int stages) {
  F32Args a = common_args(p.total_tokens, p.num_q_heads, p.num_kv_heads, p.total_seqlen, p.is_causal,
                          p.softmax_scale, p.prefix_lens, p.cu_seqlens);
  a.q = (const float*)p.q; a.k = (const float*)p.k; a.v = (const float*)p.v;
  a.out = (const float*)p.out; a.dout = (const float*)p.dout; a.olse = p.lse;
  a.dq = (float*)p.dq; a.dk = (float*)p.dk; a.dv = (float*)p.dv;
  const BwdWorkspace ws = bwd_workspace_layout(p.total_tokens, p.num_q_heads, p.numseqs, p.max_seqlen_all);
  a.delta = (float*)((char*)p.workspace + ws.delta);
  a.lse2 = (float*)((char*)p.workspace + ws.lse2);
  a.q_st = p.q_stride_token; a.q_sh = p.q_stride_head;
  a.k_st = p.k_stride_token; a.k_sh = p.k_stride_head;
  a.v_st = p.v_stride_token; a.v_sh = p.v_stride_head;
  a.o_st = p.out_stride_token; a.o_sh = p.out_stride_head;
  a.do_st = p.dout_stride_token; a.do_sh = p.dout_stride_head;
  a.dq_st = p.dq_stride_token; a.dq_sh = p.dq_stride_head;
  a.dk_st = p.dk_stride_token; a.dk_sh = p.dk_stride_head;
  a.dv_st = p.dv_stride_token; a.dv_sh = p.dv_stride_head;
  a.lse_sh = p.lse_stride_head;
  a.num_tiles = (p.max_seqlen_all + kRows - 1) / kRows;
  a.numseqs = p.numseqs;
  const int64_t rows = (int64_t)p.total_tokens * p.num_q_heads;
  if (rows > 0 && (stages & MIMIR_BWD_STAGE_DELTA))
    hipLaunchKernelGGL(delta_f32_kernel<D>, dim3((unsigned)((rows + kDeltaRows - 1) / kDeltaRows)),
                       dim3(kThreads), 0, stream, a);
  a.z0 = stages & MIMIR_BWD_STAGE_DKDV ? 0 : 1;
  const int z1 = stages & MIMIR_BWD_STAGE_DQ ? 1 + a.group : 1;
  if (a.num_tiles > 0 && p.numseqs > 0 && z1 > a.z0)
    launch_documents(a, a.group, [&](int tiles, int waves) {  // dK / dV: the tiles of the group's q heads
      F32Args b = a;
      b.num_tiles = tiles;
      const dim3 grid(p.num_kv_heads * p.numseqs, tiles, z1 - a.z0), block(waves * 64);
      if (waves == 1)
        hipLaunchKernelGGL((bwd_f32_kernel<D, 1>), grid, block, 0, stream, b);
      else if (waves == 2)
        hipLaunchKernelGGL((bwd_f32_kernel<D, 2>), grid, block, 0, stream, b);
      else
        hipLaunchKernelGGL((bwd_f32_kernel<D, 4>), grid, block, 0, stream, b);
    });
  return hipGetLastError();
}

}  // namespace

bool mimir_f32_head_dim_supported(int d) { return d == 32 || d == 64 || d == 96 || d == 128; }

hipError_t mimir_launch_fwd_f32(const MimirPrefixLMFwdParams& p, hipStream_t stream) {
  switch (p.head_dim) {
    case 32: return launch_fwd<32>(p, stream);
    case 64: return launch_fwd<64>(p, stream);
    case 96: return launch_fwd<96>(p, stream);
    case 128: return launch_fwd<128>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t mimir_launch_bwd_f32(const MimirPrefixLMBwdParams& p, hipStream_t stream, int stages) {
  switch (p.head_dim) {
    case 32: return launch_bwd<32>(p, stream, stages);
    case 64: return launch_bwd<64>(p, stream, stages);
    case 96: return launch_bwd<96>(p, stream, stages);
    case 128: return launch_bwd<128>(p, stream, stages);
    default: return hipErrorInvalidValue;
  }
}
