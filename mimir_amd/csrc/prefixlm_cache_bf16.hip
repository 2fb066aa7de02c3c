// Attention against a static KV cache (inference), bf16, for gfx950 (MI355X).
//
// Reference: src/mimir/model/layers.py:134-167 (_attention_with_cache).  The
// new keys / values go into the cache at positions cache_lengths[b] + i, then
// every query row attends the cache keys j < kv_len = cache_lengths[b] + S
// (and j <= cache_lengths[b] + i when causal).  The reference materializes the
// repeated K/V heads and a [B, S, max_kv_len] mask for SDPA; here:
//
//   cache_append_kernel      the scatter of k_new / v_new into the cache rows, first,
//                            where the attention kernels do not do it themselves
//   decode (at most 32 query rows per kv head, e.g. S = 1):
//     cache_decode_*_kernel  appends the new rows and attends, the workgroups equal
//                            shares of all key tiles of the call
//     cache_merge_kernel     adds the partial rows of the shares
//   otherwise:
//     cache_attn_kernel      one workgroup per (batch row, kv head, 128 query rows,
//                            key split): the G query heads of a kv head share its
//                            K / V tiles (rows are (token, head) pairs, token-major),
//                            64-key tiles stream through two LDS stages, S^T = K Q^T
//                            and O^T += V^T P^T on bf16 MFMA with an online softmax
//                            (the forward kernel's arithmetic)
//     cache_merge_splits_*   with several splits: adds their partial rows
#include "prefixlm_cache_layout.h"
#include "prefixlm_common.h"

namespace mimir {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kRows = kWaves * 32;  // query rows per workgroup
constexpr int kKeys = 64;           // keys per tile
constexpr int kMaxSplits = 64;      // key splits per row tile
constexpr int kMaxAppend = 1024;    // new tokens that the prefill kernel appends itself

struct CacheArgs {
  const bf16_t* q;
  const bf16_t* kn;
  const bf16_t* vn;
  bf16_t* ck;
  bf16_t* cv;
  bf16_t* out;
  const void* cache_lengths;  // int32 or int64 (idx64)
  const void* batch_indices;  // int32 or int64, or null
  int idx64;
  int64_t q_sb, q_st, q_sh, kn_sb, kn_st, kn_sh, vn_sb, vn_st, vn_sh;
  int64_t ck_sb, ck_st, ck_sh, cv_sb, cv_st, cv_sh, o_sb, o_st, o_sh;
  int B, S, L, rows, Hkv, G, causal, D;
  int n_rt;        // row tiles per (batch row, kv head)
  int splits;      // key splits per row tile (each batch row's key tiles spread evenly over them)
  float scale_log2;
  float* part_o;   // [unit, kRows, D] unnormalized O of each split (splits > 1)
  float* part_ml;  // [unit, kRows, 2]: running max (exp2 domain) and sum
  int shares;      // decode: runs of key tiles, one workgroup per kv head each
  int cus;         // CUs of the device
  int append;      // the attention kernel appends the new rows itself
};

__device__ __forceinline__ int64_t load_index(const void* p, int i, int idx64) {
  return idx64 ? ((const int64_t*)p)[i] : (int64_t)((const int32_t*)p)[i];
}
__device__ __forceinline__ int64_t cache_row(const CacheArgs& a, int b) {
  return a.batch_indices != nullptr ? load_index(a.batch_indices, b, a.idx64) : b;
}
// cache_lengths[b] clamped to [0, L]
__device__ __forceinline__ int cache_len_of(const CacheArgs& a, int b) {
  const int64_t c = load_index(a.cache_lengths, b, a.idx64);
  return c < 0 ? 0 : (c > a.L ? a.L : (int)c);
}

// k_new / v_new [b, i, h] -> cache [row(b), cache_lengths[b] + i, h]; 16 bytes per thread.
__global__ __launch_bounds__(256) void cache_append_kernel(const CacheArgs a) {
  const int chunks = a.D / 8;
  const int64_t total = (int64_t)a.B * a.S * a.Hkv * chunks;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int c = (int)(idx % chunks);
    int64_t t = idx / chunks;
    const int h = (int)(t % a.Hkv);
    t /= a.Hkv;
    const int i = (int)(t % a.S);
    const int b = (int)(t / a.S);
    const int64_t pos = load_index(a.cache_lengths, b, a.idx64) + i;
    const int64_t r = cache_row(a, b);
    if (pos < 0 || pos >= a.L || r < 0 || r >= a.rows) continue;  // outside the cache: dropped
    *(bf16x8*)&a.ck[r * a.ck_sb + (int64_t)pos * a.ck_st + (int64_t)h * a.ck_sh + c * 8] =
        *(const bf16x8*)&a.kn[(int64_t)b * a.kn_sb + (int64_t)i * a.kn_st + (int64_t)h * a.kn_sh + c * 8];
    *(bf16x8*)&a.cv[r * a.cv_sb + (int64_t)pos * a.cv_st + (int64_t)h * a.cv_sh + c * 8] =
        *(const bf16x8*)&a.vn[(int64_t)b * a.vn_sb + (int64_t)i * a.vn_st + (int64_t)h * a.vn_sh + c * 8];
  }
}

// One output row (at `orow`) from its n partial rows (max in the exp2 domain, sum,
// unnormalized O) at part_ml / part_o row slot(c), c < n:
// out = sum_c O_c 2^(m_c - M) / sum_c l_c 2^(m_c - M).  One wave: lane c takes part
// c's (max, sum), and the O rows are read one part per D / 4 lanes with kChunk
// loads in flight beside it, so up to 32 parts (D 128) cost one memory round trip.
template <int D, int kChunk = 16, typename Slot>
__device__ __forceinline__ void merge_row(const CacheArgs& a, int n, int lane, Slot&& slot, bf16_t* orow) {
  constexpr int kLanes = D / 4;        // lanes per part row, four columns each
  constexpr int kParts = 64 / kLanes;  // part rows per load
  const int sub = lane / kLanes, col = lane % kLanes * 4;
  float M = -INFINITY, lsum = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};  // this lane's columns over the parts of its lane group
  for (int c0 = 0; c0 < n; c0 += 64) {
    const int c = c0 + lane, in_chunk = min(n - c0, 64);
    const int row = slot(min(c, n - 1));
    f32x2 ml = *(const f32x2*)&a.part_ml[2 * (int64_t)row];
    f32x4 ov[kChunk];
    auto load_rows = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kChunk; ++i) {
        if (i0 + i * kParts >= in_chunk) break;  // uniform
        ov[i] = *(const f32x4*)&a.part_o[(int64_t)__shfl(row, min(i0 + i * kParts + sub, in_chunk - 1), 64) * D + col];
      }
    };
    load_rows(0);  // in flight beside the weights
    if (c >= n) ml = f32x2{-INFINITY, 0.f};
    float m = ml[0];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    const float m_new = fmaxf(M, m);
    const float alpha = M == -INFINITY ? 0.f : fast_exp2(M - m_new);
    const float w = ml[0] == -INFINITY ? 0.f : fast_exp2(ml[0] - m_new);  // -inf: no allowed key in this part
    float l = ml[1] * w;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) l += __shfl_xor(l, off, 64);
    lsum = lsum * alpha + l;
    acc *= alpha;
    M = m_new;
    for (int i0 = 0;;) {
#pragma unroll
      for (int i = 0; i < kChunk; ++i) {
        if (i0 + i * kParts >= in_chunk) break;
        const int src = i0 + i * kParts + sub;
        const float wi = __shfl(w, min(src, 63), 64);
        if (src < in_chunk && wi != 0.f) acc += ov[i] * wi;
      }
      i0 += kChunk * kParts;
      if (i0 >= in_chunk) break;
      load_rows(i0);
    }
  }
#pragma unroll
  for (int off = kLanes; off < 64; off <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (sub == 0) *(bf16x4*)&orow[col] = __builtin_convertvector(acc * inv, bf16x4);
}

// Key splits of a batch row with `keys` keys (cache_attn_kernel): tiles per split
// and the splits that hold keys.
struct RowSplit {
  int per, n;
};
__device__ __forceinline__ RowSplit row_split(const CacheArgs& a, int keys) {
  const int tiles = (keys + kKeys - 1) / kKeys;
  RowSplit r;
  r.per = max(1, (tiles + a.splits - 1) / a.splits);
  r.n = (tiles + r.per - 1) / r.per;
  return r;
}

// Whether the batch rows (at most 64) hold about as many cached keys: none differs from the
// first by more than an eighth of the chunk.
__device__ __forceinline__ bool even_lengths(const CacheArgs& a) {
  if (a.B > 64) return false;
  const int n = cache_len_of(a, min((int)threadIdx.x & 63, a.B - 1));
  const int64_t off = n - __builtin_amdgcn_readfirstlane(n);
  return __builtin_amdgcn_ballot_w64(8 * (off < 0 ? -off : off) > a.S) == 0;
}

// kAppend: the kernel reads the chunk's keys in place and appends them; without it they
// are in the cache already.  (One kernel for both: what the first needs, sixteen registers
// among it, slowed the second by 1 to 2%.)
template <int D, bool kAppend>
__global__ __launch_bounds__(kThreads, 2) void cache_attn_kernel(const CacheArgs a) {
  constexpr int DT = D / 32;
  constexpr int KS = D / 16;
  using L = TileLayout<D>;
  __shared__ __attribute__((aligned(16))) bf16_t sK0[L::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sV0[L::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sK1[L::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sV1[L::kElems];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hi = lane >> 5;

  // Later row tiles of a causal chunk see more keys, and workgroups b and b + (CUs) share a
  // CU.  Where the row tile decides (an unsplit chunk on rows of about the same length), the
  // workgroups take them by rank, the latest first over all pairs, and every other CU-sized
  // run backwards: a CU's two are then a long and a short one, and what is left over at the
  // end is short.  Against the row tiles of a pair in a row: 8 x 512 on 1536 keys 76.0 -> 68.0
  // us, 8 x 1024 on none 74.4 -> 56.4, 8 x 2048 on none 193 -> 142 (16 / 4 heads of 128), 12 x 700
  // on none 31.0 -> 25.2, 8 x 1024 on 1536 66.7 -> 52 (8 / 8 heads of 64); on rows of 100 to 2200
  // keys 8 x 300 would go from 98.9 to 107.  With the key range split, the runs of pairs alone
  // alternate (33 on 300 keys 15.1 -> 13.7, 8 x 139 on 60 to 145 25.2 -> 23.6).  Unsplit, that
  // alternation took the row tiles of some pairs the wrong way round: 12 x 700 on none 32.7.
  int u = blockIdx.x, split = 0, rt;
  if (a.splits == 1 && a.causal && even_lengths(a)) {
    const int run = u / a.cus, pairs = gridDim.x / a.n_rt;
    if (run % 2 == 1 && (run + 1) * a.cus <= (int)gridDim.x) u = (2 * run + 1) * a.cus - 1 - u;
    rt = a.n_rt - 1 - u / pairs;
    u %= pairs;
  } else {
    split = u % a.splits;
    u /= a.splits;
    rt = u % a.n_rt;
    u /= a.n_rt;
    if (a.splits > 1 && u * a.n_rt * a.splits / a.cus % 2 == 1) rt = a.n_rt - 1 - rt;
  }
  const int hk = u % a.Hkv;
  const int b = u / a.Hkv;

  const int64_t crow = cache_row(a, b);
  const bool row_in_cache = crow >= 0 && crow < a.rows;
  const int clen = cache_len_of(a, b);
  const int kv = row_in_cache ? min(clen + a.S, a.L) : 0;  // keys of this batch row
  // This batch row's key tiles, spread evenly over the splits; n_valid splits
  // hold keys.  A row without keys (outside the cache) gets zeros from split 0.
  const RowSplit rs = row_split(a, kv);
  const int per = rs.per, n_valid = rs.n;
  if (split > 0 && split >= n_valid) return;
  const int k0 = split * per * kKeys;
  const int k1 = min(kv, k0 + per * kKeys);
  const int R = a.S * a.G;  // query rows (token-major (token, head) pairs)

  // This lane's row and its key limit.
  const int row = rt * kRows + wave * 32 + l32;
  const bool row_ok = row < R;
  const int ti = row_ok ? row / a.G : 0;
  const int h = hk * a.G + (row_ok ? row - ti * a.G : 0);
  const int kend_lane = row_ok ? (a.causal ? min(clen + ti + 1, kv) : kv) : 0;
  // Wave-wide bounds (rows are token-major, so the wave's last row has the largest limit).
  const int r0 = rt * kRows + wave * 32;
  const bool wave_active = r0 < R;
  const int r_last = min(r0 + 31, R - 1);
  const int w_kend_max = wave_active ? (a.causal ? min(clen + r_last / a.G + 1, kv) : kv) : 0;
  const int w_kend_min = wave_active ? (a.causal ? min(clen + r0 / a.G + 1, kv) : kv) : 0;
  // Workgroup range of key tiles inside this split.
  const int wg_r_last = min(rt * kRows + kRows - 1, R - 1);
  const int wg_kend = a.causal ? min(clen + wg_r_last / a.G + 1, kv) : kv;
  const int kt0 = k0 / kKeys;
  const int kt1 = (min(k1, wg_kend) + kKeys - 1) / kKeys;  // may be <= kt0: nothing to attend

  const bf16_t* kbase = a.ck + (row_in_cache ? crow : 0) * a.ck_sb + (int64_t)hk * a.ck_sh;
  const bf16_t* vbase = a.cv + (row_in_cache ? crow : 0) * a.cv_sb + (int64_t)hk * a.cv_sh;
  const TileLoader<D, kWaves> ldk(a.ck_st, wave, lane), ldv(a.cv_st, wave, lane);
  // With `append`, keys [new_lo, new_hi) come from the new rows, which are on their
  // way into the cache: key j from new row j - pos.  A tile of new rows alone is copied
  // like one of the cache, from another base; a tile that holds both takes an address
  // per lane (at most two tiles of a row: with such copies for all tiles of new rows the
  // launch took longer than the append launch it saves, 8 x 512 on 1536: 78 -> 89 us).
  // 16 / 4 heads, head_dim 128, against the append launch: 8 x 512 on 1536 keys 81 ->
  // 78 us, 8 x 100 on 100 to 3000 46 -> 42, 100 on 3000 27 -> 24.5; 8 x 1024 on 1536,
  // 8 / 8 heads of 64, 68 -> 65.
  const int64_t pos_raw = kAppend ? load_index(a.cache_lengths, b, a.idx64) : 0;
  const int pos = pos_raw < -(int64_t)a.S ? -a.S : (pos_raw > a.L ? a.L : (int)pos_raw);
  const int new_lo = max(pos, 0), new_hi = min(pos + a.S, kv);
  const bf16_t* knb = a.kn + (int64_t)b * a.kn_sb + (int64_t)hk * a.kn_sh;
  const bf16_t* vnb = a.vn + (int64_t)b * a.vn_sb + (int64_t)hk * a.vn_sh;
  // Both kinds in one tile: every lane takes its 16 bytes from the row's own place
  // (keys past the last one repeat it; they are masked).
  auto issue_mixed = [&](int kb, bf16_t* tk, bf16_t* tv) {
    using Loader = TileLoader<D, kWaves>;
#pragma unroll
    for (int i = 0; i < Loader::kPerWave; ++i) {
      if (i == Loader::kPerWave - 1 && !ldk.has_last) break;
      const int u = ldk.lds[i] / 8 + lane;  // 16-byte unit of the tile
      const int c = min(u % L::kRowUnits, L::kUnits - 1) * 8;
      const int key = min(kb + L::unperm(u / L::kRowUnits), kv - 1);
      const bool fresh = key >= new_lo && key < new_hi;
      const bf16_t* ks = fresh ? knb + (int64_t)(key - pos) * a.kn_st : kbase + (int64_t)key * a.ck_st;
      const bf16_t* vs = fresh ? vnb + (int64_t)(key - pos) * a.vn_st : vbase + (int64_t)key * a.cv_st;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ks + c),
                                       (__attribute__((address_space(3))) void*)(tk + ldk.lds[i]), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vs + c),
                                       (__attribute__((address_space(3))) void*)(tv + ldk.lds[i]), 16, 0, 0);
    }
  };
  auto issue = [&](int kt, bf16_t* tk, bf16_t* tv) __attribute__((always_inline)) {
    const int kb = kt * kKeys;
    if constexpr (!kAppend) {
      ldk.issue_at(kbase + (int64_t)kb * a.ck_st, rows_bytes32(kv - kb, (uint32_t)a.ck_st, D), tk);
      ldv.issue_at(vbase + (int64_t)kb * a.cv_st, rows_bytes32(kv - kb, (uint32_t)a.cv_st, D), tv);
      return;
    }
    const bool some = kb + kKeys > new_lo && kb < new_hi;
    if (some && (kb < new_lo || new_hi < min(kb + kKeys, kv))) {
      issue_mixed(kb, tk, tv);
    } else {
      const int key0 = some ? kb - pos : kb;
      ldk.issue_at((some ? knb : kbase) + (int64_t)key0 * a.ck_st, rows_bytes32(kv - kb, (uint32_t)a.ck_st, D), tk);
      ldv.issue_at((some ? vnb : vbase) + (int64_t)key0 * a.cv_st, rows_bytes32(kv - kb, (uint32_t)a.cv_st, D), tv);
    }
  };
  if (kt0 < kt1) issue(kt0, sK0, sV0);

  // Q^T B-operand fragments: lane holds row `row`, d = 16*ks + 8*hi .. +7 (0 for rows >= R).
  bf16x8 qf[KS];
  {
    const bf16_t* qrow = a.q + (int64_t)b * a.q_sb + (int64_t)ti * a.q_st + (int64_t)h * a.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = row_ok ? *(const bf16x8*)&qrow[16 * ks + 8 * hi] : bf16x8{};
  }

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x16{};
  float m_run = -INFINITY;
  float l_run = 0.f;
  const float c2 = a.scale_log2;
  const TileLanes<D> tl(lane);

  auto compute = [&](int kt, const bf16_t* sK, const bf16_t* sV) {
    const int kb = kt * kKeys;
    if (!wave_active || kb >= w_kend_max) return;
    f32x16 st[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      st[mt] = f32x16{};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bf16x8 kf = *(const bf16x8*)&sK[tl.op_base + mt * 32 * L::kRowElems + ks * 16];
        st[mt] = mfma32(kf, qf[ks], st[mt]);
      }
    }
    if (kb + kKeys > w_kend_min) {
      __asm__ volatile("");
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kpos = kb + 32 * mt + 8 * (r >> 2) + 4 * hi + (r & 3);
          if (kpos >= kend_lane) st[mt][r] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[mt][r]);
    mx = xor32_max(mx);
    // Lazy rescaling, as in the forward kernel: the reference max moves only
    // when it grows by more than 2^8 in probability terms.
    const float m_cand = fmaxf(m_run, mx);
    const bool grow = (m_cand - m_run) * c2 > 8.f;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float m_new = grow ? m_cand : m_run;
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2((m_run - m_new) * c2);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
      m_run = m_new;
    }
    const float mb = m_run == -INFINITY ? 0.f : m_run * c2;
    float lsum = 0.f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = fast_exp2(__builtin_fmaf(st[mt][r], c2, -mb));
        st[mt][r] = pr;
        lsum += pr;
      }
    l_run += lsum;
    bf16x8 pf[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int mt = kk >> 1, s8 = (kk & 1) * 8;
      f32x8 t;
#pragma unroll
      for (int e = 0; e < 8; ++e) t[e] = st[mt][s8 + e];
      pf[kk] = to_bf16x8(t);
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const bf16_t* vp = &sV[tl.tr_base + kk * 16 * L::kRowElems + dt * 32];
        oacc[dt] = mfma32(cat8(lds_read_tr16(vp), lds_read_tr16(vp + L::kTrSecond)), pf[kk], oacc[dt]);
      }
  };

  // The new tokens whose first row lies in this row tile go into the cache here (no
  // workgroup reads these cache rows): with a kv head per q head all 128 rows are tokens,
  // and one load after another held up the first tile (8 x 1024 on 150 to 2000 keys, 6 / 6
  // heads of 128: 126.0 us, 121.6 with four in flight; 12 x 700 on none 87.6 -> 84.8).
  if (kAppend && split == 0 && row_in_cache) {
    constexpr int kUnits = D / 8, kStep = kThreads / kUnits, kBatch = 4;
    const int first = max((rt * kRows + a.G - 1) / a.G, -pos);
    const int last = min(((rt + 1) * kRows + a.G - 1) / a.G, min(a.S, a.L - pos));
    const int c = tid % kUnits * 8;
    for (int t0 = first + tid / kUnits; t0 < last; t0 += kBatch * kStep) {
      bf16x8 kx[kBatch], vx[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int t = min(t0 + i * kStep, last - 1);
        kx[i] = *(const bf16x8*)&knb[(int64_t)t * a.kn_st + c];
        vx[i] = *(const bf16x8*)&vnb[(int64_t)t * a.vn_st + c];
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int t = t0 + i * kStep;
        if (t >= last) break;
        *(bf16x8*)&a.ck[crow * a.ck_sb + (int64_t)(pos + t) * a.ck_st + (int64_t)hk * a.ck_sh + c] = kx[i];
        *(bf16x8*)&a.cv[crow * a.cv_sb + (int64_t)(pos + t) * a.cv_st + (int64_t)hk * a.cv_sh + c] = vx[i];
      }
    }
  }

  for (int kt = kt0; kt < kt1; kt += 2) {
    wait_vmem();
    __syncthreads();
    if (kt + 1 < kt1) issue(kt + 1, sK1, sV1);
    compute(kt, sK0, sV0);
    if (kt + 1 >= kt1) break;
    wait_vmem();
    __syncthreads();
    if (kt + 2 < kt1) issue(kt + 2, sK0, sV0);
    compute(kt + 1, sK1, sV1);
  }

  const float l_tot = xor32_sum(l_run);
  if (n_valid <= 1) {
    if (!wave_active || !row_ok) return;
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;  // no keys (row outside the cache): zeros
    bf16_t* orow = a.out + (int64_t)b * a.o_sb + (int64_t)ti * a.o_st + (int64_t)h * a.o_sh;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        f32x4 t;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = oacc[dt][4 * rg + e] * inv;
        *(bf16x4*)&orow[32 * dt + 8 * rg + 4 * hi] = __builtin_convertvector(t, bf16x4);
      }
    return;
  }

  // Several splits hold keys of this row tile: this split's partial rows --
  // unnormalized O, the max in the exp2 domain (-inf: no allowed key) and the sum.
  if (!wave_active) return;
  const int64_t slot = (((int64_t)u * a.n_rt + rt) * a.splits + split) * kRows + wave * 32 + l32;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      f32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = oacc[dt][4 * rg + e];
      *(f32x4*)&a.part_o[slot * D + 32 * dt + 8 * rg + 4 * hi] = t;
    }
  if (hi == 0) *(f32x2*)&a.part_ml[slot * 2] = f32x2{m_run == -INFINITY ? -INFINITY : m_run * c2, l_tot};
}

// By name: of several instantiations launched below, this toolchain drops host stubs.
template __global__ void cache_attn_kernel<128, true>(const CacheArgs);
template __global__ void cache_attn_kernel<128, false>(const CacheArgs);
template __global__ void cache_attn_kernel<64, true>(const CacheArgs);
template __global__ void cache_attn_kernel<64, false>(const CacheArgs);

// Adds the partial rows of cache_attn_kernel's key splits, one wave per query row.
// In the last split to arrive, four waves took the up to 128 rows of a tile in
// turn, two round trips of device-coherent loads each: a chunk of 100 tokens on
// 3000 cached ones (Hq 16, Hkv 4, D 128) 171 -> 27 us, of 512 on none 69 -> 29, 8 x
// 100 on 100 to 3000 81 -> 49 (append, attention and merge together).
template <int D>
__device__ __forceinline__ void cache_merge_splits_body(const CacheArgs& a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int R = a.S * a.G;
  const int groups = (R + kWaves - 1) / kWaves;  // workgroups per (batch row, kv head)
  const int row = blockIdx.x % groups * kWaves + wave;
  const int pair = blockIdx.x / groups;
  const int b = pair / a.Hkv, hk = pair - b * a.Hkv;
  if (row >= R) return;
  const int64_t crow = cache_row(a, b);
  const int keys = crow >= 0 && crow < a.rows ? min(cache_len_of(a, b) + a.S, a.L) : 0;
  const int n = row_split(a, keys).n;
  if (n <= 1) return;  // written by its split
  const int64_t unit0 = ((int64_t)pair * a.n_rt + row / kRows) * a.splits;
  const int t = row / a.G;
  merge_row<D>(a, n, lane, [&](int c) { return (int)((unit0 + c) * kRows + row % kRows); },
               a.out + (int64_t)b * a.o_sb + (int64_t)t * a.o_st + (int64_t)(hk * a.G + row - t * a.G) * a.o_sh);
}
__global__ __launch_bounds__(kThreads) void cache_merge_splits_d128_kernel(const CacheArgs a) {
  cache_merge_splits_body<128>(a);
}
__global__ __launch_bounds__(kThreads) void cache_merge_splits_d64_kernel(const CacheArgs a) {
  cache_merge_splits_body<64>(a);
}

// ---------------------------------------------------------------------------
// Decode: at most 32 query rows per kv head (R = S * G <= 32, e.g. S = 1); bound
// by the read of the cache, and for a few rows by the chain of memory round
// trips.  The 32-key tiles of all batch rows form one line, in units of
// kShareUnit, which is dealt evenly to shares (Shares), each of one workgroup per
// kv head, so rows of very different lengths keep all CUs busy to the end.  A
// share covers one or more segments (tiles of one batch row).  The query rows of a
// segment fit one wave, so instead of sharing 64-key tiles behind workgroup
// barriers, each of the kShareWaves waves streams its own tiles of the segment
// through two LDS stages of its own and waits only for its own copies: two
// independent copy pipelines per workgroup, two workgroups per CU.  The waves'
// partial rows are merged through LDS.  A (batch row, kv head) pair inside one
// share is finished there; the parts of the others go to the workspace and
// cache_merge_* adds them.  A second kernel needs no arrival counters, whose
// clearing took a launch of its own, and no device-coherent round trips: merging in
// the last share to arrive (flags with a value of the call's own instead of
// counters) left one launch, but 12.5 us of it instead of 7.4 + 4.4 for one row and
// 22.5 instead of 12.6 + 4.3 for eight.  Where pairs fill the chip about evenly
// (cache_split) each takes one workgroup of kPairWaves waves instead, and nothing
// is left to merge.
//
// The new rows are appended here too: the wave whose tile holds one stores it to
// the cache and to its LDS copy of the tile.  Batch rows that share a cache row
// see each other's new rows as if all had been appended first: the tile copy is
// overlaid with the new rows of every batch row of the same cache row.
//
// Measured against an append kernel, one workgroup of four waves per (pair, equal
// split) and a counted merge in it (Hq 16, Hkv 4, D 128): 64 rows of 512 to 8000 keys
// 140 -> 117 us (5.1 TB/s), 32 rows of 100 to 4000 41 -> 33, one row of 8000 22 -> 14;
// 8 rows of 1000 to 3600 17.4 -> 15.0, of which the two launches and their chains of
// round trips (lengths, tiles, parts) are 9.
// ---------------------------------------------------------------------------
constexpr int kDecKeys = 32;  // keys per wave tile
constexpr int kDecRows = 32;  // query rows of the decode kernel (one wave's columns)
constexpr float kRefRange = 30.f;  // how far (log2) a tile's reference may lie below the row's maximum
// Shares of the line: two waves and two (or three, cache_split) workgroups per CU, whose
// starts and ends overlap; a unit of the line is both stages of every wave.
constexpr int kShareWaves = 2;
constexpr int kShareUnit = 2 * kShareWaves;
// One workgroup per pair: four waves, one workgroup per CU; every pair is whole,
// nothing is left to merge, and only the pair's own batch row is looked up (1024 rows of
// 10 to 200 keys, 4 kv heads: 205 us with the line of all of them, 93 so).
constexpr int kPairWaves = 4;

template <int D>
struct DecTile {
  using L = TileLayout<D>;
  static constexpr int kUnits = kDecKeys * L::kRowUnits;  // 16-byte units of a 32-row tile
  static constexpr int kInst = (kUnits + 63) / 64;        // wave copy instructions per tile
  static constexpr int kElems = kInst * 512;              // bf16 elements incl. the last instruction's tail
};

// s_waitcnt vmcnt(N) for N < 64 (expcnt and lgkmcnt left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vmcnt_wide() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// Workgroup barrier for LDS data alone: unlike __syncthreads(), tile copies and
// stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __asm__ volatile("" ::: "memory");
  wait_lds();
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
}

// Inclusive sum over the wave's lanes (DPP adds; LDS-permute shuffles would cost
// six LDS round trips before the first copy).
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return x;
}

// The line of key tiles (of one kv head; they are alike), in units of kShareUnit, as
// one wave sees it: 64 batch rows at a time, one per lane.
struct TileLine {
  int first;  // batch row of lane 0
  int pos;    // position of the lane's batch row: cache_lengths clamped to [-S, L] (new row i goes to pos + i)
  int row;    // its cache row, -1 outside the cache
  int keys;   // keys it attends: cached and new ones inside the cache
  int units;  // units per kv head
  int incl;   // units per kv head of all batch rows up to this one
  struct Raw {
    int64_t length, row;
  };
  static __device__ __forceinline__ Raw fetch(const CacheArgs& a, int first, int lane) {
    const int b = first + lane;
    Raw r = {0, -1};
    if (b < a.B) r = {load_index(a.cache_lengths, b, a.idx64), cache_row(a, b)};
    return r;
  }
  __device__ __forceinline__ void set(const CacheArgs& a, Raw r, int first_, int before) {
    place(a, r.length < -(int64_t)a.S ? -a.S : (r.length > a.L ? a.L : (int)r.length),
          r.row >= 0 && r.row < a.rows ? (int)r.row : -1, first_, before);
  }
  __device__ __forceinline__ void place(const CacheArgs& a, int pos_, int row_, int first_, int before) {
    first = first_;
    pos = pos_;
    row = row_;
    keys = row >= 0 ? min(max(pos, 0) + a.S, a.L) : 0;
    units = ((keys + kDecKeys - 1) / kDecKeys + kShareUnit - 1) / kShareUnit;
    incl = before + wave_inclusive_sum(units);
  }
  __device__ __forceinline__ void load(const CacheArgs& a, int first_, int before, int lane) {
    set(a, fetch(a, first_, lane), first_, before);
  }
  __device__ __forceinline__ int end() const { return __builtin_amdgcn_readlane(incl, 63); }
};

// The line of a batch of more than 64 rows (at most kLineRows): lane c holds the units
// per kv head of batch rows 64 c .. 64 c + 63, and of all up to the last of them; the rows
// themselves stay in registers, 64 to a chunk.  All of them are loaded together, and with
// indices the batch rows on one cache row are found without a look at memory, so that the
// new rows need no launch of their own.  (Four chunks at a time and the needed one again,
// new rows appended first with indices: 128 rows of 2000 keys, 8 / 2 heads of 64, 30.9 us, so
// 30.3, with indices 34.6 -> 30.9; 300 of 0 to 100, 4 kv heads of 128, 26.2 -> 24.7 and 28.8 ->
// 25.7.)  Past kLineRows there is a workgroup per pair, which needs no line: 1000 rows of 0 to
// 300 keys, one kv head, 38.5 us with the line, 30.1 with pairs.
constexpr int kLineChunks = 8;
constexpr int kLineRows = 64 * kLineChunks;
struct LineChunks {
  int units, incl;
  int pos[kLineChunks], row[kLineChunks];
  template <typename F>
  __device__ __forceinline__ void scan(const CacheArgs& a, int lane, F&& each) {
    TileLine::Raw raw[kLineChunks];
#pragma unroll
    for (int c = 0; c < kLineChunks; ++c) {
      raw[c] = {0, -1};
      if (64 * c < a.B) raw[c] = TileLine::fetch(a, 64 * c, lane);
    }
    units = 0;
#pragma unroll
    for (int c = 0; c < kLineChunks; ++c) {
      pos[c] = 0, row[c] = -1;
      if (64 * c >= a.B) continue;  // uniform
      TileLine line;
      line.set(a, raw[c], 64 * c, 0);
      each(line);
      pos[c] = line.pos, row[c] = line.row;
      const int n = line.end();
      if (lane == c) units = n;
    }
    incl = wave_inclusive_sum(units);
  }
  __device__ __forceinline__ int total() const { return __builtin_amdgcn_readlane(incl, 63); }
  // Chunk c (uniform): its positions and cache rows, and its part of the line.
  __device__ __forceinline__ void rows(int c, int& p, int& r) const {
    p = pos[0], r = row[0];
#pragma unroll
    for (int i = 1; i < kLineChunks; ++i) p = c == i ? pos[i] : p, r = c == i ? row[i] : r;
  }
  // How many batch rows have cache row r.
  __device__ __forceinline__ int on_row(const CacheArgs& a, int r) const {
    int n = 0;
#pragma unroll
    for (int c = 0; c < kLineChunks; ++c)
      if (64 * c < a.B) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(row[c] == r));
    return n;
  }
  __device__ __forceinline__ void line(const CacheArgs& a, int c, TileLine& l) const {
    int p, r;
    rows(c, p, r);
    l.place(a, p, r, 64 * c, __builtin_amdgcn_readlane(incl, c) - __builtin_amdgcn_readlane(units, c));
  }
};

// The line's units dealt to the shares: q each, and one more to the first r.  A share is
// a run of the line for each kv head, one workgroup per head, so that the heads of a
// batch row, whose keys are adjacent in memory, stream the same positions at the same
// time.  (With the heads' lines one after another, a share somewhere in one of them, 128
// bytes of each key at a time, 64 rows of 0 to 2500 keys, 8 / 8 heads of 64, took 43.7 us, 38.0
// with a workgroup for each pair and key split, which starts the heads together; so
// 34.7.  Of 0 to 3780 54.8 -> 54.5 and 59.7 -> 49.1, of equal length 2000 53.8 -> 45.4; 64 of 500
// to 8000, 16 / 4 heads of 128, 119.4 -> 116.7.)  In whole units, the last shares empty, 24 rows
// of 500 to 2500, 8 / 8 heads of 64, 22.7 us instead of 21.1, 64 of 500 to 8000 118.6 instead of
// 116.7; but one row of 120000, 4 kv heads of 128, 51.5 instead of 53.0.
struct Shares {
  int q, r;
  __device__ __forceinline__ Shares(const CacheArgs& a, int total) : q(total / a.shares), r(total - q * a.shares) {}
  __device__ __forceinline__ int begin(int share) const { return share * q + min(share, r); }
  // the share that unit u < total lies in
  __device__ __forceinline__ int of(int u) const {
    const int longer = r * (q + 1);  // units of the first r shares, all of them if q is 0
    return u < longer ? u / (q + 1) : r + (u - longer) / q;
  }
};
// Part slot (of two per share) of a segment: the one the share begins with, or a later one.
__device__ __forceinline__ int part_slot(int share, bool first) { return 2 * share + !first; }

// Zero output for `heads` heads from h0 on of batch row b.
template <int D>
__device__ __forceinline__ void zero_rows(const CacheArgs& a, int b, int h0, int heads) {
  for (int i = threadIdx.x; i < a.S * heads * (D / 8); i += blockDim.x) {
    const int c = i % (D / 8), row = i / (D / 8);
    *(bf16x8*)&a.out[(int64_t)b * a.o_sb + (int64_t)(row / heads) * a.o_st + (int64_t)(h0 + row % heads) * a.o_sh +
                     c * 8] = bf16x8{};
  }
}

// The same for the batch rows without keys (outside the cache) among the loaded ones,
// dealt to the workgroups.
template <int D>
__device__ __forceinline__ void zero_keyless(const CacheArgs& a, const TileLine& line, int lane) {
  uint64_t none = __builtin_amdgcn_ballot_w64(line.first + lane < a.B && line.keys == 0);
  for (; none != 0; none &= none - 1) {
    const int b = line.first + __builtin_ctzll(none);
    if (b % (int)gridDim.x == (int)blockIdx.x) zero_rows<D>(a, b, 0, a.Hkv * a.G);
  }
}

template <int D, int kDecWaves, bool kPairs>
__device__ __forceinline__ void cache_decode_body(const CacheArgs& a) {
  constexpr int DT = D / 32;
  constexpr int KS = D / 16;
  using L = TileLayout<D>;
  using T = DecTile<D>;
  // two stages of (K, V) per wave; each stage array holds all waves' tiles
  __shared__ __attribute__((aligned(16))) bf16_t sK0[kDecWaves * T::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sV0[kDecWaves * T::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sK1[kDecWaves * T::kElems];
  __shared__ __attribute__((aligned(16))) bf16_t sV1[kDecWaves * T::kElems];
  // The merge's area per wave, in the second stages, which are free between a segment's
  // last tile and the second of the next: partial O [kDecRows][kPitch] (the padding keeps
  // the rows in distinct banks), then per row the reference (exp2 domain) and the sum.
  // (In an area of its own, four rows at a time, since two workgroups share the CU's LDS,
  // a segment of 32 query rows took eight passes between barriers: 64 rows of 100 to 3900
  // keys, 32 query rows a head, 87.5 -> 68.1 us, 32 of 100 to 3000, 8 / 8 heads of 64, 41.6 -> 33.6; 8
  // rows of 500 to 3000 24.2 -> 18.5, with 4 query rows a head 16.7 -> 15.9.)
  constexpr int kPitch = D + 4;
  constexpr int kArea = kDecRows * (kPitch + 2);
  static_assert(kArea * 4 <= 2 * T::kElems * 2, "two waves' K (or V) stages hold a wave's area");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hi = lane >> 5;

  // This share [u_begin, u_end) of the line, and the first batch row it touches: lane j
  // of the loaded rows.  One workgroup per pair: its batch row, and no line.
  TileLine line;
  LineChunks chunks;  // of more than 64 batch rows, not for pairs
  const int share = blockIdx.x / a.Hkv, hk = blockIdx.x - share * a.Hkv;  // share: the batch row, for pairs
  int j, u_begin = 0, u_end = 1;
  if constexpr (kPairs) {
    line.load(a, share & ~63, 0, lane);
    j = share & 63;
    if (__builtin_amdgcn_readlane(line.keys, j) == 0) {
      zero_rows<D>(a, share, hk * a.G, a.G);
      return;
    }
  } else {
    int total;
    if (a.B <= 64) {
      line.load(a, 0, 0, lane);
      zero_keyless<D>(a, line, lane);
      total = line.end();
    } else {
      chunks.scan(a, lane, [&](const TileLine& l) { zero_keyless<D>(a, l, lane); });
      total = chunks.total();
    }
    const Shares shares(a, total);
    u_begin = shares.begin(share);
    u_end = shares.begin(share + 1);
    if (u_begin >= u_end) return;
    if (a.B > 64) {
      chunks.line(a, __builtin_ctzll(__builtin_amdgcn_ballot_w64(chunks.incl > u_begin)), line);
    }
    j = __builtin_ctzll(__builtin_amdgcn_ballot_w64(line.incl > u_begin));
  }

  const int R = a.S * a.G;  // <= kDecRows
  const bool row_ok = l32 < R;
  const int ti = row_ok ? l32 / a.G : 0;
  const float c2 = a.scale_log2;
  const TileLanes<D> tl(lane);
  bf16_t* const mk0 = sK0 + wave * T::kElems;
  bf16_t* const mv0 = sV0 + wave * T::kElems;
  bf16_t* const mk1 = sK1 + wave * T::kElems;
  bf16_t* const mv1 = sV1 + wave * T::kElems;
  // This wave's copies of one 32-key tile: instruction i writes units
  // [64 i, 64 i + 64) of the wave's region; units past the 32 rows read zeros.
  uint32_t voffk[T::kInst], voffv[T::kInst];
  {
    const uint32_t stk = (uint32_t)a.ck_st * 2u, stv = (uint32_t)a.cv_st * 2u;
    int prow = lane / L::kRowUnits, c = lane % L::kRowUnits;  // of unit 64 i + lane
#pragma unroll
    for (int i = 0; i < T::kInst; ++i) {
      const uint32_t k = (uint32_t)L::unperm(prow);
      const bool ok = c < L::kUnits && prow < kDecKeys;
      voffk[i] = ok ? k * stk + c * 16 : 0x80000000u;
      voffv[i] = ok ? k * stv + c * 16 : 0x80000000u;
      prow += 64 / L::kRowUnits;
      c += 64 % L::kRowUnits;
      const int carry = c >= L::kRowUnits ? 1 : 0;
      prow += carry;
      c -= carry * L::kRowUnits;
    }
  }
  // The arguments that only a segment's start, its new rows and its end need,
  // loaded there: held across the tile loop they would spill.
  auto cold_args = []() __attribute__((always_inline)) -> const CacheArgs& {
    uint64_t seg = kernel_segment();
    __asm__ volatile("" : "+s"(seg));
    return segment_args<CacheArgs>(seg);
  };
  // The current segment: tiles [t0, t_end) of (batch row b, kv head hk), the
  // first at position u0 of the line.
  const int ck_st = (int)a.ck_st, cv_st = (int)a.cv_st;  // a span check bounds them
  int u0 = u_begin;
  int b, kv, pos_b, crow, t0, n_my, kend_lane, kend_min, u_next;
  bool whole;
  int new_lo, new_hi;  // positions [new_lo, new_hi) may hold new rows
  bool shared;         // other batch rows are on its cache row
  bf16_t *kbase, *vbase;
  bf16x8 qf[KS];

  // The other batch rows on the segment's cache row: f(batch row, its position).  (Pairs:
  // calls with indices have at most 64 batch rows here, all of them in the line.)
  auto for_others = [&](auto&& f) __attribute__((always_inline)) {
    if (!shared) return;
    for (int o0 = 0; o0 < a.B; o0 += 64) {
      int pos = line.pos, row = line.row;
      if (!kPairs && a.B > 64) chunks.rows(o0 / 64, pos, row);
      uint64_t same = __builtin_amdgcn_ballot_w64(row == crow && o0 + lane != b);
      for (; same != 0; same &= same - 1) {
        const int o = __builtin_ctzll(same);
        f(o0 + o, __builtin_amdgcn_readlane(pos, o));
      }
    }
  };
  // Overlay tile t's copy with the new rows (of batch row o, at position p on)
  // among its keys; the batch row's own are also stored to the cache.
  auto overlay_from = [&](int o, int p, int t, bf16_t* tk, bf16_t* tv) {
    constexpr int kUnits = D / 8;
    const CacheArgs& c = cold_args();
    const bf16_t* kn = c.kn + (int64_t)o * c.kn_sb + (int64_t)hk * c.kn_sh;
    const bf16_t* vn = c.vn + (int64_t)o * c.vn_sb + (int64_t)hk * c.vn_sh;
    const int64_t kn_st = c.kn_st, vn_st = c.vn_st;
    const int key0 = t * kDecKeys;
    const int lo = max(key0 - p, 0), end = min(a.S, min(key0 + kDecKeys, kv) - p);  // new rows inside the tile
    for (int i0 = lo; i0 < end; i0 += 64 / kUnits) {
      const int i = i0 + lane / kUnits, col = lane % kUnits * 8;
      if (i < end) {
        const bf16x8 kx = *(const bf16x8*)&kn[(int64_t)i * kn_st + col];
        const bf16x8 vx = *(const bf16x8*)&vn[(int64_t)i * vn_st + col];
        *(bf16x8*)&tk[L::off(p + i - key0, col)] = kx;
        *(bf16x8*)&tv[L::off(p + i - key0, col)] = vx;
        if (o == b) {
          *(bf16x8*)&kbase[(int64_t)(p + i) * ck_st + col] = kx;
          *(bf16x8*)&vbase[(int64_t)(p + i) * cv_st + col] = vx;
        }
      }
    }
  };
  auto overlay = [&](int t, bf16_t* tk, bf16_t* tv) {
    const int key0 = t * kDecKeys;
    if (key0 >= new_hi || key0 + kDecKeys <= new_lo) return;
    for_others([&](int o, int p) { overlay_from(o, p, t, tk, tv); });
    overlay_from(b, pos_b, t, tk, tv);
    __asm__ volatile("" ::: "memory");
    wait_lds();
  };


  auto issue = [&](int t, bf16_t* tk, bf16_t* tv) {
    const int key0 = t * kDecKeys;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbase + (int64_t)key0 * ck_st, rows_bytes32(kv - key0, ck_st, D));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vbase + (int64_t)key0 * cv_st, rows_bytes32(kv - key0, cv_st, D));
#pragma unroll
    for (int i = 0; i < T::kInst; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(tk + i * 512), 16,
                                               voffk[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < T::kInst; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (__attribute__((address_space(3))) void*)(tv + i * 512), 16,
                                               voffv[i], 0, 0, 0);
  };
  // Makes the segment at u0 (lane j of the line) the current one: its Q rows and
  // this wave's first tile are requested; its second tile's stages may still be in use.
  auto begin = [&]() __attribute__((always_inline)) {
    const CacheArgs& c = cold_args();
    b = line.first + j;
    kv = __builtin_amdgcn_readlane(line.keys, j);
    pos_b = __builtin_amdgcn_readlane(line.pos, j);
    crow = __builtin_amdgcn_readlane(line.row, j);
    int t_end = (kv + kDecKeys - 1) / kDecKeys;
    if constexpr (kPairs) {
      whole = true;
      u_next = u_end;
      t0 = 0;
    } else {
      const int units_b = __builtin_amdgcn_readlane(line.units, j);
      const int unit0 = u0 - (__builtin_amdgcn_readlane(line.incl, j) - units_b);
      const int unit1 = min(units_b, unit0 + u_end - u0);
      whole = unit0 == 0 && unit1 == units_b;
      u_next = u0 + unit1 - unit0;
      t0 = unit0 * kShareUnit;
      t_end = min(unit1 * kShareUnit, t_end);
    }
    n_my = t0 + wave < t_end ? (t_end - t0 - wave + kDecWaves - 1) / kDecWaves : 0;  // this wave's tiles
    const int clen = max(pos_b, 0);
    kend_lane = row_ok ? (c.causal ? min(clen + ti + 1, kv) : kv) : 0;
    kend_min = c.causal ? min(clen + 1, kv) : kv;
    kbase = c.ck + (int64_t)crow * c.ck_sb + (int64_t)hk * c.ck_sh;
    vbase = c.cv + (int64_t)crow * c.cv_sb + (int64_t)hk * c.cv_sh;
    // Q^T B-operand fragments first (their loads are older than the tile copies);
    // lanes past the R rows take row 0: their columns are never read
    const bf16_t* qrow = c.q + (int64_t)b * c.q_sb + (int64_t)ti * c.q_st +
                         (int64_t)(hk * c.G + (row_ok ? l32 - ti * c.G : 0)) * c.q_sh + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8*)&qrow[16 * ks];
    if (n_my > 0) issue(t0 + wave, mk0, mv0);
    new_lo = new_hi = 0;  // appended by a launch of its own: the copies hold them
    if (!a.append) return;
    new_lo = pos_b;
    new_hi = pos_b + a.S;
    shared = a.batch_indices != nullptr;
    if (shared)
      shared = (!kPairs && a.B > 64 ? chunks.on_row(a, crow) : __builtin_popcountll(__builtin_amdgcn_ballot_w64(line.row == crow))) > 1;
    for_others([&](int, int p) {
      new_lo = min(new_lo, p);
      new_hi = max(new_hi, p + a.S);
    });
  };

  f32x16 oacc[DT];
  // In scores, and finite (a scale below 1e-37): a tile without keys for a row keeps a reference.
  const float ref_range = fminf(kRefRange / c2, 3e38f);
  float m_run, m_top, l_run;  // the sums' reference and the row's maximum so far (scores), the sum
  auto compute = [&](int t, const bf16_t* sK, const bf16_t* sV) {
    const int kb = t * kDecKeys;
    f32x16 st = f32x16{};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) st = mfma32(*(const bf16x8*)&sK[tl.op_base + ks * 16], qf[ks], st);
    if (kb + kDecKeys > kend_min) {
      __asm__ volatile("");
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kpos = kb + 8 * (r >> 2) + 4 * hi + (r & 3);
        if (kpos >= kend_lane) st[r] = -INFINITY;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[r]);
    mx = xor32_max(mx);
    // Every tile's probabilities are taken under the tile's own maximum (but not more than
    // 2^30 below the row's so far, which bounds the sums): its largest probability is then 1
    // and exact in bf16.  Rescaled only when the row's maximum grew, what P's rounding cost
    // a tile depended on the tiles before it in its share, and so on the split: finer equal
    // splits, one tile per wave for a few rows, were more exact there.  Error against 64
    // bits, under the growing maximum / so: one row of 700 keys 2.07e-3 / 2.03e-3, 8 rows of
    // 1000 to 3600 2.09e-3 / 2.02e-3, 64 of 100 to 3000 2.12e-3 / 2.02e-3; time 11.9 / 11.5
    // us, 17.1 / 16.7, and 64 rows of 500 to 8000 120.3 / 119.8.
    m_top = fmaxf(m_top, mx);
    const float m_new = fmaxf(mx, m_top - ref_range);
    const float alpha = m_run == -INFINITY ? 1.f : fast_exp2((m_run - m_new) * c2);
    l_run *= alpha;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
    m_run = m_new;
    const float mb = m_run == -INFINITY ? 0.f : m_run * c2;
    float lsum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pr = fast_exp2(__builtin_fmaf(st[r], c2, -mb));
      st[r] = pr;
      lsum += pr;
    }
    l_run += lsum;
    bf16x8 pf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      f32x8 tv;
#pragma unroll
      for (int e = 0; e < 8; ++e) tv[e] = st[8 * kk + e];
      pf[kk] = to_bf16x8(tv);
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16_t* vp = &sV[tl.tr_base + kk * 16 * L::kRowElems + dt * 32];
        oacc[dt] = mfma32(cat8(lds_read_tr16(vp), lds_read_tr16(vp + L::kTrSecond)), pf[kk], oacc[dt]);
      }
  };

  begin();
  if (n_my > 1) issue(t0 + wave + kDecWaves, mk1, mv1);
  for (;;) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x16{};
    m_run = m_top = -INFINITY;
    l_run = 0.f;
    // Each wave waits only for its own copies: tile i has landed once at most the
    // copies of tile i + 1 are outstanding.
    for (int i = 0; i < n_my; i += 2) {
      if (i + 1 < n_my)
        wait_vmcnt_wide<2 * T::kInst>();
      else
        wait_vmcnt_wide<0>();
      overlay(t0 + wave + kDecWaves * i, mk0, mv0);
      compute(t0 + wave + kDecWaves * i, mk0, mv0);
      if (i + 2 < n_my) {
        wait_lds();  // this wave's reads of the stage are done before it is refilled
        issue(t0 + wave + kDecWaves * (i + 2), mk0, mv0);
      }
      if (i + 1 >= n_my) break;
      if (i + 2 < n_my)
        wait_vmcnt_wide<2 * T::kInst>();
      else
        wait_vmcnt_wide<0>();
      overlay(t0 + wave + kDecWaves * (i + 1), mk1, mv1);
      compute(t0 + wave + kDecWaves * (i + 1), mk1, mv1);
      if (i + 3 < n_my) {
        wait_lds();
        issue(t0 + wave + kDecWaves * (i + 3), mk1, mv1);
      }
    }

    // The next segment's first copies go out before this one's merge (this wave's
    // reads of its stages are done; the merge uses the second ones), so that a share
    // of several short segments does not pay a memory round trip for each.
    const int cur_b = b;
    const bool cur_whole = whole;
    const int64_t slot = ((int64_t)part_slot(share, u0 == u_begin) * a.Hkv + hk) * R;
    const bool more = u_next < u_end;
    wait_lds();
    if (more) {
      u0 = u_next;  // the next batch row with keys
      if constexpr (!kPairs)
        while (line.end() <= u0) chunks.line(a, line.first / 64 + 1, line);
      j = __builtin_ctzll(__builtin_amdgcn_ballot_w64(line.incl > u0));
      begin();
    }
    // Merge the waves' partial rows through LDS.
    const float l_tot = xor32_sum(l_run);
    auto area = [&](int w) __attribute__((always_inline)) {  // of wave w
      return (float*)(w < kDecWaves / 2 ? sK1 : sV1) + w % (kDecWaves / 2) * kArea;
    };
    auto row_ml = [&](int w, int row) __attribute__((always_inline)) {
      return (f32x2*)(area(w) + kDecRows * kPitch) + row;
    };
    lds_barrier();  // every wave is done with its second stage
    if (l32 < R) {
      if (hi == 0) *row_ml(wave, l32) = f32x2{m_run == -INFINITY ? -INFINITY : m_run * c2, l_tot};
      float* po = area(wave) + l32 * kPitch;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          f32x4 tv;
#pragma unroll
          for (int e = 0; e < 4; ++e) tv[e] = oacc[dt][4 * rg + e];
          *(f32x4*)&po[32 * dt + 8 * rg + 4 * hi] = tv;
        }
    }
    lds_barrier();
    constexpr int kLanes = D / 4;        // lanes per row, four columns each
    constexpr int kRowsAt = 64 / kLanes; // rows a wave takes at a time
    const int dcol = lane % kLanes * 4;
    const CacheArgs& c = cold_args();
    for (int r0 = wave * kRowsAt; r0 < R; r0 += kDecWaves * kRowsAt) {
      const int rr = min(r0 + lane / kLanes, R - 1);  // past the last row: that row again
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) M = fmaxf(M, (*row_ml(w, rr))[0]);
      float lsum = 0.f;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) {
        const f32x2 ml = *row_ml(w, rr);
        const float wt = ml[0] == -INFINITY ? 0.f : fast_exp2(ml[0] - M);
        lsum += ml[1] * wt;
        acc += *(const f32x4*)&area(w)[rr * kPitch + dcol] * wt;
      }
      if (cur_whole) {
        const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
        const int ti_r = rr / a.G;
        const int h_r = hk * a.G + (rr - ti_r * a.G);
        bf16_t* orow = c.out + (int64_t)cur_b * c.o_sb + (int64_t)ti_r * c.o_st + (int64_t)h_r * c.o_sh;
        *(bf16x4*)&orow[dcol] = __builtin_convertvector(acc * inv, bf16x4);
      } else {
        *(f32x4*)&c.part_o[(slot + rr) * D + dcol] = acc;
        if (dcol == 0) *(f32x2*)&c.part_ml[(slot + rr) * 2] = f32x2{M, lsum};
      }
    }
    if (!more) return;
    lds_barrier();  // the merge's area is the second stages again
    if (n_my > 1) issue(t0 + wave + kDecWaves, mk1, mv1);
  }
}

// One kernel per head_dim, by name: two instantiations of one kernel template
// launched from the two branches below lost one host stub in this toolchain.
__global__ __launch_bounds__(kShareWaves * 64, 1) void cache_decode_d128_kernel(const CacheArgs a) {
  cache_decode_body<128, kShareWaves, false>(a);
}
__global__ __launch_bounds__(kShareWaves * 64, 1) void cache_decode_d64_kernel(const CacheArgs a) {
  cache_decode_body<64, kShareWaves, false>(a);
}
__global__ __launch_bounds__(kPairWaves * 64, 1) void cache_decode_pairs_d128_kernel(const CacheArgs a) {
  cache_decode_body<128, kPairWaves, true>(a);
}
__global__ __launch_bounds__(kPairWaves * 64, 1) void cache_decode_pairs_d64_kernel(const CacheArgs a) {
  cache_decode_body<64, kPairWaves, true>(a);
}

// Output rows of the (batch row, kv head) pairs whose key tiles lie in several
// shares, one wave per row, from the parts in the order of the line.
template <int D, int kChunk>
__device__ __forceinline__ void cache_merge_body(const CacheArgs& a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int R = a.S * a.G;
  const int groups = (R + kWaves - 1) / kWaves;  // workgroups per pair
  const int rr = blockIdx.x % groups * kWaves + wave;
  const int pair = blockIdx.x / groups;
  const int b = pair / a.Hkv, hk = pair - b * a.Hkv;
  TileLine line;
  int total;
  if (a.B <= 64) {
    line.load(a, 0, 0, lane);
    total = line.end();
  } else {
    LineChunks chunks;
    chunks.scan(a, lane, [](const TileLine&) {});
    total = chunks.total();
    chunks.line(a, b / 64, line);
  }
  const int units_b = __builtin_amdgcn_readlane(line.units, b & 63);
  const int before = __builtin_amdgcn_readlane(line.incl, b & 63) - units_b;
  const Shares shares(a, total);
  if (units_b == 0 || rr >= R) return;
  const int w0 = shares.of(before), n = shares.of(before + units_b - 1) - w0 + 1;  // shares it lies in
  if (n == 1) return;  // written by its share
  const int slot0 = part_slot(w0, before == shares.begin(w0));
  const int t = rr / a.G;
  merge_row<D, kChunk>(a, n, lane, [&](int c) { return ((c == 0 ? slot0 : part_slot(w0 + c, true)) * a.Hkv + hk) * R + rr; },
               a.out + (int64_t)b * a.o_sb + (int64_t)t * a.o_st + (int64_t)(hk * a.G + rr - t * a.G) * a.o_sh);
}
__global__ __launch_bounds__(kThreads) void cache_merge_d128_kernel(const CacheArgs a) { cache_merge_body<128, 16>(a); }
__global__ __launch_bounds__(kThreads) void cache_merge_d64_kernel(const CacheArgs a) { cache_merge_body<64, 16>(a); }
// For more than 16 query rows per kv head: many more waves than the chip holds, and few
// parts for each; with fewer loads in flight (and registers) per wave twice as many fit
// (256 pairs of 32 rows, head_dim 64: the two launches 32.4 -> 30.7 us).
__global__ __launch_bounds__(kThreads, 8) void cache_merge_rows_d128_kernel(const CacheArgs a) {
  cache_merge_body<128, 4>(a);
}
__global__ __launch_bounds__(kThreads, 8) void cache_merge_rows_d64_kernel(const CacheArgs a) {
  cache_merge_body<64, 4>(a);
}

unsigned grid_for(int64_t items) {
  const int64_t blocks = (items + 255) / 256;
  return (unsigned)(blocks < 16384 ? (blocks > 0 ? blocks : 1) : 16384);
}

}  // namespace

CacheSplit cache_split(const MimirCacheAttnParams& p) {
  CacheSplit s = {};
  const int G = p.num_kv_heads > 0 ? p.num_q_heads / p.num_kv_heads : 1;
  const int64_t R = (int64_t)p.seqlen * G;
  s.decode = R <= kDecRows;  // the decode kernels: 32-key wave tiles
  s.n_rt = (int)((R + kRows - 1) / kRows);
  int max_kv = p.max_kv_len < p.cache_len ? p.max_kv_len : p.cache_len;
  if (max_kv < 1) max_kv = 1;
  const int tile_keys = s.decode ? kDecKeys : kKeys;
  const int tiles = (max_kv + tile_keys - 1) / tile_keys;
  s.groups = (int64_t)p.batch * p.num_kv_heads * s.n_rt;
  if (s.decode) {
    // One workgroup per pair while that fills the chip about evenly: from 256 keys
    // for any batch (two rounds of copies) up to 2048 for a pair per CU.  64 x 4
    // pairs (one launch against two, no merge): 100 to 1000 keys 25.5 -> 19.0 us, 100
    // to 2000 keys 37.5 / 37.9, 100 to 4000 keys 65 / 72 (the longest pair runs alone).
    // And for a batch past kLineRows, where a share would look for its pairs too long, and
    // for more than 16 query rows if the pairs fill the chip twice: then the parts of the
    // cut pairs are much of what there is to move (64 rows of 100 to 3000 keys, 8 / 8 heads
    // of 64, 32 query rows: 53 us, 62 dealt evenly, 57 with equal splits per pair).
    const int64_t pair_keys = 8 * s.groups;
    s.pairs = p.batch > kLineRows || (R > 16 && s.groups >= 2 * (int64_t)device_cu_count()) || max_kv <= (pair_keys < 256 ? 256 : (pair_keys < 2048 ? pair_keys : 2048));
    if (s.pairs) {  // one workgroup per pair
      s.units = s.groups;
    } else {
      // Two workgroups per CU, or one per unit and kv head if there cannot be as many (head_dim
      // 64: if those are at most four per CU, which its LDS allows: 16 rows of 10 to 4000 keys,
      // 8 / 2 heads, 13.2 -> 11.8 us); two part slots each: partial O, then (max, sum) rows.
      // Three at head_dim 64 with up to four kv heads, whose key rows of at most 512 bytes keep
      // fewer bytes in flight (two / three: 8 / 2 heads, 252 rows of 2009 to 2068 keys 55.4 / 51.6
      // us, 400 of 500 to 2000 57.8 / 53.6, 24 of 500 to 2400 13.3 / 11.4, 64 of 2000 19.0 / 20.0;
      // 8 / 8 heads, 128 of 2000 110.6 / 124.1).
      const int64_t cus = device_cu_count(), most = (int64_t)p.batch * ((tiles + kShareUnit - 1) / kShareUnit);
      int64_t shares = (p.head_dim == 64 && p.num_kv_heads <= 4 ? 3 : 2) * cus / p.num_kv_heads;
      if (shares < 1) shares = 1;
      if (p.head_dim == 64 && most * p.num_kv_heads <= 4 * cus) shares = most;
      s.units = p.num_kv_heads * (most < shares ? most : shares);
      s.workspace_bytes = (size_t)s.units * 2 * (size_t)R * ((size_t)p.head_dim + 2) * sizeof(float);
    }
    s.splits = 1;
    return s;
  }
  const int64_t target = 2 * (int64_t)device_cu_count();  // two workgroups per CU
  int64_t splits = s.groups > 0 ? (target + s.groups - 1) / s.groups : 1;
  if (splits < 1) splits = 1;
  if (splits > tiles) splits = tiles;
  if (splits > kMaxSplits) splits = kMaxSplits;
  s.splits = (int)splits;
  s.units = s.groups * s.splits;
  // partial O, then (max, sum) per unit row
  s.workspace_bytes = s.splits > 1 ? (size_t)s.units * kRows * ((size_t)p.head_dim + 2) * sizeof(float) : 0;
  return s;
}

hipError_t launch_cache_attn_bf16(const MimirCacheAttnParams& p, hipStream_t stream) {
  const CacheSplit sp = cache_split(p);
  CacheArgs a = {};
  a.q = (const bf16_t*)p.q;
  a.kn = (const bf16_t*)p.k_new;
  a.vn = (const bf16_t*)p.v_new;
  a.ck = (bf16_t*)p.cache_k;
  a.cv = (bf16_t*)p.cache_v;
  a.out = (bf16_t*)p.out;
  a.cache_lengths = p.cache_lengths;
  a.batch_indices = p.batch_indices;
  a.q_sb = p.q_stride_batch; a.q_st = p.q_stride_token; a.q_sh = p.q_stride_head;
  a.kn_sb = p.kn_stride_batch; a.kn_st = p.kn_stride_token; a.kn_sh = p.kn_stride_head;
  a.vn_sb = p.vn_stride_batch; a.vn_st = p.vn_stride_token; a.vn_sh = p.vn_stride_head;
  a.ck_sb = p.ck_stride_batch; a.ck_st = p.ck_stride_token; a.ck_sh = p.ck_stride_head;
  a.cv_sb = p.cv_stride_batch; a.cv_st = p.cv_stride_token; a.cv_sh = p.cv_stride_head;
  a.o_sb = p.out_stride_batch; a.o_st = p.out_stride_token; a.o_sh = p.out_stride_head;
  a.B = p.batch;
  a.S = p.seqlen;
  a.L = p.cache_len;
  a.rows = p.cache_rows;
  a.Hkv = p.num_kv_heads;
  a.G = p.num_q_heads / p.num_kv_heads;
  a.causal = p.causal != 0;
  a.D = p.head_dim;
  a.idx64 = p.index_int64 != 0;
  a.n_rt = sp.n_rt;
  a.splits = sp.splits;
  a.scale_log2 = p.softmax_scale * kLog2e;
  a.part_o = (float*)p.workspace;
  // Where the attention kernels append the new rows themselves, no workgroup reads them
  // from the cache, which asks for cache rows that share no memory: a batch row's new
  // rows are then seen through its own cache row alone.  (Shared, e.g. a cache expanded
  // over the batch, every batch row sees all new rows, as after appending all of them.)
  // Decode finds the batch rows on one cache row by their indices (a workgroup per pair
  // looks at up to 64 batch rows);
  // prefill does not, and needs one set of copy offsets for the new rows and the cache.
  // Longer chunks outweigh the launch that this saves: the kernel without it is 1 to 4%
  // faster (append launch / in place, rows on 150 to 2000 keys: 8 x 2048, 6 / 6 heads of 128,
  // 181 / 189 us, 8 / 8 of 64 137 / 143, 32 / 8 of 128 657 / 673; 4 x 1024, 8 / 8 of 64, 58.6 / 57.7,
  // 16 / 4 of 128 90.0 / 88.1; 12 x 700 on none, 8 / 8 of 64, 26.8 / 20.5).
  a.append = cache_rows_distinct(p) &&
             (sp.decode ? a.batch_indices == nullptr || a.B <= 64 || !sp.pairs
                        : a.batch_indices == nullptr && a.kn_st == a.ck_st && a.vn_st == a.cv_st && a.S <= kMaxAppend);
  const int64_t appends = (int64_t)a.B * a.S * a.Hkv * (a.D / 8);
  if ((sp.decode ? !sp.pairs : sp.splits > 1) && p.workspace == nullptr) return hipErrorInvalidValue;
  if (appends > 0 && !a.append) hipLaunchKernelGGL(cache_append_kernel, dim3(grid_for(appends)), dim3(256), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || sp.units == 0) return e;
  if (sp.decode) {
    const int64_t rows = (int64_t)a.S * a.G;
    a.shares = (int)(sp.units / a.Hkv);
    a.part_ml = a.part_o + (size_t)sp.units * 2 * rows * p.head_dim;
    const dim3 grid((unsigned)sp.units);
    if (sp.pairs) {
      if (p.head_dim == 128)
        hipLaunchKernelGGL(cache_decode_pairs_d128_kernel, grid, dim3(kPairWaves * 64), 0, stream, a);
      else
        hipLaunchKernelGGL(cache_decode_pairs_d64_kernel, grid, dim3(kPairWaves * 64), 0, stream, a);
      return hipGetLastError();
    }
    const dim3 merge((unsigned)(sp.groups * ((rows + kWaves - 1) / kWaves)));
    if (p.head_dim == 128) {
      hipLaunchKernelGGL(cache_decode_d128_kernel, grid, dim3(kShareWaves * 64), 0, stream, a);
      hipLaunchKernelGGL(rows > 16 ? cache_merge_rows_d128_kernel : cache_merge_d128_kernel, merge, dim3(kThreads), 0,
                         stream, a);
    } else {
      hipLaunchKernelGGL(cache_decode_d64_kernel, grid, dim3(kShareWaves * 64), 0, stream, a);
      hipLaunchKernelGGL(rows > 16 ? cache_merge_rows_d64_kernel : cache_merge_d64_kernel, merge, dim3(kThreads), 0,
                         stream, a);
    }
    return hipGetLastError();
  }
  a.part_ml = a.part_o + (size_t)sp.units * kRows * p.head_dim;
  a.cus = device_cu_count();
  const dim3 grid((unsigned)sp.units);
  if (p.head_dim == 128 && a.append)
    hipLaunchKernelGGL((cache_attn_kernel<128, true>), grid, dim3(kThreads), 0, stream, a);
  else if (p.head_dim == 128)
    hipLaunchKernelGGL((cache_attn_kernel<128, false>), grid, dim3(kThreads), 0, stream, a);
  else if (a.append)
    hipLaunchKernelGGL((cache_attn_kernel<64, true>), grid, dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((cache_attn_kernel<64, false>), grid, dim3(kThreads), 0, stream, a);
  if (sp.splits > 1) {
    const int64_t rows = (int64_t)a.S * a.G;
    const dim3 merge((unsigned)((int64_t)a.B * a.Hkv * ((rows + kWaves - 1) / kWaves)));
    if (p.head_dim == 128)
      hipLaunchKernelGGL(cache_merge_splits_d128_kernel, merge, dim3(kThreads), 0, stream, a);
    else
      hipLaunchKernelGGL(cache_merge_splits_d64_kernel, merge, dim3(kThreads), 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace mimir
