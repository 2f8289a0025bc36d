// Exact causal attention over full-width keys: the prompt pass of the attention forward
// (fourier_attn_triton/modeling_llama_fourier.py:623-633, flash_attn_func(q, k, v, causal=True)).
//
// Everything is computed transposed, so that no operand ever has to change lanes between the two products:
//   S^T[keys x rows] = K[keys x D] . Q^T[D x rows]        A = K rows as they lie in memory (a lane takes 16 bytes
//                                                          of one key), B = query rows (16 bytes of one row)
//   P^T = exp2(S^T - m)                                    per row = per lane column: running reference, base 2
//   O^T[D x rows] += V^T[D x keys] . P^T[keys x rows]      B = the lane's own eight probabilities of a 32-key tile
// The accumulator layout gives a lane the keys 4 lg .. 4 lg + 3 of each 16-key block; taking the two blocks of a
// 32-key tile as ONE contraction step whose slots are ordered {4 lg .. 4 lg + 3 of block 0, the same of block 1}
// makes those eight values the B operand as they are.  The A operand of that step, V^T with the keys in the same
// slot order, is prepared once per call by a transposing pass over V (prefill_vt_kernel): 1 KiB fragments that
// the main kernel streams into LDS unchanged.
//
// What bounds it: power, then issue.  On random operands the device runs this kernel at 1.8 - 1.9 GHz, so what counts is
// energy and instructions per score, not the order of the work.  Vector and matrix instructions of a SIMD overlap only in
// part (a 16x16x32 instruction holds the issue for half of its 16 clocks).  The softmax of a tile therefore costs a lane one
// multiply-add, half a three-way maximum, one exponential, half a conversion and one addition per score, and one vote per
// sixteen rows: only where a row's maximum rises do lanes exchange it and rescale.  Consecutive matrix instructions change one
// operand at a time.  32768 tokens, 32 / 8 heads of 128 dims, bf16, behind the other kernels of a prompt: 9.47 ms (an exchange on
// every tile) -> 8.70 ms, 1011 TFLOP/s; four sequences of 3001 tokens, 24 / 8 heads: 344 -> 329 us, where maxima still rise
// on most tiles.  A reference that lags behind the maximum by up to 8 would rescale next to nothing (8.27 ms), but rounds
// the largest weights, which are exact against the maximum: the error of peaked rows against 64 bits rose by a fifth; so did
// denominators from the f16 weights.  Slower: 32x32x16 instructions (half the count, but twice the accumulator traffic per
// product), denominators on the matrix unit, two waves per SIMD, a third stage.
//
// Workgroup: one KV head, HW query heads of it (all that share its keys, up to four) times RW blocks of 32 query
// rows, one wave each.  The key tiles travel HBM -> LDS once per workgroup (global_load_lds, two stages, one
// meeting per tile) in fragment order, so every LDS read of a wave is one conflict-free 16 bytes per lane.
#include "fa_common.h"
#include "fa_mfma_util.h"

namespace {
using namespace fa_mfma;

constexpr int kTileKeys = 32;
// a row's softmax reference moves only when a score exceeds it by more than this (base 2): the probabilities stay below
// 2^8, exact to f16's eleven bits, and most tiles rescale nothing
constexpr float kMaxLag = 0.f;
constexpr float kNoReference = -1e30f;   // before a row's first key: finite, so that a masked score is -inf against it

template <typename E>
struct PrefillParams {
  const E* q;          // (B, Hq, q_len, D) through strides, D contiguous
  int64_t q_bs, q_hs, q_rs;
  const E* k;          // (B, S, Hkv * D) token-major
  int64_t k_bs, k_rs;
  const f16_t* vt;     // [B][Hkv][tiles][D / 16][64 lanes][8]: V^T fragments, always f16 (see prefill_vt_kernel)
  E* out;              // (B, q_len, Hq, D) contiguous
  int B, Hq, Hkv, S, q_len, n_tiles, HW, RW;
  float sm_log2e;
};

// slot e of lane group lg in a 32-key tile
__device__ __forceinline__ int slot_key(int lg, int e) { return e < 4 ? 4 * lg + e : 16 + 4 * lg + (e - 4); }

// A wave transposes kVtTiles key tiles on its own: a lane holds eight keys (its slots of a tile) of eight dims, so that the
// 16-bit values change places inside the lane, and LDS only turns the lanes' 128-byte runs into whole rows of fragments
// (the pieces of a run are permuted so that neither side meets a bank twice).  All eight loads are on their way at once.
// Before, a block of 256 threads turned the tile with 2-byte reads of LDS behind two loads in a row.  us, before -> now: two
// sequences of 700 rows x 8 heads of 128 16.5 -> 6.5, four of 3001 19.2 -> 10.4 (4.7 TB/s), one of 8192 18.9 -> 9.6, eight of
// 1000 x 4 heads of 64 16.8 -> 6.4, one of 65 x 2 heads of 64 3.4 -> 3.6.
template <int D>
constexpr int kVtTiles = 128 / D;

template <typename E, int D>
__global__ __launch_bounds__(64) void prefill_vt_kernel(const E* __restrict__ v, int64_t v_bs, int64_t v_rs,
                                                        f16_t* __restrict__ vt, int S, int Hkv, int n_tiles) {
  // The second product runs in f16 whatever the storage type: the reference computes this attention as
  // flash_attn_func(q.half(), k.half(), v.half()) (MODEL:633), with probabilities of 11 significant bits; a bf16
  // operand would keep 8.  bf16 -> f16 is exact between 2^-14 and 65504 (larger magnitudes are clamped there).
  struct alignas(sizeof(E) * 8) Piece { E e[8]; };
  struct alignas(16) PieceOut { f16_t e[8]; };
  __shared__ PieceOut s_out[8 * 64];
  constexpr int C = D / 8;                        // pieces of a row
  const int lane = threadIdx.x, c = lane % C, lg = lane / C & 3, tl = lane / (4 * C);
  const int t0 = blockIdx.x * kVtTiles<D>, h = blockIdx.y, b = blockIdx.z;
  const E* src = v + (int64_t)b * v_bs + (int64_t)h * D + c * 8;
  const int key0 = (t0 + tl) * kTileKeys;
  Piece pc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) pc[e] = *(const Piece*)(src + (int64_t)min(key0 + slot_key(lg, e), S - 1) * v_rs);
  // piece x of the tiles (16 bytes of f16): eight to a run, run k = x / 8, kept at place (x ^ swz(k)) of the run
  auto swz = [](int k) { return (k ^ (k >> 3)) & 7; };
  const int run = ((tl * (D / 16) + (c >> 1)) * 4 + lg) * 2 + (c & 1);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    PieceOut o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = key0 + slot_key(lg, e) < S ? fa_to_float(pc[e].e[j]) : 0.f;
      o.e[e] = f16_t{(_Float16)fminf(fmaxf(x, -65504.f), 65504.f)};
    }
    s_out[run * 8 + (j ^ swz(run))] = o;
  }
  __syncthreads();
  PieceOut* dst = (PieceOut*)(vt + (((int64_t)b * Hkv + h) * n_tiles + t0) * (int64_t)(kTileKeys * D));
  const int here = min(kVtTiles<D>, n_tiles - t0) * (kTileKeys * D / 8);   // pieces of the tiles that there are
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int x = it * 64 + lane;
    if (x < here) dst[x] = s_out[(x & ~7) | ((x & 7) ^ swz(x >> 3))];
  }
}

template <typename E, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(3, 3))) void prefill_attn_kernel(const PrefillParams<E> p) {
  using M = Mma<E>;
  using vec8 = typename M::vec8;
  constexpr int KS = D / 32, DG = D / 16;
  constexpr int NF = 2 * KS + DG;                 // fragments (1 KiB) of one key tile: K (block, kstep), then V^T
  constexpr int OPS = (NF + WAVES - 1) / WAVES;   // fragments a wave brings in per tile
  __shared__ __attribute__((aligned(16))) unsigned char s_tile[2][NF * 1024];

  const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = p.Hq / p.Hkv;
  const int groups = G / p.HW;                    // workgroups per KV head along the heads
  const int kvh = blockIdx.y / groups, hg = blockIdx.y - kvh * groups;
  const int b = blockIdx.z;
  const int head = kvh * G + hg * p.HW + (w % p.HW);
  const int rblk = ((int)gridDim.x - 1 - (int)blockIdx.x) * p.RW + w / p.HW;   // long rows first
  const int r0 = rblk * 32;
  const int offset = p.S - p.q_len;               // row i sees keys 0 .. i + offset
  const int wg_last_row = min(p.q_len, ((int)gridDim.x - (int)blockIdx.x) * p.RW * 32) - 1;
  const int n_t = min(p.n_tiles, (wg_last_row + offset) / kTileKeys + 1);

  // this wave's share of a tile: fragments w, w + WAVES, ... (clamped to the last one: every wave issues OPS loads).
  // Addresses are a wave-uniform base plus one 32-bit lane offset for K and one for V^T; only a last tile that reaches
  // past the keys computes its (clamped) rows afresh.
  const E* kb_base = p.k + (int64_t)b * p.k_bs + (int64_t)kvh * D;
  const f16_t* vt_base = p.vt + ((int64_t)b * p.Hkv + kvh) * p.n_tiles * (int64_t)(kTileKeys * D);
  const unsigned k_off = (unsigned)((lc * p.k_rs + 8 * lg) * (int64_t)sizeof(E)), vt_off = lane * 16;
  const bool ragged_keys = (p.S % kTileKeys) != 0;
  auto issue = [&](int t, int buf) {
    const bool clamp = ragged_keys && t == p.n_tiles - 1;   // wave-uniform
    const E* k_tile = kb_base + (int64_t)t * kTileKeys * p.k_rs;
    const f16_t* v_tile = vt_base + (int64_t)t * (kTileKeys * D);
#pragma unroll
    for (int i = 0; i < OPS; ++i) {
      const int f = min(w + i * WAVES, NF - 1);
      const bool is_k = f < 2 * KS;
      const char* base = is_k ? (const char*)(k_tile + (int64_t)(16 * (f / KS)) * p.k_rs + 32 * (f % KS))
                              : (const char*)(v_tile + (f - 2 * KS) * 512);
      unsigned off = is_k ? k_off : vt_off;
      if (clamp && is_k) {
        const int first = t * kTileKeys + 16 * (f / KS);   // (may itself lie past the keys: the base then moves back)
        base = (const char*)(kb_base + 32 * (f % KS)) + (int64_t)min(first, p.S - 1) * p.k_rs * (int64_t)sizeof(E);
        off = (unsigned)((max(min(first + lc, p.S - 1) - first, 0) * p.k_rs + 8 * lg) * (int64_t)sizeof(E));
      }
      load_frag_to_lds((const E*)(base + off), &s_tile[buf][f * 1024]);
    }
  };
  if (n_t > 0) issue(0, 0);

  // query rows of this wave as B operands: row 16 rb + lc, dims 32 ks + 8 lg ..
  vec8 Qf[2][KS];
  {
    const E* qb = p.q + (int64_t)b * p.q_bs + (int64_t)head * p.q_hs + 8 * lg;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int row = min(r0 + 16 * rb + lc, p.q_len - 1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        Qf[rb][ks] = __builtin_bit_cast(vec8, *(const uint4v*)(qb + (int64_t)row * p.q_rs + 32 * ks));
    }
  }
  float4v oacc[DG][2];
#pragma unroll
  for (int dg = 0; dg < DG; ++dg) oacc[dg][0] = oacc[dg][1] = float4v{0.f, 0.f, 0.f, 0.f};
  float m_run[2] = {kNoReference, kNoReference}, l_run[2] = {0.f, 0.f};
  // the query loads above must not be confused with the tile loads by the counted waits below
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(Qf[rb][ks]));

  for (int t = 0; t < n_t; ++t) {
    const int buf = t & 1;
    wait_vmcnt<0>();        // this wave's fragments of tile t have landed (nothing else is outstanding)
    barrier_lds_only();     // everybody's have, and everybody is done with the other stage
    if (t + 1 < n_t) issue(t + 1, buf ^ 1);
    if (t * kTileKeys > r0 + 31 + offset) continue;   // this wave's rows end before the tile (a lower row block)
    const unsigned base = lds_addr_of(&s_tile[buf][0]) + lane * 16;
    // ---- S^T = K . Q^T
    float4v sacc[2][2] = {{float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}},
                          {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}}};
    // K fragments f = block * KS + kstep, two at a time into alternating halves of kf: the reads of a pair are on
    // their way while the matrix unit works on the pair before
    uint4v kf[4];
    constexpr int NFK = 2 * KS;
    auto s_pair = [&](uint4v& f0, uint4v& f1, int f) {   // fragments f, f + 1 (f is a constant after unrolling)
      sacc[f / KS][0] = M::mma(__builtin_bit_cast(vec8, f0), Qf[0][f % KS], sacc[f / KS][0]);
      sacc[f / KS][1] = M::mma(__builtin_bit_cast(vec8, f0), Qf[1][f % KS], sacc[f / KS][1]);
      sacc[(f + 1) / KS][1] = M::mma(__builtin_bit_cast(vec8, f1), Qf[1][(f + 1) % KS], sacc[(f + 1) / KS][1]);
      sacc[(f + 1) / KS][0] = M::mma(__builtin_bit_cast(vec8, f1), Qf[0][(f + 1) % KS], sacc[(f + 1) / KS][0]);
    };
    kf[0] = lds_read_b128_async_at<0 * 1024>(base);
    kf[1] = lds_read_b128_async_at<1 * 1024>(base);
    kf[2] = lds_read_b128_async_at<2 * 1024>(base);
    kf[3] = lds_read_b128_async_at<3 * 1024>(base);
    if constexpr (NFK == 8) {
      lds_wait_for2<2>(kf[0], kf[1]);
      s_pair(kf[0], kf[1], 0);
      kf[0] = lds_read_b128_async_at<4 * 1024>(base);
      kf[1] = lds_read_b128_async_at<5 * 1024>(base);
      lds_wait_for2<2>(kf[2], kf[3]);
      s_pair(kf[2], kf[3], 2);
      kf[2] = lds_read_b128_async_at<6 * 1024>(base);
      kf[3] = lds_read_b128_async_at<7 * 1024>(base);
      lds_wait_for2<2>(kf[0], kf[1]);
      s_pair(kf[0], kf[1], 4);
      lds_wait_for2<0>(kf[2], kf[3]);
      s_pair(kf[2], kf[3], 6);
    } else {   // heads of 64 dims: four fragments
      static_assert(NFK == 4, "head dims of 64 or 128");
      lds_wait_for2<2>(kf[0], kf[1]);
      s_pair(kf[0], kf[1], 0);
      lds_wait_for2<0>(kf[2], kf[3]);
      s_pair(kf[2], kf[3], 2);
    }
    // V^T fragments of the first half of the dims are requested now and used after the softmax
    uint4v vf[4];
    const unsigned vbase = base + 2 * KS * 1024;
    vf[0] = lds_read_b128_async_at<0>(vbase);
    vf[1] = lds_read_b128_async_at<1024>(vbase);
    vf[2] = lds_read_b128_async_at<2048>(vbase);
    vf[3] = lds_read_b128_async_at<3072>(vbase);
    // ---- softmax of the tile (base 2), per row = per lane column
    if (t * kTileKeys + 31 > r0 + offset || t * kTileKeys + 31 >= p.S) {   // wave-uniform
      asm volatile("");   // a real branch: as selects these masks would run on every tile
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int lim = min(r0 + 16 * rb + lc + offset, p.S - 1) - t * kTileKeys;   // last key of the tile this row may see
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (slot_key(lg, e) > lim) sacc[e >> 2][rb][e & 3] = -INFINITY;
      }
    }
    // distance of every score from its row's reference, the running maximum (the scale of the softmax rides in the
    // subtraction).  Most tiles raise no row's maximum: a vote per sixteen rows finds that out without a lane exchange.
    float x[2][8];
    auto distances = [&](int rb) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[rb][e] = __builtin_fmaf(sacc[e >> 2][rb][e & 3], p.sm_log2e, -m_run[rb]);
    };
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      distances(rb);
      // always on the first tile: every row sees its first key.  (Not "> 0": the maximum hands a NaN on)
      if (__any(!(fa_fmax8(x[rb]) <= 0.f))) {
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = sacc[e >> 2][rb][e & 3];
        const float m_new = fa_fmax(m_run[rb], fa_rows_max(fa_fmax8(s)) * p.sm_log2e);   // (the scale is positive)
        const float alpha = __builtin_amdgcn_exp2f(m_run[rb] - m_new);
        m_run[rb] = m_new;
        l_run[rb] *= alpha;
#pragma unroll
        for (int dg = 0; dg < DG; ++dg) oacc[dg][rb] *= alpha;
        distances(rb);
      }
    }
    half8 pb[2];   // probabilities as f16 operands; the denominators add the exponentials themselves
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float pv = __builtin_amdgcn_exp2f(x[rb][e]);
        psum += pv;
        pb[rb][e] = (_Float16)pv;
      }
      l_run[rb] += psum;
    }
    // ---- O^T += V^T . P^T (the fragments in pairs, like the K fragments above)
    auto o_pair = [&](uint4v& f0, uint4v& f1, int dg) {
      oacc[dg][0] = Mma<f16_t>::mma(__builtin_bit_cast(half8, f0), pb[0], oacc[dg][0]);
      oacc[dg][1] = Mma<f16_t>::mma(__builtin_bit_cast(half8, f0), pb[1], oacc[dg][1]);
      oacc[dg + 1][1] = Mma<f16_t>::mma(__builtin_bit_cast(half8, f1), pb[1], oacc[dg + 1][1]);
      oacc[dg + 1][0] = Mma<f16_t>::mma(__builtin_bit_cast(half8, f1), pb[0], oacc[dg + 1][0]);
    };
    if constexpr (DG == 8) {
      lds_wait_for2<2>(vf[0], vf[1]);
      o_pair(vf[0], vf[1], 0);
      vf[0] = lds_read_b128_async_at<4 * 1024>(vbase);
      vf[1] = lds_read_b128_async_at<5 * 1024>(vbase);
      lds_wait_for2<2>(vf[2], vf[3]);
      o_pair(vf[2], vf[3], 2);
      vf[2] = lds_read_b128_async_at<6 * 1024>(vbase);
      vf[3] = lds_read_b128_async_at<7 * 1024>(vbase);
      lds_wait_for2<2>(vf[0], vf[1]);
      o_pair(vf[0], vf[1], 4);
      lds_wait_for2<0>(vf[2], vf[3]);
      o_pair(vf[2], vf[3], 6);
    } else {
      static_assert(DG == 4, "head dims of 64 or 128");
      lds_wait_for2<2>(vf[0], vf[1]);
      o_pair(vf[0], vf[1], 0);
      lds_wait_for2<0>(vf[2], vf[3]);
      o_pair(vf[2], vf[3], 2);
    }
  }

  // ---- out[b, row, head, :] = O / l
  typedef typename M::elem elem4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const float l = fa_rows_sum(l_run[rb]);
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    const int row = r0 + 16 * rb + lc;
    if (row < p.q_len) {
      E* o = p.out + (((int64_t)b * p.q_len + row) * p.Hq + head) * D + 4 * lg;
#pragma unroll
      for (int dg = 0; dg < DG; ++dg) {
        elem4 e4;
#pragma unroll
        for (int v = 0; v < 4; ++v) e4[v] = (typename M::elem)(oacc[dg][rb][v] * inv);
        *(elem4*)(o + 16 * dg) = e4;
      }
    }
  }
}

template <typename E, int D>
int launch_prefill(const void* q, int64_t q_bs, int64_t q_hs, int64_t q_rs, const void* k, int64_t k_bs, int64_t k_rs,
                   const void* v, int64_t v_bs, int64_t v_rs, void* out, void* workspace, int B, int Hq, int Hkv, int S,
                   int q_len, float sm_scale, hipStream_t st) {
  const int n_tiles = fa_cdiv(S, kTileKeys);
  f16_t* vt = (f16_t*)workspace;
  prefill_vt_kernel<E, D><<<dim3(fa_cdiv(n_tiles, kVtTiles<D>), Hkv, B), 64, 0, st>>>((const E*)v, v_bs, v_rs, vt, S, Hkv, n_tiles);
  const int G = Hq / Hkv;
  PrefillParams<E> p{};
  p.q = (const E*)q; p.q_bs = q_bs; p.q_hs = q_hs; p.q_rs = q_rs;
  p.k = (const E*)k; p.k_bs = k_bs; p.k_rs = k_rs;
  p.vt = vt; p.out = (E*)out;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.S = S; p.q_len = q_len; p.n_tiles = n_tiles;
  p.HW = G % 4 == 0 ? 4 : G % 3 == 0 ? 3 : G % 2 == 0 ? 2 : 1;   // query heads of one KV head per workgroup
  p.RW = 4 / p.HW;                                                // blocks of 32 query rows per workgroup
  p.sm_log2e = sm_scale * 1.4426950408889634f;
  const int waves = p.HW * p.RW;
  dim3 grid(fa_cdiv(q_len, 32 * p.RW), Hkv * (G / p.HW), B);
  if (waves == 3) prefill_attn_kernel<E, D, 3><<<grid, 192, 0, st>>>(p);
  else prefill_attn_kernel<E, D, 4><<<grid, 256, 0, st>>>(p);
  return fa_check_launch("fa_prefill_attn");
}

}  // namespace

extern "C" size_t fa_prefill_attn_workspace_bytes(int B, int Hkv, int D, int S) {
  if (B <= 0 || Hkv <= 0 || D <= 0 || S <= 0) return 0;
  return (size_t)B * Hkv * fa_cdiv(S, kTileKeys) * kTileKeys * D * 2;
}

extern "C" int fa_prefill_attn(const void* q, int64_t q_batch_stride, int64_t q_head_stride, int64_t q_row_stride,
                               const void* k, const void* v, int64_t kv_batch_stride, int64_t kv_row_stride, void* out,
                               int dtype, int B, int Hq, int Hkv, int D, int S, int q_len, float sm_scale,
                               void* workspace, size_t workspace_bytes, fa_stream_t stream) {
  FA_REQUIRE(q && k && v && out, FA_ERR_NULL_POINTER, "fa_prefill_attn: null pointer");
  FA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && S > 0 && q_len > 0 && q_len <= S && Hq % Hkv == 0, FA_ERR_BAD_SHAPE,
             "fa_prefill_attn: B=%d Hq=%d Hkv=%d S=%d q_len=%d", B, Hq, Hkv, S, q_len);
  FA_REQUIRE(dtype == FA_BF16 || dtype == FA_FP16, FA_ERR_BAD_DTYPE,
             "fa_prefill_attn: dtype %d (the matrix cores take 16-bit operands)", dtype);
  FA_REQUIRE(D == 64 || D == 128, FA_ERR_UNSUPPORTED, "fa_prefill_attn: head_dim %d (64 or 128)", D);
  const size_t need = fa_prefill_attn_workspace_bytes(B, Hkv, D, S);
  FA_REQUIRE(workspace && workspace_bytes >= need, FA_ERR_WORKSPACE, "fa_prefill_attn: workspace %zu < %zu",
             workspace_bytes, need);
  FA_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)workspace) & 15) == 0 &&
                 ((q_batch_stride | q_head_stride | q_row_stride | kv_batch_stride | kv_row_stride) & 7) == 0,
             FA_ERR_MISALIGNED, "fa_prefill_attn: rows must be 16-byte aligned");
  FA_REQUIRE(B <= 65535 && Hq <= 65535, FA_ERR_UNSUPPORTED, "fa_prefill_attn: batch or head count above 65535");
  const float sm = sm_scale > 0.f ? sm_scale : 1.0f / sqrtf((float)D);
  hipStream_t st = fa_hip_stream(stream);
#define FA_PREFILL(E, DD)                                                                                              \
  return launch_prefill<E, DD>(q, q_batch_stride, q_head_stride, q_row_stride, k, kv_batch_stride, kv_row_stride, v,   \
                               kv_batch_stride, kv_row_stride, out, workspace, B, Hq, Hkv, S, q_len, sm, st)
  if (dtype == FA_BF16) {
    if (D == 128) FA_PREFILL(bf16_t, 128);
    FA_PREFILL(bf16_t, 64);
  }
  if (D == 128) FA_PREFILL(f16_t, 128);
  FA_PREFILL(f16_t, 64);
#undef FA_PREFILL
}
