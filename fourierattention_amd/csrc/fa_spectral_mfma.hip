// Spectral compression of a long prefill on the matrix cores (gfx950, wave64):
//   c[b, n, m]     = sum_k cos(2 pi (k + k_start) n / T) a[b, k, cols[m]]
//   c[b, N + n, m] = sum_k sin(...)                       a[b, k, cols[m]]
// (mat_fourier_triton TRI:81-102 / the FFT branch of MultiDimHiPPO2.forward TRI:858-865).
//
// The token axis is cut into steps of 128 tokens.  Inside a step the basis depends on the token offset
// only, E[n, i] = e^{i theta n i}, a constant f16 MFMA operand that every wave keeps in registers for its
// frequencies; the position of the step enters as one complex rotation per step and frequency:
//   sum_k e^{i theta n (p0 + k)} a[k] = e^{i theta n p0} * Horner_s( e^{i theta n 128}, G_s[n] ),
//   G_s[n] = sum_{i<128} E[n, i] a[128 s + i]
// so the steps are walked from the last to the first, acc <- G_s + e^{i theta n 128} acc, with the
// accumulators (fp32) never leaving registers.  Three kernels:
//   pack    evaluates the basis table, gathers the compressed columns of the token-major input, converts them to f16 and
//           writes them as ready-made MFMA B operands (column tile of 16, kstep of 32 tokens, 64 lanes x 8 tokens)
//   gemm    one workgroup = 128 frequencies x 64 columns x one chunk of steps; the operands of a step
//           travel HBM -> LDS with global_load_lds, one barrier per step
//   reduce  sums the chunks into c
#include "fa_mfma_util.h"

namespace fa_mfma {

constexpr int kStepTokens = 128;               // tokens per step (four MFMA ksteps)
constexpr int kStepK = kStepTokens / 32;
constexpr int kWgFreqs = 128;                  // frequencies per workgroup (four waves x four row tiles of 8)
constexpr int kWgCols = 64;                    // columns per workgroup (four column tiles of 16)

// ---- basis table: A operands E[row tile rt][kstep][lane] x half8, row r of a tile = frequency rt*8 + r/2,
// cos (r even) or sin (r odd); lane l holds row l % 16, tokens 8 * (l / 16) + e of the kstep ----------------
// A thread takes two tokens of a frequency and writes both rows: one evaluation per phase (a thread per row would
// evaluate every phase twice), short chains (7.4 -> 5.6 us for 512 frequencies).
// It needs nothing but N and T: the blocks of the table ride in the launch that packs the columns (as a launch of its own
// in front of the products: 3.8 - 6 us).
constexpr int kTableThreads = kStepK * 128;    // per row tile
__host__ __device__ inline int table_blocks(int N) { return (N / 8 * kTableThreads + 255) / 256; }
__device__ __forceinline__ void spectral_table_block(half2v* __restrict__ tab, int N, int T, int block) {
  const int idx = block * 256 + threadIdx.x;
  if (idx >= (N / 8) * kTableThreads) return;
  const int ep = idx & 3, f = (idx >> 2) & 7, lg = (idx >> 5) & 3, frag = idx >> 7;   // frag = rt * kStepK + ks
  const int n = frag / kStepK * 8 + f, token = frag % kStepK * 32 + 8 * lg + 2 * ep;
  half2v c, s;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    float sn, co;
    fa_sincos_phase(n, token + e, T, &sn, &co);
    c[e] = (_Float16)co;
    s[e] = (_Float16)sn;
  }
  half2v* out = tab + ((int64_t)frag * 64 + lg * 16 + 2 * f) * 4 + ep;
  out[0] = c;
  out[4] = s;
}
struct SpectralTable {
  half2v* tab;
  int N, T;
};

// ---- pack: block = 32 tokens x 256 columns; lanes run along the columns for the gather, the transposition to
// token-contiguous fragments goes through LDS.  grid (ksteps + blocks of the basis table, column blocks, parts * B): part p of
// the input starts p * a_part elements behind the first and its fragments p * out_part behind the first's; with
// col_inv_scale the columns are scaled ------
template <typename E>
__global__ __launch_bounds__(256) void spectral_pack_kernel(
    const E* __restrict__ a, int64_t a_bs, int64_t a_rs, const int32_t* __restrict__ cols,
    const float* __restrict__ col_inv_scale, half8* __restrict__ out, int K, int Mc, int CT, int KS32, int B, int64_t a_part,
    int64_t out_part, const SpectralTable st) {
  constexpr int kPitch = 256 + 4;   // f16 elements per LDS row: 8 rows apart = 16 banks apart
  __shared__ _Float16 tile[32][kPitch];
  if ((int)blockIdx.x >= KS32) {
    spectral_table_block(st.tab, st.N, st.T, ((int)blockIdx.x - KS32) * gridDim.y * gridDim.z + blockIdx.z * gridDim.y + blockIdx.y);
    return;
  }
  const int tid = threadIdx.x;
  const int ks = blockIdx.x, m0 = blockIdx.y * 256, part = blockIdx.z / B, b = blockIdx.z - part * B;
  a += part * a_part;
  out += part * out_part;
  const int m = m0 + tid;
  const bool mok = m < Mc;
  const int col = mok ? (cols ? cols[m] : m) : 0;
  const E* ab = a + (int64_t)b * a_bs + col;
  const float mul = (col_inv_scale && mok) ? col_inv_scale[(int64_t)b * Mc + m] : 1.f;
  float v[32];
#pragma unroll
  for (int kk = 0; kk < 32; ++kk) {
    const int k = ks * 32 + kk;
    v[kk] = fa_to_float(ab[(int64_t)min(k, K - 1) * a_rs]);
  }
#pragma unroll
  for (int kk = 0; kk < 32; ++kk) {
    const int k = ks * 32 + kk;
    // f16 holds every bf16 / f16 value of magnitude below 65504 exactly (tiny ones as subnormals)
    const float x = (mok && k < K) ? fminf(fmaxf(v[kk] * mul, -65504.f), 65504.f) : 0.f;
    tile[kk][tid] = (_Float16)x;
  }
  __syncthreads();
  // 16 column tiles x 64 lanes of fragments, four per thread
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int f = i * 256 + tid;
    const int ctl = f >> 6, lane = f & 63;
    const int lc = lane & 15, lg = lane >> 4;
    const int ct = (m0 >> 4) + ctl;
    if (ct >= CT) continue;
    half8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = tile[8 * lg + e][ctl * 16 + lc];
    out[(((int64_t)b * CT + ct) * KS32 + ks) * 64 + lane] = o;
  }
}

// ---- one pass over the prompt's K (or V) rows for everything the cache's prefill needs from them -------------------
// block = (PPB consecutive pages of 32 tokens, KV head, batch element); the head's slice of the rows goes through LDS
// once and leaves as
//   pages      the stored dims in the page layout of the decode kernels (what fa_mid_pack writes),
//   fragments  the compressed dims as f16 B operands of the compression GEMM (what spectral_pack_kernel writes; a
//              column tile that two heads share is written by both, each its own 16-byte pieces),
//   partials   sum / max / min of every compressed column over the block's tokens (what col_stats_partial_kernel
//              leaves, finished by the same final launch).
// Blocks take up to four pages one after the other; a prompt too short to fill the chip that way - four blocks for every
// compute unit - takes fewer a block.  Packing and compressing, us, four pages -> by this rule: 3001 tokens x 4 sequences
// x 8 heads 55.6 -> 50.8, 3000 x 1 x 8 32.7 -> 27.3, 1800 x 1 x 8 29.5 -> 24.4; from 1024 blocks on (5000 x 8 x 8,
// 32768 x 1 x 8 and 12000 x 2 x 8) the rule is the same as before: 57, 77.6 and 102.6 both.
inline int pack_pages_per_block(int n_pages, int heads_x_batch) {
  int per = 4;
  while (per > 1 && (int64_t)fa_cdiv(n_pages, per) * heads_x_batch < 1024) per >>= 1;
  return per;
}

template <typename E>
struct PrefillPackParams {
  const E* src;
  int64_t src_bs, src_rs, row0;
  int L, K_fft;                 // mid rows; rows that enter the transform (K_fft <= L)
  E* store;                     // paged store of the stored dims
  int64_t st_bs;
  int cap_pages;
  const int32_t* n_list; const int32_t* n_h; const int32_t* pad_h;   // stored dims: flat h*D + d, per-head offsets
  const int32_t* c_list; const int32_t* c_h;                         // compressed dims, likewise
  half8* packed;                // [B][CT][KS32][64]
  float* psum; float* pmax; float* pmin;   // [B][n_blocks][Mc]
  int Mc, CT, KS32, n_pages, per_block, n_blocks, Hkv, D, is_v;
  SpectralTable table;          // the blocks of x behind n_blocks evaluate the basis of the products
};

template <typename E>
__global__ __launch_bounds__(256) void prefill_pack_kernel(const PrefillPackParams<E> p) {
  constexpr int kMaxD = 256;
  constexpr int kPitch = kMaxD + 8;                 // elements; keeps rows 16-byte aligned
  struct alignas(sizeof(E) * 8) Piece { E v[8]; };
  __shared__ __attribute__((aligned(32))) E tile[32][kPitch];
  __shared__ int s_col[kMaxD];                      // dim within the head of every stored position
  __shared__ int s_ccol[kMaxD];                     // ... of every compressed position
  const int h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, D = p.D;
  if ((int)blockIdx.x >= p.n_blocks) {
    spectral_table_block(p.table.tab, p.table.N, p.table.T, ((int)blockIdx.x - p.n_blocks) * gridDim.y * gridDim.z + b * gridDim.y + h);
    return;
  }
  const int n0 = p.n_h[h], n_len = p.n_h[h + 1] - n0;
  const int p0 = p.pad_h[h], dp = p.pad_h[h + 1] - p0;
  const int c0 = p.c_h[h], c_len = p.c_h[h + 1] - c0;
  for (int j = tid; j < dp; j += 256) s_col[j] = n_len > 0 ? min(max(p.n_list[n0 + min(j, n_len - 1)] - h * D, 0), D - 1) : 0;
  for (int j = tid; j < c_len; j += 256) s_ccol[j] = min(max(p.c_list[c0 + j] - h * D, 0), D - 1);
  const E* sb = p.src + (int64_t)b * p.src_bs + p.row0 * p.src_rs + (int64_t)h * D;
  const int ppr = D >> 3;                           // 16-byte pieces per row of the head
  const int pages_of_rows = (p.L + 31) >> 5;
  // columns past the last compressed dim in the last column tile belong to nobody: the last head clears them
  const int c_extra = h == p.Hkv - 1 ? p.CT * 16 - p.Mc : 0;
  float sum = 0.f, mx = -INFINITY, mn = INFINITY;   // thread j < c_len: statistics of its column
  for (int pp = 0; pp < p.per_block; ++pp) {
    const int page = blockIdx.x * p.per_block + pp;
    if (page >= p.n_pages) break;
    __syncthreads();                                // the tile of the page before has been read (and the lists stored)
    if (page < pages_of_rows) {
      const int64_t last = (int64_t)p.L - 1;
      for (int q = tid; q < 32 * ppr; q += 256) {
        const int t = q / ppr, c = q - t * ppr;
        const int64_t token = (int64_t)page * 32 + t;
        *(Piece*)&tile[t][c * 8] = *(const Piece*)(sb + (token < last ? token : last) * p.src_rs + c * 8);
      }
    }
    __syncthreads();
    // ---- pages of the stored dims
    if (page < pages_of_rows && n_len > 0) {
      Piece* out = (Piece*)(p.store + (int64_t)b * p.st_bs + (int64_t)p0 * 32 * p.cap_pages + (int64_t)page * dp * 32);
      const int n_pieces = dp * 32 / 8;
      for (int piece = tid; piece < n_pieces; piece += 256) {
        const int frag = piece >> 6, lane = piece & 63;
        Piece o;
        if (!p.is_v) {
          const int nks = dp >> 5;
          const int tb = frag / nks, s_ = frag - tb * nks;
          const int t = tb * 16 + (lane & 15), j0 = s_ * 32 + 8 * (lane >> 4);
          const bool row_ok = (int64_t)page * 32 + t < p.L;
#pragma unroll
          for (int e = 0; e < 8; ++e) o.v[e] = (row_ok && j0 + e < n_len) ? tile[t][s_col[j0 + e]] : E{};
        } else {
          const int j = frag * 16 + (lane & 15);
          const int col = s_col[j];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int t = 8 * (lane >> 4) + i;
            o.v[i] = (j < n_len && (int64_t)page * 32 + t < p.L) ? tile[t][col] : E{};
          }
        }
        out[piece] = o;
      }
    }
    // ---- f16 fragments of the compressed dims (tokens past the transform's rows are zero)
    if (page < p.KS32) {
      for (int idx = tid; idx < (c_len + c_extra) * 4; idx += 256) {
        const int j = idx >> 2, lg = idx & 3;
        const int m = c0 + j;                       // column of the compressed matrix
        half8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int t = 8 * lg + e;
          float x = 0.f;
          if (j < c_len && (int64_t)page * 32 + t < p.K_fft) x = fminf(fmaxf(fa_to_float(tile[t][s_ccol[j]]), -65504.f), 65504.f);
          o[e] = (_Float16)x;
        }
        p.packed[(((int64_t)b * p.CT + (m >> 4)) * p.KS32 + page) * 64 + lg * 16 + (m & 15)] = o;
      }
    }
    // ---- column statistics over the mid rows
    if (tid < c_len && page < pages_of_rows) {
      const int col = s_ccol[tid];
      const int n_t = min(32, p.L - page * 32);
      for (int t = 0; t < n_t; ++t) {
        const float v = fa_to_float(tile[t][col]);
        sum += v;
        mx = fmaxf(mx, v);
        mn = fminf(mn, v);
      }
    }
  }
  if (tid < c_len) {
    const int64_t o = ((int64_t)b * p.n_blocks + blockIdx.x) * p.Mc + c0 + tid;
    p.psum[o] = sum;
    p.pmax[o] = mx;
    p.pmin[o] = mn;
  }
}

// One step of the Horner walk: acc <- E * (the step's four column tiles in LDS) + rotation * acc.  The tiles of a kstep
// ((j, ks) at lds + (4 j + ks) KiB) are requested one kstep ahead of the products that take them, the first ones in
// front of the rotation, which has 128 vector instructions to cover them: a wave that read and then waited spent longer
// on LDS latency than on its matrix instructions.  No branch between a request and its wait (accumulators start as
// zeros, which rotate to zeros).  32768 rows x 512 columns, 512 frequencies: 37.8 -> 34.8 us (990 TFLOP/s).
__device__ __forceinline__ void spectral_step(float4v (&acc)[4][4], const half8 (&Ea)[4][kStepK], const float (&rc)[4][2],
                                              const float (&rs)[4][2], unsigned lds) {
  uint4v b0[4], b1[4];
#define FA_STEP_READ(B, ks)                                   \
  B[0] = lds_read_b128_async_at<(0 * kStepK + (ks)) * 1024>(lds); \
  B[1] = lds_read_b128_async_at<(1 * kStepK + (ks)) * 1024>(lds); \
  B[2] = lds_read_b128_async_at<(2 * kStepK + (ks)) * 1024>(lds); \
  B[3] = lds_read_b128_async_at<(3 * kStepK + (ks)) * 1024>(lds)
  auto products = [&](const uint4v (&b)[4], int ks) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ea[i][ks], __builtin_bit_cast(half8, b[j]), acc[i][j], 0, 0, 0);
  };
  static_assert(kStepK == 4, "four ksteps, two register sets");
  FA_STEP_READ(b0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int f2 = 0; f2 < 2; ++f2) {
        const float c = acc[i][j][2 * f2], sn = acc[i][j][2 * f2 + 1];
        // (spelled out: left to itself the compiler rounds the one product for some tiles and the other for the rest)
        acc[i][j][2 * f2] = __builtin_fmaf(rc[i][f2], c, -(rs[i][f2] * sn));
        acc[i][j][2 * f2 + 1] = __builtin_fmaf(rc[i][f2], sn, rs[i][f2] * c);
      }
  FA_STEP_READ(b1, 1);
  lds_wait_for4<4>(b0);
  products(b0, 0);
  FA_STEP_READ(b0, 2);
  lds_wait_for4<4>(b1);
  products(b1, 1);
  FA_STEP_READ(b1, 3);
  lds_wait_for4<4>(b0);
  products(b0, 2);
  lds_wait_for4<0>(b1);
  products(b1, 3);
#undef FA_STEP_READ
}

struct SpectralGemmParams {
  const half8* tab;      // basis table
  const half8* packed;   // [B][CT][KS32][64] fragments
  float* part;           // [S][B][2N][Mc]; with a single chunk: the result c itself (no reduction launch)
  int add_to_part;       // single chunk only: add to what part holds instead of overwriting it
  int B, N, Mc, CT, KS32, T;
  int n_steps, steps_per_chunk, n_chunks;
  int64_t k_start;
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void spectral_gemm_kernel(const SpectralGemmParams p) {
  constexpr int NST = 4;   // steps in LDS: the one in use and three on their way
  __shared__ __attribute__((aligned(16))) unsigned char s_stage[NST][4][kStepK][1024];
  const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.z / p.n_chunks, chunk = blockIdx.z - b * p.n_chunks;
  const int rt0 = (blockIdx.y * 4 + w) * 4;          // first of this wave's four row tiles
  const int ct0 = blockIdx.x * 4;                    // first of the workgroup's four column tiles
  const int n_rt = p.N / 8;
  const int s_beg = chunk * p.steps_per_chunk;
  const int s_end = min(p.n_steps, s_beg + p.steps_per_chunk);
  const int n_it = s_end - s_beg;

  // this wave stages column tile w of every step (clamped: a tile past the end repeats the last one)
  const int ct_mine = min(ct0 + w, p.CT - 1);
  const _Float16* src = (const _Float16*)(p.packed + (((int64_t)b * p.CT + ct_mine) * p.KS32) * 64) + lane * 8;
  auto issue = [&](int s, int stage) {
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks)
      load_frag_to_lds(src + (int64_t)(s * kStepK + ks) * 512, &s_stage[stage][w][ks][0]);
  };
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < n_it) issue(s_end - 1 - i, i);

  half8 Ea[4][kStepK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks) Ea[i][ks] = p.tab[((int64_t)min(rt0 + i, n_rt - 1) * kStepK + ks) * 64 + lane];
  // per frequency of this lane (row tile i, pair f2): rotation of one step
  float rc[4][2], rs[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int f2 = 0; f2 < 2; ++f2) fast_sincos_phase(min(rt0 + i, n_rt - 1) * 8 + lg * 2 + f2, kStepTokens, p.T, &rs[i][f2], &rc[i][f2]);
  float4v acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  // the table loads must have landed before the loop: inside it the only waits on vector memory are explicit
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks) asm volatile("" ::"v"(Ea[i][ks]));

  for (int it = 0; it < n_it; ++it) {
    const int s = s_end - 1 - it, stage = it % NST;
    if (it + NST - 2 < n_it) wait_vmcnt<(NST - 2) * kStepK>();   // the steps behind this one may still be in flight
    else wait_vmcnt<0>();
    barrier_lds_only();   // every wave's share of step s has landed; nobody still reads the stage refilled next
    if (it + NST - 1 < n_it) issue(s - (NST - 1), (it + NST - 1) % NST);
    spectral_step(acc, Ea, rc, rs, lds_addr_of(&s_stage[stage][0][0][lane * 16]));
  }

  // into the common frame (phase of the chunk's first token) and out
  const int64_t p0 = (int64_t)s_beg * kStepTokens + p.k_start;
  float* out = p.part + ((int64_t)chunk * p.B + b) * 2 * p.N * p.Mc;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (rt0 + i >= n_rt) continue;
#pragma unroll
    for (int f2 = 0; f2 < 2; ++f2) {
      const int n = (rt0 + i) * 8 + lg * 2 + f2;
      float sn, co;
      fast_sincos_phase(n, p0, p.T, &sn, &co);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = (ct0 + j) * 16 + lc;
        if (m < p.Mc) {
          const float c = acc[i][j][2 * f2], s_ = acc[i][j][2 * f2 + 1];
          float* oc = out + (int64_t)n * p.Mc + m;
          float* os = out + (int64_t)(p.N + n) * p.Mc + m;
          const float vc = co * c - sn * s_, vs = sn * c + co * s_;
          *oc = p.add_to_part ? *oc + vc : vc;
          *os = p.add_to_part ? *os + vs : vs;
        }
      }
    }
  }
}

__global__ __launch_bounds__(256) void spectral_reduce_kernel(const float* __restrict__ part, float* __restrict__ c,
                                                              int64_t total, int n_chunks, int accumulate) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;   // total is a multiple of 16 whatever Mc is: 2N is one
  float4 a = accumulate ? *(const float4*)(c + i) : make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s = 0; s < n_chunks; ++s) {
    const float4 v = *(const float4*)(part + (int64_t)s * total + i);
    a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
  }
  *(float4*)(c + i) = a;
}

// ---------------------------------------------------------------------------------------------------------
// Statistics of the reconstruction (mat_fourier_avg_std_triton, TRI:285-326):
//   r[k, m] = (1/N) sum_n cos(theta k n) c[n, m] + sin(theta k n) s[n, m],     s[n] = c[N + n]
// The roles of position and frequency are those of the compression exchanged: rows are the positions k, and the
// contraction runs over the coefficient index n, cut into steps of 127.  A step is taken from its centre n_c = 127 t:
// with the coefficients folded, c+ = c[n_c + j] + c[n_c - j] and c- = c[n_c + j] - c[n_c - j] for the 64 offsets j = 0 .. 63
// (c+ = c- = c[n_c] for j = 0),
//   sum over the step of cos(theta k n) c[n] = cos(phi) . (E_cos c+) - sin(phi) . (E_sin c-)
//   sum over the step of sin(theta k n) s[n] = sin(phi) . (E_cos s+) + cos(phi) . (E_sin s-),      phi = theta k n_c
// so that the matrix cores compute real sums only, half of what two complex ones (basis rows cos and sin for every
// coefficient, one accumulator of the two used) take, and a step ends in two multiply-adds per sum instead of a complex
// rotation.  The fold happens in 32 bits ahead of the rounding to f16, scaled by a power of two per column (the range of
// coefficients is not bounded).
// The lowest frequencies carry the mean, the drift and the slow oscillations of a signal, often its largest part, and theirs
// are the largest errors.  Step 0 has no lower half, so cosines meet c and sines meet s, and the fragments that
// c- and s+ would take hold what the rounding of c and s leaves over; the extremes of a slow column fall on a basis of one.
// The coefficient of frequency 0 stays out of the products altogether and is added in 32 bits.  (Steps of 128 from
// their centres 63.5, .. need one step less, but there c[1] meets the rounded basis of offset 62.5: columns with a drift
// had their deviation off by 1.07e-4 instead of the 7.6e-5 of a basis that is not folded.)
// Position k gives r[k] = A_k + B_k (A cosine, B sine part) and, because the period is a whole number of positions, also
// its mirror image r[T - k] = A_k - B_k: only the positions up to T / 2 are computed, each standing for two where the
// sequence reaches past T / 2.
// Bound by the matrix cores and the LDS reads that feed them (a fragment feeds four products).
// us, all launches (complex sums on coefficients packed by launches of their own -> now; steps of 128 without the second
// term of step 0 in brackets): 32768 positions x 512 columns, 512 frequencies 73.1 -> 48.9 (44.3); eight tensors of 31740 positions
// 296 -> 190 (164), four of 1977 x 910 54.7 -> 39.9 (36.4), two of 9000 x 300 with 128 frequencies 26.2 -> 18.5 (17.1).  Relative
// error of the deviation against 64 bits, rms over the columns, same three: 31740 x 512 of a period of 130044, noise
// 4.04e-5 -> 3.77e-5 (4.03e-5), mean of twice the noise 1.67e-4 -> 8.4e-5 (1.87e-4), drift 7.6e-5 -> 4.3e-5 (1.07e-4); 32768 of 32768,
// drift 5.3e-5 -> 4.3e-5 (7.9e-5).  The mean, over the deviation: 2.1e-4 -> 1.8e-6 (1.1e-4) with a mean, 2.8e-6 -> 1.9e-7 (1.7e-6)
// without.
// ---------------------------------------------------------------------------------------------------------
constexpr int kRecPos = 256;      // positions of a workgroup: four waves x four tiles of 16
constexpr int kRecCols = 32;      // columns of a unit of work: two tiles of 16
constexpr int kRecStep = 127;     // coefficient indices of a step: its centre and 63 to either side (step 0: above it only)
constexpr int kRecHalf = 64;      // offsets of a step
constexpr int kRecFrags = 8;      // fragments of a step and column tile: {c+, c-, s+, s-} x two ksteps of 32 offsets
__host__ __device__ inline int recon_steps(int N) { return N <= kRecHalf ? 1 : 1 + (N - kRecHalf + kRecStep - 1) / kRecStep; }
constexpr int kMaxColShare = 8;   // units of a workgroup at most

struct ReconPrepParams {
  const float* c;     // [B][2N][Mc]
  half8* packed;      // [B][CT][n_steps][kRecFrags][64]
  float* scale;       // [B][Mc]
  half2v* tab;        // [position tiles][cos k0, cos k1, sin k0, sin k1][64] x half8
  float* phi;         // [row blocks][n_steps][cos, sin][kRecPos]
  int B, N, Mc, CT, T, n_steps;
};

// Everything the statistics need, in one launch of 1024 threads a block: the first CT * B blocks fold and pack a column tile
// each (thread = column, offset), the rest evaluate the basis of 32 positions and their phases at the steps.
__global__ __launch_bounds__(1024) void recon_prep_kernel(const ReconPrepParams p) {
  constexpr int kHold = 8;   // steps whose coefficients a thread holds between the maximum and the scaling
  constexpr int kOut = 4;    // steps that leave through LDS at a time
  __shared__ float s_mx[64][16];
  __shared__ __attribute__((aligned(16))) _Float16 s_out[kOut * kRecFrags * 512];
  const int tid = threadIdx.x;
  int blk = blockIdx.x;
  if (blk >= p.CT * p.B) {
    blk -= p.CT * p.B;   // 32 positions: two tiles, thread = (tile, kstep, lane group, position, pair of offsets)
    const int ep = tid & 3, lc = (tid >> 2) & 15, lg = (tid >> 6) & 3, kk = (tid >> 8) & 1, tile = blk * 2 + (tid >> 9);
    half2v co2, sn2;
    float own = 0.f;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float sn, co;
      fa_sincos_phase(tile * 16 + lc, 32 * kk + 8 * lg + 2 * ep + e, p.T, &sn, &co);
      co2[e] = (_Float16)co;
      sn2[e] = (_Float16)sn;
      own = fmaf((float)co2[e], co, fmaf((float)sn2[e], sn, own));
    }
    half2v* out = p.tab + ((int64_t)(tile * 4 + kk) * 64 + lg * 16 + lc) * 4 + ep;
    out[0] = co2;
    out[2 * 64 * 4] = sn2;
    // A rounded basis answers its own position with a sum of squares that is not quite 64: the phases carry the
    // reciprocal, so that what is coherent with the position - the signal at its extremes - comes out unscaled.  (Step 0
    // takes no phases.)
    float* s_own = &s_mx[0][0];   // [32 positions][32]
    s_own[((tid >> 9) * 16 + lc) * 32 + (kk * 4 + lg) * 4 + ep] = own;
    __syncthreads();
    const int pos = tid & 31;
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < 32; ++k) sum += s_own[pos * 32 + ((k + pos) & 31)];   // (rotated: no two lanes on one bank)
    const float unit = 64.0f / sum;
    const int k = blk * 32 + pos, rb = k / kRecPos;
    for (int t = tid >> 5; t < p.n_steps; t += 32) {
      float sn, co;
      fa_sincos_phase(k, kRecStep * t, p.T, &sn, &co);
      float* o = p.phi + ((int64_t)(rb * p.n_steps + t) * 2) * kRecPos + k % kRecPos;
      o[0] = co * unit;
      o[kRecPos] = sn * unit;
    }
    return;
  }
  const int ct = blk % p.CT, b = blk / p.CT;
  const int lc = tid & 15, i = tid >> 4, m = ct * 16 + lc;
  const float* cb = p.c + (int64_t)b * 2 * p.N * p.Mc + min(m, p.Mc - 1);
  float v[kHold][4];   // cos rows above and below the centre, sin rows likewise; zeros where there are none
  auto load = [&](int t0) {
#pragma unroll
    for (int u = 0; u < kHold; ++u)
      if (t0 + u < p.n_steps) {
        const int hi = (t0 + u) * kRecStep + i, lo = (t0 + u) * kRecStep - i;
        const int hc = min(hi, p.N - 1), lc0 = min(max(lo, 0), p.N - 1);
        v[u][0] = cb[(int64_t)hc * p.Mc];
        v[u][1] = cb[(int64_t)lc0 * p.Mc];
        v[u][2] = cb[(int64_t)(p.N + hc) * p.Mc];
        v[u][3] = cb[(int64_t)(p.N + lc0) * p.Mc];
        // (frequency 0 is added behind the products; step 0 has nothing below its centre, and the centre counts once)
        if (hi == 0 || hi >= p.N) v[u][0] = v[u][2] = 0.f;
        if (lo <= 0 || lo >= p.N || i == 0) v[u][1] = v[u][3] = 0.f;
      }
  };
  float mx = 0.f;
  for (int t0 = 0; t0 < p.n_steps; t0 += kHold) {
    load(t0);
#pragma unroll
    for (int u = 0; u < kHold; ++u)
      if (t0 + u < p.n_steps)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[u][0]), fabsf(v[u][1])), fmaxf(fabsf(v[u][2]), fabsf(v[u][3]))));
  }
  s_mx[i][lc] = mx;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 64; ++k) mx = fmaxf(mx, s_mx[k][lc]);
  // power of two: scaling is exact.  (Columns of nothing but tiny values are not scaled into the denormals' reciprocal.)
  const float sc = mx > 0.f ? exp2f(fmaxf(ceilf(log2f(mx)), -100.f)) : 1.f, inv = 1.0f / sc;
  if (i == 0 && m < p.Mc) p.scale[(int64_t)b * p.Mc + m] = sc;
  half8* out = p.packed + ((int64_t)(b * p.CT + ct) * p.n_steps) * kRecFrags * 64;
  const int at = ((i >> 5) * 64 + ((i >> 3) & 3) * 16 + lc) * 8 + (i & 7);   // of offset i in a pair of fragments
  for (int t0 = 0; t0 < p.n_steps; t0 += kHold) {
    if (p.n_steps > kHold) load(t0);
#pragma unroll
    for (int u0 = 0; u0 < kHold; u0 += kOut) {
      if (t0 + u0 >= p.n_steps) break;
#pragma unroll
      for (int u = 0; u < kOut; ++u)
        if (t0 + u0 + u < p.n_steps) {
          const float own = m < p.Mc ? inv : 0.f;
          const float ch = v[u0 + u][0] * own, cl = v[u0 + u][1] * own, sh = v[u0 + u][2] * own, sl = v[u0 + u][3] * own;
          const bool first = t0 + u0 + u == 0;
          const _Float16 cp = (_Float16)(ch + cl), sp = (_Float16)(sh + sl);
          _Float16* o = s_out + u * kRecFrags * 512 + at;
          o[0 * 1024] = cp;
          o[1 * 1024] = (_Float16)(ch - (first ? (float)cp : cl));   // step 0: what the rounding leaves over
          o[2 * 1024] = sp;
          o[3 * 1024] = (_Float16)(sh - (first ? (float)sp : sl));
        }
      __syncthreads();
      const int n = min(kOut, p.n_steps - t0 - u0) * kRecFrags * 64;
      for (int k = tid; k < n; k += 1024) out[(int64_t)(t0 + u0) * kRecFrags * 64 + k] = ((const half8*)s_out)[k];
      __syncthreads();
    }
  }
}

struct ReconStatsParams {
  const float* c;
  const half8* tab;
  const half8* packed;
  const float* phi;
  const float* scale;
  float* psum;
  float* pmax;
  float* pmin;   // [B][RB][Mc]
  int B, N, Mc, CT, K, T, n_steps, RB;
  int cb_per;    // units (column blocks) of a workgroup
  int Kd;        // positions computed directly: min(K, T / 2 + 1)
  int half;      // T / 2: mirror images beyond it count as positions of their own (a value no position exceeds
                 // when the sequence is longer than the period and every position is computed directly)
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void spectral_recon_stats_kernel(
    const ReconStatsParams p) {
  constexpr int NST = 3;                                // steps in LDS: the one in use and two on their way
  constexpr int kStage = 2 * kRecFrags * 1024 + 2048;   // the fragments of two column tiles, the phases of the positions
  __shared__ __attribute__((aligned(16))) unsigned char s_stage[NST][kStage];
  __shared__ float s_stat[3][4][kMaxColShare * kRecCols];   // sum / max / min, by wave and column
  const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rb = blockIdx.x, b = blockIdx.y;
  const int S = p.n_steps;
  const int cb0 = blockIdx.z * p.cb_per;
  const int n_cb = min((p.Mc + kRecCols - 1) / kRecCols - cb0, p.cb_per);
  const int Q = n_cb * S;

  int next_cb = cb0, next_s = 0;   // the step requested next
  auto issue = [&](int stage) {
    // wave w: four fragments of column tile w / 2 (clamped: a tile past the end repeats the last one); the first two
    // waves bring the phases as well
    const int ct = min(next_cb * 2 + (w >> 1), p.CT - 1);
    const half8* src = p.packed + (((int64_t)(b * p.CT + ct) * S + next_s) * kRecFrags + (w & 1) * 4) * 64 + lane;
#pragma unroll
    for (int f = 0; f < 4; ++f) load_frag_to_lds(src + f * 64, &s_stage[stage][(w * 4 + f) * 1024]);
    if (w < 2) load_frag_to_lds(p.phi + ((int64_t)(rb * S + next_s) * 2 + w) * kRecPos + 4 * lane, &s_stage[stage][(16 + w) * 1024]);
    if (++next_s == S) {
      next_s = 0;
      ++next_cb;
    }
  };
  half8 Ec[4][2], Es[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half8* t = p.tab + ((int64_t)(rb * (kRecPos / 16) + w * 4 + i) * 4) * 64 + lane;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      Ec[i][kk] = t[kk * 64];
      Es[i][kk] = t[(2 + kk) * 64];
    }
  }
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < Q) issue(i);
  float4v A[4][2], Bs[4][2];   // (step 0 of a column block starts them)
  // (the table must have landed before the loop: inside it the only waits on vector memory are explicit)
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) asm volatile("" ::"v"(Ec[i][kk]), "v"(Es[i][kk]));

  const int kw = rb * kRecPos + w * 64;   // first position of the wave
  const bool all_in = kw + 63 < p.Kd;
  const bool mirror_all = all_in && p.T - (kw + 63) > p.half && p.T - kw < p.K;
  const bool mirror_none = p.T - kw <= p.half || p.T - (kw + 63) >= p.K;
  int it = -1, cbl = 0;
  for (int q = 0; q < Q; ++q) {
    if (++it == S) {
      it = 0;
      ++cbl;
    }
    const int stage = q % NST;
    if (q + NST - 2 >= Q) wait_vmcnt<0>();
    else if (w < 2) wait_vmcnt<(NST - 2) * 5>();
    else wait_vmcnt<(NST - 2) * 4>();
    barrier_lds_only();   // every wave's share of the step has landed; nobody still reads the stage refilled next
    if (q + NST - 1 < Q) issue((q + NST - 1) % NST);
    const unsigned st = lds_addr_of(&s_stage[stage][0]), fr = st + lane * 16, ph = st + 16 * 1024 + (w * 64 + 4 * lg) * 4;
    uint4v pc[4], ps[4], b0[4], b1[4];
    pc[0] = lds_read_b128_async_at<0>(ph);
    pc[1] = lds_read_b128_async_at<64>(ph);
    pc[2] = lds_read_b128_async_at<128>(ph);
    pc[3] = lds_read_b128_async_at<192>(ph);
    ps[0] = lds_read_b128_async_at<1024 + 0>(ph);
    ps[1] = lds_read_b128_async_at<1024 + 64>(ph);
    ps[2] = lds_read_b128_async_at<1024 + 128>(ph);
    ps[3] = lds_read_b128_async_at<1024 + 192>(ph);
#define FA_REC_READ(B, G)                                       \
  B[0] = lds_read_b128_async_at<((G) * 4 + 0) * 1024>(fr);      \
  B[1] = lds_read_b128_async_at<((G) * 4 + 1) * 1024>(fr);      \
  B[2] = lds_read_b128_async_at<((G) * 4 + 2) * 1024>(fr);      \
  B[3] = lds_read_b128_async_at<((G) * 4 + 3) * 1024>(fr)
    // one column tile's cosine or sine coefficients: f = {+ k0, + k1, - k0, - k1}; step 0: {c k0, c k1, rest k0, rest k1}
    auto products = [&](const uint4v (&f)[4], float4v (&acc)[4][2], int j, bool sine) {
      float4v C[4], D[4];
      if (it == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(sine ? Es[i][k & 1] : Ec[i][k & 1], __builtin_bit_cast(half8, f[k]),
                                                               k ? acc[i][j] : float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        return;
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          C[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ec[i][kk], __builtin_bit_cast(half8, f[kk]),
                                                        kk ? C[i] : float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          D[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Es[i][kk], __builtin_bit_cast(half8, f[2 + kk]),
                                                        kk ? D[i] : float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4v co = __builtin_bit_cast(float4v, pc[i]), sn = __builtin_bit_cast(float4v, ps[i]);
        acc[i][j] += (sine ? sn : co) * C[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4v co = __builtin_bit_cast(float4v, pc[i]), sn = __builtin_bit_cast(float4v, ps[i]);
        if (sine) acc[i][j] += co * D[i];
        else acc[i][j] -= sn * D[i];
      }
    };
    FA_REC_READ(b0, 0);
    lds_wait_for4<8>(pc);
    lds_wait_for4<4>(ps);
    FA_REC_READ(b1, 1);
    lds_wait_for4<4>(b0);
    products(b0, A, 0, false);
    FA_REC_READ(b0, 2);
    lds_wait_for4<4>(b1);
    products(b1, Bs, 0, true);
    FA_REC_READ(b1, 3);
    lds_wait_for4<4>(b0);
    products(b0, A, 1, false);
    lds_wait_for4<0>(b1);
    products(b1, Bs, 1, true);
#undef FA_REC_READ
    if (it != S - 1) continue;
    // the column block is complete: r = A +- B (the scale follows behind the loop) at this lane's 16 positions per column
    // and at their mirror images
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float sum = 0.f, mx = -INFINITY, mn = INFINITY;
      if (mirror_all) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float a = A[i][j][v], bb = Bs[i][j][v], hi = a + bb, lo = a - bb;
            sum += a;
            mx = fa_fmax(fa_fmax(mx, hi), lo);
            mn = fa_fmin(fa_fmin(mn, hi), lo);
          }
        sum += sum;
      } else if (all_in && mirror_none) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float r = A[i][j][v] + Bs[i][j][v];
            sum += r;
            mx = fa_fmax(mx, r);
            mn = fa_fmin(mn, r);
          }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int k = kw + i * 16 + 4 * lg + v;
            const float r = A[i][j][v] + Bs[i][j][v], r2 = A[i][j][v] - Bs[i][j][v];
            if (k < p.Kd) {
              sum += r;
              mx = fa_fmax(mx, r);
              mn = fa_fmin(mn, r);
            }
            const int km = p.T - k;   // the mirror image counts where it is a position of its own beyond T / 2
            if (k < p.Kd && km > p.half && km < p.K) {
              sum += r2;
              mx = fa_fmax(mx, r2);
              mn = fa_fmin(mn, r2);
            }
          }
      }
      sum = fa_rows_sum(sum);
      mx = fa_rows_max(mx);
      mn = fa_rows_min(mn);
      if (lg == 0) {
        // (written past the compiler, which would wait for the tiles on their way first)
        const unsigned at = lds_addr_of(&s_stat[0][w][cbl * kRecCols + j * 16 + lc]);
        constexpr int kKind = 4 * kMaxColShare * kRecCols * 4;   // bytes
        asm volatile("ds_write_b32 %0, %1\n\tds_write_b32 %0, %2 offset:%4\n\tds_write_b32 %0, %3 offset:%5" ::"v"(at), "v"(sum),
                     "v"(mx), "v"(mn), "n"(kKind), "n"(2 * kKind)
                     : "memory");
      }
    }
  }
  barrier_lds_only();   // (behind the wait for the writes above)
  const float inv_n = 1.0f / (float)p.N;
  // positions and mirror images the workgroup stands for
  const int k0 = rb * kRecPos, k1 = min(k0 + kRecPos, p.Kd);
  const int n_pos = k1 - k0 + (p.half < p.T ? max(0, min(k1, p.T - p.half) - max(k0, p.T - p.K + 1)) : 0);
  for (int c = tid; c < n_cb * kRecCols; c += 256) {
    const int m = cb0 * kRecCols + c;
    if (m >= p.Mc) break;
    const float sc = p.scale[(int64_t)b * p.Mc + m] * inv_n, c0 = p.c[(int64_t)b * 2 * p.N * p.Mc + m] * inv_n;
    const int64_t o = ((int64_t)b * p.RB + rb) * p.Mc + m;
    p.psum[o] = ((s_stat[0][0][c] + s_stat[0][1][c]) + (s_stat[0][2][c] + s_stat[0][3][c])) * sc + (float)n_pos * c0;
    p.pmax[o] = fa_fmax(fa_fmax(s_stat[1][0][c], s_stat[1][1][c]), fa_fmax(s_stat[1][2][c], s_stat[1][3][c])) * sc + c0;
    p.pmin[o] = fa_fmin(fa_fmin(s_stat[2][0][c], s_stat[2][1][c]), fa_fmin(s_stat[2][2][c], s_stat[2][3][c])) * sc + c0;
  }
}

// The statistics of a cache in single precision: complex sums, one pass over the cosine and one over the sine coefficients
// on the walk of the compression, from which the real and the imaginary part are taken.  Twice the work of the kernel above and
// further from 64 bits (deviations 4e-5 .. 2e-4, means 1e-4 of the deviation): it is kept for unchanged results, not for its
// accuracy.  The statistics are rounded to fp16, where a place is up to 1e-3 of a value, and with any other order of roundings some
// columns round the other way: the attention over them moves by 5e-4, nothing beside the roundings of a 16-bit model, but
// fifty times the 1e-5 to which results in single precision are to stay what they are.
__global__ __launch_bounds__(1024) void coef_colscale_kernel(const float* __restrict__ c, float* __restrict__ scale,
                                                             float* __restrict__ inv_scale, int N2, int Mc) {
  // 16 columns x 64 row classes: 64 bytes of a row per access, and four times the blocks of whole waves of columns
  __shared__ float s_mx[64][16];
  const int lane = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int m = blockIdx.x * 16 + lane, b = blockIdx.y;
  float mx = 0.f;
  if (m < Mc) {
    const float* cp = c + (int64_t)b * N2 * Mc + m;
    for (int n0 = g; n0 < N2; n0 += 64 * 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = cp[(int64_t)min(n0 + 64 * u, N2 - 1) * Mc];
#pragma unroll
      for (int u = 0; u < 8; ++u) mx = fmaxf(mx, fabsf(v[u]));
    }
  }
  s_mx[g][lane] = mx;
  __syncthreads();
  if (g == 0 && m < Mc) {
#pragma unroll
    for (int i = 1; i < 64; ++i) mx = fmaxf(mx, s_mx[i][lane]);
    const float sc = mx > 0.f ? exp2f(ceilf(log2f(mx))) : 1.f;   // power of two: scaling is exact
    scale[(int64_t)b * Mc + m] = sc;
    inv_scale[(int64_t)b * Mc + m] = 1.0f / sc;
  }
}

constexpr int kWalkColShare = 16;   // column blocks of a workgroup at most

struct ReconWalkParams {
  const half8* tab;        // basis rows of the positions: [ceil(K/8)][kStepK][64]
  const half8* packed[2];  // cos / sin coefficients, [B][CT][KS32][64] fragments
  const float* scale;      // [B][Mc]
  float* psum;
  float* pmax;
  float* pmin;             // [B][RB][Mc]
  int B, N, Mc, CT, KS32, K, T, n_steps, RB;
  int cb_per; // column blocks of a workgroup
  int Kd;     // positions computed directly: min(K, T / 2 + 1)
  int half;   // T / 2: mirror images beyond it count as positions of their own (a value no position exceeds
              // when the sequence is longer than the period and every position is computed directly)
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void spectral_recon_walk_kernel(
    const ReconWalkParams p) {
  constexpr int NST = 4;
  __shared__ __attribute__((aligned(16))) unsigned char s_stage[NST][4][kStepK][1024];
  __shared__ float s_red[3][4][kWgCols];
  __shared__ float s_scale[kWalkColShare * kWgCols];   // scale / N of this workgroup's columns
  const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rb = blockIdx.x, b = blockIdx.y;
  const int rt0 = (rb * 4 + w) * 4;
  const int n_rt = (p.Kd + 7) / 8;
  const int S = p.n_steps;
  const int cb0 = blockIdx.z * p.cb_per;
  const int n_cb = min((p.Mc + kWgCols - 1) / kWgCols - cb0, p.cb_per);
  const int Q = n_cb * 2 * S;   // steps of this workgroup: column block, pass (cos, sin), step (last to first)

  int next_cb = cb0, next_pass = 0, next_s = S - 1;   // the step requested next (walked, not divided out of a step number)
  auto issue = [&](int stage) {
    const int ct = min(next_cb * 4 + w, p.CT - 1);
    const half8* frags = next_pass ? p.packed[1] : p.packed[0];
    const _Float16* src = (const _Float16*)(frags + (((int64_t)b * p.CT + ct) * p.KS32) * 64) + lane * 8;
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks)
      load_frag_to_lds(src + (int64_t)(next_s * kStepK + ks) * 512, &s_stage[stage][w][ks][0]);
    if (--next_s < 0) {
      next_s = S - 1;
      next_cb += next_pass;
      next_pass ^= 1;
    }
  };
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < Q) issue(i);

  half8 Ea[4][kStepK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks) Ea[i][ks] = p.tab[((int64_t)min(rt0 + i, n_rt - 1) * kStepK + ks) * 64 + lane];
  float rc[4][2], rs[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int f2 = 0; f2 < 2; ++f2) fast_sincos_phase(min(rt0 + i, n_rt - 1) * 8 + lg * 2 + f2, kStepTokens, p.T, &rs[i][f2], &rc[i][f2]);
  float4v acc[4][4];
  float re[4][4][2];   // real part left by the cos pass
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int ks = 0; ks < kStepK; ++ks) asm volatile("" ::"v"(Ea[i][ks]));

  // (read here once: a load behind the walk of a column block would wait for every tile on its way)
  const float inv_n = 1.0f / (float)p.N;
  for (int i = tid; i < n_cb * kWgCols; i += 256) {
    const int m = cb0 * kWgCols + i;
    s_scale[i] = m < p.Mc ? p.scale[(int64_t)b * p.Mc + m] * inv_n : 0.f;
  }
  int cb = cb0, pass = 0, it = -1;
  for (int q = 0; q < Q; ++q) {
    if (++it == S) {
      it = 0;
      cb += pass;
      pass ^= 1;
    }
    const int stage = q % NST;
    if (q + NST - 2 < Q) wait_vmcnt<(NST - 2) * kStepK>();
    else wait_vmcnt<0>();
    barrier_lds_only();
    if (q + NST - 1 < Q) issue((q + NST - 1) % NST);
    spectral_step(acc, Ea, rc, rs, lds_addr_of(&s_stage[stage][0][0][lane * 16]));
    if (it != S - 1) continue;
    if (pass == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          re[i][j][0] = acc[i][j][0];
          re[i][j][1] = acc[i][j][2];
          acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
        }
      continue;
    }
    // both passes done for this column block: r = (re +- im) * scale / N at this lane's 8 positions per column and
    // at their mirror images
    const int half = p.half;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float sc = s_scale[((cb - cb0) * 4 + j) * 16 + lc];
      float sum = 0.f, mx = -INFINITY, mn = INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int f2 = 0; f2 < 2; ++f2) {
          const int k = (rt0 + i) * 8 + lg * 2 + f2;
          const float r = (re[i][j][f2] + acc[i][j][2 * f2 + 1]) * sc;
          if (k < p.Kd) {
            sum += r;
            mx = fmaxf(mx, r);
            mn = fminf(mn, r);
          }
          const int km = p.T - k;   // the mirror image counts where it is a position of its own beyond T / 2
          const float r2 = (re[i][j][f2] - acc[i][j][2 * f2 + 1]) * sc;
          if (k < p.Kd && km > half && km < p.K) {
            sum += r2;
            mx = fmaxf(mx, r2);
            mn = fminf(mn, r2);
          }
        }
      sum = fa_rows_sum(sum);
      mx = fa_rows_max(mx);
      mn = fa_rows_min(mn);
      if (lg == 0) {
        s_red[0][w][j * 16 + lc] = sum;
        s_red[1][w][j * 16 + lc] = mx;
        s_red[2][w][j * 16 + lc] = mn;
      }
    }
    __syncthreads();
    if (tid < kWgCols) {
      const int m = cb * kWgCols + tid;
      if (m < p.Mc) {
        const int64_t o = ((int64_t)b * p.RB + rb) * p.Mc + m;
        p.psum[o] = (s_red[0][0][tid] + s_red[0][1][tid]) + (s_red[0][2][tid] + s_red[0][3][tid]);
        p.pmax[o] = fmaxf(fmaxf(s_red[1][0][tid], s_red[1][1][tid]), fmaxf(s_red[1][2][tid], s_red[1][3][tid]));
        p.pmin[o] = fminf(fminf(s_red[2][0][tid], s_red[2][1][tid]), fminf(s_red[2][2][tid], s_red[2][3][tid]));
      }
    }
    // the next barrier (top of the loop) orders these reads before s_red is written again
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  }
}

}  // namespace fa_mfma

namespace {
struct SpectralPlan {
  int CT, KS32, n_steps, n_chunks, steps_per_chunk;
  size_t off_tab, off_packed, off_part, total;
};
SpectralPlan spectral_plan(int B, int K, int Mc, int N) {
  using namespace fa_mfma;
  SpectralPlan p{};
  p.CT = fa_cdiv(Mc, 16);
  p.n_steps = fa_cdiv(K, kStepTokens);
  p.KS32 = p.n_steps * kStepK;
  const int64_t tiles = (int64_t)B * fa_cdiv(N, kWgFreqs) * fa_cdiv(Mc, kWgCols);
  // Chunks of the walk, at least four steps each: two workgroups fit a compute unit, so the launch takes as many rounds as
  // there are 512s of workgroups, each as long as a chunk and about three steps of prologue and store.  (Always rounded up to
  // 512 workgroups, 240 tiles of 16 steps ran as 720 workgroups of 6 steps in two rounds: 50.8 us a call against 39.7.)
  const int max_chunks = p.n_steps / 4 > 0 ? p.n_steps / 4 : 1;
  int64_t best = INT64_MAX;
  for (int n = 1; n <= max_chunks && (n == 1 || tiles * n <= 1024); ++n) {
    const int per = fa_cdiv(p.n_steps, n);
    const int64_t cost = (int64_t)fa_cdiv(tiles * fa_cdiv(p.n_steps, per), 512) * (per + 3);
    if (cost < best) { best = cost; p.steps_per_chunk = per; }
  }
  p.n_chunks = fa_cdiv(p.n_steps, p.steps_per_chunk);
  size_t o = 0;
  auto take = [&](size_t bytes) { size_t at = o; o += fa_align_up(bytes, 256); return at; };
  p.off_tab = take((size_t)(N / 8) * kStepK * 64 * 16);
  p.off_packed = take((size_t)B * p.CT * p.KS32 * 1024);
  p.off_part = take((size_t)p.n_chunks * B * 2 * N * Mc * 4);
  p.total = o;
  return p;
}
}  // namespace

bool fa_spectral_mfma_ok(int a_dtype, int K, int Mc, int N) {
  return (a_dtype == FA_BF16 || a_dtype == FA_FP16) && N % 8 == 0 && K >= 4 * fa_mfma::kStepTokens;
}

size_t fa_spectral_mfma_workspace(int B, int K, int Mc, int N) { return spectral_plan(B, K, Mc, N).total; }

namespace {
// GEMM and chunk reduction on the table and the fragments that are already in the workspace
int spectral_after_pack(const SpectralPlan& pl, float* c, int B, int Mc, int N, int T, int64_t k_start, int accumulate,
                        void* workspace, hipStream_t st);
}  // namespace

int fa_spectral_mfma_launch(const void* a, int a_dtype, int64_t a_bs, int64_t a_rs, const int32_t* cols, float* c, int B,
                            int K, int Mc, int N, int T, int64_t k_start, int accumulate, void* workspace,
                            hipStream_t st) {
  using namespace fa_mfma;
  const SpectralPlan pl = spectral_plan(B, K, Mc, N);
  half8* packed = (half8*)((char*)workspace + pl.off_packed);
  const SpectralTable table{(half2v*)((char*)workspace + pl.off_tab), N, T};
  dim3 pgrid(pl.KS32 + fa_cdiv(table_blocks(N), (int64_t)fa_cdiv(Mc, 256) * B), fa_cdiv(Mc, 256), B);
  if (a_dtype == FA_BF16)
    spectral_pack_kernel<bf16_t><<<pgrid, 256, 0, st>>>((const bf16_t*)a, a_bs, a_rs, cols, nullptr, packed, K, Mc, pl.CT, pl.KS32, B, 0, 0, table);
  else
    spectral_pack_kernel<f16_t><<<pgrid, 256, 0, st>>>((const f16_t*)a, a_bs, a_rs, cols, nullptr, packed, K, Mc, pl.CT, pl.KS32, B, 0, 0, table);
  return spectral_after_pack(pl, c, B, Mc, N, T, k_start, accumulate, workspace, st);
}

namespace {
int spectral_after_pack(const SpectralPlan& pl, float* c, int B, int Mc, int N, int T, int64_t k_start, int accumulate,
                        void* workspace, hipStream_t st) {
  using namespace fa_mfma;
  char* ws = (char*)workspace;
  half8* tab = (half8*)(ws + pl.off_tab);
  half8* packed = (half8*)(ws + pl.off_packed);
  float* part = (float*)(ws + pl.off_part);
  SpectralGemmParams gp{};
  const bool direct = pl.n_chunks == 1;   // nothing to sum: the GEMM writes (or adds to) c itself
  gp.tab = tab; gp.packed = packed; gp.part = direct ? c : part;
  gp.add_to_part = direct && accumulate;
  gp.B = B; gp.N = N; gp.Mc = Mc; gp.CT = pl.CT; gp.KS32 = pl.KS32; gp.T = T;
  gp.n_steps = pl.n_steps; gp.steps_per_chunk = pl.steps_per_chunk; gp.n_chunks = pl.n_chunks;
  gp.k_start = k_start;
  dim3 ggrid(fa_cdiv(Mc, kWgCols), fa_cdiv(N, kWgFreqs), B * pl.n_chunks);
  spectral_gemm_kernel<<<ggrid, 256, 0, st>>>(gp);
  const int64_t total = (int64_t)B * 2 * N * Mc;
  if (!direct) spectral_reduce_kernel<<<fa_cdiv(total / 4, 256), 256, 0, st>>>(part, c, total, pl.n_chunks, accumulate);
  return fa_check_launch("fa_mat_fourier");
}

struct PrefillPlan {
  SpectralPlan sp;
  int n_pages;
  size_t off_sum, off_max, off_min, total;
};
PrefillPlan prefill_plan(int B, int L, int K_fft, int Mc, int N) {
  PrefillPlan p{};
  p.sp = spectral_plan(B, K_fft, Mc, N);
  const int pages_of_rows = fa_cdiv(L, 32);
  p.n_pages = pages_of_rows > p.sp.KS32 ? pages_of_rows : p.sp.KS32;
  // (room for as many blocks as the smallest number of KV heads, one, could ask for)
  const size_t blocks = fa_cdiv(p.n_pages, fa_mfma::pack_pages_per_block(p.n_pages, B));
  size_t o = p.sp.total;
  auto take = [&](size_t bytes) { size_t at = o; o += fa_align_up(bytes, 256); return at; };
  p.off_sum = take((size_t)B * blocks * Mc * 4);
  p.off_max = take((size_t)B * blocks * Mc * 4);
  p.off_min = take((size_t)B * blocks * Mc * 4);
  p.total = o;
  return p;
}
}  // namespace

extern "C" int fa_prefill_compress_ok(int dtype, int L, int K_fft, int Mc, int N, int D) {
  return fa_spectral_mfma_ok(dtype, K_fft, Mc, N) && L >= K_fft && K_fft > 0 && D % 8 == 0 && D <= 256;
}

extern "C" size_t fa_prefill_compress_workspace_bytes(int B, int L, int K_fft, int Mc, int N) {
  if (B <= 0 || L <= 0 || K_fft <= 0 || Mc <= 0 || N <= 0) return 0;
  return prefill_plan(B, L, K_fft, Mc, N).total;
}

extern "C" int fa_prefill_compress(const void* src, int dtype, int64_t src_bs, int64_t src_rs, int64_t row0, int L, int K_fft,
                                   void* store, int64_t st_bs, int cap_pages, const int32_t* n_list, const int32_t* n_h,
                                   const int32_t* pad_h, const int32_t* c_list, const int32_t* c_h, int Mc, float* coef,
                                   float* avg, float* max_dev, int stats_round_dtype, int B, int Hkv, int D, int N, int T,
                                   int is_v, void* workspace, size_t workspace_bytes, fa_stream_t stream) {
  using namespace fa_mfma;
  FA_REQUIRE(src && store && n_h && pad_h && c_list && c_h && coef && avg && max_dev, FA_ERR_NULL_POINTER,
             "fa_prefill_compress: null pointer");
  FA_REQUIRE(B > 0 && Hkv > 0 && L > 0 && cap_pages > 0 && row0 >= 0 && T > 0, FA_ERR_BAD_SHAPE, "fa_prefill_compress: bad shape");
  FA_REQUIRE((int64_t)cap_pages * 32 >= L, FA_ERR_BAD_SHAPE, "fa_prefill_compress: %d rows do not fit %d pages", L, cap_pages);
  FA_REQUIRE(fa_prefill_compress_ok(dtype, L, K_fft, Mc, N, D), FA_ERR_UNSUPPORTED,
             "fa_prefill_compress: dtype=%d L=%d K=%d Mc=%d N=%d D=%d is for the separate calls", dtype, L, K_fft, Mc, N, D);
  FA_REQUIRE(src_rs >= (int64_t)Hkv * D && src_rs % 8 == 0 && src_bs % 8 == 0 && ((uintptr_t)src & 15) == 0,
             FA_ERR_MISALIGNED, "fa_prefill_compress: rows of %lld elements (need %d, 16-byte aligned)", (long long)src_rs, Hkv * D);
  const PrefillPlan pl = prefill_plan(B, L, K_fft, Mc, N);
  FA_REQUIRE(workspace && workspace_bytes >= pl.total, FA_ERR_WORKSPACE, "fa_prefill_compress: workspace %zu < %zu",
             workspace_bytes, pl.total);
  FA_REQUIRE(((uintptr_t)workspace & 255) == 0 && ((uintptr_t)coef & 15) == 0, FA_ERR_MISALIGNED,
             "fa_prefill_compress: workspace not 256-byte or coefficients not 16-byte aligned");
  hipStream_t st = fa_hip_stream(stream);
  char* ws = (char*)workspace;
  float* psum = (float*)(ws + pl.off_sum);
  float* pmax = (float*)(ws + pl.off_max);
  float* pmin = (float*)(ws + pl.off_min);
  const int per_block = pack_pages_per_block(pl.n_pages, Hkv * B), n_blocks = fa_cdiv(pl.n_pages, per_block);
  auto launch = [&](auto tag) {
    using E = decltype(tag);
    PrefillPackParams<E> pp{};
    pp.src = (const E*)src; pp.src_bs = src_bs; pp.src_rs = src_rs; pp.row0 = row0; pp.L = L; pp.K_fft = K_fft;
    pp.store = (E*)store; pp.st_bs = st_bs; pp.cap_pages = cap_pages;
    pp.n_list = n_list; pp.n_h = n_h; pp.pad_h = pad_h; pp.c_list = c_list; pp.c_h = c_h;
    pp.packed = (half8*)(ws + pl.sp.off_packed);
    pp.psum = psum; pp.pmax = pmax; pp.pmin = pmin;
    pp.Mc = Mc; pp.CT = pl.sp.CT; pp.KS32 = pl.sp.KS32; pp.n_pages = pl.n_pages; pp.per_block = per_block; pp.n_blocks = n_blocks;
    pp.Hkv = Hkv; pp.D = D; pp.is_v = is_v;
    pp.table = SpectralTable{(half2v*)(ws + pl.sp.off_tab), N, T};
    prefill_pack_kernel<E><<<dim3(n_blocks + fa_cdiv(table_blocks(N), (int64_t)Hkv * B), Hkv, B), 256, 0, st>>>(pp);
  };
  if (dtype == FA_BF16) launch(bf16_t{}); else launch(f16_t{});
  int rc = spectral_after_pack(pl.sp, coef, B, Mc, N, T, 0, 0, workspace, st);
  if (rc != FA_OK) return rc;
  fa_stats_finalize_launch(psum, pmax, pmin, avg, max_dev, B, L, Mc, n_blocks, stats_round_dtype, st);
  return fa_check_launch("fa_prefill_compress");
}

namespace {
struct ReconPlan {
  int CT, n_steps, RB;
  size_t off_tab, off_packed, off_phi, off_scale, off_sum, off_max, off_min, total;
};
ReconPlan recon_plan(int B, int N, int Mc, int K) {
  using namespace fa_mfma;
  ReconPlan p{};
  p.CT = fa_cdiv(Mc, 16);
  p.n_steps = recon_steps(N);
  p.RB = fa_cdiv(K, kRecPos);
  size_t o = 0;
  auto take = [&](size_t bytes) { size_t at = o; o += fa_align_up(bytes, 256); return at; };
  p.off_tab = take((size_t)p.RB * (kRecPos / 16) * 4 * 1024);
  p.off_packed = take((size_t)B * p.CT * p.n_steps * kRecFrags * 1024);
  p.off_phi = take((size_t)p.RB * p.n_steps * 2 * kRecPos * 4);
  p.off_scale = take((size_t)B * Mc * 4);
  p.off_sum = take((size_t)B * p.RB * Mc * 4);
  p.off_max = take((size_t)B * p.RB * Mc * 4);
  p.off_min = take((size_t)B * p.RB * Mc * 4);
  p.total = o;
  return p;
}
}  // namespace

namespace {
// Column blocks per workgroup of the reconstruction statistics.  Two workgroups fit a compute unit, and a workgroup
// pays about half a column block for its basis rows before the first product: take the share whose rounds over the
// device, times the length of a round, come out shortest.
int recon_col_share(int row_groups, int n_cb, int most) {
  int best = n_cb < most ? n_cb : most;
  float best_cost = 1e30f;
  for (int cs = 1; cs <= n_cb; ++cs) {
    const int per = fa_cdiv(n_cb, cs);
    if (per > most) continue;
    const float cost = (float)fa_cdiv((int64_t)row_groups * fa_cdiv(n_cb, per), 512) * ((float)per + 0.5f);
    if (cost < best_cost) { best_cost = cost; best = per; }
  }
  return best;
}
}  // namespace

namespace {
struct ReconWalkPlan {
  int CT, KS32, n_steps, RB;
  size_t off_tab, off_pc, off_ps, off_scale, off_inv, off_sum, off_max, off_min, total;
};
ReconWalkPlan recon_walk_plan(int B, int N, int Mc, int K) {
  using namespace fa_mfma;
  ReconWalkPlan p{};
  p.CT = fa_cdiv(Mc, 16);
  p.n_steps = fa_cdiv(N, kStepTokens);
  p.KS32 = p.n_steps * kStepK;
  p.RB = fa_cdiv(K, kWgFreqs);
  size_t o = 0;
  auto take = [&](size_t bytes) { size_t at = o; o += fa_align_up(bytes, 256); return at; };
  p.off_tab = take((size_t)fa_cdiv(K, 8) * kStepK * 64 * 16);
  p.off_pc = take((size_t)B * p.CT * p.KS32 * 1024);
  p.off_ps = take((size_t)B * p.CT * p.KS32 * 1024);
  p.off_scale = take((size_t)B * Mc * 4);
  p.off_inv = take((size_t)B * Mc * 4);
  p.off_sum = take((size_t)B * p.RB * Mc * 4);
  p.off_max = take((size_t)B * p.RB * Mc * 4);
  p.off_min = take((size_t)B * p.RB * Mc * 4);
  p.total = o;
  return p;
}
}  // namespace

namespace {
int recon_walk_launch(const float* c, int B, int N, int Mc, int K, int T, void* workspace, float** psum, float** pmax, float** pmin,
                      hipStream_t st) {
  using namespace fa_mfma;
  const ReconWalkPlan pl = recon_walk_plan(B, N, Mc, K);
  char* ws = (char*)workspace;
  half8* tab = (half8*)(ws + pl.off_tab);
  half8* pc = (half8*)(ws + pl.off_pc);
  half8* ps = (half8*)(ws + pl.off_ps);
  float* scale = (float*)(ws + pl.off_scale);
  float* inv = (float*)(ws + pl.off_inv);
  *psum = (float*)(ws + pl.off_sum);
  *pmax = (float*)(ws + pl.off_max);
  *pmin = (float*)(ws + pl.off_min);
  // positions 0 .. T / 2 stand for their mirror images as well (unless the sequence is longer than the period)
  const bool mirror = K <= T + 1;
  const int Kd = mirror && T / 2 + 1 < K ? T / 2 + 1 : K;
  const int RBd = fa_cdiv(Kd, kWgFreqs);
  const int kp8 = fa_cdiv(Kd, 8) * 8;
  coef_colscale_kernel<<<dim3(fa_cdiv(Mc, 16), B), 1024, 0, st>>>(c, scale, inv, 2 * N, Mc);
  // the cosine rows and, behind them, the sine rows; the basis of the positions beside them
  const int col_blocks = fa_cdiv(Mc, 256);
  const dim3 pgrid(pl.KS32 + fa_cdiv(table_blocks(kp8), col_blocks * 2 * B), col_blocks, 2 * B);
  spectral_pack_kernel<float><<<pgrid, 256, 0, st>>>(c, (int64_t)2 * N * Mc, Mc, nullptr, inv, pc, N, Mc, pl.CT, pl.KS32, B,
                                                     (int64_t)N * Mc, ps - pc, SpectralTable{(half2v*)tab, kp8, T});
  ReconWalkParams rp{};
  rp.tab = tab; rp.packed[0] = pc; rp.packed[1] = ps; rp.scale = scale;
  rp.psum = *psum; rp.pmax = *pmax; rp.pmin = *pmin;
  rp.B = B; rp.N = N; rp.Mc = Mc; rp.CT = pl.CT; rp.KS32 = pl.KS32; rp.K = K; rp.T = T; rp.n_steps = pl.n_steps; rp.RB = RBd;
  rp.Kd = Kd;
  rp.half = mirror ? T / 2 : 0x7fffffff;
  const int n_cb = fa_cdiv(Mc, kWgCols);
  rp.cb_per = recon_col_share(RBd * B, n_cb, kWalkColShare);
  spectral_recon_walk_kernel<<<dim3(RBd, B, fa_cdiv(n_cb, rp.cb_per)), 256, 0, st>>>(rp);
  return RBd;
}
}  // namespace

bool fa_recon_stats_mfma_ok(int N, int Mc, int K) { return N >= 32 && Mc >= 16 && K >= 1024; }

size_t fa_recon_stats_mfma_workspace(int B, int N, int Mc, int K) {
  const size_t a = recon_plan(B, N, Mc, K).total, b = recon_walk_plan(B, N, Mc, K).total;
  return a > b ? a : b;
}

int fa_recon_stats_mfma_launch(const float* c, int B, int N, int Mc, int K, int T, bool single, void* workspace, float** psum,
                               float** pmax, float** pmin, hipStream_t st) {
  using namespace fa_mfma;
  if (single) return recon_walk_launch(c, B, N, Mc, K, T, workspace, psum, pmax, pmin, st);
  const ReconPlan pl = recon_plan(B, N, Mc, K);
  char* ws = (char*)workspace;
  half8* tab = (half8*)(ws + pl.off_tab);
  half8* packed = (half8*)(ws + pl.off_packed);
  float* phi = (float*)(ws + pl.off_phi);
  float* scale = (float*)(ws + pl.off_scale);
  *psum = (float*)(ws + pl.off_sum);
  *pmax = (float*)(ws + pl.off_max);
  *pmin = (float*)(ws + pl.off_min);
  // positions 0 .. T / 2 stand for their mirror images as well (unless the sequence is longer than the period)
  const bool mirror = K <= T + 1;
  const int Kd = mirror && T / 2 + 1 < K ? T / 2 + 1 : K;
  const int RBd = fa_cdiv(Kd, kRecPos);
  ReconPrepParams pp{};
  pp.c = c; pp.packed = packed; pp.scale = scale; pp.tab = (half2v*)tab; pp.phi = phi;
  pp.B = B; pp.N = N; pp.Mc = Mc; pp.CT = pl.CT; pp.T = T; pp.n_steps = pl.n_steps;
  recon_prep_kernel<<<pl.CT * B + RBd * (kRecPos / 32), 1024, 0, st>>>(pp);
  ReconStatsParams rp{};
  rp.c = c; rp.tab = tab; rp.packed = packed; rp.phi = phi; rp.scale = scale;
  rp.psum = *psum; rp.pmax = *pmax; rp.pmin = *pmin;
  rp.B = B; rp.N = N; rp.Mc = Mc; rp.CT = pl.CT; rp.K = K; rp.T = T; rp.n_steps = pl.n_steps; rp.RB = RBd;
  rp.Kd = Kd;
  rp.half = mirror ? T / 2 : 0x7fffffff;
  const int n_cb = fa_cdiv(Mc, kRecCols);
  rp.cb_per = recon_col_share(RBd * B, n_cb, kMaxColShare);
  spectral_recon_stats_kernel<<<dim3(RBd, B, fa_cdiv(n_cb, rp.cb_per)), 256, 0, st>>>(rp);
  return RBd;
}
