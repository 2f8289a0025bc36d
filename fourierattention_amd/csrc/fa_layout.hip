// Page layout of the stored mid dims: pack (prefill), append (eviction) and unpack.
#include "fa_common.h"

namespace {

// element offset inside one (batch, head) run of pages
__device__ __forceinline__ int64_t page_elem_offset(bool is_v, int dp, int64_t token, int j) {
  const int64_t page = token >> 5;
  const int t = (int)(token & 31);
  int frag, lane, e;
  if (!is_v) {
    frag = (t >> 4) * (dp >> 5) + (j >> 5);
    lane = ((j & 31) >> 3) * 16 + (t & 15);
    e = j & 7;
  } else {
    frag = j >> 4;
    lane = (t >> 3) * 16 + (j & 15);
    e = t & 7;
  }
  return page * dp * 32 + (int64_t)frag * 512 + lane * 8 + e;
}

// one block per page (32 tokens) of one (b, h): the gather reads run along the stored dims of a token row,
// the page is assembled in LDS and leaves as whole fragments (16 bytes per lane); grid (pages, Hkv, B)
template <typename E>
__global__ __launch_bounds__(256) void mid_pack_kernel(
    const E* __restrict__ src, int64_t src_bs, int64_t src_rs, int64_t row0, int L, E* __restrict__ store,
    int64_t st_bs, int cap_pages, const int32_t* __restrict__ n_list, const int32_t* __restrict__ n_h,
    const int32_t* __restrict__ pad_h, int is_v) {
  constexpr int kMaxDp = 256;                       // padded stored dims of a head
  constexpr int kPitch = kMaxDp + 8;                // elements; keeps rows 16-byte aligned
  struct alignas(sizeof(E) * 8) Piece { E v[8]; };  // what one lane of a fragment holds
  __shared__ __attribute__((aligned(32))) E tile[32][kPitch];
  const int page = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int n0 = n_h[h], n_len = n_h[h + 1] - n0;
  const int p0 = pad_h[h], dp = pad_h[h + 1] - p0;
  if (n_len == 0) return;
  const int tid = threadIdx.x;
  __shared__ int s_col[kMaxDp];
  for (int j = tid; j < dp; j += 256) s_col[j] = n_list[n0 + min(j, n_len - 1)];
  __syncthreads();
  // gather: consecutive threads take consecutive stored dims of one token; eight loads in flight per thread,
  // all unconditional (clamped to the last real dim / row, masked afterwards)
  const E* sb = src + (int64_t)b * src_bs + row0 * src_rs;
  const int64_t last = (int64_t)L - 1;
  for (int base = tid; base < 32 * dp; base += 256 * 8) {
    E v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int idx = min(base + 256 * u, 32 * dp - 1);
      const int t = idx / dp, j = idx - t * dp;
      const int64_t token = (int64_t)page * 32 + t;
      v[u] = sb[(token < last ? token : last) * src_rs + s_col[j]];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int idx = base + 256 * u;
      if (idx < 32 * dp) {
        const int t = idx / dp, j = idx - t * dp;
        const bool ok = j < n_len && (int64_t)page * 32 + t < L;
        tile[t][j] = ok ? v[u] : E{};
      }
    }
  }
  __syncthreads();
  Piece* out = (Piece*)(store + (int64_t)b * st_bs + (int64_t)p0 * 32 * cap_pages + (int64_t)page * dp * 32);
  const int n_pieces = dp * 32 / 8;
  for (int piece = tid; piece < n_pieces; piece += 256) {
    const int frag = piece >> 6, lane = piece & 63;
    Piece o;
    if (!is_v) {
      const int nks = dp >> 5;
      const int tb = frag / nks, s_ = frag - tb * nks;
      o = *(const Piece*)&tile[tb * 16 + (lane & 15)][s_ * 32 + 8 * (lane >> 4)];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) o.v[i] = tile[8 * (lane >> 4) + i][frag * 16 + (lane & 15)];
    }
    out[piece] = o;
  }
}

// The same for 16-bit rows that are 16-byte aligned: the head's whole slice of the 32 token rows is read with
// 16-byte loads into LDS (every line of the source is needed anyway: stored and compressed dims interleave), and
// the gather along the stored dims happens on the way out of LDS.
template <typename E>
__global__ __launch_bounds__(256) void mid_pack_rows_kernel(
    const E* __restrict__ src, int64_t src_bs, int64_t src_rs, int64_t row0, int L, E* __restrict__ store,
    int64_t st_bs, int cap_pages, const int32_t* __restrict__ n_list, const int32_t* __restrict__ n_h,
    const int32_t* __restrict__ pad_h, int D, int is_v) {
  constexpr int kMaxD = 256;                        // head dim, and padded stored dims of a head
  constexpr int kPitch = kMaxD + 8;                 // elements; keeps rows 16-byte aligned
  struct alignas(sizeof(E) * 8) Piece { E v[8]; };
  __shared__ __attribute__((aligned(32))) E tile[32][kPitch];
  __shared__ int s_col[kMaxD];
  const int page = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int n0 = n_h[h], n_len = n_h[h + 1] - n0;
  const int p0 = pad_h[h], dp = pad_h[h + 1] - p0;
  if (n_len == 0) return;
  const int tid = threadIdx.x;
  // dim within the head of every stored position (clamped into the head: the reads below stay inside the tile)
  for (int j = tid; j < dp; j += 256) s_col[j] = min(max(n_list[n0 + min(j, n_len - 1)] - h * D, 0), D - 1);
  const E* sb = src + (int64_t)b * src_bs + row0 * src_rs + (int64_t)h * D;
  const int ppr = D >> 3;                           // 16-byte pieces per row of the head
  const int64_t last = (int64_t)L - 1;
  for (int p = tid; p < 32 * ppr; p += 256) {
    const int t = p / ppr, c = p - t * ppr;
    const int64_t token = (int64_t)page * 32 + t;
    *(Piece*)&tile[t][c * 8] = *(const Piece*)(sb + (token < last ? token : last) * src_rs + c * 8);
  }
  __syncthreads();
  Piece* out = (Piece*)(store + (int64_t)b * st_bs + (int64_t)p0 * 32 * cap_pages + (int64_t)page * dp * 32);
  const int n_pieces = dp * 32 / 8;
  for (int piece = tid; piece < n_pieces; piece += 256) {
    const int frag = piece >> 6, lane = piece & 63;
    Piece o;
    if (!is_v) {
      const int nks = dp >> 5;
      const int tb = frag / nks, s_ = frag - tb * nks;
      const int t = tb * 16 + (lane & 15), j0 = s_ * 32 + 8 * (lane >> 4);
      const bool row_ok = (int64_t)page * 32 + t < L;
#pragma unroll
      for (int e = 0; e < 8; ++e) o.v[e] = (row_ok && j0 + e < n_len) ? tile[t][s_col[j0 + e]] : E{};
    } else {
      const int j = frag * 16 + (lane & 15);
      const int col = s_col[j];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = 8 * (lane >> 4) + i;
        o.v[i] = (j < n_len && (int64_t)page * 32 + t < L) ? tile[t][col] : E{};
      }
    }
    out[piece] = o;
  }
}

// Rows whose columns are the stored dims already, head by head (the reference's own k_uncompressed / v_uncompressed): head
// h's run of n_h[h+1] - n_h[h] columns is read in pieces of eight, at whatever alignment the run has, and no index list is
// involved.  A piece of a K fragment is eight neighbouring dims of one token, i.e. one piece of the source: it goes from
// register to store.  V pieces hold eight tokens of one dim and turn round in LDS, kRunPages pages per block.
// Bound by the chain of a block (offsets, rows, LDS, store) with eight blocks per compute unit: 15356 rows x 512 columns of
// two sequences in 16 us (4 TB/s read and written), against 33 us through mid_pack_kernel's index list, whose loads
// bring one element per lane.  Two pages per block let a thread have two pieces in flight.
constexpr int kRunPages = 2;

template <typename E, int MAXD>
__global__ __launch_bounds__(256) void mid_pack_runs_kernel(
    const E* __restrict__ src, int64_t src_bs, int64_t src_rs, int64_t row0, int L, E* __restrict__ store,
    int64_t st_bs, int cap_pages, const int32_t* __restrict__ n_h, const int32_t* __restrict__ pad_h, int is_v) {
  constexpr int kPitch = MAXD + 8;
  struct alignas(sizeof(E) * 8) Piece { E v[8]; };
  typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
  __shared__ __attribute__((aligned(32))) E tile[kRunPages * 32][kPitch];
  const int h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
  const int page0 = blockIdx.x * kRunPages;
  const int n0 = n_h[h], n_len = n_h[h + 1] - n0;
  const int p0 = pad_h[h], dp = pad_h[h + 1] - p0;
  if (n_len <= 0) return;
  const int n_pages = min(kRunPages, ((L + 31) >> 5) - page0);
  const E* sb = src + (int64_t)b * src_bs + (row0 + (int64_t)page0 * 32) * src_rs + n0;
  const int rows = min(n_pages * 32, L - page0 * 32);          // rows of the source behind this block's pages
  // dims j0 .. j0 + 7 of row t; zeros past the head's dims and past the rows
  auto fetch = [&](int t, int j0) {
    const E* row = sb + (int64_t)min(t, rows - 1) * src_rs;
    if constexpr (sizeof(E) == 2) if (n_len >= 8) {
      // one load at whatever alignment the run has; the last piece of a run is read so that it ends with the run
      const int s0 = min(j0, n_len - 8), past = t < rows ? j0 - s0 : 8;     // past: elements the load starts too early
      u64x2 x;
      __builtin_memcpy(&x, row + s0, 16);
      const int by = past * 16;
      const uint64_t lo = by == 0 ? x.x : by < 64 ? (x.x >> by) | (x.y << (64 - by)) : by < 128 ? x.y >> (by - 64) : 0;
      const uint64_t hi = by < 64 ? x.y >> by : 0;
      x.x = lo;
      x.y = hi;
      return __builtin_bit_cast(Piece, x);
    }
    Piece o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const E x = row[min(j0 + e, n_len - 1)];
      o.v[e] = (t < rows && j0 + e < n_len) ? x : E{};
    }
    return o;
  };
  Piece* out = (Piece*)(store + (int64_t)b * st_bs + (int64_t)p0 * 32 * cap_pages + (int64_t)page0 * dp * 32);
  const int per_page = dp * 4;                                 // pieces of a page
  const int n_pieces = n_pages * per_page;
  if (!is_v) {
    const int nks = dp >> 5;
#pragma unroll 2
    for (int q = tid; q < n_pieces; q += 256) {
      const int f = q >> 6, lane = q & 63;                     // fragment (page, tb, s) of the block, lane of the fragment
      const int ptb = f / nks, s_ = f - ptb * nks;
      out[q] = fetch(ptb * 16 + (lane & 15), s_ * 32 + 8 * (lane >> 4));
    }
    return;
  }
  const int ppr = dp >> 3;                                     // pieces per row
#pragma unroll 2
  for (int q = tid; q < n_pages * 32 * ppr; q += 256) {
    const int t = q / ppr, c = q - t * ppr;
    *(Piece*)&tile[t][c * 8] = fetch(t, c * 8);
  }
  __syncthreads();
  const int frags = dp >> 4;
  for (int q = tid; q < n_pieces; q += 256) {
    const int f = q >> 6, lane = q & 63;
    const int pg = f / frags, dg = f - pg * frags;
    Piece o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = tile[pg * 32 + 8 * (lane >> 4) + i][dg * 16 + (lane & 15)];
    out[q] = o;
  }
}

// New rows of K and of V behind those a window buffer holds, both in one launch; U: the unit that strides and widths allow.
template <typename U>
__global__ __launch_bounds__(256) void append_rows_kernel(const U* __restrict__ k, const U* __restrict__ v, int64_t src_bs,
                                                          int64_t src_rs, U* __restrict__ k_dst, U* __restrict__ v_dst,
                                                          int64_t dst_bs, int64_t dst_rs, int width, int B) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= width) return;
  const bool is_v = (int)blockIdx.z >= B;
  const int64_t b = is_v ? blockIdx.z - B : blockIdx.z, t = blockIdx.y;
  (is_v ? v_dst : k_dst)[b * dst_bs + t * dst_rs + i] = (is_v ? v : k)[b * src_bs + t * src_rs + i];
}

// The rows of a prompt: token-major copies and the near rows (sink, window, spare slot) in one pass.  A block takes 16 rows of
// K or V; a thread moves 16 bytes at a time, neighbouring threads along a row of the copy, four loads ahead of their
// stores.  Bound by HBM: 4 x 3001 rows of 1024 16-bit values, K and V, head-major: 22 us (4.5 TB/s) where a copy of each
// and six small ones took 18 + 18 + 25.
constexpr int kPromptRows = 16;
struct PromptRowsParams {
  const uint4 *k, *v;      // strides in pieces of 16 bytes
  int64_t bs, hs, rs;
  uint4 *k_tok, *v_tok, *k_near, *v_near;
  int64_t near_bs;
  int n_first, n_last, spare, S, heads, ppd;   // ppd: pieces of a head's row
};

__global__ __launch_bounds__(256) void prompt_rows_kernel(const PromptRowsParams p) {
  const bool is_v = blockIdx.y != 0;
  const int64_t b = blockIdx.z;
  const uint4* src = (is_v ? p.v : p.k) + b * p.bs;
  uint4* tok = is_v ? p.v_tok : p.k_tok;
  uint4* near_rows = is_v ? p.v_near : p.k_near;
  if (near_rows) near_rows += b * p.near_bs;
  const int ppr = p.heads * p.ppd;   // pieces of a row
  const int n_near = p.n_first + p.n_last;
  // rows of the launch: with copies every row of the prompt, otherwise the near ones; behind them the row of zeros
  const int rows = tok ? p.S : n_near;
  const int r0 = blockIdx.x * kPromptRows, r1 = min(rows + (near_rows ? p.spare : 0), r0 + kPromptRows);
  const int n = (r1 - r0) * ppr;
  for (int i0 = threadIdx.x; i0 < n; i0 += 4 * 256) {
    uint4 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = min(i0 + u * 256, n - 1), r = r0 + i / ppr, c = i % ppr, h = c / p.ppd;
      const int s = tok ? min(r, p.S - 1) : r < p.n_first ? r : min(p.S - p.n_last + (r - p.n_first), p.S - 1);
      x[u] = src[h * p.hs + s * p.rs + (c - h * p.ppd)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * 256;
      if (i >= n) break;
      const int r = r0 + i / ppr, c = i % ppr;
      int slot = -1;
      if (r >= rows) {
        slot = n_near;
        x[u] = uint4{0, 0, 0, 0};
      } else if (!tok) {
        slot = r;
      } else {
        tok[(b * p.S + r) * ppr + c] = x[u];
        slot = r < p.n_first ? r : r >= p.S - p.n_last ? p.n_first + r - (p.S - p.n_last) : -1;
      }
      if (near_rows && slot >= 0) near_rows[(int64_t)slot * ppr + c] = x[u];
    }
  }
}

// Operands of a call in the types the kernels take, all in one launch: a grid row per item, items in the argument block.
constexpr int kMaxConvert = 16;
struct ConvertArgs { fa_convert_item item[kMaxConvert]; };

__global__ __launch_bounds__(256) void convert_kernel(const ConvertArgs a) {
  const fa_convert_item it = a.item[blockIdx.y];
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < it.count; i += step) {
    switch (it.kind) {
      case FA_CONVERT_I64_I32: ((int32_t*)it.dst)[i] = (int32_t)((const int64_t*)it.src)[i]; break;
      case FA_CONVERT_BF16_F32: ((float*)it.dst)[i] = fa_to_float(((const bf16_t*)it.src)[i]); break;
      case FA_CONVERT_F16_F32: ((float*)it.dst)[i] = fa_to_float(((const f16_t*)it.src)[i]); break;
      default: {   // offsets of counts rounded up to whole units (at most a few dozen heads: every entry sums for itself)
        int32_t sum = 0;
        for (int64_t h = 0; h < i; ++h) {
          const int32_t n = it.kind == FA_CONVERT_PAD_I64 ? (int32_t)(((const int64_t*)it.src)[h + 1] - ((const int64_t*)it.src)[h])
                                                          : ((const int32_t*)it.src)[h + 1] - ((const int32_t*)it.src)[h];
          sum += (n + it.unit - 1) / it.unit * it.unit;
        }
        ((int32_t*)it.dst)[i] = sum;
      }
    }
  }
}

template <typename E>
__global__ __launch_bounds__(256) void mid_append_kernel(
    const E* __restrict__ row, int64_t row_bs, int64_t pos, E* __restrict__ store, int64_t st_bs, int cap_pages,
    const int32_t* __restrict__ n_list, const int32_t* __restrict__ n_h, const int32_t* __restrict__ pad_h, int Hkv,
    int Cn, int is_v) {
  const int b = blockIdx.y;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= Cn) return;
  int h = 0;
  while (h + 1 < Hkv && n_h[h + 1] <= c) ++h;
  const int j = c - n_h[h];
  const int p0 = pad_h[h], dp = pad_h[h + 1] - p0;
  store[(int64_t)b * st_bs + (int64_t)p0 * 32 * cap_pages + page_elem_offset(is_v, dp, pos, j)] =
      row[(int64_t)b * row_bs + n_list[c]];
}

template <typename E>
__global__ __launch_bounds__(256) void mid_unpack_kernel(
    const E* __restrict__ store, int64_t st_bs, int cap_pages, int L, E* __restrict__ dst,
    const int32_t* __restrict__ n_h, const int32_t* __restrict__ pad_h, int Cn, int is_v) {
  const int h = blockIdx.y, b = blockIdx.z;
  const int n0 = n_h[h], n_len = n_h[h + 1] - n0;
  const int p0 = pad_h[h], dp = pad_h[h + 1] - p0;
  if (n_len == 0) return;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)L * n_len) return;
  const int64_t token = idx / n_len;
  const int j = (int)(idx % n_len);
  dst[((int64_t)b * L + token) * Cn + n0 + j] =
      store[(int64_t)b * st_bs + (int64_t)p0 * 32 * cap_pages + page_elem_offset(is_v, dp, token, j)];
}

template <typename F>
int dispatch16(int dtype, const char* what, F&& f) {
  switch (dtype) {
    case FA_BF16: f(bf16_t{}); return FA_OK;
    case FA_FP16: f(f16_t{}); return FA_OK;
    case FA_FP32: f(float{}); return FA_OK;
    default: fa_set_error("%s: dtype %d", what, dtype); return FA_ERR_BAD_DTYPE;
  }
}

}  // namespace

extern "C" int fa_mid_pack(const void* src, int dtype, int64_t src_bs, int64_t src_rs, int64_t row0, int L,
                           void* store, int64_t st_bs, int cap_pages, const int32_t* n_list, const int32_t* n_h,
                           const int32_t* pad_h, int B, int Hkv, int D, int is_v, int cols_kind, fa_stream_t stream) {
  FA_REQUIRE(src && store && n_h && pad_h, FA_ERR_NULL_POINTER, "fa_mid_pack: null pointer");
  FA_REQUIRE(cols_kind == FA_COLS_ANY || cols_kind == FA_COLS_HEAD_DIMS || cols_kind == FA_COLS_IN_ORDER, FA_ERR_BAD_SHAPE,
             "fa_mid_pack: cols_kind %d", cols_kind);
  FA_REQUIRE(B > 0 && Hkv > 0 && L >= 0 && cap_pages > 0 && row0 >= 0, FA_ERR_BAD_SHAPE, "fa_mid_pack: bad shape");
  FA_REQUIRE((int64_t)cap_pages * 32 >= L, FA_ERR_BAD_SHAPE, "fa_mid_pack: %d rows do not fit %d pages", L, cap_pages);
  if (L == 0) return FA_OK;
  hipStream_t st = fa_hip_stream(stream);
  FA_REQUIRE(D > 0, FA_ERR_BAD_SHAPE, "fa_mid_pack: head_dim %d", D);
  FA_REQUIRE(D <= 256, FA_ERR_UNSUPPORTED, "fa_mid_pack: head_dim %d above 256", D);
  dim3 grid(fa_cdiv(L, 32), Hkv, B);
  // the row kernel reads head h's slice [h*D, (h+1)*D) of every source row and picks the stored dims out of it:
  // only the caller knows whether the index list means that (it cannot be told from the strides)
  const bool rows16 = cols_kind == FA_COLS_HEAD_DIMS && ((uintptr_t)src & 15) == 0 && src_bs % 8 == 0 &&
                      src_rs % 8 == 0 && D % 8 == 0;
  FA_REQUIRE(cols_kind != FA_COLS_HEAD_DIMS || src_rs >= (int64_t)Hkv * D, FA_ERR_BAD_SHAPE,
             "fa_mid_pack: rows of %lld elements cannot hold %d heads of %d dims", (long long)src_rs, Hkv, D);
  int rc = dispatch16(dtype, "fa_mid_pack", [&](auto tag) {
    using E = decltype(tag);
    if (cols_kind == FA_COLS_IN_ORDER) {
      const dim3 rgrid(fa_cdiv(fa_cdiv(L, 32), kRunPages), Hkv, B);
      if (D <= 128)
        mid_pack_runs_kernel<E, 128><<<rgrid, 256, 0, st>>>((const E*)src, src_bs, src_rs, row0, L, (E*)store, st_bs, cap_pages,
                                                           n_h, pad_h, is_v);
      else
        mid_pack_runs_kernel<E, 256><<<rgrid, 256, 0, st>>>((const E*)src, src_bs, src_rs, row0, L, (E*)store, st_bs, cap_pages,
                                                           n_h, pad_h, is_v);
      return;
    }
    if constexpr (sizeof(E) == 2) {
      if (rows16) {
        mid_pack_rows_kernel<E><<<grid, 256, 0, st>>>((const E*)src, src_bs, src_rs, row0, L, (E*)store, st_bs, cap_pages,
                                                     n_list, n_h, pad_h, D, is_v);
        return;
      }
    }
    mid_pack_kernel<E><<<grid, 256, 0, st>>>((const E*)src, src_bs, src_rs, row0, L, (E*)store, st_bs, cap_pages, n_list,
                                            n_h, pad_h, is_v);
  });
  return rc != FA_OK ? rc : fa_check_launch("fa_mid_pack");
}

extern "C" int fa_append_rows(const void* k, const void* v, int64_t src_bs, int64_t src_rs, void* k_dst, void* v_dst, int64_t dst_bs,
                              int64_t dst_rs, int64_t pos, int B, int rows, int width, int dtype, fa_stream_t stream) {
  FA_REQUIRE(k && v && k_dst && v_dst, FA_ERR_NULL_POINTER, "fa_append_rows: null pointer");
  FA_REQUIRE(B > 0 && B <= 32767 && rows >= 0 && rows <= 65535 && width > 0 && pos >= 0, FA_ERR_BAD_SHAPE,
             "fa_append_rows: B=%d rows=%d width=%d", B, rows, width);
  FA_REQUIRE(dtype == FA_BF16 || dtype == FA_FP16 || dtype == FA_FP32, FA_ERR_BAD_DTYPE, "fa_append_rows: dtype %d", dtype);
  if (rows == 0) return FA_OK;
  hipStream_t st = fa_hip_stream(stream);
  const int es = dtype == FA_FP32 ? 4 : 2;
  char *kd = (char*)k_dst + pos * dst_rs * es, *vd = (char*)v_dst + pos * dst_rs * es;
  auto go = [&](auto tag) {
    using U = decltype(tag);
    const int per = (int)sizeof(U) / es;
    append_rows_kernel<U><<<dim3(fa_cdiv(width / per, 256), rows, 2 * B), 256, 0, st>>>(
        (const U*)k, (const U*)v, src_bs / per, src_rs / per, (U*)kd, (U*)vd, dst_bs / per, dst_rs / per, width / per, B);
  };
  const uintptr_t ptrs = (uintptr_t)k | (uintptr_t)v | (uintptr_t)kd | (uintptr_t)vd;
  const uint64_t steps = (uint64_t)((src_bs | src_rs | dst_bs | dst_rs | (int64_t)width) * es);
  if (((ptrs | steps) & 15) == 0) go(uint4{});
  else if (es == 4) go(uint32_t{});
  else go(uint16_t{});
  return fa_check_launch("fa_append_rows");
}

extern "C" int fa_prompt_rows(const void* k, const void* v, int64_t bs, int64_t hs, int64_t rs, void* k_tok, void* v_tok,
                              void* k_near, void* v_near, int64_t near_bs, int n_first, int n_last, int spare, int dtype, int B,
                              int S, int heads, int D, fa_stream_t stream) {
  FA_REQUIRE(k && v && (!k_tok == !v_tok) && (!k_near == !v_near) && (k_tok || k_near), FA_ERR_NULL_POINTER,
             "fa_prompt_rows: null pointer");
  FA_REQUIRE(B > 0 && B <= 65535 && S > 0 && heads > 0 && D > 0 && n_first >= 0 && n_last >= 0 && (int64_t)n_first + n_last <= S &&
                 (spare == 0 || spare == 1), FA_ERR_BAD_SHAPE,
             "fa_prompt_rows: B=%d S=%d heads=%d D=%d near rows %d + %d + %d", B, S, heads, D, n_first, n_last, spare);
  FA_REQUIRE(dtype == FA_BF16 || dtype == FA_FP16 || dtype == FA_FP32, FA_ERR_BAD_DTYPE, "fa_prompt_rows: dtype %d", dtype);
  const int64_t es = dtype == FA_FP32 ? 4 : 2;
  const uintptr_t ptrs = (uintptr_t)k | (uintptr_t)v | (uintptr_t)k_tok | (uintptr_t)v_tok | (uintptr_t)k_near | (uintptr_t)v_near;
  FA_REQUIRE(((ptrs | (uint64_t)((bs | hs | rs | near_bs | D) * es)) & 15) == 0, FA_ERR_MISALIGNED,
             "fa_prompt_rows: rows, strides and pointers must be multiples of 16 bytes");
  const int64_t row = (int64_t)heads * D;
  FA_REQUIRE(!k_near || near_bs >= (n_first + n_last + spare) * row, FA_ERR_BAD_SHAPE, "fa_prompt_rows: near rows overlap");
  FA_REQUIRE(row * es / 16 * kPromptRows <= INT32_MAX - 1024, FA_ERR_UNSUPPORTED, "fa_prompt_rows: rows of %lld elements", (long long)row);
  const int per = (int)(16 / es);
  PromptRowsParams p{};
  p.k = (const uint4*)k; p.v = (const uint4*)v; p.bs = bs / per; p.hs = hs / per; p.rs = rs / per;
  p.k_tok = (uint4*)k_tok; p.v_tok = (uint4*)v_tok; p.k_near = (uint4*)k_near; p.v_near = (uint4*)v_near; p.near_bs = near_bs / per;
  p.n_first = n_first; p.n_last = n_last; p.spare = spare; p.S = S; p.heads = heads; p.ppd = D / per;
  const int rows = (k_tok ? S : n_first + n_last) + (k_near ? spare : 0);
  if (rows == 0) return FA_OK;
  prompt_rows_kernel<<<dim3(fa_cdiv(rows, kPromptRows), 2, B), 256, 0, fa_hip_stream(stream)>>>(p);
  return fa_check_launch("fa_prompt_rows");
}

extern "C" int fa_convert(const fa_convert_item* items, int n, fa_stream_t stream) {
  FA_REQUIRE(items || n == 0, FA_ERR_NULL_POINTER, "fa_convert: null pointer");
  FA_REQUIRE(n >= 0 && n <= kMaxConvert, FA_ERR_BAD_SHAPE, "fa_convert: %d items (at most %d)", n, kMaxConvert);
  ConvertArgs a{};
  int64_t most = 0;
  for (int i = 0; i < n; ++i) {
    const fa_convert_item& it = items[i];
    FA_REQUIRE(it.count >= 0 && (it.count == 0 || (it.src && it.dst)), FA_ERR_NULL_POINTER, "fa_convert: item %d", i);
    FA_REQUIRE(it.kind >= FA_CONVERT_I64_I32 && it.kind <= FA_CONVERT_PAD_I32, FA_ERR_BAD_DTYPE, "fa_convert: kind %d", it.kind);
    FA_REQUIRE(it.kind < FA_CONVERT_PAD_I64 || it.unit > 0, FA_ERR_BAD_SHAPE, "fa_convert: unit %d", it.unit);
    a.item[i] = it;
    if (it.count > most) most = it.count;
  }
  if (most == 0) return FA_OK;
  const int64_t blocks = (most + 255) / 256;
  convert_kernel<<<dim3((unsigned)(blocks < 64 ? blocks : 64), n), 256, 0, fa_hip_stream(stream)>>>(a);
  return fa_check_launch("fa_convert");
}

extern "C" int fa_mid_append(const void* row, int dtype, int64_t row_bs, int64_t pos, void* store, int64_t st_bs,
                             int cap_pages, const int32_t* n_list, const int32_t* n_h, const int32_t* pad_h, int B,
                             int Hkv, int Cn, int is_v, fa_stream_t stream) {
  FA_REQUIRE(row && store && n_h && pad_h, FA_ERR_NULL_POINTER, "fa_mid_append: null pointer");
  FA_REQUIRE(B > 0 && Hkv > 0 && Cn >= 0 && pos >= 0 && cap_pages > 0, FA_ERR_BAD_SHAPE, "fa_mid_append: bad shape");
  FA_REQUIRE(pos < (int64_t)cap_pages * 32, FA_ERR_BAD_SHAPE, "fa_mid_append: position %lld beyond %d pages",
             (long long)pos, cap_pages);
  if (Cn == 0) return FA_OK;
  FA_REQUIRE(n_list, FA_ERR_NULL_POINTER, "fa_mid_append: index list null");
  hipStream_t st = fa_hip_stream(stream);
  dim3 grid(fa_cdiv(Cn, 256), B);
  int rc = dispatch16(dtype, "fa_mid_append", [&](auto tag) {
    using E = decltype(tag);
    mid_append_kernel<E><<<grid, 256, 0, st>>>((const E*)row, row_bs, pos, (E*)store, st_bs, cap_pages, n_list, n_h, pad_h,
                                              Hkv, Cn, is_v);
  });
  return rc != FA_OK ? rc : fa_check_launch("fa_mid_append");
}

extern "C" int fa_mid_unpack(const void* store, int dtype, int64_t st_bs, int cap_pages, int L, void* dst,
                             const int32_t* n_h, const int32_t* pad_h, int B, int Hkv, int D, int Cn, int is_v,
                             fa_stream_t stream) {
  FA_REQUIRE(store && n_h && pad_h, FA_ERR_NULL_POINTER, "fa_mid_unpack: null pointer");
  FA_REQUIRE(B > 0 && Hkv > 0 && L >= 0 && Cn >= 0 && cap_pages > 0, FA_ERR_BAD_SHAPE, "fa_mid_unpack: bad shape");
  FA_REQUIRE((int64_t)cap_pages * 32 >= L, FA_ERR_BAD_SHAPE, "fa_mid_unpack: %d rows beyond %d pages", L, cap_pages);
  if (L == 0 || Cn == 0) return FA_OK;
  FA_REQUIRE(dst, FA_ERR_NULL_POINTER, "fa_mid_unpack: dst null");
  FA_REQUIRE(D > 0, FA_ERR_BAD_SHAPE, "fa_mid_unpack: head_dim %d", D);
  hipStream_t st = fa_hip_stream(stream);
  dim3 grid(fa_cdiv((int64_t)L * D, 256), Hkv, B);
  int rc = dispatch16(dtype, "fa_mid_unpack", [&](auto tag) {
    using E = decltype(tag);
    mid_unpack_kernel<E><<<grid, 256, 0, st>>>((const E*)store, st_bs, cap_pages, L, (E*)dst, n_h, pad_h, Cn, is_v);
  });
  return rc != FA_OK ? rc : fa_check_launch("fa_mid_unpack");
}
