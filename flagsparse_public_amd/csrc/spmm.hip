// spmm.hip -- CSR SpMM for gfx950: C = alpha * A B + beta * C, row-major B and C.
//
// A group of G lanes owns one row and a tile of G*VW dense columns; each lane
// owns VW consecutive columns and gathers them from the B row of every entry
// with one vector load (16 bytes: fp32 x4, fp64 x2, 16-bit x8, complex64 x2), so
// a group reads one contiguous B-row segment per entry.  U entries are kept in
// flight per lane.  Rows longer than short_max are cut into chunks reduced by
// whole wavefronts (64/G groups interleave over the chunk's entries and are
// combined with xor exchanges); a row spanning several chunks stores one
// partial row per chunk, and spmm_fixup_kernel (a second, small launch) sums
// them in chunk order.
//
// Bound (B beyond L2): the 128-byte lines of the gathered B rows, which the
// Infinity Cache delivers at about 7 TB/s whatever the element type: 250,000
// rows with 5M random entries take 181 us for 256-byte B rows both in bf16
// (N = 128) and fp32 (N = 64).  16-bit values were bound by the lane instead:
// one 2-byte element per lane and load, one row per wavefront, 374 us for
// bf16 N = 128, 190 us for N = 64 (now 97 us); odd widths by scalar loads:
// fp32 N = 33 191 -> 167 us, bf16 N = 47 194 -> 138 us (a 94-byte row touches
// 1.7 lines on average).
//
// Replaces the reference's ALG1 row x column-tile kernel (spmm_csr.py:92-134,
// 525-599) and the bucketed opt / alg2 kernels (spmm_csr.py:602-919,
// spmm_csr_opt_alg2.py:338-629).
#include "spmm_kernel.hpp"

namespace fs {

template <typename V, typename I, typename P>
struct SpmmParams {
  const P* ptr;
  const I* idx;
  const V* val;
  const V* B;
  V* C;
  int64_t ldb, ldc, n_dense;
  int64_t n_rows;
  int64_t n_tiles;  // column tiles of G*VW columns
  double alpha, beta;
  int64_t short_max;
  int64_t n_chunk_blocks;
  int64_t n_chunks;
  int64_t chunk_nnz;
  const int64_t* long_rows;
  const int64_t* long_chunk_ptr;
  const int32_t* chunk_long;
  void* partials;     // [n_chunks * n_dense] accumulators
  int64_t n_blocks;   // of all launches of the kernel
  int64_t block0;     // first block of this one
  int xcd_remap;
};

// A launch holds fewer than 2^32 work-items: larger grids go in several.
constexpr int64_t kMmMostBlocks = ((int64_t)1 << 32) / kMmBlock - 1;

template <typename V, typename A, typename I, typename P, int G, int VW, int U>
__device__ __forceinline__ void spmm_chunk_role(const SpmmParams<V, I, P>& p, int64_t bid) {
  using CA = typename MmChunkAcc<A>::T;
  constexpr int kGroups = kWave / G;
  const int lane = threadIdx.x % kWave;
  const int64_t item = bid * kMmWaves + threadIdx.x / kWave;
  const int64_t c = item / p.n_tiles, tile = item % p.n_tiles;
  if (c >= p.n_chunks) return;
  const int grp = lane / G, g = lane % G;
  int64_t n0 = tile * (G * VW) + (int64_t)g * VW;
  const bool colok = n0 < p.n_dense;
  const int skip = shift_tail<VW>(n0, p.n_dense);
  const int64_t li = p.chunk_long[c];
  const int64_t row = p.long_rows[li];
  const int64_t c0 = p.long_chunk_ptr[li];
  const int64_t nc = p.long_chunk_ptr[li + 1] - c0;
  const int64_t rs = (int64_t)p.ptr[row], re = (int64_t)p.ptr[row + 1];
  const int64_t s = rs + (c - c0) * p.chunk_nnz;
  const int64_t e = s + p.chunk_nnz < re ? s + p.chunk_nnz : re;
  CA acc[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) acc[k].init();
  // four compensated columns a lane: seven entries of a chunk in flight, not the
  // eight of the other roles, keep the kernel at 80 registers and six wavefronts
  // per SIMD (1,048,576 rows of 15 entries, none of them in chunks, N = 64: 376 us,
  // 394 at five; with six entries 379, and 300 rows of 400 entries 5% slower)
  constexpr int UC = std::is_same<CA, Comp>::value && VW == 4 && U == 8 ? 7 : U;
  if (colok) mm_accumulate<VW, UC>(acc, p.idx, p.val, p.B, p.ldb, n0, s + grp, e, kGroups);
#pragma unroll
  for (int k = 0; k < VW; ++k) cross_group_reduce<G>(acc[k]);
  if (nc == 1) {
    if (grp == 0 && colok) write_vec<G, VW>(p.C, row * p.ldc + n0, acc, p.alpha, p.beta, skip);
    return;
  }
  CA* parts = reinterpret_cast<CA*>(p.partials);  // summed by spmm_fixup_kernel
  if (grp == 0 && colok)
#pragma unroll
    for (int k = 0; k < VW; ++k)
      if (k >= skip) parts[c * p.n_dense + n0 + k] = acc[k];
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Adds the partials of the kU chunks from k on at column n, all loads in flight.
template <int kU, typename CA>
__device__ __forceinline__ void fixup_batch(CA& tot, const CA* __restrict__ parts, int64_t n_dense,
                                            int64_t n, int64_t k) {
  CA q[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) q[u] = parts[(k + u) * n_dense + n];
#pragma unroll
  for (int u = 0; u < kU; ++u) tot.merge(q[u]);
}

// Sum of the partials of chunks [k0, k1) at column n, in chunk order.
template <typename CA>
__device__ __forceinline__ CA fixup_sum(const CA* __restrict__ parts, int64_t n_dense, int64_t n,
                                        int64_t k0, int64_t k1) {
  CA tot;
  tot.init();
  int64_t k = k0;
  for (; k + 8 <= k1; k += 8) fixup_batch<8>(tot, parts, n_dense, n, k);
  for (; k + 2 <= k1; k += 2) fixup_batch<2>(tot, parts, n_dense, n, k);
  if (k < k1) fixup_batch<1>(tot, parts, n_dense, n, k);
  return tot;
}

// Second pass for rows cut into several chunks.  Lanes take `cols` columns
// (a power of two, at most a wavefront) times 64 / cols ways, each way a
// contiguous range of the row's chunks; the ways' sums meet in LDS and are
// added in order.  A row of up to kFixWave chunks per way belongs to one
// wavefront; a longer one is summed by the block's four.  Bound by the
// latency of the longest row's chain of partial loads: one wavefront per row
// with one load at a time took 73 us where power-law rows of up to 100,000
// entries leave 391 chunks (N = 47, fp64 sums), this form 10 us; with two
// chunks in every row (20,000 rows of about 300 entries, N = 64) SpMM and
// fix-up take 137 us in both forms.
constexpr int kFixWave = 16;

template <typename A, typename V, typename I, typename P>
__global__ __launch_bounds__(kMmBlock) void spmm_fixup_kernel(SpmmParams<V, I, P> p, int64_t n_long,
                                                              int col_shift) {
  using CA = typename MmChunkAcc<A>::T;
  __shared__ CA part[kMmBlock];
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  const int cols = 1 << col_shift, ways = kWave >> col_shift;
  const int c = lane & (cols - 1), way = lane >> col_shift;
  const CA* parts = reinterpret_cast<const CA*>(p.partials);
  const int64_t l0 = (int64_t)blockIdx.x * kMmWaves;
  int64_t bound[kMmWaves + 1];  // all loaded together; past n_long: no chunks
#pragma unroll
  for (int r = 0; r <= kMmWaves; ++r)
    bound[r] = p.long_chunk_ptr[l0 + r < n_long ? l0 + r : n_long];
#pragma unroll
  for (int r = 0; r < kMmWaves; ++r) {  // the long rows of this block, uniform control flow
    const int64_t li = l0 + r;
    const int64_t c0 = bound[r];
    const int64_t nc = bound[r + 1] - c0;
    if (nc <= 1) continue;  // written by its chunk
    const bool whole = nc > (int64_t)kFixWave * ways;
    if (!whole && wv != r) continue;
    const int64_t row = p.long_rows[li];
    const int nw = whole ? ways * kMmWaves : ways;
    const int w = whole ? wv * ways + way : way;
    const int64_t per = (nc + nw - 1) / nw;
    // ways that have chunks (adding all 64 took 2 us more at N = 1, two chunks a row)
    const int used = (int)((nc + per - 1) / per);
    const int64_t k0 = c0 + (w * per < nc ? w * per : nc);
    const int64_t k1 = c0 + ((w + 1) * per < nc ? (w + 1) * per : nc);
    for (int64_t n0 = 0; n0 < p.n_dense; n0 += cols) {
      const int64_t n = n0 + c;
      CA tot;
      tot.init();
      if (n < p.n_dense) tot = fixup_sum(parts, p.n_dense, n, k0, k1);
      if (nw > 1) {
        part[threadIdx.x] = tot;
        if (whole) __syncthreads(); else wave_lds_sync();
        if (w == 0)
          for (int i = 1; i < used; ++i) tot.merge(part[(whole ? 0 : wv * kWave) + (i << col_shift) + c]);
        if (whole) __syncthreads(); else wave_lds_sync();
      }
      if (w == 0 && n < p.n_dense) write_out(p.C, row * p.ldc + n, tot.value(), p.alpha, p.beta);
    }
  }
}

template <typename V, typename I>
constexpr bool kHotSpmm = (std::is_same<V, float>::value || std::is_same<V, double>::value) &&
                          std::is_same<I, int32_t>::value;

// Short rows load their entries group-cooperatively in the int32-column
// kernels whose lane groups hold whole batches.
template <typename V, typename I, int G, int U>
constexpr bool kGroupLoads = std::is_same<I, int32_t>::value && G >= U && G % U == 0;

// Widest lane segment: 16 bytes (int64-column kernels: one column per lane).
template <typename V, typename I>
constexpr int kMaxVw = !std::is_same<I, int32_t>::value ? 1
                       : sizeof(V) == 2 ? 8 : sizeof(V) == 4 ? 4 : sizeof(V) == 8 ? 2 : 1;

// Lane groups narrower than a batch (G < U: few dense columns) take the
// wavefront's 64 / G consecutive rows together: their entries are
// contiguous, so the wavefront copies them into its LDS window with coalesced
// loads (64 consecutive entries per instruction) and each group reads its
// row's columns and values from there.  A wavefront whose rows hold more than
// kMmStageMax entries (a long row among them) loads per group instead.
template <typename V, typename I, int G, int U>
constexpr bool kWaveStaged = kHotSpmm<V, I> && G < U;

constexpr int kMmStage = 512;          // entries per wavefront window
constexpr int kMmStageMax = 8 * kMmStage;

template <typename A, int G, int VW, int U, typename V, typename I, typename P>
__device__ __forceinline__ void spmm_staged_rows(const SpmmParams<V, I, P>& p, int64_t rb,
                                                 int64_t row, int64_t n0, int skip) {
  using C = typename A::compute_t;
  __shared__ int32_t st_col[kMmWaves][kMmStage];
  __shared__ C st_val[kMmWaves][kMmStage];
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  const int64_t wrow0 = rb * (kMmBlock / G) + (int64_t)wv * (kWave / G);
  if (wrow0 >= p.n_rows) return;  // the whole wavefront
  const int64_t wrow1 = wrow0 + kWave / G < p.n_rows ? wrow0 + kWave / G : p.n_rows;
  const int64_t wb = (int64_t)p.ptr[wrow0], we = (int64_t)p.ptr[wrow1];
  const bool live = row < wrow1;
  const int64_t rs = live ? (int64_t)p.ptr[row] : we, re = live ? (int64_t)p.ptr[row + 1] : we;
  const bool mine = live && re - rs <= p.short_max && n0 < p.n_dense;  // longer: chunked
  A acc[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) acc[k].init();
  if (we - wb > kMmStageMax) {
    if (!mine) return;
    mm_accumulate<VW, U>(acc, p.idx, p.val, p.B, p.ldb, n0, rs, re, 1);
  } else {
    int32_t* sc = st_col[wv];
    C* sv = st_val[wv];
    for (int64_t w0 = wb; w0 < we; w0 += kMmStage) {
      const int64_t cnt = we - w0 < kMmStage ? we - w0 : kMmStage;
      // all of the window's loads first, then its LDS stores: a load whose
      // store sits in the same per-lane branch is waited for there, one slice
      // of the window at a time.  Slices wholly past cnt are skipped by the
      // wavefront (cnt is uniform); lanes past cnt re-read entry w0.
      constexpr int kPer = kMmStage / kWave;
      const int cntu = __builtin_amdgcn_readfirstlane((int)cnt);
      int32_t lc[kPer];
      V lv[kPer];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        if (k * kWave < cntu) {
          const int i = k * kWave + lane;
          const int64_t jj = w0 + (i < cntu ? i : 0);
          lc[k] = (int32_t)p.idx[jj];
          lv[k] = p.val[jj];
        } else {
          lc[k] = 0;
          lv[k] = V(0);
        }
      }
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        asm volatile("" : "+v"(lc[k]));
        asm volatile("" : "+v"(lv[k]));
      }
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int i = k * kWave + lane;
        if (i < cntu) {
          sc[i] = lc[k];
          sv[i] = (C)lv[k];
        }
      }
      wave_lds_sync();
      const int64_t lo = rs > w0 ? rs : w0;
      const int64_t hi = re < w0 + cnt ? re : w0 + cnt;
      if (mine) {
        for (int64_t j = lo; j < hi; j += U) {
          int64_t col[U];
          C a[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            // unconditional LDS reads (past hi: entry j again), as above
            const int64_t jj = j + u < hi ? j + u : j;
            col[u] = (int64_t)sc[jj - w0];
            a[u] = sv[jj - w0];
          }
          unsigned ok = 0;
#pragma unroll
          for (int u = 0; u < U; ++u) ok |= (unsigned)(j + u < hi) << u;
          RawVec<V, VW> r[U];
          gather_masked(r, p.B, p.ldb, col, n0, ok);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            C b[VW];
            widen_row(b, r[u]);
            if (j + u < hi)
#pragma unroll
              for (int k = 0; k < VW; ++k) acc[k].add_prod(a[u], b[k]);
          }
        }
      }
      wave_lds_sync();  // the window is rewritten next
    }
    if (!mine) return;
  }
  write_vec<G, VW>(p.C, row * p.ldc + n0, acc, p.alpha, p.beta, skip);
}

template <typename V, typename A, typename I, typename P, int G, int VW, int U>
__global__ __launch_bounds__(kMmBlock) void spmm_csr_kernel(SpmmParams<V, I, P> p) {
  const int64_t bid = p.block0 + blockIdx.x;
  if (bid < p.n_chunk_blocks) {
    spmm_chunk_role<V, A, I, P, G, VW, U>(p, bid);
    return;
  }
  int64_t sb = bid - p.n_chunk_blocks;
  if (p.xcd_remap) sb = xcd_remap_block(sb, p.n_blocks - p.n_chunk_blocks);
  const int64_t tile = sb % p.n_tiles, rb = sb / p.n_tiles;
  const int64_t row = rb * (kMmBlock / G) + threadIdx.x / G;
  const int g = threadIdx.x % G;
  int64_t n0 = tile * (G * VW) + (int64_t)g * VW;
  const int skip = shift_tail<VW>(n0, p.n_dense);
  if constexpr (kWaveStaged<V, I, G, U>) {
    spmm_staged_rows<A, G, VW, U>(p, rb, row, n0, skip);
    return;
  }
  if (row >= p.n_rows) return;  // the whole group
  const int64_t rs = (int64_t)p.ptr[row], re = (int64_t)p.ptr[row + 1];
  if (re - rs > p.short_max) return;  // chunked elsewhere (the whole group)
  A acc[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) acc[k].init();
  if constexpr (kGroupLoads<V, I, G, U>) {
    using C = typename A::compute_t;
    constexpr int F = kMmFill<G>;
    __shared__ int32_t slot_col[kMmBlock * F];
    __shared__ C slot_val[kMmBlock * F];
    const int first = (threadIdx.x - g) * F;  // the group's F * G slots
    const bool colok = n0 < p.n_dense;
    mm_accumulate_group<VW, U, G>(acc, slot_col + first, slot_val + first, p.idx, p.val, p.B,
                                  p.ldb, n0, colok, rs, re, g);
    if (!colok) return;
  } else {
    if (n0 >= p.n_dense) return;  // lanes past the last column own nothing
    mm_accumulate<VW, U>(acc, p.idx, p.val, p.B, p.ldb, n0, rs, re, 1);
  }
  write_vec<G, VW>(p.C, row * p.ldc + n0, acc, p.alpha, p.beta, skip);
}

// Whether each XCD takes a contiguous range of rows (xcd_remap_block) where the
// plan leaves it to the launch.  Neighbouring rows of matrices from meshes gather
// the same B rows, which one L2 then holds once; dealt in turn, blocks bring them
// into all eight.  fp32 / fp64, banded rows of 15: 1M rows N = 64 362 -> 351 us,
// N = 100 705 -> 643; 300,000 rows N = 100 210 -> 194, fp64 405 -> 345 us.  Random
// rows of 16: between -5% and +1%.  Not taken: B below 24 MB (20,000 rows N = 8 to
// 64: up to 8% slower), rows of under 12 entries (1M banded rows of 9, N = 64 234
// -> 241 us), 16-bit values (1M rows of 9, N = 100 303 -> 312 us), long rows, and
// column tiles, whose neighbours belong on different XCDs, unless the last tile
// holds a few columns only: it reads the lines where the tile before it ends, and
// finds them in the L2 of its own XCD.  Random rows of 15, fp64 N = 129 / 131: 344 ->
// 250 / 339 -> 242 us, fp32 N = 257 338 -> 235 us, bf16 N = 513 347 -> 300; rows of 5,
// power-law and banded rows, B of 2 to 400 MB: from -30% to +2%.  Tiles a quarter
// full: +8% on banded fp64 N = 158.
template <typename V>
static inline bool spmm_xcd_rows(const fs_csr* M, int64_t n_dense, int64_t tile, int64_t n_tiles,
                                 const fs_plan* pl) {
  if (n_tiles > 1) return n_dense % tile != 0 && n_dense % tile <= tile / 8;
  return (std::is_same<V, float>::value || std::is_same<V, double>::value) &&
         M->n_cols * n_dense * (int64_t)sizeof(V) >= ((int64_t)24 << 20) &&
         M->nnz >= 12 * M->n_rows && pl->n_long <= M->n_rows / 128;
}

template <typename V, typename A, typename I, typename P, int G, int VW>
int launch_spmm_gv(const fs_csr* M, const void* B, int64_t ldb, void* C, int64_t ldc,
                   int64_t n_dense, double alpha, double beta, const fs_plan* pl, hipStream_t st) {
  SpmmParams<V, I, P> p;
  p.ptr = static_cast<const P*>(M->row_ptr);
  p.idx = static_cast<const I*>(M->col_idx);
  p.val = static_cast<const V*>(M->values);
  p.B = static_cast<const V*>(B);
  p.C = static_cast<V*>(C);
  p.ldb = ldb;
  p.ldc = ldc;
  p.n_dense = n_dense;
  p.n_rows = M->n_rows;
  p.n_tiles = (n_dense + G * VW - 1) / (G * VW);
  p.alpha = alpha;
  p.beta = beta;
  p.short_max = pl->short_max;
  p.n_chunks = pl->n_chunks;
  p.n_chunk_blocks = (pl->n_chunks * p.n_tiles + kMmWaves - 1) / kMmWaves;
  p.chunk_nnz = pl->chunk_nnz;
  p.long_rows = pl->long_rows;
  p.long_chunk_ptr = pl->long_chunk_ptr;
  p.chunk_long = pl->chunk_long;
  p.partials = pl->partials;
  p.xcd_remap = pl->xcd_remap == FS_XCD_AUTO ? spmm_xcd_rows<V>(M, n_dense, G * VW, p.n_tiles, pl)
                                             : pl->xcd_remap != 0;
  const int64_t rows_per_block = kMmBlock / G;
  const int64_t short_blocks = ((M->n_rows + rows_per_block - 1) / rows_per_block) * p.n_tiles;
  const int64_t grid = p.n_chunk_blocks + short_blocks;
  if (grid == 0) return FS_OK;
  if (grid > 0x7fffffffLL)
    return fail(FS_ERR_UNSUPPORTED, "fs_spmm_csr: grid of %lld blocks too large", (long long)grid);
  // entries in flight per lane: 8 on request for fp32 / fp64 with int32
  // columns (short rows then finish in one or two batches), else 4
  auto kernel = spmm_csr_kernel<V, A, I, P, G, VW, 4>;
  if constexpr (kHotSpmm<V, I>)
    if (pl->unroll >= 8) kernel = spmm_csr_kernel<V, A, I, P, G, VW, 8>;
  p.n_blocks = grid;
  for (p.block0 = 0; p.block0 < grid; p.block0 += kMmMostBlocks) {
    const int64_t n = grid - p.block0 < kMmMostBlocks ? grid - p.block0 : kMmMostBlocks;
    kernel<<<dim3((unsigned)n), dim3(kMmBlock), 0, st>>>(p);
    const int rc = check_launch("fs_spmm_csr");
    if (rc) return rc;
  }
  if (pl->n_chunks <= pl->n_long) return FS_OK;  // no row spans several chunks
  const int64_t blocks = (pl->n_long + kMmWaves - 1) / kMmWaves;
  int col_shift = 0;
  while (col_shift < 6 && ((int64_t)1 << col_shift) < n_dense) ++col_shift;
  spmm_fixup_kernel<A><<<dim3((unsigned)blocks), dim3(kMmBlock), 0, st>>>(p, pl->n_long, col_shift);
  return check_launch("fs_spmm_csr");
}

// Lane groups built per vector width (spmm_tile_shape picks no others): the
// widest takes 8 to 64 lanes, narrower ones serve B with too few columns for
// eight lanes of the next width, hence at most 16 lanes.
template <typename V, typename A, typename I, typename P, int VW>
int launch_spmm_g(int G, const fs_csr* M, const void* B, int64_t ldb, void* C, int64_t ldc,
                  int64_t n_dense, double alpha, double beta, const fs_plan* pl, hipStream_t st) {
  constexpr int kMax = kMaxVw<V, I>;
  if constexpr (VW == 1) {
    if constexpr (kHotSpmm<V, I>) {
      if (G == 1) return launch_spmm_gv<V, A, I, P, 1, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
      if (G == 2) return launch_spmm_gv<V, A, I, P, 2, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
    }
    if (G <= 4) return launch_spmm_gv<V, A, I, P, 4, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  }
  if constexpr (std::is_same<I, int32_t>::value) {
    if (G <= 8) return launch_spmm_gv<V, A, I, P, 8, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  }
  if constexpr (VW < kMax) {
    return launch_spmm_gv<V, A, I, P, 16, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  } else {
    if (G <= 16) return launch_spmm_gv<V, A, I, P, 16, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
    if constexpr (std::is_same<I, int32_t>::value) {
      if (G <= 32) return launch_spmm_gv<V, A, I, P, 32, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
    }
    return launch_spmm_gv<V, A, I, P, 64, VW>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  }
}

// Whether B rows are cut into tiles of one 128-byte line, where plan and column
// tile leave it to the launch.  Tiles of one row go
// to neighbouring blocks, which the XCDs take in turn, so with 2, 4 or 8 tiles
// an XCD gathers only its part of every B row, and its L2 (4 MB) holds that many
// times as many rows.  That pays where B does not fit one L2 and one tile of it
// nearly does, rows have enough entries to pay for reading them once per tile,
// and no long rows dominate (their chunks bring the wide launch its
// parallelism).  Random rows of 20, fp32, N = 64 / 128 / 256: 32,000 rows 20.2 ->
// 17.8 / 39.9 -> 31.2 / 85.8 -> 59.3 us, 64,000 rows 42.3 -> 38.1 / 86.6 -> 68.6 /
// 181 -> 142 us, 96,000 rows 64.3 -> 59.4 / 134 -> 117 us; 160,000 rows 111 -> 109
// / 230 -> 221 us (not taken: banded ones 118 -> 118).  Against it: rows of 5,
// 64,000 rows, N = 128 29.6 -> 30.5 us; rows of 40 on a B of 8 MB, which the
// lines' repeated use keeps in L2 anyway, fp64 25.3 -> 27.1 us; power-law rows,
// 64,000, 66 -> 75 us.
static inline bool spmm_line_tiles(const fs_csr* M, int64_t row_bytes, const fs_plan* pl) {
  const int64_t lines = row_bytes / 128, panel = M->n_cols * 128, mb = 1 << 20;
  return row_bytes % 128 == 0 && (lines == 2 || lines == 4 || lines == 8) &&
         panel * lines > (M->nnz > 32 * M->n_rows ? 12 : 6) * mb &&
         panel <= (lines == 8 ? 8 : 12) * mb && M->nnz >= 8 * M->n_rows &&
         pl->n_long <= M->n_rows / 128;
}

template <typename V, typename A, typename I, typename P>
int launch_spmm(const fs_csr* M, const void* B, int64_t ldb, void* C, int64_t ldc, int64_t n_dense,
                double alpha, double beta, const fs_plan* pl, int32_t col_tile, hipStream_t st) {
  constexpr int kMax = kMaxVw<V, I>;
  if constexpr (std::is_same<I, int32_t>::value && kMax * sizeof(V) == 16 && kMax > 1)
    if (col_tile == 0 && pl->xcd_remap == FS_XCD_AUTO &&
        spmm_line_tiles(M, n_dense * (int64_t)sizeof(V), pl))
      return launch_spmm_g<V, A, I, P, kMax>(8, M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  // fp64, B rows of 1 KB and more: tiles of 512 bytes unless the last would be
  // mostly idle.  Tiles of one row go to neighbouring blocks, so with two
  // tiles each XCD (round-robin by block) gathers only its half of every B
  // row: N = 128, 250,000 rows of 20 random entries 742 -> 715 us, banded
  // 200,000 rows 319 -> 292 us; N = 100 (a 36-column last tile) 251 -> 279 us.
  // fp32 rows of 1 KB gain on random columns (730 -> 703 us) but lose on a
  // 1M-row band (1744 -> 1820 us).
  if (std::is_same<V, double>::value && kMax > 1 && col_tile == 0 && n_dense >= 128 &&
      (n_dense % 64 == 0 || n_dense % 64 >= 32))
    col_tile = 64;
  // complex64 rows of 1 KB and more keep one 512-byte tile per wavefront, one
  // column per lane (100,000 rows of 20 random entries, N = 128 / 192: 275 /
  // 426 us against 280 / 457 with two columns per lane)
  if constexpr (std::is_same<V, c64_t>::value && kMax > 1)
    if (col_tile == 0 && n_dense >= 128)
      return launch_spmm_gv<V, A, I, P, 64, 1>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  int vw, G;
  spmm_tile_shape<kMax>(n_dense, col_tile, &vw, &G);
  if constexpr (kMax >= 8)
    if (vw == 8) return launch_spmm_g<V, A, I, P, 8>(G, M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  if constexpr (kMax >= 4)
    if (vw == 4) return launch_spmm_g<V, A, I, P, 4>(G, M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  if constexpr (kMax >= 2)
    if (vw == 2) return launch_spmm_g<V, A, I, P, 2>(G, M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
  return launch_spmm_g<V, A, I, P, 1>(G, M, B, ldb, C, ldc, n_dense, alpha, beta, pl, st);
}

template <typename V, typename A>
int launch_spmm_idx(const fs_csr* M, const void* B, int64_t ldb, void* C, int64_t ldc, int64_t n_dense,
                    double alpha, double beta, const fs_plan* pl, int32_t col_tile, hipStream_t st) {
  if (M->index_type == FS_I32 && M->ptr_type == FS_I32) return launch_spmm<V, A, int32_t, int32_t>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, col_tile, st);
  if (M->index_type == FS_I32 && M->ptr_type == FS_I64) return launch_spmm<V, A, int32_t, int64_t>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, col_tile, st);
  if (M->index_type == FS_I64 && M->ptr_type == FS_I32) return launch_spmm<V, A, int64_t, int32_t>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, col_tile, st);
  return launch_spmm<V, A, int64_t, int64_t>(M, B, ldb, C, ldc, n_dense, alpha, beta, pl, col_tile, st);
}

}  // namespace fs

using namespace fs;

extern "C" int fs_spmm_csr(const fs_csr* A, const void* B, int64_t ldb, void* C, int64_t ldc,
                           int64_t n_dense, double alpha, double beta, const fs_plan* plan,
                           int32_t col_tile, void* stream) {
  int rc = check_csr(A, "fs_spmm_csr");
  if (rc) return rc;
  if (n_dense < 0) return fail(FS_ERR_VALUE, "fs_spmm_csr: n_dense must be >= 0");
  if (col_tile < 0) return fail(FS_ERR_VALUE, "fs_spmm_csr: col_tile must be >= 0");
  rc = check_plan(plan, A, n_dense, "fs_spmm_csr");
  if (rc) return rc;
  if (A->n_rows == 0 || n_dense == 0) return FS_OK;
  if (!C) return fail(FS_ERR_VALUE, "fs_spmm_csr: C is null");
  if (A->n_cols > 0 && !B) return fail(FS_ERR_VALUE, "fs_spmm_csr: B is null");
  if (ldc < n_dense || (A->n_cols > 0 && ldb < n_dense))
    return fail(FS_ERR_VALUE, "fs_spmm_csr: leading dimensions must be >= n_dense");
  hipStream_t st = as_stream(stream);
  const bool wide = plan->accumulate == FS_ACC_WIDE;
  switch (A->value_type) {
    case FS_F16: return launch_spmm_idx<f16_t, Plain<float>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_BF16: return launch_spmm_idx<bf16_t, Plain<float>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_F32:
      return wide ? launch_spmm_idx<float, Plain<double>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st)
                  : launch_spmm_idx<float, Plain<float>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_F64: return launch_spmm_idx<double, Plain<double>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_C32: return launch_spmm_idx<c32_t, Plain<cplx<float>>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_C64: return launch_spmm_idx<c64_t, Plain<cplx<float>>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    case FS_C128: return launch_spmm_idx<c128_t, Plain<cplx<double>>>(A, B, ldb, C, ldc, n_dense, alpha, beta, plan, col_tile, st);
    default: return fail(FS_ERR_TYPE, "fs_spmm_csr: unsupported value_type %d", A->value_type);
  }
}
