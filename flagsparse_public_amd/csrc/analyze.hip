// analyze.hip -- one device pass that replaces the reference's host-synchronising
// validation reductions (spmv_csr.py:525-542, spmm_csr.py:226-252: indptr[0],
// indptr[-1], monotonicity, min/max column, max row length) and gathers the
// row-length statistics the kernel selector reads.  The caller copies the
// FS_STATS_LEN results to the host once.
//
// All statistics are integers, combined with integer atomics, so the result is
// exact and independent of scheduling.
#include "fs_host.hpp"

namespace fs {

constexpr int kAnBlock = 1024;
constexpr int kAnRows = 4;  // row pointer pairs in flight per thread

enum {
  ST_PTR0 = 0, ST_PTRN = 1, ST_DEC = 2, ST_CMIN = 3, ST_CMAX = 4, ST_LMAX = 5, ST_LMIN = 6,
  ST_SUMSQ = 7, ST_EMPTY = 8, ST_HIST = 9, ST_LONGNNZ = 15
};
static_assert(ST_LONGNNZ + 1 == FS_STATS_LEN, "statistics layout");

// Row-split outputs of fs_csr_analyze_split (see the header).  st[ST_SPLIT]
// counts long rows and chunks together, chunks in the low kSplitBits bits, so
// that one atomic gives a group of rows consecutive long-row ordinals and
// consecutive chunks at once.  That leaves the count 27 bits below the sign,
// which the entry point checks.
constexpr int ST_SPLIT = FS_STATS_LEN;
constexpr int kSplitBits = 36;

struct SplitOut {
  int64_t short_max = 0, cap_long = 0;
  uint32_t chunk_nnz = 1, cap_chunks = 0;
  int64_t* long_rows = nullptr;
  int64_t* long_chunk_ptr = nullptr;
  int32_t* chunk_long = nullptr;
  int32_t* cols32 = nullptr;
};

// Lists the block's long rows among kAnRows rows a thread (`row` + u * stride,
// long where bit u of `lg` is set).  The rows of a block take consecutive
// ordinals and chunks, so the counter sees one atomic per block and iteration;
// same-address atomics serialise, and with one per 64 rows that hold a long row
// they were most of the pass (both launches: 170,000 power-law rows, 2M 64-bit
// columns 40.5 -> 18.2 us; 1M such rows, 12M 32-bit columns 175 -> 24.6 us; no
// long row, 4.5M columns 14.2 -> 14.8 us).  The order of blocks is free, and so
// is the order of rows in the list: a row's chunks are its own and are summed in
// chunk order wherever they lie.  Row pointers are not validated yet, so every
// write is bounded by the capacities.
//
// Kept small (rolled loops, lengths read again): where no row is long, the
// pass pays for this only by the size of its code.
template <typename P>
__device__ __forceinline__ void split_rows(const SplitOut& s, int64_t* st, const P* ptr,
                                           uint32_t lg, int64_t row, int64_t stride, int turn) {
  // two turns' sums: those of one turn are written again only after the
  // barrier of the next, when nobody reads them any more
  __shared__ uint64_t wave_sum[2][kAnBlock / kWave];
  __shared__ uint64_t block_base;
  uint64_t* sums = wave_sum[turn & 1];
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  auto chunks = [&](int u) {
    const int64_t i = row + u * stride, l = (int64_t)ptr[i + 1] - (int64_t)ptr[i];
    const uint32_t c = (uint32_t)((l < INT32_MAX ? l : INT32_MAX) - 1) / s.chunk_nnz + 1;
    return c > s.cap_chunks ? s.cap_chunks + 1 : c;
  };
  uint64_t own = 0, scan = 0;  // scan: inclusive over the wavefront
  const bool some = __ballot(lg != 0) != 0;
  if (some) {
#pragma unroll 1
    for (uint32_t m = lg; m; m &= m - 1)
      own += ((uint64_t)1 << kSplitBits) + chunks(__builtin_ctz(m));
    scan = own;
#pragma unroll 1
    for (int k = 1; k < kWave; k <<= 1) {
      const uint64_t o = __shfl_up(scan, k);
      if (lane >= k) scan += o;
    }
  }
  if (lane == kWave - 1) sums[wv] = scan;
  __syncthreads();
  if (!__ballot(sums[lane % (kAnBlock / kWave)] != 0)) return;  // uniform over the block
  uint64_t before = 0, total = 0;
#pragma unroll 1
  for (int i = 0; i < kAnBlock / kWave; ++i) {
    before += i < wv ? sums[i] : 0;
    total += sums[i];
  }
  if (threadIdx.x == 0)
    block_base = __hip_atomic_fetch_add(reinterpret_cast<unsigned long long*>(st + ST_SPLIT), total,
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (!some) return;
  uint64_t at = block_base + before + scan - own;
#pragma unroll 1
  for (int u = 0; u < kAnRows; ++u) {
    const bool is_long = lg >> u & 1;
    const uint32_t per = is_long ? chunks(u) : 0;
    const int64_t li = (int64_t)(at >> kSplitBits);
    const int64_t c0 = (int64_t)(at & (((uint64_t)1 << kSplitBits) - 1));
    if (is_long && li < s.cap_long) {
      s.long_rows[li] = row + u * stride;
      s.long_chunk_ptr[li + 1] = c0 + per;  // where the next ordinal's chunks begin
      if (per == 1 && c0 < s.cap_chunks) s.chunk_long[c0] = (int32_t)li;
    }
    // rows of several chunks: the whole wavefront fills each row's chunk list
    for (uint64_t rest = __ballot(is_long && per > 1); rest; rest &= rest - 1) {
      const int src = __builtin_ctzll(rest);
      const uint32_t n = __shfl(per, src);
      const int64_t c = __shfl(c0, src), o = __shfl(li, src);
      for (uint32_t k = lane; k < n; k += kWave)
        if (o < s.cap_long && c + k < s.cap_chunks) s.chunk_long[c + k] = (int32_t)o;
    }
    at += ((uint64_t)is_long << kSplitBits) + per;
  }
}

template <typename P>
__global__ void analyze_init(const P* ptr, int64_t n_rows, int64_t* st, int64_t* long_chunk_ptr) {
  const int t = threadIdx.x;
  if (t == 0 && long_chunk_ptr) {
    st[ST_SPLIT] = 0;
    long_chunk_ptr[0] = 0;
  }
  if (t < FS_STATS_LEN) {
    int64_t v = 0;
    if (t == ST_CMIN) v = INT64_MAX;
    else if (t == ST_CMAX) v = -1;
    else if (t == ST_LMIN) v = n_rows > 0 ? INT64_MAX : 0;
    else if (t == ST_PTR0) v = ptr ? (int64_t)ptr[0] : 0;
    else if (t == ST_PTRN) v = ptr ? (int64_t)ptr[n_rows] : 0;
    st[t] = v;
  }
}

// Wave reductions by a butterfly of DPP / swizzle moves (fs_device.hpp: every
// lane of a 2K group holds the group's value after step K, so the mirror
// partners are as good as xor partners).
struct OpSum { template <typename T> __device__ static T of(T a, T b) { return a + b; } };
struct OpMax { template <typename T> __device__ static T of(T a, T b) { return a > b ? a : b; } };
struct OpMin { template <typename T> __device__ static T of(T a, T b) { return a < b ? a : b; } };

template <int K> __device__ __forceinline__ int32_t an_move(int32_t v) { return xmov_i32<K>(v); }
template <int K> __device__ __forceinline__ int64_t an_move(int64_t v) {
  const int lo = xmov_i32<K>((int)(v & 0xffffffff));
  const int hi = xmov_i32<K>((int)(v >> 32));
  return ((int64_t)hi << 32) | (uint32_t)lo;
}
template <typename Op, typename T> __device__ __forceinline__ T wave_reduce(T v) {
  v = Op::of(v, an_move<1>(v));
  v = Op::of(v, an_move<2>(v));
  v = Op::of(v, an_move<4>(v));
  v = Op::of(v, an_move<8>(v));
  v = Op::of(v, an_move<16>(v));
  return Op::of(v, an_move<32>(v));
}

// Reduction of statistic k: 0 sum, 1 max, 2 min (PTR0 / PTRN are set by
// analyze_init and not reduced).
__device__ __forceinline__ int stat_op(int k) {
  return (k == ST_LMAX || k == ST_CMAX) ? 1 : (k == ST_LMIN || k == ST_CMIN) ? 2 : 0;
}

// Reduces the block's statistics v[2..FS_STATS_LEN), each already reduced over
// its wavefront: one LDS exchange and one barrier, then thread k applies
// statistic k with one atomic.
__device__ __forceinline__ void block_apply_all(const int64_t (&v)[FS_STATS_LEN], int64_t* st) {
  __shared__ int64_t red[FS_STATS_LEN][kAnBlock / kWave];
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0)
#pragma unroll
    for (int k = 2; k < FS_STATS_LEN; ++k) red[k][w] = v[k];
  __syncthreads();
  const int k = threadIdx.x;
  if (k >= 2 && k < FS_STATS_LEN) {
    const int op = stat_op(k);
    int64_t r = red[k][0];
#pragma unroll
    for (int i = 1; i < kAnBlock / kWave; ++i) {
      const int64_t o = red[k][i];
      r = op == 0 ? r + o : op == 1 ? (o > r ? o : r) : (o < r ? o : r);
    }
    int64_t* dst = st + k;
    if (op == 0) { if (r) __hip_atomic_fetch_add(dst, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    else if (op == 1) __hip_atomic_fetch_max(dst, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_fetch_min(dst, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Memory-bound on large matrices and a latency chain on small ones, where the
// reduction used to be most of it (fourteen 64-bit wave reductions through
// ds_bpermute).  Counts are ballots summed in scalar registers, and the six
// statistics left are reduced with DPP moves.  With both launches: 16,384 rows
// of 16 entries 13.9 -> 8.6 us, 1M rows of 16 34.8 -> 22.8 us (67 MB), 4M rows
// of 12 51.0 -> 42.9 us (208 MB, 4.8 TB/s); with 64-bit arrays, whose columns
// took 8-byte loads, 15.6 -> 10.5, 41.3 -> 31.0, 82.0 -> 71.3 us (5.8 TB/s).
template <typename I, typename P, bool SPLIT, bool NT>
__global__ __launch_bounds__(kAnBlock) void analyze_pass(const P* __restrict__ ptr,
                                                          const I* __restrict__ idx,
                                                          int64_t n_rows, int64_t nnz,
                                                          int64_t* st, SplitOut split) {
  const int64_t stride = (int64_t)gridDim.x * kAnBlock;
  const int64_t t0 = (int64_t)blockIdx.x * kAnBlock + threadIdx.x;
  const int lane = threadIdx.x % kWave;
  int64_t lmax = 0, lmin = INT64_MAX, sumsq = 0, longnnz = 0;
  // wavefront totals: rows of length < 0, 0, and above each histogram edge
  int64_t dec = 0, empty = 0, g0 = 0, g4 = 0, g16 = 0, g64 = 0, g256 = 0, g4096 = 0;
  // rows: four row pointer pairs in flight; lanes past the end re-read the
  // last row and skip it.  The loop is uniform over the wavefront (ballots),
  // and where long rows are listed over the block (barriers).
  int turn = 0;
  for (int64_t w0 = SPLIT ? t0 - threadIdx.x : t0 - lane; w0 < n_rows; w0 += kAnRows * stride) {
    const int64_t w = SPLIT ? w0 + threadIdx.x : w0 + lane;
    uint32_t lg = 0;
    int64_t len[kAnRows];
#pragma unroll
    for (int u = 0; u < kAnRows; ++u) {
      const int64_t i = w + u * stride < n_rows ? w + u * stride : n_rows - 1;
      len[u] = (int64_t)ptr[i + 1] - (int64_t)ptr[i];
    }
#pragma unroll
    for (int u = 0; u < kAnRows; ++u) {
      const bool live = w + u * stride < n_rows;
      const int64_t l = len[u];
      dec += __popcll(__ballot(live && l < 0));
      empty += __popcll(__ballot(live && l == 0));
      g0 += __popcll(__ballot(live && l > 0));
      g4 += __popcll(__ballot(live && l > 4));
      g16 += __popcll(__ballot(live && l > 16));
      g64 += __popcll(__ballot(live && l > 64));
      g256 += __popcll(__ballot(live && l > 256));
      g4096 += __popcll(__ballot(live && l > 4096));
      if (live) {
        lmax = l > lmax ? l : lmax;
        lmin = l < lmin ? l : lmin;
        sumsq += l * l;
        if (l > 256) longnnz += l;
      }
      if constexpr (SPLIT) lg |= (uint32_t)(live && l > split.short_max) << u;
    }
    if constexpr (SPLIT) split_rows(split, st, ptr, lg, w, stride, turn++);
  }
  // columns: only min and max are kept, so a lane past the end re-reads the
  // iteration's first column instead of branching.  16-byte loads (four 32-bit
  // or two 64-bit columns), eight in flight per thread, over the aligned body
  // of the column array.  NT (non-temporal): see kAnNtBytes.
  typedef I vec_t __attribute__((ext_vector_type(16 / sizeof(I))));
  constexpr int kPer = 16 / (int)sizeof(I);
  I mn = sizeof(I) == 4 ? (I)INT32_MAX : (I)INT64_MAX, mx = -1;
  const int64_t head = (int64_t)(((16 - ((uintptr_t)idx & 15)) & 15) / sizeof(I));
  const int64_t h0 = head < nnz ? head : nnz;
  const int64_t nv = (nnz - h0) / kPer;
  const vec_t* q = reinterpret_cast<const vec_t*>(idx + h0);
  for (int64_t k = t0; k < nv; k += 8 * stride) {
    vec_t c[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const vec_t* at = q + (k + u * stride < nv ? k + u * stride : k);
      if constexpr (NT) c[u] = __builtin_nontemporal_load(at);
      else c[u] = *at;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        mn = c[u][e] < mn ? c[u][e] : mn;
        mx = c[u][e] > mx ? c[u][e] : mx;
      }
    if constexpr (SPLIT && sizeof(I) == 8) {
      // 32-bit copy of the columns; a vector past the end is vector k again
      if (split.cols32) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int64_t j = h0 + 2 * (k + u * stride < nv ? k + u * stride : k);
          split.cols32[j] = (int32_t)c[u][0];
          split.cols32[j + 1] = (int32_t)c[u][1];
        }
      }
    }
  }
  // the unaligned head and the tail: fewer than two vectors of columns
  const int64_t tail = h0 + kPer * nv;
  if (t0 < h0 + (nnz - tail)) {
    const int64_t j = t0 < h0 ? t0 : tail + (t0 - h0);
    const I c = idx[j];
    if constexpr (SPLIT && sizeof(I) == 8)
      if (split.cols32) split.cols32[j] = (int32_t)c;
    mn = c < mn ? c : mn;
    mx = c > mx ? c : mx;
  }
  // no columns at all: the initial INT64_MAX stays (every 32-bit column is
  // at most the narrower start value)
  const int64_t cmin = nnz > 0 ? (int64_t)wave_reduce<OpMin>(mn) : INT64_MAX;
  const int64_t v[FS_STATS_LEN] = {
      0, 0, dec, cmin, (int64_t)wave_reduce<OpMax>(mx), wave_reduce<OpMax>(lmax),
      wave_reduce<OpMin>(lmin), wave_reduce<OpSum>(sumsq), empty, g0 - g4, g4 - g16, g16 - g64,
      g64 - g256, g256 - g4096, g4096, wave_reduce<OpSum>(longnnz)};
  block_apply_all(v, st);
}

// Columns of more bytes than this are read past the caches.  An unprepared
// call's product follows at once and reads the columns again.  Smaller ones it
// finds where this pass left them (whole calls, non-temporal -> cached: 4.5M
// 32-bit columns in fp64 55.8 -> 53.7 us, 4.4M 64-bit ones in bf16 72.5 -> 65.0,
// 20M 32-bit ones in fp32 116.6 -> 114.5); larger ones only push its other data
// out (24M 32-bit columns 142 -> 149 us, 48M 243 -> 257, 36M 64-bit 288 -> 293).
constexpr int64_t kAnNtBytes = (int64_t)80 << 20;

template <typename I, typename P>
int launch_analyze(const fs_csr* A, int64_t* st, const SplitOut* split, hipStream_t s) {
  const P* ptr = static_cast<const P*>(A->row_ptr);
  const I* idx = static_cast<const I*>(A->col_idx);
  analyze_init<P><<<1, 64, 0, s>>>(ptr, A->n_rows, st, split ? split->long_chunk_ptr : nullptr);
  int rc = check_launch("fs_csr_analyze");
  if (rc) return rc;
  const int64_t work = A->n_rows > A->nnz ? A->n_rows : A->nnz;
  if (work == 0) return FS_OK;
  // few, wide blocks (one per CU): each reduces in LDS first, so every
  // statistic sees at most `blocks` same-address atomics (they serialise: with
  // two blocks per CU 1M rows of 16 take 28.2 instead of 22.8 us), while each
  // thread keeps eight 16-byte column loads in flight
  int64_t blocks = (work + kAnBlock * 32 - 1) / (kAnBlock * 32);
  if (blocks > 256) blocks = 256;
  const bool nt = A->nnz * (int64_t)sizeof(I) > kAnNtBytes;
  const SplitOut out = split ? *split : SplitOut{};
  auto run = split ? (nt ? analyze_pass<I, P, true, true> : analyze_pass<I, P, true, false>)
                   : (nt ? analyze_pass<I, P, false, true> : analyze_pass<I, P, false, false>);
  run<<<(unsigned)blocks, kAnBlock, 0, s>>>(ptr, idx, A->n_rows, A->nnz, st, out);
  return check_launch("fs_csr_analyze");
}

static int analyze_checked(const fs_csr* A, int64_t* stats, const SplitOut* split, void* stream,
                           const char* who) {
  if (!A) return fail(FS_ERR_VALUE, "%s: matrix descriptor is null", who);
  if ((A->index_type != FS_I32 && A->index_type != FS_I64) ||
      (A->ptr_type != FS_I32 && A->ptr_type != FS_I64))
    return fail(FS_ERR_TYPE, "%s: index and row-pointer types must be FS_I32 or FS_I64", who);
  if (A->n_rows < 0 || A->nnz < 0) return fail(FS_ERR_VALUE, "%s: negative size", who);
  if (!stats) return fail(FS_ERR_VALUE, "%s: stats is null", who);
  if (!A->row_ptr) return fail(FS_ERR_VALUE, "%s: row_ptr is null", who);
  if (A->nnz > 0 && !A->col_idx) return fail(FS_ERR_VALUE, "%s: col_idx is null", who);
  hipStream_t s = as_stream(stream);
  if (A->index_type == FS_I32 && A->ptr_type == FS_I32) return launch_analyze<int32_t, int32_t>(A, stats, split, s);
  if (A->index_type == FS_I32 && A->ptr_type == FS_I64) return launch_analyze<int32_t, int64_t>(A, stats, split, s);
  if (A->index_type == FS_I64 && A->ptr_type == FS_I32) return launch_analyze<int64_t, int32_t>(A, stats, split, s);
  return launch_analyze<int64_t, int64_t>(A, stats, split, s);
}

}  // namespace fs

using namespace fs;

extern "C" int fs_csr_analyze(const fs_csr* A, int64_t* stats, void* stream) {
  return analyze_checked(A, stats, nullptr, stream, "fs_csr_analyze");
}

extern "C" int fs_csr_analyze_split(const fs_csr* A, int64_t* stats, int64_t short_max,
                                    int64_t chunk_nnz, int64_t* long_rows, int64_t* long_chunk_ptr,
                                    int64_t cap_long, int32_t* chunk_long, int64_t cap_chunks,
                                    int32_t* cols32, void* stream) {
  const char* who = "fs_csr_analyze_split";
  if (A && A->nnz > INT32_MAX) return fail(FS_ERR_UNSUPPORTED, "%s: more than 2^31 - 1 entries", who);
  if (short_max < 1) return fail(FS_ERR_VALUE, "%s: short_max must be >= 1", who);
  if (chunk_nnz <= 0 || chunk_nnz % kWave != 0)
    return fail(FS_ERR_VALUE, "%s: chunk_nnz must be a positive multiple of 64", who);
  if (A && (A->n_rows < cap_long ? A->n_rows : cap_long) >= (int64_t)1 << (63 - kSplitBits))
    return fail(FS_ERR_UNSUPPORTED, "%s: room for 2^27 long rows or more", who);
  if (cap_long < 0 || cap_chunks < 0 || cap_long > INT32_MAX || cap_chunks > INT32_MAX)
    return fail(FS_ERR_VALUE, "%s: capacities must be in [0, 2^31)", who);
  if (!long_chunk_ptr || (cap_long > 0 && !long_rows) || (cap_chunks > 0 && !chunk_long))
    return fail(FS_ERR_VALUE, "%s: null list", who);
  SplitOut s;
  s.short_max = short_max;
  s.chunk_nnz = (uint32_t)(chunk_nnz < INT32_MAX ? chunk_nnz : INT32_MAX);  // rows are no longer
  s.cap_long = cap_long;
  s.cap_chunks = (uint32_t)cap_chunks;
  s.long_rows = long_rows;
  s.long_chunk_ptr = long_chunk_ptr;
  s.chunk_long = chunk_long;
  s.cols32 = cols32;
  return analyze_checked(A, stats, &s, stream, who);
}
