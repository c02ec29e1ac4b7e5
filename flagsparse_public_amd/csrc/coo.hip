// coo.hip -- COO entries to CSR order on the device (entry point fs_coo_sort):
// the entries ordered by (row, column), equal pairs in input order, and the row
// pointer they imply, with the index-range checks in the same passes.
//
// A sample sort of packed keys row | column | input position (the bit widths
// of n_rows, n_cols and nnz, at most 64 together), so that keys are distinct
// and one comparison decides.  A stratified sample gives splitters for up to
// 4096 buckets; one pass over the entries finds every entry's bucket and
// counts; neighbouring buckets are joined into groups of about group_size
// entries; a second pass moves the keys and values into their groups; each
// group is sorted in LDS by one workgroup, so the result does not depend on the
// order in which the second pass placed the entries.  Skewed rows and repeated
// pairs need no special case: splitters are whole keys.
//
// Why not a radix sort of the key: it takes a pass of key and payload over
// memory per byte of row bits + column bits, and the row pointer's bincount on
// top (82 us of same-line atomics for 1.8M entries); here each entry moves
// twice.  Bound by LDS traffic, the latency of its short launches and the
// atomics with which tiles reserve their places rather than by bytes: 1.8M
// entries in 89 us (64-bit radix sort, index gathers, range reductions and
// bincount took 550 us), 4M power-law entries 190 us.
//
// Above 2^22 entries, where groups would outgrow the LDS, the same passes first
// move the entries into parts of about 1.8M keys (runs of hundreds of entries, at
// the rate of a copy) and then sort all parts at once, one per grid row, with
// the parts' sizes read on the device: 4.25M random entries 217 us, 14.4M banded
// 532 us (with the 64-bit radix sort and its follow-up passes about 2.9 ms).
//
// Bucket sizes vary with the sample (gamma distributed, four samples each).
// A group beyond kCooLargeCap entries, 4 times the mean group (8 times the mean
// bucket) at the size limit, is reported in *flags, and the caller sorts by
// other means.
#include "fs_host.hpp"

namespace fs {

// Entries per bucket aimed at: at 768 a group of 1.8M entries now and then
// passed kCooSmallCap, and sorting that one took 13 us more.
constexpr int kCooTarget = 448;
constexpr int kCooMaxBuckets = 4096;
constexpr int kCooOver = 4;          // sampled entries per bucket
constexpr int kCooItems = 8;         // entries per thread in the LDS sorts
constexpr int kCooSmallCap = 3584;   // group sizes of the two sort launches
constexpr int kCooLargeCap = 8192;
constexpr int kCooMinGroup = 512;    // entries per group aimed at
constexpr int kCooMaxGroup = 2048;
constexpr int kCooMaxGroups = 2048;
constexpr int kCooBins = 2048;       // bins of the in-group sort
constexpr int kCooBinMax = 32;       // entries of one bin it takes
constexpr int kCooTable = 2048;      // leading key bits that narrow the bucket search
constexpr int kCooTile = 8192;       // entries per workgroup of the two passes
constexpr int kCooBlock = 1024;
constexpr int64_t kCooMaxNnz = (int64_t)kCooMaxGroups * kCooMaxGroup;  // one part
// Larger inputs are first moved into parts of about this size (kCooMaxBuckets
// buckets of kCooTarget entries each); a part may be half as large again.
constexpr int64_t kCooPart = (int64_t)kCooMaxBuckets * kCooTarget;
constexpr int kCooMaxParts = 64;
constexpr int kCooMaxSamples = kCooOver * kCooMaxBuckets;
static_assert(kCooPart * 3 / 2 <= kCooMaxNnz, "part sizes");

constexpr int kCooBadRow = 1, kCooBadCol = 2, kCooOverflow = 4;

struct CooWork {
  uint64_t* sample;     // [kCooMaxSamples]; this and the next five: one per part
  uint64_t* splitters;  // [kCooMaxBuckets]
  uint32_t* counts;     // [kCooMaxBuckets]
  uint16_t* group_of;   // [kCooMaxBuckets]
  uint32_t* starts;     // [kCooMaxGroups + 1] first entry of each group
  uint32_t* cursor;     // [kCooMaxGroups]
  uint32_t* large;      // [parts * kCooMaxGroups + 1]: count, then part << 16 | group
  uint64_t* keys;       // [nnz] by group
  int32_t* rows;        // [nnz] sorted rows
  uint16_t* bucket;     // [nnz] bucket of each input entry
  uint64_t* part_keys;  // [nnz] by part, if there are several (then rows lie here too)
  char* part_values;    // [8 * nnz] likewise
  uint32_t* part_start; // [parts + 1]
};

struct CooShape {
  int64_t nnz, n_rows, n_cols;
  int col_shift, row_shift;  // key = row << row_shift | column << col_shift | position
  int table_shift;           // key >> table_shift < kCooTable for rows in range
  int parts;
  int64_t total;  // entries of all parts
  int n_buckets, n_samples, n_groups, group_size, over;  // over: samples per bucket
};

// The sizes that follow from nnz (at most kCooMaxNnz).
__host__ __device__ inline void coo_sizes(CooShape& s) {
  const uint32_t n = (uint32_t)s.nnz, nb = (n + kCooTarget - 1) / kCooTarget;
  s.over = kCooOver;
  s.n_buckets = (int)(nb > kCooMaxBuckets ? kCooMaxBuckets : nb);
  s.n_samples = s.n_buckets == 1 ? 0 : s.n_buckets * kCooOver;
  // about 1024 groups (four per CU, all resident), within the size limits
  uint32_t g = n / 1024;
  g = g < kCooMinGroup ? kCooMinGroup : g > kCooMaxGroup ? kCooMaxGroup : g;
  s.group_size = (int)g;
  s.n_groups = (int)((n - 1) / g + 1);
}

static int bits_for(int64_t n) {  // bits of 0 .. n - 1
  int b = 0;
  while (b < 63 && ((int64_t)1 << b) < n) ++b;
  return b;
}

// False where the packed key or the size does not fit.
static bool coo_shape(CooShape* s, int64_t nnz, int64_t n_rows, int64_t n_cols) {
  if (nnz < 1 || nnz > kCooPart * kCooMaxParts || n_rows < 0 || n_cols < 0 || n_rows > INT32_MAX || n_cols > INT32_MAX)
    return false;
  s->nnz = s->total = nnz;
  s->n_rows = n_rows;
  s->n_cols = n_cols;
  s->col_shift = bits_for(nnz);
  s->row_shift = s->col_shift + bits_for(n_cols);
  const int bits = s->row_shift + bits_for(n_rows);
  if (bits > 64 || s->row_shift > 63) return false;
  s->table_shift = bits > 11 ? bits - 11 : 0;
  static_assert(kCooTable == 1 << 11, "table bits");
  s->parts = nnz <= kCooMaxNnz ? 1 : (int)((nnz + kCooPart - 1) / kCooPart);
  if (s->parts == 1) {
    coo_sizes(*s);
  } else {  // the buckets and groups of the first move are the parts
    s->n_buckets = s->n_groups = s->parts;
    s->over = kCooMaxSamples / s->parts;
    s->n_samples = s->parts * s->over;
    s->group_size = 0;
  }
  return true;
}

// Carves the workspace (base may be null: only the size is wanted).
static int64_t coo_carve(CooWork* w, char* base, const CooShape& s) {
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + at : nullptr;
    at += (bytes + 255) / 256 * 256;
    return p;
  };
  const int64_t sets = s.parts == 1 ? 1 : s.parts + 1;  // the last for the move into parts
  w->sample = reinterpret_cast<uint64_t*>(take(8 * sets * kCooMaxSamples));
  w->splitters = reinterpret_cast<uint64_t*>(take(8 * sets * kCooMaxBuckets));
  w->counts = reinterpret_cast<uint32_t*>(take(4 * sets * kCooMaxBuckets));
  w->group_of = reinterpret_cast<uint16_t*>(take(2 * sets * kCooMaxBuckets));
  w->starts = reinterpret_cast<uint32_t*>(take(4 * sets * (kCooMaxGroups + 1)));
  w->cursor = reinterpret_cast<uint32_t*>(take(4 * sets * kCooMaxGroups));
  w->large = reinterpret_cast<uint32_t*>(take(4 * (sets * kCooMaxGroups + 1)));
  w->keys = reinterpret_cast<uint64_t*>(take(8 * s.nnz));
  w->bucket = reinterpret_cast<uint16_t*>(take(2 * s.nnz));
  w->part_keys = nullptr;
  w->part_values = nullptr;
  w->part_start = nullptr;
  if (s.parts == 1) {
    w->rows = reinterpret_cast<int32_t*>(take(4 * s.nnz));
  } else {
    w->part_keys = reinterpret_cast<uint64_t*>(take(8 * s.nnz));
    w->part_values = take(8 * s.nnz);
    w->part_start = reinterpret_cast<uint32_t*>(take(4 * (s.parts + 1)));
    w->rows = reinterpret_cast<int32_t*>(w->part_keys);  // read for the last time before
  }
  return at;
}

// Set p of the work arrays that there is one of per part.
__host__ __device__ inline void coo_set(CooWork& w, int64_t p) {
  w.sample += p * kCooMaxSamples;
  w.splitters += p * kCooMaxBuckets;
  w.counts += p * kCooMaxBuckets;
  w.group_of += p * kCooMaxBuckets;
  w.starts += p * (kCooMaxGroups + 1);
  w.cursor += p * kCooMaxGroups;
}

// Turns to part p: its sizes and its share of the arrays; returns its first
// entry, or -1 if there is nothing to do (coo_parts flags a part that is too
// large).  PARTS: whether there are several.
template <bool PARTS>
__device__ __forceinline__ int64_t coo_enter(CooShape& s, CooWork& w, int p) {
  if constexpr (!PARTS) return 0;
  const int64_t a = w.part_start[p], n = (int64_t)w.part_start[p + 1] - a;
  if (n < 1 || n > kCooPart * 3 / 2) return -1;
  s.nnz = n;
  coo_sizes(s);
  coo_set(w, p);
  w.keys += a;
  w.rows += a;
  w.bucket += a;
  w.part_keys += a;
  return a;
}

// The entries a pass reads: index pairs, or the keys of a part.
template <typename I> struct CooPairs {
  static constexpr bool kParts = false;
  typedef struct { I row, col; } entry;
  const I* __restrict__ row;
  const I* __restrict__ col;
  __device__ entry load(const CooWork&, int64_t e) const { return {row[e], col[e]}; }
  // Out-of-range rows and columns give some key (they are flagged by coo_count
  // and the outputs are not used): any 64-bit value sorts.
  __device__ uint64_t key(const CooShape& s, entry x, int64_t e) const {
    return ((uint64_t)x.row << s.row_shift) | ((uint64_t)x.col << s.col_shift) | (uint64_t)e;
  }
  __device__ int bad(const CooShape& s, entry x) const {
    return ((int64_t)x.row < 0 || (int64_t)x.row >= s.n_rows ? kCooBadRow : 0) |
           ((int64_t)x.col < 0 || (int64_t)x.col >= s.n_cols ? kCooBadCol : 0);
  }
};
struct CooKeys {
  static constexpr bool kParts = true;
  typedef uint64_t entry;
  __device__ entry load(const CooWork& w, int64_t e) const { return w.part_keys[e]; }
  __device__ uint64_t key(const CooShape&, entry x, int64_t) const { return x; }
  __device__ int bad(const CooShape&, entry) const { return 0; }
};

// Sample i: from the i-th of equal ranges of the input, at a hashed place
// inside it.  Also clears the counters of the passes that follow.
template <typename In>
__global__ __launch_bounds__(256) void coo_sample(In in, CooShape s, CooWork w, int64_t* flags) {
  if (coo_enter<In::kParts>(s, w, blockIdx.y) < 0) return;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < s.n_buckets) w.counts[i] = 0;
  if (i == 0 && !In::kParts) {
    w.large[0] = 0;
    *flags = 0;
  }
  if (i >= s.n_samples) return;
  const int64_t a = (int64_t)i * s.nnz / s.n_samples, z = (int64_t)(i + 1) * s.nnz / s.n_samples;
  uint32_t h = (uint32_t)i * 2654435761u;
  h = (h ^ (h >> 15)) * 2246822519u;
  const int64_t e = a + (int64_t)((h ^ (h >> 13)) % (uint32_t)(z - a));
  w.sample[i] = in.key(s, in.load(w, e), e);
}

// Splitters: every workgroup bins the whole sample by its leading key bits in
// LDS and ranks some of its members, 16 lanes counting the smaller keys of the
// member's bin; the members of rank over * k are the splitters (keys are
// distinct).  A bin may hold any part of the sample (skewed rows), hence the
// many workgroups.  Counting over the whole sample instead took 15 us where
// this takes 7 (9,400 samples).
constexpr int kCooRanked = 64;  // members a workgroup ranks at a time

template <bool PARTS>
__global__ __launch_bounds__(kCooBlock) void coo_splitters(CooShape s, CooWork w) {
  extern __shared__ uint64_t binned[];
  __shared__ uint32_t bin[kCooTable + 1];
  __shared__ uint32_t part[kCooBlock / kWave];
  if (coo_enter<PARTS>(s, w, blockIdx.y) < 0) return;
  constexpr int kU = kCooMaxSamples / kCooBlock;
  static_assert(kCooTable == 2 * kCooBlock, "two bins a thread");
  const int t = threadIdx.x, lane = t % kWave, wv = t / kWave, n = s.n_samples;
  auto bin_of = [&](uint64_t key) {
    const uint64_t h = key >> s.table_shift;
    return h < kCooTable ? (int)h : kCooTable - 1;
  };
  uint64_t k[kU];
  uint32_t r[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (t + u * kCooBlock < n) k[u] = w.sample[t + u * kCooBlock];
  bin[t] = bin[t + kCooBlock] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (t + u * kCooBlock < n) r[u] = atomicAdd(&bin[bin_of(k[u])], 1u);
  __syncthreads();
  const uint32_t n0 = bin[2 * t], n1 = bin[2 * t + 1];
  uint32_t scan = n0 + n1;
#pragma unroll
  for (int q = 1; q < kWave; q <<= 1) {
    const uint32_t o = __shfl_up(scan, q);
    if (lane >= q) scan += o;
  }
  if (lane == kWave - 1) part[wv] = scan;
  __syncthreads();
  uint32_t at = scan - n0 - n1;
  for (int i = 0; i < wv; ++i) at += part[i];
  bin[2 * t] = at;
  bin[2 * t + 1] = at + n0;
  if (t == 0) bin[kCooTable] = (uint32_t)n;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (t + u * kCooBlock < n) binned[bin[bin_of(k[u])] + r[u]] = k[u];
  __syncthreads();
  for (int i = blockIdx.x * kCooRanked + t / 16; i < n; i += gridDim.x * kCooRanked) {
    const uint64_t m = w.sample[i];
    const int b = bin_of(m);
    uint32_t rank = 0;
    for (uint32_t q = bin[b] + t % 16; q < bin[b + 1]; q += 16) rank += binned[q] < m;
#pragma unroll
    for (int q = 1; q < 16; q <<= 1) rank += __shfl_xor(rank, q);
    rank += bin[b];
    if (t % 16 == 0 && rank > 0 && rank % s.over == 0) w.splitters[rank / s.over - 1] = m;
  }
}

// Bucket of every entry (the number of splitters <= its key), bucket sizes,
// and the range checks.  A table over the leading key bits leaves a step or two
// of the search where rows are filled evenly (3.7M entries, 4096 buckets: 44 ->
// 21 us; 1.8M: 17 -> 15 us, the rest being atomics).
template <typename In>
__global__ __launch_bounds__(kCooBlock) void coo_count(In in, CooShape s, CooWork w, int64_t* flags) {
  __shared__ uint64_t split[kCooMaxBuckets];
  __shared__ uint32_t hist[kCooMaxBuckets];
  __shared__ uint16_t table[kCooTable + 1];
  if (coo_enter<In::kParts>(s, w, blockIdx.y) < 0) return;
  const int t = threadIdx.x, last = s.n_buckets - 1;
  const int64_t e0 = (int64_t)blockIdx.x * kCooTile + t;
  if (e0 - t >= s.nnz) return;  // uniform: a part of fewer tiles
  constexpr int kU = kCooTile / kCooBlock;
  typename In::entry x[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u)
    x[u] = in.load(w, e0 + u * kCooBlock < s.nnz ? e0 + u * kCooBlock : s.nnz - 1);
  for (int b = t; b < s.n_buckets; b += kCooBlock) {
    hist[b] = 0;
    if (b < last) split[b] = w.splitters[b];
  }
  __syncthreads();
  // splitters in an earlier slot of the table; keys past the table's range
  // (flagged rows) search from its last slot on
  for (int h = t; h <= kCooTable; h += kCooBlock) {
    int lo = 0, hi = last;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (split[mid] >> s.table_shift < (uint64_t)h) lo = mid + 1; else hi = mid;
    }
    table[h] = (uint16_t)(h < kCooTable ? lo : last);
  }
  __syncthreads();
  int bad = 0;
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int64_t e = e0 + u * kCooBlock;
    if (e >= s.nnz) break;
    bad |= in.bad(s, x[u]);
    const uint64_t key = in.key(s, x[u], e);
    const uint64_t h = key >> s.table_shift;
    const int slot = h < kCooTable ? (int)h : kCooTable - 1;
    int lo = table[slot], hi = table[slot + 1];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (split[mid] <= key) lo = mid + 1; else hi = mid;
    }
    w.bucket[e] = (uint16_t)lo;
    atomicAdd(&hist[lo], 1u);
  }
  if (bad) atomicOr(reinterpret_cast<unsigned long long*>(flags), (unsigned long long)bad);
  __syncthreads();
  // blocks begin at different buckets, so that they do not queue for one line
  const int turn = (int)(blockIdx.x * kWave % (unsigned)s.n_buckets);
  for (int i = t; i < s.n_buckets; i += kCooBlock) {
    const int b = i + turn < s.n_buckets ? i + turn : i + turn - s.n_buckets;
    if (hist[b]) atomicAdd(&w.counts[b], hist[b]);
  }
}

// Groups: bucket b belongs to group (entries before b) / group_size, so a
// group holds neighbouring buckets of group_size entries and at most one
// bucket more; starts of the groups (groups that begin no bucket are empty).
template <bool PARTS>
__global__ __launch_bounds__(kCooBlock) void coo_groups(CooShape s, CooWork w) {
  __shared__ uint32_t part[kCooBlock / kWave];
  __shared__ uint32_t start[kCooMaxGroups + 1];
  const int t = threadIdx.x, lane = t % kWave, wv = t / kWave;
  if (coo_enter<PARTS>(s, w, blockIdx.y) < 0) return;
  constexpr int kPer = kCooMaxBuckets / kCooBlock;
  for (int g = t; g <= s.n_groups; g += kCooBlock) start[g] = ~0u;
  uint32_t c[kPer], sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int b = t * kPer + k;
    c[k] = b < s.n_buckets ? w.counts[b] : 0;
    sum += c[k];
  }
  uint32_t scan = sum;
#pragma unroll
  for (int k = 1; k < kWave; k <<= 1) {
    const uint32_t o = __shfl_up(scan, k);
    if (lane >= k) scan += o;
  }
  if (lane == kWave - 1) part[wv] = scan;
  __syncthreads();
  uint32_t at = scan - sum;
  for (int i = 0; i < wv; ++i) at += part[i];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int b = t * kPer + k;
    if (b < s.n_buckets) {
      // a bucket without entries may begin at nnz: it goes to the last group
      const uint32_t g = at / (uint32_t)s.group_size;
      const uint32_t grp = g < (uint32_t)s.n_groups ? g : (uint32_t)(s.n_groups - 1);
      w.group_of[b] = (uint16_t)grp;
      atomicMin(&start[grp], at);
      at += c[k];
    }
  }
  __syncthreads();
  for (int g = t; g <= s.n_groups; g += kCooBlock) {
    // an empty group starts where the next one that is not empty does
    uint32_t v = ~0u;
    for (int h = g; h < s.n_groups && v == ~0u; ++h) v = start[h];
    if (v == ~0u) v = (uint32_t)s.nnz;
    w.starts[g] = v;
    if (g < s.n_groups) w.cursor[g] = v;
  }
}

// The parts of the first move: its buckets, each a group of its own (w: its
// set of the work arrays).  One wavefront.
__global__ __launch_bounds__(kWave) void coo_parts(CooShape s, CooWork w, int64_t* flags) {
  static_assert(kCooMaxParts == kWave, "one part a lane");
  const int p = threadIdx.x;
  const uint32_t n = p < s.parts ? w.counts[p] : 0;
  uint32_t scan = n;
#pragma unroll
  for (int k = 1; k < kWave; k <<= 1) {
    const uint32_t o = __shfl_up(scan, k);
    if (p >= k) scan += o;
  }
  if (p < s.parts) {
    w.group_of[p] = (uint16_t)p;
    w.cursor[p] = w.part_start[p] = scan - n;
    if (p == s.parts - 1) w.part_start[s.parts] = scan;
  }
  if ((int64_t)n > kCooPart * 3 / 2)
    atomicOr(reinterpret_cast<unsigned long long*>(flags), (unsigned long long)kCooOverflow);
}

template <typename O, int VB> struct CooOut {
  const char* values;
  char* out_values;
  O* out_row;  // or null
  O* out_col;
};

template <int VB> struct CooValue {
  typedef uint64_t type __attribute__((ext_vector_type(2)));
  type x;
};
template <> struct CooValue<2> { uint16_t x; };
template <> struct CooValue<4> { uint32_t x; };
template <> struct CooValue<8> { uint64_t x; };

// Values are aligned to their components only (8 bytes of a 16-byte one).
template <int VB> __device__ __forceinline__ CooValue<VB> load_value(const char* p, int64_t i) {
  CooValue<VB> v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p + i * VB, VB < 8 ? VB : VB == 8 ? 4 : 8), VB);
  return v;
}
template <int VB> __device__ __forceinline__ void store_value(char* p, int64_t i, CooValue<VB> v) {
  __builtin_memcpy(__builtin_assume_aligned(p + i * VB, VB < 8 ? VB : VB == 8 ? 4 : 8), &v, VB);
}

// Moves the keys and the values into their groups: a workgroup reserves its
// share of every group with one atomic and places its entries there, brought
// into group order in LDS first, so that a group's share is one run of a store.
// Stores from input order to scattered places bound this pass (1.8M entries: 19
// us for the keys alone, 44 us with 4-byte values; 18.6 and 22 us in runs), and
// with the values here the sort reads them in order instead of at random.
// 16-byte values stay where they are: the sort gathers them.  Tiles of 6144 and
// 4096 entries: 30 and 32 us (more atomics).
template <typename In, int VB>
__global__ __launch_bounds__(kCooBlock) void coo_scatter(In in, CooShape s, CooWork w,
                                                         const char* __restrict__ values,
                                                         uint64_t* __restrict__ out_keys,
                                                         char* __restrict__ out_values) {
  __shared__ uint64_t stage[kCooTile];
  __shared__ uint16_t owner[kCooTile];
  __shared__ uint32_t hist[kCooMaxGroups];   // entries, then first place of the tile's share
  __shared__ uint16_t first[kCooMaxGroups];  // first slot in the stage
  __shared__ uint32_t part[kCooBlock / kWave];
  uint16_t* group_of = reinterpret_cast<uint16_t*>(stage);  // until the stage is filled
  const int t = threadIdx.x, lane = t % kWave, wv = t / kWave;
  const int64_t a = coo_enter<In::kParts>(s, w, blockIdx.y);
  const int64_t tile0 = (int64_t)blockIdx.x * kCooTile, e0 = tile0 + t;
  if (a < 0 || tile0 >= s.nnz) return;  // uniform
  values += a * VB;
  out_keys += a;
  out_values += a * VB;
  for (int g = t; g < s.n_groups; g += kCooBlock) hist[g] = 0;
  for (int b = t; b < s.n_buckets; b += kCooBlock) group_of[b] = w.group_of[b];
  constexpr int kU = kCooTile / kCooBlock;
  uint64_t key[kU];
  CooValue<VB> v[kU];
  uint32_t g[kU], r[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int64_t e = e0 + u * kCooBlock < s.nnz ? e0 + u * kCooBlock : s.nnz - 1;
    key[u] = in.key(s, in.load(w, e), e);
    g[u] = w.bucket[e];
    if (VB <= 8) v[u] = load_value<VB>(values, e);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    g[u] = group_of[g[u]];
    if (e0 + u * kCooBlock < s.nnz) r[u] = atomicAdd(&hist[g[u]], 1u);
  }
  __syncthreads();
  // slots: exclusive scan of the counts, two groups a thread
  static_assert(kCooMaxGroups == 2 * kCooBlock, "two groups a thread");
  const uint32_t n0 = 2 * t < s.n_groups ? hist[2 * t] : 0;
  const uint32_t n1 = 2 * t + 1 < s.n_groups ? hist[2 * t + 1] : 0;
  uint32_t scan = n0 + n1;
#pragma unroll
  for (int k = 1; k < kWave; k <<= 1) {
    const uint32_t o = __shfl_up(scan, k);
    if (lane >= k) scan += o;
  }
  if (lane == kWave - 1) part[wv] = scan;
  __syncthreads();
  uint32_t at = scan - n0 - n1;
  for (int i = 0; i < wv; ++i) at += part[i];
  first[2 * t] = (uint16_t)at;
  first[2 * t + 1] = (uint16_t)(at + n0);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (e0 + u * kCooBlock < s.nnz) {
      r[u] += first[g[u]];
      stage[r[u]] = key[u];
      owner[r[u]] = (uint16_t)g[u];
    }
  __syncthreads();
  // the thread that holds group k's count reserves its places
  if (n0) hist[2 * t] = atomicAdd(&w.cursor[2 * t], n0) - at;
  if (n1) hist[2 * t + 1] = atomicAdd(&w.cursor[2 * t + 1], n1) - (at + n0);
  __syncthreads();
  const int n = s.nnz - tile0 < kCooTile ? (int)(s.nnz - tile0) : kCooTile;
  uint32_t to[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int i = t + u * kCooBlock;
    if (i < n) {
      to[u] = hist[owner[i]] + i;  // < nnz: the same entries were counted
      out_keys[to[u]] = stage[i];
    }
  }
  if constexpr (VB <= 8) {
    __syncthreads();
    CooValue<VB>* vs = reinterpret_cast<CooValue<VB>*>(stage);
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (e0 + u * kCooBlock < s.nnz) vs[r[u]] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (t + u * kCooBlock < n) store_value<VB>(out_values, to[u], vs[t + u * kCooBlock]);
  }
}

// One LDS slot of padding per thread's items keeps the blocked accesses off
// each other's banks.
__device__ __forceinline__ int coo_pad(int i) { return i + i / kCooItems; }
template <int CAP> constexpr int kCooLds = CAP + CAP / kCooItems;

// Merge sort of the n keys from entry s on into key[coo_pad(0 .. n - 1)]: every
// thread sorts eight keys in registers, then runs of 8, 16, ... are merged
// pairwise, each thread finding its eight outputs by a merge-path search.  n
// is rounded up to whole threads with keys above all others.
__device__ void coo_merge_sort(const CooWork& w, uint32_t s, int n, uint64_t* key) {
  constexpr int kN = kCooItems;
  const int t = threadIdx.x, m = (n + kN - 1) / kN * kN;
  const bool live = t * kN < m;
  uint64_t k[kN];
  if (live) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int j = t * kN + i;
      k[i] = j < n ? w.keys[s + j] : ~(uint64_t)0;
    }
#pragma unroll
    for (int r = 0; r < kN; ++r)
#pragma unroll
      for (int i = r & 1; i + 1 < kN; i += 2) {
        const uint64_t a = k[i], b = k[i + 1];
        k[i] = a < b ? a : b;
        k[i + 1] = a < b ? b : a;
      }
#pragma unroll
    for (int i = 0; i < kN; ++i) key[coo_pad(t * kN + i)] = k[i];
  }
  __syncthreads();
  for (int run = kN; run < m; run <<= 1) {
    if (live) {
      const int out0 = t * kN, a0 = out0 & ~(2 * run - 1), d = out0 - a0;
      const int la = run < m - a0 ? run : m - a0;  // the last runs may be short
      const int b0 = a0 + la, lb = run < m - b0 ? run : m - b0;
      int lo = d > lb ? d - lb : 0, hi = d < la ? d : la;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (key[coo_pad(b0 + d - 1 - mid)] < key[coo_pad(a0 + mid)]) hi = mid; else lo = mid + 1;
      }
      int a = lo, b = d - lo;
      uint64_t ka = a < la ? key[coo_pad(a0 + a)] : ~(uint64_t)0;
      uint64_t kb = b < lb ? key[coo_pad(b0 + b)] : ~(uint64_t)0;
#pragma unroll
      for (int i = 0; i < kN; ++i) {
        // an exhausted run reads as the largest key, which only the padding
        // equals: either side then gives the same value
        if (ka <= kb) {
          k[i] = ka;
          ++a;
          ka = a < la ? key[coo_pad(a0 + a)] : ~(uint64_t)0;
        } else {
          k[i] = kb;
          ++b;
          kb = b < lb ? key[coo_pad(b0 + b)] : ~(uint64_t)0;
        }
      }
    }
    __syncthreads();
    if (live)
#pragma unroll
      for (int i = 0; i < kN; ++i) key[coo_pad(t * kN + i)] = k[i];
    __syncthreads();
  }
}

struct CooBlockStats {
  uint64_t lo[16], hi[16];
  uint32_t sum[16], most[16];
};

// at: the sum over the threads before this one; most: the maximum over all.
template <int WAVES>
__device__ __forceinline__ void coo_scan(uint32_t sum, uint32_t& most, uint32_t& at, CooBlockStats& bs) {
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  uint32_t scan = sum;
#pragma unroll
  for (int q = 1; q < kWave; q <<= 1) {
    const uint32_t a = __shfl_up(scan, q), b = __shfl_xor(most, q);
    if (lane >= q) scan += a;
    most = b > most ? b : most;
  }
  if (lane == kWave - 1) {
    bs.sum[wv] = scan;
    bs.most[wv] = most;
  }
  __syncthreads();
  at = scan - sum;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    at += i < wv ? bs.sum[i] : 0;
    most = bs.most[i] > most ? bs.most[i] : most;
  }
}

// Sorts the n <= CAP keys from entry s on and writes the entries out.  Keys
// are binned by their leading bits below the group's range (about one key a
// bin where columns spread evenly inside rows), placed bin by bin, and ranked
// by counting the smaller keys of their bin.  Where a long row crowds one bin
// among many short ones, the bins are cut once more by their own ranges (2M
// power-law entries: 58 + 33 -> 38 + 15 us in the two launches, the rest from
// the values in place); groups that crowd there too (clustered columns) are
// merge-sorted.  1.8M even entries: 44 us with the merge sort alone, 34 us
// binned, 25 us with the values in place.
template <int CAP, typename O, int VB>
__device__ void coo_sort_group(const CooShape& sh, const CooWork& w, const CooOut<O, VB>& o,
                               uint32_t s, int n, char* smem, CooBlockStats& bs) {
  constexpr int kT = CAP / kCooItems, kWaves = kT / kWave, kU = kCooItems;
  uint64_t* key = reinterpret_cast<uint64_t*>(smem);
  uint32_t* bin = reinterpret_cast<uint32_t*>(smem + 8 * CAP);
  const int t = threadIdx.x, lane = t % kWave, wv = t / kWave;
  if (n == 0) return;  // uniform
  // values from coo_scatter: read before the barriers, written back after them
  CooValue<VB> v[kU];
  uint64_t k[kU], lo = ~(uint64_t)0, hi = 0;
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int j = t + u * kT;
    k[u] = w.keys[s + (j < n ? j : 0)];
    if (VB <= 8) v[u] = load_value<VB>(o.out_values, s + (j < n ? j : 0));
  }
  for (int b = t; b < kCooBins; b += kT) bin[b] = 0;
#pragma unroll
  for (int u = 0; u < kU; ++u) {  // past n: key 0 of the group again
    lo = k[u] < lo ? k[u] : lo;
    hi = k[u] > hi ? k[u] : hi;
  }
#pragma unroll
  for (int q = 32; q >= 1; q >>= 1) {
    const uint64_t a = __shfl_xor(lo, q), b = __shfl_xor(hi, q);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  if (lane == 0) {
    bs.lo[wv] = lo;
    bs.hi[wv] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    lo = bs.lo[i] < lo ? bs.lo[i] : lo;
    hi = bs.hi[i] > hi ? bs.hi[i] : hi;
  }
  // (hi - lo) >> shift < kCooBins
  const int width = 64 - (hi > lo ? __builtin_clzll(hi - lo) : 64);
  constexpr int kBinBits = 11;
  static_assert(kCooBins == 1 << kBinBits, "bin bits");
  const int shift = width > kBinBits ? width - kBinBits : 0;
  uint32_t r[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (t + u * kT < n) r[u] = atomicAdd(&bin[(k[u] - lo) >> shift], 1u);
  __syncthreads();
  // exclusive scan of the bins in place; a bin keeps its size in the top bits
  constexpr int kPer = (kCooBins + kT - 1) / kT;
  uint32_t c[kPer], sum = 0, most = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = t * kPer + i;
    c[i] = b < kCooBins ? bin[b] : 0;
    sum += c[i];
    most = c[i] > most ? c[i] : most;
  }
  uint32_t at;
  coo_scan<kWaves>(sum, most, at, bs);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int b = t * kPer + i;
    if (b < kCooBins) bin[b] = at | c[i] << 16;  // at <= CAP < 2^16
    at += c[i];
  }
  __syncthreads();
  uint32_t start[kU], size[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const uint32_t b = t + u * kT < n ? bin[(k[u] - lo) >> shift] : 0;
    start[u] = b & 0xffffu;
    size[u] = b >> 16;
  }
  if (most > (uint32_t)kCooBinMax) {  // uniform
    // second level: a bin of m keys is cut into m equal parts, which the places
    // of the sorted keys count; then as above
    uint32_t* part = reinterpret_cast<uint32_t*>(smem);
    for (int i = t; i < CAP; i += kT) part[i] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (t + u * kT < n) {
        const uint64_t in = (k[u] - lo) & (((uint64_t)1 << shift) - 1);
        const int drop = shift > 32 ? shift - 32 : 0;
        start[u] += (uint32_t)((in >> drop) * size[u] >> (shift - drop));
        r[u] = atomicAdd(&part[start[u]], 1u);
      }
    __syncthreads();
    uint32_t d[kU];
    sum = most = 0;
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      d[i] = part[t * kU + i];
      sum += d[i];
      most = d[i] > most ? d[i] : most;
    }
    coo_scan<kWaves>(sum, most, at, bs);
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      part[t * kU + i] = at | d[i] << 16;
      at += d[i];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t b = t + u * kT < n ? part[start[u]] : 0;
      start[u] = b & 0xffffu;
      size[u] = b >> 16;
    }
    __syncthreads();
  }
  const bool binned = most <= (uint32_t)kCooBinMax;  // uniform
  if (binned) {
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (t + u * kT < n) key[start[u] + r[u]] = k[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      r[u] = start[u];
      for (uint32_t i = 0; i < size[u]; ++i) r[u] += key[start[u] + i] < k[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (t + u * kT < n) {
        key[r[u]] = k[u];
        if (VB <= 8) store_value<VB>(o.out_values, (int64_t)s + r[u], v[u]);
      }
    __syncthreads();
  } else {
    __syncthreads();  // the bins' memory is the merge sort's
    coo_merge_sort(w, s, n, key);
  }
  const uint64_t pos_mask = ((uint64_t)1 << sh.col_shift) - 1;
  const uint64_t col_mask = ((uint64_t)1 << (sh.row_shift - sh.col_shift)) - 1;
  for (int i = t; i < n; i += kT) {
    const uint64_t kk = key[binned ? i : coo_pad(i)];
    const int64_t at = (int64_t)s + i;
    const int32_t row = (int32_t)(kk >> sh.row_shift);
    w.rows[at] = row;
    if (o.out_row) o.out_row[at] = (O)row;
    o.out_col[at] = (O)(int32_t)((kk >> sh.col_shift) & col_mask);
    // the position of a valid key; flagged input may hold any bits there
    const int64_t p = (int64_t)(kk & pos_mask);
    if (VB > 8 || !binned) store_value<VB>(o.out_values, at, load_value<VB>(o.values, p < sh.total ? p : 0));
  }
}

// keys and bins of the binned sort, or the padded keys of the merge sort
template <int CAP> constexpr int kCooSmem =
    8 * CAP + 4 * kCooBins > 8 * kCooLds<CAP> ? 8 * CAP + 4 * kCooBins : 8 * kCooLds<CAP>;

// Turns the outputs to the part that begins at entry a.
template <typename O, int VB> __device__ __forceinline__ void coo_out(CooOut<O, VB>& o, int64_t a) {
  o.out_values += a * VB;
  o.out_col += a;
  if (o.out_row) o.out_row += a;
}

template <typename O, int VB, bool PARTS>
__global__ __launch_bounds__(kCooSmallCap / kCooItems) void coo_sort_small(CooShape sh, CooWork w,
                                                                           CooOut<O, VB> o,
                                                                           int64_t* flags) {
  __shared__ __align__(8) char smem[kCooSmem<kCooSmallCap>];
  __shared__ CooBlockStats bs;
  const int64_t a = coo_enter<PARTS>(sh, w, blockIdx.y);
  if (a < 0 || (int)blockIdx.x >= sh.n_groups) return;  // uniform
  coo_out(o, a);
  const uint32_t s = w.starts[blockIdx.x];
  const int n = (int)(w.starts[blockIdx.x + 1] - s);
  if (n > kCooSmallCap) {  // left to coo_sort_large
    if (threadIdx.x == 0) {
      if (n > kCooLargeCap)
        atomicOr(reinterpret_cast<unsigned long long*>(flags), (unsigned long long)kCooOverflow);
      else
        w.large[1 + atomicAdd(w.large, 1u)] = blockIdx.y << 16 | blockIdx.x;
    }
    return;
  }
  coo_sort_group<kCooSmallCap, O, VB>(sh, w, o, s, n, smem, bs);
}

template <typename O, int VB, bool PARTS>
__global__ __launch_bounds__(kCooLargeCap / kCooItems) void coo_sort_large(CooShape sh, CooWork w,
                                                                           CooOut<O, VB> o) {
  __shared__ __align__(8) char smem[kCooSmem<kCooLargeCap>];
  __shared__ CooBlockStats bs;
  const uint32_t n_large = w.large[0];
  for (uint32_t i = blockIdx.x; i < n_large; i += gridDim.x) {
    const uint32_t id = w.large[1 + i], g = id & 0xffffu;
    CooShape ps = sh;
    CooWork pw = w;
    CooOut<O, VB> po = o;
    coo_out(po, coo_enter<PARTS>(ps, pw, (int)(id >> 16)));  // a listed part is not refused
    const uint32_t s = pw.starts[g];
    coo_sort_group<kCooLargeCap, O, VB>(ps, pw, po, s, (int)(pw.starts[g + 1] - s), smem, bs);
    __syncthreads();  // the next group reuses the LDS
  }
}

// Row pointer of the sorted rows: ptr[r] = entries in rows before r, by binary
// search (no dependence on gaps between rows).
template <typename P>
__global__ __launch_bounds__(256) void coo_row_ptr(const int32_t* __restrict__ rows, int64_t nnz,
                                                   int64_t n_rows, P* __restrict__ ptr) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r > n_rows) return;
  int64_t lo = 0, hi = nnz;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)rows[mid] < r) lo = mid + 1; else hi = mid;
  }
  ptr[r] = (P)lo;
}

// The passes over one input, or over all parts at once (grid y).
template <typename In, typename O, int VB>
int coo_passes(const In& in, const CooShape& s, const CooWork& w, const char* values,
               const CooOut<O, VB>& o, int64_t* flags, hipStream_t st) {
  constexpr bool kP = In::kParts;
  const unsigned parts = (unsigned)s.parts;
  // of one part at most
  const int64_t most = kP ? kCooPart * 3 / 2 : s.nnz;
  const int samples = kP ? kCooMaxSamples : s.n_samples, groups = kP ? kCooMaxGroups : s.n_groups;
  const dim3 tiles((unsigned)((most + kCooTile - 1) / kCooTile), parts);
  const int first = samples > s.n_buckets ? samples : s.n_buckets;
  coo_sample<In><<<dim3((first + 255) / 256, parts), 256, 0, st>>>(in, s, w, flags);
  if (kP || s.n_buckets > 1) {
    // parts: few workgroups each, the binning of the sample is most of it
    const dim3 grid(kP ? 32 : (samples + kCooRanked - 1) / kCooRanked, parts);
    coo_splitters<kP><<<grid, kCooBlock, sizeof(uint64_t) * samples, st>>>(s, w);
  }
  coo_count<In><<<tiles, kCooBlock, 0, st>>>(in, s, w, flags);
  coo_groups<kP><<<dim3(1, parts), kCooBlock, 0, st>>>(s, w);
  coo_scatter<In, VB><<<tiles, kCooBlock, 0, st>>>(in, s, w, values, w.keys, o.out_values);
  coo_sort_small<O, VB, kP><<<dim3(groups, parts), kCooSmallCap / kCooItems, 0, st>>>(s, w, o, flags);
  if (s.nnz > kCooSmallCap) {
    const int blocks = kP ? 256 : groups < 64 ? groups : 64;
    coo_sort_large<O, VB, kP><<<blocks, kCooLargeCap / kCooItems, 0, st>>>(s, w, o);
  }
  return check_launch("fs_coo_sort");
}

template <typename I, typename O, int VB>
int coo_run(const CooShape& s, const CooWork& w, const void* values, const I* row, const I* col,
            void* out_values, O* out_row, O* out_col, int64_t* flags, hipStream_t st) {
  const CooPairs<I> in{row, col};
  const CooOut<O, VB> o{static_cast<const char*>(values), static_cast<char*>(out_values), out_row, out_col};
  if (s.parts == 1) return coo_passes<CooPairs<I>, O, VB>(in, s, w, o.values, o, flags, st);
  // move the entries into the parts, with the same passes
  CooWork pw = w;
  coo_set(pw, s.parts);
  const unsigned tiles = (unsigned)((s.nnz + kCooTile - 1) / kCooTile);
  coo_sample<CooPairs<I>><<<(s.n_samples + 255) / 256, 256, 0, st>>>(in, s, pw, flags);
  coo_splitters<false><<<(s.n_samples + kCooRanked - 1) / kCooRanked, kCooBlock, sizeof(uint64_t) * s.n_samples, st>>>(s, pw);
  coo_count<CooPairs<I>><<<tiles, kCooBlock, 0, st>>>(in, s, pw, flags);
  coo_parts<<<1, kWave, 0, st>>>(s, pw, flags);
  coo_scatter<CooPairs<I>, VB><<<tiles, kCooBlock, 0, st>>>(in, s, pw, o.values, w.part_keys, w.part_values);
  return coo_passes<CooKeys, O, VB>(CooKeys{}, s, w, w.part_values, o, flags, st);
}

template <typename I, typename O>
int coo_run_vb(int vb, const CooShape& s, const CooWork& w, const void* values, const void* row,
               const void* col, void* out_values, void* out_row, void* out_col, int64_t* flags,
               hipStream_t st) {
  const I* r = static_cast<const I*>(row);
  const I* c = static_cast<const I*>(col);
  O* orow = static_cast<O*>(out_row);
  O* ocol = static_cast<O*>(out_col);
  switch (vb) {
    case 2: return coo_run<I, O, 2>(s, w, values, r, c, out_values, orow, ocol, flags, st);
    case 4: return coo_run<I, O, 4>(s, w, values, r, c, out_values, orow, ocol, flags, st);
    case 8: return coo_run<I, O, 8>(s, w, values, r, c, out_values, orow, ocol, flags, st);
    default: return coo_run<I, O, 16>(s, w, values, r, c, out_values, orow, ocol, flags, st);
  }
}

}  // namespace fs

using namespace fs;

extern "C" int64_t fs_coo_sort_workspace(int64_t nnz, int64_t n_rows, int64_t n_cols) {
  CooShape s;
  CooWork w;
  return coo_shape(&s, nnz, n_rows, n_cols) ? coo_carve(&w, nullptr, s) : 0;
}

extern "C" int fs_coo_sort(int32_t value_bytes, const void* values, int32_t index_type,
                           const void* row, const void* col, int64_t nnz, int64_t n_rows,
                           int64_t n_cols, void* out_values, int32_t out_index_type, void* out_row,
                           void* out_col, int32_t ptr_type, void* out_ptr, void* workspace,
                           int64_t workspace_bytes, int64_t* flags, void* stream) {
  const char* who = "fs_coo_sort";
  if (value_bytes != 2 && value_bytes != 4 && value_bytes != 8 && value_bytes != 16)
    return fail(FS_ERR_TYPE, "%s: values must have 2, 4, 8 or 16 bytes", who);
  if ((index_type != FS_I32 && index_type != FS_I64) ||
      (out_index_type != FS_I32 && out_index_type != FS_I64) ||
      (ptr_type != FS_I32 && ptr_type != FS_I64))
    return fail(FS_ERR_TYPE, "%s: index types must be FS_I32 or FS_I64", who);
  if (nnz < 1 || n_rows < 0 || n_cols < 0) return fail(FS_ERR_VALUE, "%s: bad size", who);
  CooShape s;
  if (!coo_shape(&s, nnz, n_rows, n_cols)) return fail(FS_ERR_UNSUPPORTED, "%s: too large", who);
  if (!values || !row || !col || !out_values || !out_col || !out_ptr || !workspace || !flags)
    return fail(FS_ERR_VALUE, "%s: null pointer", who);
  CooWork w;
  if (workspace_bytes < coo_carve(&w, static_cast<char*>(workspace), s))
    return fail(FS_ERR_VALUE, "%s: workspace too small", who);
  hipStream_t st = as_stream(stream);
  int rc;
  if (index_type == FS_I32)
    rc = out_index_type == FS_I32
             ? coo_run_vb<int32_t, int32_t>(value_bytes, s, w, values, row, col, out_values, out_row, out_col, flags, st)
             : coo_run_vb<int32_t, int64_t>(value_bytes, s, w, values, row, col, out_values, out_row, out_col, flags, st);
  else
    rc = out_index_type == FS_I32
             ? coo_run_vb<int64_t, int32_t>(value_bytes, s, w, values, row, col, out_values, out_row, out_col, flags, st)
             : coo_run_vb<int64_t, int64_t>(value_bytes, s, w, values, row, col, out_values, out_row, out_col, flags, st);
  if (rc) return rc;
  const unsigned blocks = (unsigned)((n_rows + 256) / 256);
  if (ptr_type == FS_I32)
    coo_row_ptr<int32_t><<<blocks, 256, 0, st>>>(w.rows, nnz, n_rows, static_cast<int32_t*>(out_ptr));
  else
    coo_row_ptr<int64_t><<<blocks, 256, 0, st>>>(w.rows, nnz, n_rows, static_cast<int64_t*>(out_ptr));
  return check_launch(who);
}
