// batched.hip -- many independent fp32 CSR SpMV / SpMM problems in one launch.
//
// The work list (device memory, built once per batch) holds items of
// (matrix, kind, row range), one block each: a few passes of the block's lane
// groups over SpMV rows, one over SpMM rows.  Rows are computed with the
// single-matrix kernels' short-row procedures (lane-group width, unroll,
// reduction tree), so a row's result is bit-identical to the single-matrix
// launch with the same group width.  A single-row item longer than a lane
// group's bound is reduced by the whole block instead.
//
// The hardware hands the blocks out: there is no queue to wait for and no item
// end at which a block's lane groups wait for the longest row of many, and
// blocks of both kinds share a CU.  32 matrices of 1,000 to 200,000 rows of 34
// (44M entries), one SpMV and one 8-column SpMM each: persistent blocks on a
// queue of 96 KB items, two lanes per SpMM row, 744 us; this form 587 us (SpMV
// alone 440 -> 248, SpMM alone 515 -> 376).  What bounds it: the requests of the
// gathers to L2 and, for B beyond L2, the 128-byte lines behind them.  Small
// batches no longer start and drain 2,048 blocks: 8 matrices of 15 to 3,000 rows
// of 10 69.8 -> 6.2 us; 16 of 500 to 100,000 rows of 8, N = 12, 145 -> 69 us.
// No counterpart in the reference (one launch per matrix and bucket there).
#include "spmm_kernel.hpp"
#include "spmv_kernel.hpp"

namespace fs {

constexpr int kBatBlock = 256;

struct BatchMatrix {
  const void* row_ptr;
  const int32_t* col;
  const float* val;
  const float* x;
  float* y;
  const float* B;
  float* C;
  int64_t n_rows, n_cols, nnz, n_dense, ldb, ldc;
  int32_t group_lanes, ptr64;
  int32_t mm_lanes, mm_vw;  // SpMM lane group and vector width
};

__device__ __forceinline__ int64_t bm_ptr(const BatchMatrix& m, int64_t r) {
  return m.ptr64 ? static_cast<const int64_t*>(m.row_ptr)[r]
                 : (int64_t) static_cast<const int32_t*>(m.row_ptr)[r];
}

// acc[r] += the products of row r's entries s[r] .. e[r] - 1 for lane g of S
// (entries g, g + S, ...: accumulate_span's order), two entries of each of the
// R rows in flight.
template <int R, int S>
__device__ __forceinline__ void bat_accumulate(Plain<float> (&acc)[R], const BatchMatrix& m,
                                               const int64_t (&s)[R], const int64_t (&e)[R], int g) {
  constexpr int U = 2;
  int64_t j[R];
  bool more = false;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    j[r] = s[r] + g;
    more |= j[r] < e[r];
  }
  while (more) {
    int32_t ci[R][U];
    float a[R][U], x[R][U];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = j[r] + u * S < e[r];
        ci[r][u] = ok ? m.col[j[r] + u * S] : 0;
        a[r][u] = ok ? m.val[j[r] + u * S] : 0.f;
      }
    // the empty asm keeps each index's use (and the wait for its load) out of
    // the masked load's branch, so all loads are issued before the first wait
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) asm volatile("" : "+v"(ci[r][u]));
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) x[r][u] = j[r] + u * S < e[r] ? m.x[(int64_t)ci[r][u]] : 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) asm volatile("" : "+v"(x[r][u]));
    more = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j[r] + u * S < e[r]) acc[r].add_prod(a[r][u], x[r][u]);
      j[r] += U * S;
      more |= j[r] < e[r];
    }
  }
}

// --- SpMV rows of an item with groups of S lanes (the single-matrix short
// role's lane order and group_reduce<S>).  A row of at most 2 S entries is one
// round of loads for its group; wide groups take two rows at once, whose rounds
// then overlap (32 matrices of rows of 34, SpMV alone: 268 -> 248 us, with the
// SpMMs 605 -> 587; four rows: 315 and 796 us, their registers cost the whole
// kernel wavefronts; 4-lane groups with two: 68.6 -> 69.5 us).  Rows over 8 S
// entries take accumulate_span's deeper batches one by one.
template <int S>
__device__ void bat_spmv_rows(const BatchMatrix& m, int64_t r0, int64_t r1, double alpha, double beta) {
  constexpr int kGroups = kBatBlock / S, R = S >= 16 ? 2 : 1;
  const int grp = threadIdx.x / S, g = threadIdx.x % S;
  DirectVals<float> vs{m.val};
  // every group runs the same number of iterations so the S-lane exchange in
  // group_reduce always sees its whole group active
  for (int64_t base = r0; base < r1; base += kGroups * R) {
    int64_t s[R], e[R];
    Plain<float> acc[R];
    bool deep = R == 1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t row = base + grp + r * kGroups;
      const int64_t q = row < r1 ? row : r1 - 1;
      s[r] = bm_ptr(m, q);
      e[r] = bm_ptr(m, q + 1);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (base + grp + r * kGroups >= r1) e[r] = s[r];
      deep |= e[r] - s[r] > 8 * S;
      acc[r].init();
    }
    if (deep) {
#pragma unroll
      for (int r = 0; r < R; ++r) accumulate_span<S, 4>(acc[r], m.col, vs, m.x, s[r], e[r], g);
    } else if constexpr (R > 1) {
      bat_accumulate<R, S>(acc, m, s, e, g);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) group_reduce<S>(acc[r]);
    if (g == 0)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (base + grp + r * kGroups < r1)
          write_out(m.y, base + grp + r * kGroups, acc[r].value(), alpha, beta);
  }
}

// --- one long SpMV row with the whole block: lanes stride by 256, wave
// reduction, then the 4 wave totals summed in order through LDS.
__device__ void bat_spmv_long_row(const BatchMatrix& m, int64_t row, double alpha, double beta,
                                  float* lds) {
  DirectVals<float> vs{m.val};
  Comp acc;
  acc.init();
  const int64_t rs = bm_ptr(m, row), re = bm_ptr(m, row + 1);
  accumulate_span<kBatBlock, 4>(acc, m.col, vs, m.x, rs, re, threadIdx.x);
  group_reduce<kWave>(acc);
  const int w = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) { lds[2 * w] = acc.s; lds[2 * w + 1] = acc.c; }
  __syncthreads();
  if (threadIdx.x == 0) {
    Comp t;
    t.init();
    for (int i = 0; i < kBatBlock / kWave; ++i) {
      Comp o;
      o.s = lds[2 * i];
      o.c = lds[2 * i + 1];
      t.merge(o);
    }
    write_out(m.y, row, t.value(), alpha, beta);
  }
  __syncthreads();
}

// --- SpMM rows: the single-matrix short role (G lanes a row, VW columns a
// lane, entries loaded by the group through its LDS slots).  A row of its own
// that is longer than FS_BATCH_LONG_MM belongs to the whole block: its groups
// take equal ranges of the entries, and their sums are added in order,
// compensated.  One group would walk it alone while the rest of the launch is
// done: six power-law matrices of 30,000 rows (up to 20,000 entries), N = 3 / 8 /
// 40 / 260, by one group 2137 / 2137 / 3099 / 5276 us (by the former two lanes with
// eight entries in flight 1050 / 1567 / 1749 / 3016), here 102 / 119 / 272 / 1530.
constexpr int kBatMmU = 4;                // SpMM entries in flight per lane
constexpr int kBatSlots = kBatBlock * 2;  // at most two fills per lane (kMmFill)
union BatLds {
  struct {
    int32_t col[kBatSlots];
    float val[kBatSlots];
  } slot;
  float part[kBatBlock * 4];  // sums of a long row's groups
};

template <int G, int VW>
__device__ void bat_spmm_rows(const BatchMatrix& m, int64_t r0, int64_t r1, double alpha, double beta,
                              BatLds& lds) {
  constexpr int kGroups = kBatBlock / G, F = kMmFill<G>;
  static_assert(kBatBlock * F <= kBatSlots, "slots");
  const int grp = threadIdx.x / G, g = threadIdx.x % G;
  const int first = grp * (G * F);
  // uniform over the block
  const bool whole = r1 - r0 == 1 && bm_ptr(m, r1) - bm_ptr(m, r0) > FS_BATCH_LONG_MM;
  const int64_t tiles = (m.n_dense + G * VW - 1) / (G * VW);
  for (int64_t t = 0; t < tiles; ++t) {
    int64_t n0 = t * (G * VW) + (int64_t)g * VW;
    const bool colok = n0 < m.n_dense;
    const int skip = shift_tail<VW>(n0, m.n_dense);
    for (int64_t row = whole ? r0 : r0 + grp; row < r1; row += kGroups) {
      int64_t rs = bm_ptr(m, row), re = bm_ptr(m, row + 1);
      if (whole) {
        const int64_t per = (re - rs + kGroups - 1) / kGroups;
        rs = rs + grp * per < re ? rs + grp * per : re;
        re = rs + per < re ? rs + per : re;
      }
      Plain<float> acc[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) acc[k].init();
      mm_accumulate_group<VW, kBatMmU, G>(acc, lds.slot.col + first, lds.slot.val + first, m.col,
                                          m.val, m.B, m.ldb, n0, colok, rs, re, g);
      if (whole) {
        __syncthreads();  // the slots' memory is the sums'
#pragma unroll
        for (int k = 0; k < VW; ++k) lds.part[threadIdx.x * VW + k] = acc[k].value();
        __syncthreads();
        if (grp == 0 && colok) {
          Comp sum[VW];
#pragma unroll
          for (int k = 0; k < VW; ++k) sum[k].init();
#pragma unroll 1
          for (int i = 0; i < kGroups; ++i)
#pragma unroll
            for (int k = 0; k < VW; ++k) sum[k].add_value(lds.part[(i * G + g) * VW + k]);
          write_vec<G, VW>(m.C, row * m.ldc + n0, sum, alpha, beta, skip);
        }
        __syncthreads();  // the next tile's slots
      } else if (colok) {
        write_vec<G, VW>(m.C, row * m.ldc + n0, acc, alpha, beta, skip);
      }
    }
  }
}

__device__ void bat_spmv_dispatch(const BatchMatrix& m, int64_t r0, int64_t r1, double alpha, double beta) {
  switch (m.group_lanes) {
    case 1: bat_spmv_rows<1>(m, r0, r1, alpha, beta); break;
    case 2: bat_spmv_rows<2>(m, r0, r1, alpha, beta); break;
    case 4: bat_spmv_rows<4>(m, r0, r1, alpha, beta); break;
    case 8: bat_spmv_rows<8>(m, r0, r1, alpha, beta); break;
    case 16: bat_spmv_rows<16>(m, r0, r1, alpha, beta); break;
    case 32: bat_spmv_rows<32>(m, r0, r1, alpha, beta); break;
    default: bat_spmv_rows<64>(m, r0, r1, alpha, beta); break;
  }
}

// The (VW, G) pairs that spmm_tile_shape<4> gives.
__device__ void bat_spmm_dispatch(const BatchMatrix& m, int64_t r0, int64_t r1, double alpha,
                                  double beta, BatLds& lds) {
  if (m.mm_vw == 4) {
    switch (m.mm_lanes) {
      case 8: bat_spmm_rows<8, 4>(m, r0, r1, alpha, beta, lds); break;
      case 16: bat_spmm_rows<16, 4>(m, r0, r1, alpha, beta, lds); break;
      case 32: bat_spmm_rows<32, 4>(m, r0, r1, alpha, beta, lds); break;
      default: bat_spmm_rows<64, 4>(m, r0, r1, alpha, beta, lds); break;
    }
  } else if (m.mm_vw == 2) {
    if (m.mm_lanes <= 8) bat_spmm_rows<8, 2>(m, r0, r1, alpha, beta, lds);
    else bat_spmm_rows<16, 2>(m, r0, r1, alpha, beta, lds);
  } else {
    if (m.mm_lanes <= 4) bat_spmm_rows<4, 1>(m, r0, r1, alpha, beta, lds);
    else if (m.mm_lanes <= 8) bat_spmm_rows<8, 1>(m, r0, r1, alpha, beta, lds);
    else bat_spmm_rows<16, 1>(m, r0, r1, alpha, beta, lds);
  }
}

__global__ __launch_bounds__(kBatBlock) void batched_kernel(const BatchMatrix* __restrict__ mats,
                                                            const fs_batch_item* __restrict__ items,
                                                            int64_t long_row, double alpha,
                                                            double beta) {
  __shared__ BatLds lds;
  const fs_batch_item w = items[blockIdx.x];
  const BatchMatrix& m = mats[w.matrix];
  if (w.kind == FS_BATCH_SPMV) {
    if (w.row_end - w.row_begin == 1 && bm_ptr(m, w.row_begin + 1) - bm_ptr(m, w.row_begin) > long_row)
      bat_spmv_long_row(m, w.row_begin, alpha, beta, lds.part);
    else
      bat_spmv_dispatch(m, w.row_begin, w.row_end, alpha, beta);
  } else {
    bat_spmm_dispatch(m, w.row_begin, w.row_end, alpha, beta, lds);
  }
}

}  // namespace fs

using namespace fs;

extern "C" int64_t fs_batch_matrix_bytes(void) { return (int64_t)sizeof(BatchMatrix); }

extern "C" int fs_batch_pack(const fs_batch_entry* entries, int64_t n_entries, void* packed_host) {
  if (n_entries < 0 || (n_entries > 0 && (!entries || !packed_host)))
    return fail(FS_ERR_VALUE, "fs_batch_pack: bad arguments");
  BatchMatrix* out = static_cast<BatchMatrix*>(packed_host);
  for (int64_t i = 0; i < n_entries; ++i) {
    const fs_batch_entry& e = entries[i];
    const fs_csr& A = e.A;
    int rc = check_csr(&A, "fs_batch_pack");
    if (rc) return rc;
    if (A.value_type != FS_F32 || A.index_type != FS_I32)
      return fail(FS_ERR_TYPE, "fs_batch_pack: entry %lld must be fp32 with int32 columns", (long long)i);
    if (e.n_dense < 0 || (e.n_dense > 0 && (e.ldb < e.n_dense || e.ldc < e.n_dense)))
      return fail(FS_ERR_VALUE, "fs_batch_pack: entry %lld has bad dense shape", (long long)i);
    const int s = e.group_lanes;
    if (s != 1 && s != 2 && s != 4 && s != 8 && s != 16 && s != 32 && s != 64)
      return fail(FS_ERR_VALUE, "fs_batch_pack: entry %lld group_lanes must be a power of two <= 64", (long long)i);
    BatchMatrix m;
    m.row_ptr = A.row_ptr;
    m.col = static_cast<const int32_t*>(A.col_idx);
    m.val = static_cast<const float*>(A.values);
    m.x = static_cast<const float*>(e.x);
    m.y = static_cast<float*>(e.y);
    m.B = static_cast<const float*>(e.B);
    m.C = static_cast<float*>(e.C);
    m.n_rows = A.n_rows;
    m.n_cols = A.n_cols;
    m.nnz = A.nnz;
    m.n_dense = e.n_dense;
    m.ldb = e.ldb;
    m.ldc = e.ldc;
    m.group_lanes = s;
    m.ptr64 = A.ptr_type == FS_I64;
    int vw = 1, lanes = 1;
    if (e.n_dense > 0) spmm_tile_shape<4>(e.n_dense, 0, &vw, &lanes);
    m.mm_vw = vw;
    m.mm_lanes = lanes;
    out[i] = m;
  }
  return FS_OK;
}

extern "C" int fs_batch_rows(int32_t group_lanes, int64_t n_dense) {
  // SpMV: four rows per lane group (8 or 64 of 32 rows: 287 / 274 against 271 us
  // on the batch above), enough to pay for a block's start; SpMM: one (two: 413
  // against 382 us, the block waits for the longer of more rows)
  // (lanes that fs_batch_pack refuses get some positive count here)
  if (n_dense <= 0)
    return group_lanes > 0 && group_lanes <= kWave ? 4 * (kBatBlock / group_lanes) : kBatBlock;
  int vw = 1, lanes = 1;
  spmm_tile_shape<4>(n_dense, 0, &vw, &lanes);
  return kBatBlock / (lanes < 4 ? 4 : lanes);
}

extern "C" int fs_batch_run(const void* packed_dev, int64_t n_matrices, const fs_batch_item* items,
                            int64_t n_items, int64_t long_row, int32_t* queue, int32_t grid,
                            double alpha, double beta, void* stream) {
  if (n_items < 0 || n_matrices < 0) return fail(FS_ERR_VALUE, "fs_batch_run: negative counts");
  if (n_items == 0) return FS_OK;
  if (!packed_dev || !items || !queue) return fail(FS_ERR_VALUE, "fs_batch_run: null pointer");
  if (grid <= 0) return fail(FS_ERR_VALUE, "fs_batch_run: grid must be positive");
  if (long_row < 1) return fail(FS_ERR_VALUE, "fs_batch_run: long_row must be >= 1");
  if (n_items + (int64_t)grid > (int64_t)INT32_MAX)
    return fail(FS_ERR_UNSUPPORTED, "fs_batch_run: n_items + grid must stay below 2^31 - 1");
  // a launch holds fewer than 2^32 work-items: long lists go in several
  constexpr int64_t kMost = (int64_t)1 << 23;
  for (int64_t i = 0; i < n_items; i += kMost) {
    const int64_t n = n_items - i < kMost ? n_items - i : kMost;
    batched_kernel<<<(unsigned)n, kBatBlock, 0, as_stream(stream)>>>(
        static_cast<const BatchMatrix*>(packed_dev), items + i, long_row, alpha, beta);
    const int rc = check_launch("fs_batch_run");
    if (rc) return rc;
  }
  return FS_OK;
}
