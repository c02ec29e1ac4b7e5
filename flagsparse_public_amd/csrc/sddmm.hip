// sddmm.hip -- CSR SDDMM for gfx950: out[p] = alpha * <x[row(p)], y[col(p)]> +
// beta * data[p] over the entries p of a CSR pattern (entry point
// fs_sddmm_csr).
//
// Replaces the reference's Triton kernel (sddmm_csr.py:108-151: a program per
// 128 entries, K in BLOCK_K steps, tl.sum reduction).  A row of x or y is cut
// into parts of 16 bytes, loaded at any alignment; a group of at most 8 lanes
// takes two entries, lane g parts g, g + 8, ..., and the group reduces with DPP /
// swizzle exchanges.  fp32 without data keeps a lane for every part up to 32
// parts: 16 lanes take four entries, 32 lanes eight (sddmm_launch).
//
// Why so few lanes: with a lane for every part (up to 64) the exchanges and the
// address work of an entry, spread over many lanes with little to do, bound the
// kernel; with 8 the 128-byte lines of the y rows do (about 7 TB/s) once y exceeds
// L2.  3M entries of a banded pattern, where the lines stay in L2, fp32 K = 160 299
// -> 197 us, fp64 K = 40 / 64 / 100: 171 -> 117 / 193 -> 157 / 393 -> 278 us; 1.6M
// random entries, K = 160 in fp32 157 -> 151, in fp64 359 -> 298 us.  Adding beta *
// data: banded fp32 K = 64 / 128 101 -> 85 / 200 -> 157 us.
// Widths that 16 bytes do not divide took element loads: fp32 K = 33 / 97, random
// 92 -> 47 / 122 -> 108 us, banded 172 -> 68 / 229 -> 156 us; fp64 K = 47 158 ->
// 106 us.  16 lanes above 32 parts: 3-5% faster on random patterns, up to 18%
// slower on banded ones; a lane for every part there: 5-7% faster on 600,000
// random entries (fp32 K = 200 / 512: 74 / 171 us against 78 / 182).
#include "fs_host.hpp"

namespace fs {

constexpr int kSdBlock = 256;

// VW consecutive elements of a row, at any address: one 16-byte load.
template <typename T, int VW> struct SdVec {
  typedef T type __attribute__((ext_vector_type(VW), aligned(sizeof(T))));
};
template <typename T> struct SdVec<T, 1> { typedef T type; };
template <int VW, typename V> __device__ __forceinline__ auto sd_elem(const V& v, int i) {
  if constexpr (VW == 1) return v;
  else return v[i];
}

// A group takes E entries, kSdBlock / G apart, so that consecutive groups read
// consecutive row ids / columns; their loads are in flight together.
//
// A lane takes the parts that NS lanes would take if there was one for every
// part (up to 64): the sums of parts that would lie in different lanes stay
// apart until the end and are added pairwise, so no sum has a longer chain of
// additions than with that many lanes, and its error is the same (fp32 sums,
// K = 64 / 160, relative to fp64: 6.80e-8 / 7.60e-8 with the lanes, 6.78e-8 /
// 7.51e-8 here).  Sums in fp64 over fp32 values need no such care and keep one.
// TAIL: the last part of a row is not whole; it is loaded VW elements from the
// row's end, and those that the part before it holds are left out.
template <typename A, typename T, typename O, int G, int VW, int NS, int E, bool TAIL>
__global__ __launch_bounds__(kSdBlock) void sddmm_kernel(
    const int32_t* __restrict__ row_ids, const int32_t* __restrict__ cols,
    const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ data,
    O* __restrict__ out, int64_t nnz, int64_t k_dim, double alpha, double beta) {
  using C = typename A::compute_t;
  using V = typename SdVec<T, VW>::type;
  constexpr int kGroups = kSdBlock / G;
  constexpr int kSums = sizeof(C) > sizeof(T) ? 1 : NS;
  // parts in flight per lane and entry (fp32 K = 160, banded: 203 us with one,
  // 200 with two, 247 with four, whose registers leave fewer wavefronts)
  constexpr int kB = NS < 2 ? NS : 2;
  const int64_t p0 = (int64_t)blockIdx.x * kGroups * E + threadIdx.x / G;
  const int g = threadIdx.x % G;
  const T* xr[E];
  const T* yr[E];
  bool live[E];  // the whole group agrees
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t p = p0 + (int64_t)e * kGroups;
    live[e] = p < nnz;
    // past nnz: the last entry again (nnz >= 1), computed and not written,
    // so that no load sits under a per-lane branch
    const int64_t q = live[e] ? p : nnz - 1;
    xr[e] = x + (int64_t)row_ids[q] * k_dim;
    yr[e] = y + (int64_t)cols[q] * k_dim;
  }
  C d[E];  // loaded ahead of the rows, not behind the sums
#pragma unroll
  for (int e = 0; e < E; ++e)
    d[e] = data && live[e] ? (C)data[p0 + (int64_t)e * kGroups] * (C)beta : (C)0;
  A acc[E][kSums];
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < kSums; ++i) acc[e][i].init();
  if constexpr (NS == 1 && !TAIL && G <= 16) {
    // a lane for every part: the parts' loads sit under the lane's own bound,
    // which takes 40 instead of 72 registers in the 16-lane kernel with four
    // entries (K = 40 / 64, 600,000 random entries: 17.6 -> 16.4 / 20.9 -> 19.9
    // us); 32 lanes with eight entries are faster below (K = 80 / 96: 29.7 / 31.3
    // against 32.4 / 33.5)
    for (int64_t k = (int64_t)g * VW; k < k_dim; k += (int64_t)G * VW)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const V a = *reinterpret_cast<const V*>(xr[e] + k);
        const V b = *reinterpret_cast<const V*>(yr[e] + k);
#pragma unroll
        for (int i = 0; i < VW; ++i)
          acc[e][0].add_prod((C)sd_elem<VW>(a, i), (C)sd_elem<VW>(b, i));
      }
  } else {
    for (int64_t k0 = 0; k0 < k_dim; k0 += (int64_t)G * VW * NS)
#pragma unroll
      for (int s0 = 0; s0 < NS; s0 += kB) {
        if (k0 + (int64_t)s0 * G * VW >= k_dim) break;  // uniform
        V a[kB][E], b[kB][E];
        bool ok[kB];
        int skip[kB];
#pragma unroll
        for (int s = 0; s < kB; ++s) {
          const int64_t k = k0 + (int64_t)((s0 + s) * G + g) * VW;
          ok[s] = k < k_dim;
          skip[s] = TAIL && ok[s] && k + VW > k_dim ? (int)(k + VW - k_dim) : 0;
          const int64_t at = ok[s] ? k - skip[s] : 0;
#pragma unroll
          for (int e = 0; e < E; ++e) {
            a[s][e] = *reinterpret_cast<const V*>(xr[e] + at);
            b[s][e] = *reinterpret_cast<const V*>(yr[e] + at);
          }
        }
#pragma unroll
        for (int s = 0; s < kB; ++s) {
          const int sum = kSums == 1 ? 0 : s0 + s;
          if (ok[s] && !(TAIL && skip[s])) {
#pragma unroll
            for (int e = 0; e < E; ++e)
#pragma unroll
              for (int i = 0; i < VW; ++i)
                acc[e][sum].add_prod((C)sd_elem<VW>(a[s][e], i), (C)sd_elem<VW>(b[s][e], i));
          } else if (TAIL && skip[s]) {
#pragma unroll
            for (int i = 1; i < VW; ++i)
              if (i >= skip[s])
#pragma unroll
                for (int e = 0; e < E; ++e)
                  acc[e][sum].add_prod((C)sd_elem<VW>(a[s][e], i), (C)sd_elem<VW>(b[s][e], i));
          }
        }
      }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
#pragma unroll
    for (int h = kSums / 2; h > 0; h /= 2)
#pragma unroll
      for (int i = 0; i < h; ++i) acc[e][i].merge(acc[e][i + h]);
    group_reduce<G>(acc[e][0]);
    if (live[e] && g == 0) {
      const int64_t p = p0 + (int64_t)e * kGroups;
      C v = acc[e][0].value() * (C)alpha;
      if (data) v += d[e];
      out[p] = (O)v;
    }
  }
}

template <typename A, typename T, typename O, int G, int VW, int NS, int E = 2>
void sddmm_launch_g(const int32_t* rid, const int32_t* cols, const T* x, const T* y,
                    const T* data, O* out, int64_t nnz, int64_t k, double alpha, double beta,
                    hipStream_t st) {
  const int64_t per_block = (int64_t)(kSdBlock / G) * E;
  const int64_t blocks = (nnz + per_block - 1) / per_block;
  const dim3 grid((unsigned)blocks), block(kSdBlock);
  if constexpr (VW > 1) {
    if (k % VW != 0) {
      sddmm_kernel<A, T, O, G, VW, NS, E, true><<<grid, block, 0, st>>>(rid, cols, x, y, data, out, nnz, k, alpha, beta);
      return;
    }
  }
  sddmm_kernel<A, T, O, G, VW, NS, E, false><<<grid, block, 0, st>>>(rid, cols, x, y, data, out, nnz, k, alpha, beta);
}

template <typename A, typename T, typename O>
int sddmm_launch(const fs_csr* P, const int32_t* rid, const void* x, const void* y, int64_t k,
                 void* out, double alpha, double beta, hipStream_t st) {
  const int32_t* cols = static_cast<const int32_t*>(P->col_idx);
  const T* xs = static_cast<const T*>(x);
  const T* ys = static_cast<const T*>(y);
  const T* data = static_cast<const T*>(P->values);
  O* o = static_cast<O*>(out);
  constexpr int kVec = sizeof(T) == 4 ? 4 : 2;
  const int64_t nnz = P->nnz, per = (k + kVec - 1) / kVec;
  if (k < kVec) {  // no whole vector in a row
    if (k <= 1) sddmm_launch_g<A, T, O, 1, 1, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
    else if (k == 2) sddmm_launch_g<A, T, O, 2, 1, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
    else sddmm_launch_g<A, T, O, 4, 1, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
    return check_launch("fs_sddmm_csr");
  }
  int lanes = 1;  // the power of two that covers the row's parts, at most 64
  while (lanes < per && lanes < 64) lanes <<= 1;
  switch (lanes) {
    case 1: sddmm_launch_g<A, T, O, 1, kVec, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st); break;
    case 2: sddmm_launch_g<A, T, O, 2, kVec, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st); break;
    case 4: sddmm_launch_g<A, T, O, 4, kVec, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st); break;
    case 8: sddmm_launch_g<A, T, O, 8, kVec, 1>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st); break;
    // fp32 without data keeps a lane for every part and more entries in flight.
    // K = 128, 2M random entries of 400,000 rows 164 us against 177, 1.6M of
    // 100,000 113 against 115; with data 181 against 177, banded 193 against 157.
    // K = 64: 84.9 against 87.6, 56.0 against 55.4, banded 82 against 80 us.
    case 16:
      if (kVec == 4 && !data && k % kVec == 0)
        sddmm_launch_g<A, T, O, 16, kVec, 1, 4>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
      else
        sddmm_launch_g<A, T, O, 8, kVec, 2>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
      break;
    case 32:
      if (kVec == 4 && !data)
        sddmm_launch_g<A, T, O, 32, kVec, 1, 8>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
      else
        sddmm_launch_g<A, T, O, 8, kVec, 4>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st);
      break;
    default: sddmm_launch_g<A, T, O, 8, kVec, 8>(rid, cols, xs, ys, data, o, nnz, k, alpha, beta, st); break;
  }
  return check_launch("fs_sddmm_csr");
}

}  // namespace fs

using namespace fs;

extern "C" int fs_sddmm_csr(const fs_csr* P, const int32_t* row_ids, const void* x,
                            const void* y, int64_t k_dim, void* out, int32_t out_type,
                            int32_t accumulate, double alpha, double beta, void* stream) {
  if (!P) return fail(FS_ERR_VALUE, "fs_sddmm_csr: pattern descriptor is null");
  if (P->value_type != FS_F32 && P->value_type != FS_F64)
    return fail(FS_ERR_TYPE, "fs_sddmm_csr: x / y must be fp32 or fp64");
  if (P->index_type != FS_I32)
    return fail(FS_ERR_TYPE, "fs_sddmm_csr: column indices must be int32");
  if (P->nnz < 0 || P->n_rows < 0 || P->n_cols < 0 || k_dim < 0)
    return fail(FS_ERR_VALUE, "fs_sddmm_csr: negative size");
  if (out_type != P->value_type && out_type != FS_F64)
    return fail(FS_ERR_TYPE, "fs_sddmm_csr: out must be the value type or fp64");
  if (accumulate != FS_ACC_NATIVE && accumulate != FS_ACC_WIDE)
    return fail(FS_ERR_VALUE, "fs_sddmm_csr: accumulate must be FS_ACC_NATIVE or FS_ACC_WIDE");
  if (P->nnz == 0) return FS_OK;
  if (!row_ids || !P->col_idx || !out || (k_dim > 0 && (!x || !y)))
    return fail(FS_ERR_VALUE, "fs_sddmm_csr: null pointer");
  hipStream_t st = as_stream(stream);
  const bool wide = accumulate == FS_ACC_WIDE;
  if (P->value_type == FS_F64)
    return out_type == FS_F64
               ? sddmm_launch<Plain<double>, double, double>(P, row_ids, x, y, k_dim, out, alpha, beta, st)
               : fail(FS_ERR_TYPE, "fs_sddmm_csr: bad out type");
  if (out_type == FS_F64)
    return wide ? sddmm_launch<Plain<double>, float, double>(P, row_ids, x, y, k_dim, out, alpha, beta, st)
                : sddmm_launch<Plain<float>, float, double>(P, row_ids, x, y, k_dim, out, alpha, beta, st);
  return wide ? sddmm_launch<Plain<double>, float, float>(P, row_ids, x, y, k_dim, out, alpha, beta, st)
              : sddmm_launch<Plain<float>, float, float>(P, row_ids, x, y, k_dim, out, alpha, beta, st);
}
