// spmm_kernel.hpp -- SpMM row procedures shared by the single-matrix kernels and
// the batched one: a lane group's gathers of B rows, its entry loads through LDS
// slots, the stores of C, and the choice of lanes and columns per lane.
#ifndef FS_SPMM_KERNEL_HPP_
#define FS_SPMM_KERNEL_HPP_
#include <type_traits>

#include "fs_host.hpp"

namespace fs {

constexpr int kMmBlock = 256;
constexpr int kMmWaves = kMmBlock / kWave;

template <typename A> struct MmChunkAcc { using T = A; };
template <> struct MmChunkAcc<Plain<float>> { using T = Comp; };

// True xor exchange (lane ^ K): quad_perm for 1 and 2, ds_swizzle for 4..16,
// ds_bpermute for 32.  Used to combine lane groups at equal positions.
template <int K> __device__ __forceinline__ int xor_i32(int v) {
  if constexpr (K == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
  else if constexpr (K == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
  else if constexpr (K == 4 || K == 8 || K == 16) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (K << 10));
  else {
    static_assert(K == 32, "bad xor distance");
    return __builtin_amdgcn_ds_bpermute((__lane_id() ^ 32) << 2, v);
  }
}
template <int K> __device__ __forceinline__ float xor_x(float v) { return __int_as_float(xor_i32<K>(__float_as_int(v))); }
template <int K> __device__ __forceinline__ double xor_x(double v) {
  int64_t b = __double_as_longlong(v);
  int lo = xor_i32<K>((int)(b & 0xffffffff));
  int hi = xor_i32<K>((int)(b >> 32));
  return __longlong_as_double(((int64_t)(uint32_t)lo) | ((int64_t)hi << 32));
}
template <int K, typename T> __device__ __forceinline__ cplx<T> xor_x(cplx<T> v) { return {xor_x<K>(v.re), xor_x<K>(v.im)}; }
template <int K, typename T> __device__ __forceinline__ Plain<T> xor_x(const Plain<T>& a) { Plain<T> o; o.s = xor_x<K>(a.s); return o; }
template <int K> __device__ __forceinline__ Comp xor_x(const Comp& a) { Comp o; o.s = xor_x<K>(a.s); o.c = xor_x<K>(a.c); return o; }

// Sum accumulators over lane groups of width G inside a wavefront (positions
// kept): after this every lane holds the sum over the 64/G groups.
template <int G, typename A> __device__ __forceinline__ void cross_group_reduce(A& a) {
  if constexpr (G <= 1) { A o = xor_x<1>(a); a.merge(o); }
  if constexpr (G <= 2) { A o = xor_x<2>(a); a.merge(o); }
  if constexpr (G <= 4) { A o = xor_x<4>(a); a.merge(o); }
  if constexpr (G <= 8) { A o = xor_x<8>(a); a.merge(o); }
  if constexpr (G <= 16) { A o = xor_x<16>(a); a.merge(o); }
  if constexpr (G <= 32) { A o = xor_x<32>(a); a.merge(o); }
}

// VW consecutive stored values of type V as loaded: 32-bit words (one 16-bit
// value in the low half for a single 2-byte element).  The vector types carry
// only the element's own alignment, so a lane's segment may start at any
// element of B or C (odd leading dimensions, offset bases, the shifted tail
// window below); gfx950 serves a misaligned global dwordx4 in hardware and the
// compiler emits the same instruction as for an aligned one.
template <typename V, int VW> struct RawVec {
  static constexpr int kBytes = (int)sizeof(V) * VW;
  static constexpr int kWords = kBytes < 4 ? 1 : kBytes / 4;
  uint32_t w[kWords];
};
// alignment of a vector access: the stored element's scalar
template <typename V> constexpr int kElemAlign = alignof(V) < sizeof(V) ? (int)alignof(V) : (int)sizeof(V);

template <int W, int AL> struct WordVec;
template <> struct WordVec<1, 2> { typedef uint32_t type __attribute__((aligned(2))); };
template <> struct WordVec<2, 2> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(2))); };
template <> struct WordVec<4, 2> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(2))); };
template <> struct WordVec<1, 4> { typedef uint32_t type __attribute__((aligned(4))); };
template <> struct WordVec<2, 4> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct WordVec<4, 4> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct WordVec<2, 8> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct WordVec<4, 8> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(8))); };

template <typename V, int VW>
__device__ __forceinline__ void load_raw(RawVec<V, VW>& r, const V* __restrict__ p, int64_t off) {
  using R = RawVec<V, VW>;
  if constexpr (R::kBytes < 4) {
    r.w[0] = *reinterpret_cast<const uint16_t*>(p + off);
  } else {
    using T = typename WordVec<R::kWords, kElemAlign<V>>::type;
    const T v = *reinterpret_cast<const T*>(p + off);
    __builtin_memcpy(r.w, &v, R::kBytes);
  }
}

template <typename V, int VW, typename C>
__device__ __forceinline__ void unpack_raw(C (&out)[VW], const RawVec<V, VW>& r) {
  V v[VW];
  __builtin_memcpy(v, r.w, sizeof(V) * VW);
#pragma unroll
  for (int k = 0; k < VW; ++k) out[k] = load_as<C>(v, k);
}

// Load VW consecutive stored values starting at element `off` as compute type.
template <typename C, int VW, typename S>
__device__ __forceinline__ void load_vec(C (&out)[VW], const S* __restrict__ p, int64_t off) {
  RawVec<S, VW> r;
  load_raw(r, p, off);
  unpack_raw(out, r);
}

// B rows of a masked batch, raw: r[u] = B[col[u] * ldb + n0 .. + VW) for the u
// whose bit is set in `ok` (others zero).
template <int VW, int U, typename V>
__device__ __forceinline__ void gather_masked(RawVec<V, VW> (&r)[U], const V* __restrict__ B,
                                              int64_t ldb, const int64_t (&col)[U], int64_t n0,
                                              unsigned ok) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if ((ok >> u) & 1u) {
      load_raw(r[u], B, col[u] * ldb + n0);
    } else {
#pragma unroll
      for (int w = 0; w < RawVec<V, VW>::kWords; ++w) r[u].w[w] = 0u;
    }
  }
}

// Widening of a gathered row.  When the compute type differs from the stored
// one (fp32 B accumulated in fp64, 16-bit values, complex), the words stay
// opaque (empty asm) until every load of the batch is issued: a widening placed
// inside a masked load's branch brings a wait for that load with it and
// serialises the batch.
template <typename V, int VW, typename C>
__device__ __forceinline__ void widen_row(C (&b)[VW], RawVec<V, VW>& r) {
  if constexpr (!std::is_same<C, V>::value) {
#pragma unroll
    for (int w = 0; w < RawVec<V, VW>::kWords; ++w) asm volatile("" : "+v"(r.w[w]));
  }
  unpack_raw(b, r);
}

// The lane's column window: columns n0 .. n0 + VW - 1 of which the last
// VW - skip are its own.  A row's last lane shifts its window back so that it
// ends at the last column (n_dense >= VW always holds): every load stays
// inside the row with no scalar tail, and the columns it shares with the lane
// before are computed but not written.
template <int VW>
__device__ __forceinline__ int shift_tail(int64_t& n0, int64_t n_dense) {
  if constexpr (VW > 1) {
    if (n0 < n_dense && n0 + VW > n_dense) {
      const int skip = (int)(n0 + VW - n_dense);
      n0 = n_dense - VW;
      return skip;
    }
  }
  return 0;
}

// C[off + skip .. off + VW) = alpha * acc + beta * C (C read only when beta is
// nonzero): write_out's arithmetic.  One vector store where the window is
// whole and the values are 16-bit, or the row's lane group is at least 32
// lanes wide.  Measured on the 1M-row banded matrix in fp32: vector stores
// took N = 128 (32 lanes) from 798 to 776 us, but were ~2 us slower than VW
// scalar stores at N = 32 / 64 (8 / 16 lanes).
template <int G, int VW, typename V, typename A>
__device__ __forceinline__ void write_vec(V* __restrict__ C, int64_t off, const A (&acc)[VW],
                                          double alpha, double beta, int skip) {
  using T = std::decay_t<decltype(acc[0].value())>;
  constexpr bool kVec = VW > 1 && (G >= 32 || sizeof(V) == 2);
  if constexpr (kVec) {
    if (skip == 0) {
      T v[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) v[k] = alpha == 1.0 ? acc[k].value() : scale(acc[k].value(), alpha);
      if (beta != 0.0) {
        T old[VW];
        load_vec<T, VW>(old, C, off);
#pragma unroll
        for (int k = 0; k < VW; ++k) v[k] = add(v[k], scale(old[k], beta));
      }
      V o[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) store_from(o, k, v[k]);
      using W = typename WordVec<RawVec<V, VW>::kWords, kElemAlign<V>>::type;
      W w;
      __builtin_memcpy(&w, o, sizeof(V) * VW);
      *reinterpret_cast<W*>(C + off) = w;
      return;
    }
  }
#pragma unroll
  for (int k = 0; k < VW; ++k)
    if (k >= skip) write_out(C, off + k, acc[k].value(), alpha, beta);
}

// One entry's products into the lane's columns.  Compensated sums take two
// columns at a time: their ten steps interleaved over a batch's entries and
// columns cost registers and with them wavefronts of all rows of the kernel
// (fp32, four columns a lane, eight entries in flight: 98, 82 so; bf16, eight
// columns: 120, 69 so).
template <typename A, typename C, int VW>
__device__ __forceinline__ void mm_products(A (&acc)[VW], C a, const C (&b)[VW]) {
#pragma unroll
  for (int k = 0; k < VW; ++k) {
    acc[k].add_prod(a, b[k]);
    if (std::is_same<A, Comp>::value && (k % 2 == 1 || k == VW - 1))
      __builtin_amdgcn_sched_barrier(0);
  }
}

// Accumulate entries j = s + first, s + first + step, ... < e into acc[VW] for
// the lane's columns n0 .. n0+VW-1.
template <int VW, int U, typename A, typename V, typename I>
__device__ __forceinline__ void mm_accumulate(A (&acc)[VW], const I* __restrict__ idx,
                                              const V* __restrict__ val,
                                              const V* __restrict__ B, int64_t ldb,
                                              int64_t n0, int64_t s, int64_t e, int64_t step) {
  using C = typename A::compute_t;
  int64_t j = s;
  for (; j + (int64_t)(U - 1) * step < e; j += (int64_t)U * step) {
    int64_t col[U];
    C a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      col[u] = ldg_index(idx, j + u * step);
      a[u] = load_as<C>(val, j + u * step);
    }
    RawVec<V, VW> r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load_raw(r[u], B, col[u] * ldb + n0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      C b[VW];
      unpack_raw(b, r[u]);
      mm_products(acc, a[u], b);
    }
  }
  if (j < e) {
    // the last, partial batch: all its loads in flight at once, entries past
    // e masked (their products are not added)
    I ci[U];
    C a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool ok = j + u * step < e;
      ci[u] = ok ? idx[j + u * step] : I(0);
      a[u] = ok ? load_as<C>(val, j + u * step) : zero<C>();
    }
    // the empty asm keeps each index's widening (and the wait for its load)
    // out of the masked load's branch, so the batch's loads are all issued
    // before the first wait
    int64_t col[U];
    unsigned ok = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      asm volatile("" : "+v"(ci[u]));
      col[u] = (int64_t)ci[u];
      ok |= (unsigned)(j + u * step < e) << u;
    }
    RawVec<V, VW> r[U];
    gather_masked(r, B, ldb, col, n0, ok);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      C b[VW];
      widen_row(b, r[u]);
      if (j + u * step < e) mm_products(acc, a[u], b);
    }
  }
}

// A short row's entries, loaded G at a time by the G lanes of its group (lane
// g loads entry j0 + g: one coalesced col / value load per G entries instead
// of one broadcast load per entry, which cuts the L2 requests of the entry
// stream), parked in the group's LDS slots and read back U at a time.  Lanes
// past the last dense column (colok false) still load their share.  The
// products are added in entry order, as in mm_accumulate.
// F fills per round: each lane loads F entries (F * G slots per group), so a
// row of up to F * G entries needs one fill round trip instead of F.  The next
// round's entries are loaded before this round's gathers, and the slots are
// ordered by LDS-only fences, which do not wait for them: fp64 N = 8, 200,000
// rows of 24 80.7 -> 73.8 us; bf16 N = 32, 100,000 rows of 34 40.3 -> 37.2 us;
// rows of one round (1M-row band of 15) unchanged.
template <int G> constexpr int kMmFill = G <= 8 ? 2 : 1;

template <int VW, int U, int G, typename A, typename V>
__device__ __forceinline__ void mm_accumulate_group(A (&acc)[VW], int32_t* slot_col,
                                                    typename A::compute_t* slot_val,
                                                    const int32_t* __restrict__ idx,
                                                    const V* __restrict__ val,
                                                    const V* __restrict__ B, int64_t ldb,
                                                    int64_t n0, bool colok, int64_t s,
                                                    int64_t e, int g) {
  using C = typename A::compute_t;
  constexpr int F = kMmFill<G>;
  static_assert(G % U == 0, "batches of U entries tile the group's G slots");
  // lane g's share of the fill from j0 on, unconditional (past e: the fill's
  // first entry again), so that the loads of a lane are in flight together;
  // the next fill is loaded before the gathers of this one, so its latency
  // (the entries stream from memory) passes behind theirs
  int32_t fc[F];
  V fv[F];
  auto fetch = [&](int64_t j0) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int64_t jj = j0 + f * G + g;
      const int64_t q = jj < e ? jj : j0;
      fc[f] = idx[q];
      fv[f] = val[q];
    }
  };
  if (s < e) fetch(s);
  for (int64_t j0 = s; j0 < e; j0 += G * F) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      slot_col[f * G + g] = fc[f];
      slot_val[f * G + g] = load_as<C>(fv, f);
    }
    if (j0 + G * F < e) fetch(j0 + G * F);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    const int cnt = e - j0 < G * F ? (int)(e - j0) : G * F;
    if (colok) {
      for (int u0 = 0; u0 < cnt; u0 += U) {
        int64_t col[U];
        C a[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          // LDS reads are unconditional (a slot past cnt re-reads slot u0):
          // under a per-lane branch each would be waited for in turn
          const int uu = u0 + u < cnt ? u0 + u : u0;
          col[u] = (int64_t)slot_col[uu];
          a[u] = slot_val[uu];
        }
        unsigned ok = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) ok |= (unsigned)(u0 + u < cnt) << u;
        RawVec<V, VW> r[U];
        gather_masked(r, B, ldb, col, n0, ok);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          C b[VW];
          widen_row(b, r[u]);
          if (u0 + u < cnt)
#pragma unroll
            for (int k = 0; k < VW; ++k) acc[k].add_prod(a[u], b[k]);
        }
      }
    }
    // the slots are rewritten by the next batch
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
}

static inline int pow2_at_least(int64_t v) {
  int g = 1;
  while (g < v && g < 64) g <<= 1;
  return g;
}

// Columns per lane and lanes per row for n_dense columns in tiles of col_tile
// (0: all).  The lane segment is the widest up to 16 bytes that leaves at
// least eight lanes to a row, so that a row's entries are loaded a whole
// batch at a time by its group; neither the alignment of B and C nor the
// divisibility of n_dense narrows it (load_raw, shift_tail).
template <int MAXV>
static inline void spmm_tile_shape(int64_t n_dense, int64_t col_tile, int* vw, int* lanes) {
  // a column tile wider than B would leave the lanes past n_dense idle
  const int64_t tile = col_tile > 0 && col_tile < n_dense ? col_tile : n_dense;
  int v = MAXV;
  while (v > 1 && tile / v < 8) v >>= 1;
  *vw = v;
  *lanes = pow2_at_least((tile + v - 1) / v);
}

}  // namespace fs

#endif
