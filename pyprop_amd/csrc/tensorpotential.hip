// Tensor-potential multiply on MI355X.
//
// Semantics follow the generated Fortran kernels of
// core/tensorpotential/tensorpotentialmultiply_generator.py:
//   dest(row_0..row_R-1) += [conj] V(i_0..i_R-1) * scaling * source(col_0..col_R-1)
// summed over each rank's (row, col, i) enumeration (Simp 302-363, Herm 370-398,
// Diag 403-432, Ident 436-462, Band 467-618, BandNH 622-762, Dense 1227-1330).
//
// Design.  The outer ranks (all but the innermost) only enumerate index tuples; the
// plan lists them on the host once, in the reference loop order, grouped by destination
// fibre (a fibre is the innermost-rank vector at fixed outer indices).  One workgroup
// owns one destination fibre, so no atomics are needed and the summation order is fixed
// (deterministic).  Its four waves split the fibre's tuple list in four contiguous parts
// whose partial sums are added in order at the end.  Workgroups are launched in order of
// decreasing tuple count (longest first) to balance the tail, those of compact plans in
// an order by XCD (xcd_order).
//
// Innermost rank:
//  * banded storages (BandNH = zgbmv, Band = zhbmv) are re-laid out once into
//    diagonal-major form D[fibre][d][i] = A(i, i + d - hb): lane i streams row i with
//    fully coalesced loads (consecutive lanes read consecutive addresses), the source
//    window is staged in LDS per wave.  If every imaginary part is zero the diagonals are
//    stored as float64 (8 B/element instead of 16).  Streamed in this form the path is
//    HBM-bound.
//    Real potentials are then stored once where they repeat (compact_term): a term whose bands
//    are all symmetric keeps the diagonals d >= hb only, row i of a lower diagonal being read at
//    row i - (hb - d) of its mirror image; fibres that are equal bit for bit are kept once.
//    Potentials of this kind repeat a lot: (i1, j1) and (j1, i1) give the same band, and so do
//    most angular pairs (c, c') and (c', c).  What differs in its last bit is kept apart: helium
//    (42 channels x 60 x 60, 2.65 GB) keeps 0.49 GB when generated from the grid, 1.09 GB when
//    expanded from the host's radial factors, whose 1/r12 bands are not symmetric to the bit.
//    Where mirror images are read the sums and their order do not change.  Where they are not
//    (all terms symmetric, n <= 64), a lower diagonal's product is v (s x) instead of s (v x) and
//    is added to its row at the end: other roundings, of the same number of operations.
//  * all other storages go through a generic per-row entry list (CSR) over the
//    reference layout; correct for every storage, not tuned.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstring>
#include <new>
#include <numeric>
#include <type_traits>
#include <utility>
#include <vector>

#include "pp_common.h"
#include "pp_internal.h"

namespace pp {

// ----------------------------------------------------------------------------------
// host: per-rank enumerations in reference loop order
// ----------------------------------------------------------------------------------
struct RankEntry {
  int row, col, pidx, toggle;
};

static std::vector<RankEntry> enumerate_rank(int id, int potExt, int srcExt, const int32_t* pairs,
                                             int pairCount) {
  std::vector<RankEntry> e;
  switch (id) {
    case PP_STORAGE_SIMP:
      PP_REQUIRE(pairs && pairCount == potExt, "Simp rank needs pairs with count == potential extent");
      for (int i = 0; i < potExt; ++i) e.push_back({pairs[2 * i], pairs[2 * i + 1], i, 0});
      break;
    case PP_STORAGE_HERM:
      PP_REQUIRE(pairs && pairCount == potExt, "Herm rank needs pairs with count == potential extent");
      for (int i = 0; i < potExt; ++i) {
        e.push_back({pairs[2 * i], pairs[2 * i + 1], i, 0});
        e.push_back({pairs[2 * i + 1], pairs[2 * i], i, 1});
      }
      break;
    case PP_STORAGE_DIAG:
      for (int i = 0; i < potExt; ++i) e.push_back({i, i, i, 0});
      break;
    case PP_STORAGE_IDENT:
      for (int r = 0; r < srcExt; ++r) e.push_back({r, r, 0, 0});
      break;
    case PP_STORAGE_DENSE:
      for (int r = 0; r < srcExt; ++r)
        for (int c = 0; c < srcExt; ++c) e.push_back({r, c, r * srcExt + c, 0});
      break;
    case PP_STORAGE_BAND: {
      PP_REQUIRE(srcExt > 0 && potExt % srcExt == 0, "Band potential extent must be a multiple of N");
      int band = potExt / srcExt;
      for (int r = 0; r < srcExt; ++r)
        for (int c = r; c < std::min(r + band, srcExt); ++c) e.push_back({r, c, r * band + c - r, 0});
      for (int hr = 0; hr < srcExt; ++hr)
        for (int hc = hr + 1; hc < std::min(hr + band, srcExt); ++hc)
          e.push_back({hc, hr, hr * band + hc - hr, 1});
      break;
    }
    case PP_STORAGE_BANDNH: {
      PP_REQUIRE(srcExt > 0 && potExt % srcExt == 0, "BandNH potential extent must be a multiple of N");
      int bw = potExt / srcExt;
      PP_REQUIRE(bw % 2 == 1, "BandNH band count must be odd");
      int b = (bw - 1) / 2;
      for (int c = 0; c < srcExt; ++c)
        for (int r = std::max(0, c - b); r <= std::min(srcExt - 1, c + b); ++r)
          e.push_back({r, c, c * bw + b + r - c, 0});
      break;
    }
    default:
      throw Error(PP_ERR_INVALID, "unknown storage id " + std::to_string(id));
  }
  for (auto& x : e) {
    PP_REQUIRE(x.row >= 0 && x.row < srcExt && x.col >= 0 && x.col < srcExt,
               "pair index out of range for rank extent");
    PP_REQUIRE(x.pidx >= 0 && x.pidx < potExt, "potential index out of range");
  }
  return e;
}

// ----------------------------------------------------------------------------------
// device kernels
// ----------------------------------------------------------------------------------
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T>
__device__ inline T cz();
template <>
__device__ inline double2 cz<double2>() { return make_double2(0.0, 0.0); }
template <>
__device__ inline float2 cz<float2>() { return make_float2(0.f, 0.f); }

// acc += (conj?) v * x for real or complex v
template <class S, class C>
__device__ inline void acc_vx(C& acc, S v, C x, bool) {
  acc.x = fma(v, x.x, acc.x);
  acc.y = fma(v, x.y, acc.y);
}
template <class C>
__device__ inline void acc_vx(C& acc, C v, C x, bool cj) {
  const auto vy = cj ? -v.y : v.y;
  acc.x = fma(v.x, x.x, acc.x);
  acc.x = fma(-vy, x.y, acc.x);
  acc.y = fma(v.x, x.y, acc.y);
  acc.y = fma(vy, x.x, acc.y);
}

template <class C>
__device__ inline void acc_scaled(C& acc, C s, C p) {
  acc.x = fma(s.x, p.x, acc.x);
  acc.x = fma(-s.y, p.y, acc.x);
  acc.y = fma(s.x, p.y, acc.y);
  acc.y = fma(s.y, p.x, acc.y);
}

// One value of a band through a buffer descriptor: byte offset lane_off per lane (kPastBand: masked,
// reads zero) plus a uniform one.  KEEP: the value is read again soon; otherwise the diagonals are
// read exactly once per product and streamed past the caches (non-temporal, bit 1 of the cache policy).
typedef unsigned pp_u2v __attribute__((ext_vector_type(2)));
typedef unsigned pp_u4v __attribute__((ext_vector_type(4)));
enum { kStreamed = 0, kMixed = 1, kSymmetric = 2 };  // how a plan's terms are stored
constexpr int kPastBand = 0x40000000;  // fibres are far smaller
template <class V, bool KEEP>
__device__ __forceinline__ V ld_band(__amdgpu_buffer_rsrc_t band, int lane_off, int off) {
  constexpr int policy = KEEP ? 0 : 2;
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(band, lane_off, off, policy));
  } else if constexpr (sizeof(V) == 8) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(band, lane_off, off, policy));
  } else {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(band, lane_off, off, policy));
  }
}

template <class C>
struct DiaArgs {
  const int4* tuples;   // {src fibre, stored potential fibre, (term << 1) | conj, 0}
  unsigned sym;         // bit t: term t keeps the diagonals d >= hb only
  const int* fib_ptr;   // per destination fibre, tuple range
  const int* fib_order; // launch order
  const void* dia[kMaxTerms];
  C scale[kMaxTerms];
  int n;                // innermost extent
  const C* src;
  C* dst;
  const C* addend;      // optional
  C alpha;
  int accumulate;       // dst_out = (accumulate ? dst_in : 0) + addend + alpha * sum
};

template <class F, int... R>
__device__ __forceinline__ void for_rows_of(F&& f, std::integer_sequence<int, R...>) {
  (f(std::integral_constant<int, R>{}), ...);
}
// f(0), ..., f(NR - 1) with compile-time arguments
template <int NR, class F>
__device__ __forceinline__ void for_rows(F&& f) {
  for_rows_of(f, std::make_integer_sequence<int, NR>{});
}

// COMPACT: kMixed, some term is stored compactly; kSymmetric, all are and keep half the diagonals (the
// offsets then are the same for every tuple).  Their values are read again soon (as a mirror image, or by
// another fibre), so they are left in the caches instead of streamed past them.  Helium's full H in
// FP64: 428 us streaming every fibre (HBM); 172 us, in which the 0.49 GB stored come into the XCDs' L2s 2.5
// times each, 1.24 GB at 7.2 TB/s, while the L1s' 8-byte loads (16 clocks of a CU each) take half the
// clocks; 251 with the mirror images read as well.
template <class V, class C, int BW, int NR, int COMPACT>
__global__ __launch_bounds__(256) void tp_dia_kernel(DiaArgs<C> a) {
  constexpr int HB = (BW - 1) / 2;
  constexpr int WIN = NR * 64 + BW;
  __shared__ C xs[4][WIN];  // per-wave source window; reused for the final reduction
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int fib = a.fib_order[blockIdx.x];
  if (fib < 0) return;
  const int t0 = a.fib_ptr[fib];
  const int cnt = a.fib_ptr[fib + 1] - t0;
  const int w0 = t0 + (int)(((long long)cnt * wave) >> 2);
  const int w1 = t0 + (int)(((long long)cnt * (wave + 1)) >> 2);
  const int n = a.n;
  C* xw = xs[wave];
  for (int j = lane; j < WIN; j += 64) xw[j] = cz<C>();
  C acc[NR];
  for_rows<NR>([&](auto r) { acc[r] = cz<C>(); });
  // One row per lane and symmetric bands throughout: element (i, i + k) is used where it is read, for
  // row i with x_{i+k} and for row i + k with lane i's own x_i.  The shift by k is the same for all
  // tuples, so those products gather in an accumulator per k and move to their rows once, at the end:
  // no mirror image is read, and half of the windows' LDS reads go.
  constexpr bool SCATTER = COMPACT == kSymmetric && NR == 1;
  constexpr int NK = SCATTER ? HB : 0;
  C below[NK + 1];  // below[k]: to be added to row i + k
#pragma unroll
  for (int k = 0; k <= NK; ++k) below[k] = cz<C>();
  wave_sync();
  // Lane t holds term t's potential and scale, and lane l the l-th of the next 64 tuples: reading them
  // from memory one by one (scalar loads, whose waits are those of LDS too) stalled every tuple.
  const int tl = min(lane, kMaxTerms - 1);
  const unsigned long long dia_l = reinterpret_cast<unsigned long long>(a.dia[tl]);
  const C scale_l = a.scale[tl];
  int4 tup_l = make_int4(0, 0, 0, 0);
  auto from_lane = [](int v, int l) { return __builtin_amdgcn_readlane(v, l); };
  auto tuple = [&](int l) {
    return make_int4(from_lane(tup_l.x, l), from_lane(tup_l.y, l), from_lane(tup_l.z, l), 0);
  };
  // Source values of a tuple, and the bands of its row r per lane (lanes past the fibre repeat its last
  // row).  Several rows through a descriptor and by components: an array of whole values copied from memory
  // and on to LDS was kept in scratch memory, 23 us instead of 7 for 8 x 40 x 96 with 3 diagonals.  One row
  // plainly (13 x 30 x 30: 13.1 us, 13.6 through a descriptor).
  typedef decltype(C::x) Pair __attribute__((ext_vector_type(2)));
  auto load_x = [&](const int4& tp, C (&x)[NR]) {
    const C* xp = a.src + (long long)tp.x * n;
    if constexpr (NR == 1) {
      x[0] = xp[min(lane, n - 1)];
    } else {
      const __amdgpu_buffer_rsrc_t fibre =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<C*>(xp), (short)0, n * (int)sizeof(C), 0x00020000);
      for_rows<NR>([&](auto r) {
        const Pair v = ld_band<Pair, true>(fibre, min(lane + 64 * r, n - 1) * (int)sizeof(C), 0);
        x[r].x = v[0];
        x[r].y = v[1];
      });
    }
  };
  auto is_sym = [&](const int4& tp) {
    return COMPACT == kSymmetric || (COMPACT == kMixed && (a.sym >> (tp.z >> 1) & 1));
  };
  auto bands = [&](const int4& tp) {  // the tuple's potential fibre
    const int term = tp.z >> 1;
    const unsigned long long base = (unsigned)from_lane((int)(dia_l & 0xffffffffu), term) |
                                    (unsigned long long)(unsigned)from_lane((int)(dia_l >> 32), term) << 32;
    const int fibre = (is_sym(tp) ? HB + 1 : BW) * n;  // stored values of a potential fibre
    return __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(base + (unsigned long long)tp.y * fibre * sizeof(V)), (short)0,
        fibre * (int)sizeof(V), 0x00020000);
  };
  auto load_row = [&](__amdgpu_buffer_rsrc_t band, bool sym, int r, V (&v)[BW]) {
    const int i = lane + 64 * r;
#pragma unroll
    for (int k = 0; k <= HB; ++k)
#pragma unroll
      for (int m = 0; m < (k && !SCATTER ? 2 : 1); ++m) {  // a diagonal and its mirror image, whose lines are the same
        const int d = m ? HB - k : HB + k;
        // stored diagonal of element (i, i + d - HB); of a mirrored one the row is i - (HB - d), and
        // rows outside the matrix, like lanes past the fibre, are masked by an offset past the buffer
        const int first = sym && m ? k : 0;
        const int off = (sym ? k : d) * n - first;
        v[d] = ld_band<V, COMPACT != 0>(band, i < n && i >= first ? i * (int)sizeof(V) : kPastBand, off * (int)sizeof(V));
      }
  };
  auto window = [&](const C (&x)[NR]) {
    if constexpr (NR == 1) {
      if (lane < n) xw[HB + lane] = x[0];
    } else {
      for_rows<NR>([&](auto r) {
        if (lane + 64 * r < n) *reinterpret_cast<Pair*>(xw + HB + lane + 64 * r) = Pair{x[r].x, x[r].y};
      });
    }
    wave_sync();
  };
  auto use_row = [&](const int4& tp, auto r, const C& x, const V (&v)[BW]) {
    const int term = tp.z >> 1;
    const bool cj = tp.z & 1;
    C s;
    if constexpr (sizeof(C) == sizeof(double2)) {
      s.x = __hiloint2double(from_lane(__double2hiint(scale_l.x), term), from_lane(__double2loint(scale_l.x), term));
      s.y = __hiloint2double(from_lane(__double2hiint(scale_l.y), term), from_lane(__double2loint(scale_l.y), term));
    } else {
      s.x = __int_as_float(from_lane(__float_as_int(scale_l.x), term));
      s.y = __int_as_float(from_lane(__float_as_int(scale_l.y), term));
    }
    const int i = lane + 64 * r;
    C part = cz<C>();
    if constexpr (SCATTER) {
      C sx = cz<C>();
      acc_scaled(sx, s, x);
      acc_vx(part, v[HB], x, cj);
#pragma unroll
      for (int k = 1; k <= NK; ++k) {
        acc_vx(part, v[HB + k], xw[i + HB + k], cj);
        acc_vx(below[k], v[HB + k], sx, cj);
      }
    } else {
#pragma unroll
      for (int d = 0; d < BW; ++d) acc_vx(part, v[d], xw[i + d], cj);
    }
    acc_scaled(acc[r], s, part);
  };
  for (int b0 = w0; b0 < w1; b0 += 64) {
    const int last = min(64, w1 - b0) - 1;
    tup_l = a.tuples[b0 + min(lane, last)];
    if constexpr (NR * BW * sizeof(V) <= 13 * sizeof(double)) {
      // the next tuple's loads are issued before the current one is used: a wave waits for memory about
      // half as often, for one more set of registers
      auto load = [&](const int4& tp, C (&x)[NR], V (&v)[NR][BW]) {
        const __amdgpu_buffer_rsrc_t band = bands(tp);
        load_x(tp, x);
        for_rows<NR>([&](auto r) { load_row(band, is_sym(tp), r, v[r]); });
      };
      auto use = [&](const int4& tp, const C (&x)[NR], const V (&v)[NR][BW]) {
        window(x);
        for_rows<NR>([&](auto r) { use_row(tp, r, x[r], v[r]); });
        wave_sync();
      };
      C xa[NR], xb[NR];
      V va[NR][BW], vb[NR][BW];
      int4 ta = tuple(0), tb;
      load(ta, xa, va);
      for (int l = 0; l <= last; l += 2) {
        tb = tuple(min(l + 1, last));
        load(tb, xb, vb);
        use(ta, xa, va);
        if (l + 1 > last) break;
        ta = tuple(min(l + 2, last));
        load(ta, xa, va);
        use(tb, xb, vb);
      }
    } else {
      // A row per lane at a time, the next one's bands loaded ahead: the bands of all rows at once take up
      // to 512 registers and scratch memory, and leave one wave to a SIMD.  3 x 24 x 512, all pairs, 21
      // diagonals: real 132 us (214 all at once, 192 by row without the next), complex 208 (777, 239);
      // 4 x 30 x 300, 13 diagonals: 68 (109, 88) and 97 (158, 103).
      constexpr int kAhead = BW * sizeof(V) <= 21 * sizeof(double) ? 1 : 0;  // rows loaded ahead
      for (int l = 0; l <= last; ++l) {
        const int4 tp = tuple(l);
        C x[NR];
        const __amdgpu_buffer_rsrc_t band = bands(tp);
        load_x(tp, x);
        V v[kAhead + 1][BW];
        load_row(band, is_sym(tp), 0, v[0]);
        window(x);
        for_rows<NR>([&](auto r) {
          constexpr int R = decltype(r)::value;
          if constexpr (kAhead == 1 && R + 1 < NR) load_row(band, is_sym(tp), R + 1, v[(R + 1) & 1]);
          if constexpr (kAhead == 0 && R > 0) load_row(band, is_sym(tp), R, v[0]);
          use_row(tp, r, x[r], v[R & kAhead]);
        });
        wave_sync();
      }
    }
  }
#pragma unroll
  for (int k = 1; k <= NK; ++k) {
    xw[lane] = below[k];
    wave_sync();
    if (lane >= k) {
      acc[0].x += xw[lane - k].x;
      acc[0].y += xw[lane - k].y;
    }
    wave_sync();
  }
  __syncthreads();
  C(*red)[WIN] = xs;
  for_rows<NR>([&](auto r) { red[wave][lane + 64 * r] = acc[r]; });
  __syncthreads();
  if (wave == 0) {
    C* out = a.dst + (long long)fib * n;
    const C* add = a.addend ? a.addend + (long long)fib * n : nullptr;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int i = lane + 64 * r;
      if (i < n) {
        C s = red[0][i];
        s.x += red[1][i].x; s.y += red[1][i].y;
        s.x += red[2][i].x; s.y += red[2][i].y;
        s.x += red[3][i].x; s.y += red[3][i].y;
        C o = a.accumulate ? out[i] : cz<C>();
        if (add) { o.x += add[i].x; o.y += add[i].y; }
        acc_scaled(o, a.alpha, s);
        out[i] = o;
      }
    }
  }
}

// generic path: entries per inner row (CSR) over the reference layout
template <class C>
struct GenArgs {
  const int4* tuples;
  const int* fib_ptr;
  const int* fib_order;
  const int* row_ptr;      // n + 1
  const int4* entries;     // {col, potential index, flags, 0}; flags: 1 conj, 2 real part, 4 ignore tuple conj
  const void* vref[kMaxTerms];
  C scale[kMaxTerms];
  long long pin;           // innermost potential extent
  int n;
  const C* src;
  C* dst;
  const C* addend;
  C alpha;
  int accumulate;
};

template <class C>
__global__ __launch_bounds__(64) void tp_generic_kernel(GenArgs<C> a) {
  const int fib = a.fib_order[blockIdx.x];
  const int t0 = a.fib_ptr[fib];
  const int t1 = a.fib_ptr[fib + 1];
  const int n = a.n;
  C* out = a.dst + (long long)fib * n;
  const C* add = a.addend ? a.addend + (long long)fib * n : nullptr;
  for (int i = threadIdx.x; i < n; i += 64) {
    C acc = cz<C>();
    const int e0 = a.row_ptr[i], e1 = a.row_ptr[i + 1];
    for (int t = t0; t < t1; ++t) {
      const int4 tp = a.tuples[t];
      const int term = tp.z >> 1;
      const bool tcj = tp.z & 1;
      const C* v = reinterpret_cast<const C*>(a.vref[term]) + (long long)tp.y * a.pin;
      const C* x = a.src + (long long)tp.x * n;
      C part = cz<C>();
      for (int e = e0; e < e1; ++e) {
        const int4 en = a.entries[e];
        C vv = v[en.y];
        if (en.z & 2) vv.y = 0;
        const bool cj = ((en.z & 4) ? false : tcj) ^ (bool)(en.z & 1);
        acc_vx(part, vv, x[en.x], cj);
      }
      acc_scaled(acc, a.scale[term], part);
    }
    C o = a.accumulate ? out[i] : cz<C>();
    if (add) { o.x += add[i].x; o.y += add[i].y; }
    acc_scaled(o, a.alpha, acc);
    out[i] = o;
  }
}

// repack reference band layouts into diagonal-major form
//   BandNH: A(i, j) = V[j*bw + hb + i - j]
//   Band  : A(i, j) = V[j*k + i - j] (i > j), conj(V[i*k + j - i]) (i < j), Re V[i*k] (i == j)
template <class OutT>
__global__ void repack_band_kernel(const double2* __restrict__ vref, OutT* __restrict__ out,
                                   long long fibres, int n, int bw, int kind, long long pin) {
  const int hb = (bw - 1) / 2;
  const long long total = fibres * bw * (long long)n;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(idx % n);
    const int d = (int)((idx / n) % bw);
    const long long f = idx / ((long long)n * bw);
    const int j = i + d - hb;
    double2 val = make_double2(0.0, 0.0);
    if (j >= 0 && j < n) {
      const double2* v = vref + f * pin;
      if (kind == PP_STORAGE_BANDNH) {
        val = v[(long long)j * bw + hb + i - j];
      } else {
        const int k = hb + 1;
        if (i > j) val = v[(long long)j * k + i - j];
        else if (i < j) { val = v[(long long)i * k + j - i]; val.y = -val.y; }
        else { val = v[(long long)i * k]; val.y = 0.0; }
      }
    }
    if constexpr (sizeof(OutT) == sizeof(double)) out[idx] = (OutT)val.x;
    else if constexpr (sizeof(OutT) == sizeof(double2)) out[idx] = val;
    else if constexpr (sizeof(OutT) == sizeof(float)) out[idx] = (OutT)val.x;
    else out[idx] = make_float2((float)val.x, (float)val.y);
  }
}

__global__ void max_abs_imag_kernel(const double2* __restrict__ v, long long n, unsigned long long* flag) {
  bool nz = false;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    nz |= (v[i].y != 0.0);
  if (__any(nz) && (threadIdx.x & 63) == 0) atomicOr(flag, 1ull);
}

// out[a][r] (+)= sum_t coeffs[t][a] radial[t][r].  Bound by the 16 bytes written per value: a thread
// takes one r, holds its T radial values in registers and walks over a range of a, whose T
// coefficients are uniform (scalar loads); each wave stores 1 KB runs that nothing reads back soon
// (non-temporal).  One value per thread with an integer division and 2 T loads each: 3.45 ms on helium's
// 1/r12 (394 x 575640, 11 terms, 3.63 GB); this form 0.70 ms (5.2 TB/s; with temporal stores 0.75).
template <int T>
__global__ __launch_bounds__(256) void expand_terms_kernel(long long p0, long long rc, long long r0, long long a_range,
                                                           const double* __restrict__ coeffs,
                                                           const double* __restrict__ radial,
                                                           double2* __restrict__ out, int accumulate) {
  const long long r = r0 + blockIdx.x * 256LL + threadIdx.x;
  const long long a0 = blockIdx.y * a_range, a1 = min(p0, a0 + a_range);
  if (r >= rc) return;
  double R[T];
#pragma unroll
  for (int t = 0; t < T; ++t) R[t] = radial[t * rc + r];
  for (long long a = a0; a < a1; ++a) {
    double v = 0.0;
#pragma unroll
    for (int t = 0; t < T; ++t) v = fma(coeffs[t * p0 + a], R[t], v);
    typedef double pp_d2v __attribute__((ext_vector_type(2)));
    pp_d2v* o = reinterpret_cast<pp_d2v*>(out + a * rc + r);
    pp_d2v w = {v, 0.0};
    if (accumulate) w += *o;
    __builtin_nontemporal_store(w, o);
  }
}

void expand_terms(int terms, long long p0, long long rc, const double* coeffs, const double* radial, double2* out,
                  int accumulate, hipStream_t s) {
  constexpr long long kSlice = 1LL << 31;  // radial values per launch, which holds fewer than 2^32 threads a row
  for (long long r0 = 0; r0 < rc; r0 += kSlice) {
    const long long nx = (std::min(kSlice, rc - r0) + 255) / 256;
    // a range per workgroup: 4096 workgroups keep every CU writing; more would re-read the radial values
    const long long ny = std::max(1LL, std::min({p0, 65535LL, (4096 + nx - 1) / nx}));
    const long long a_range = (p0 + ny - 1) / ny;
    const dim3 grid((unsigned)nx, (unsigned)((p0 + a_range - 1) / a_range));
    for (int t0 = 0; t0 < terms; t0 += 12) {
      switch (std::min(12, terms - t0)) {
#define PP_EXPAND(T)                                                                                            \
  case T:                                                                                                       \
    hipLaunchKernelGGL(expand_terms_kernel<T>, grid, dim3(256), 0, s, p0, rc, r0, a_range, coeffs + t0 * p0,     \
                       radial + t0 * rc, out, accumulate || t0 > 0);                                            \
    break;
        PP_EXPAND(1) PP_EXPAND(2) PP_EXPAND(3) PP_EXPAND(4) PP_EXPAND(5) PP_EXPAND(6) PP_EXPAND(7) PP_EXPAND(8)
        PP_EXPAND(9) PP_EXPAND(10) PP_EXPAND(11) PP_EXPAND(12)
#undef PP_EXPAND
      }
    }
  }
  PP_HIP(hipGetLastError());
}

__global__ void convert_f64_f32_kernel(const double* __restrict__ in, float* __restrict__ out, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    out[i] = (float)in[i];
}

// ----------------------------------------------------------------------------------
// plan construction
// ----------------------------------------------------------------------------------
struct Tuple {
  int dst, src, pot, conj;
};

static std::vector<Tuple> outer_tuples(const TPGeometry& g) {
  const int R = g.rank;
  std::vector<std::vector<RankEntry>> per(R > 1 ? R - 1 : 0);
  for (int r = 0; r + 1 < R; ++r)
    per[r] = enumerate_rank(g.ids[r], g.pot_ext[r], g.src_ext[r], g.pairs[r].empty() ? nullptr : g.pairs[r].data(),
                            (int)(g.pairs[r].size() / 2));
  std::vector<Tuple> out;
  if (R == 1) {
    out.push_back({0, 0, 0, 0});
    return out;
  }
  // strides over the outer dims
  std::vector<long long> sstride(R - 1), pstride(R - 1);
  long long s = 1, p = 1;
  for (int r = R - 2; r >= 0; --r) {
    sstride[r] = s;
    pstride[r] = p;
    s *= g.src_ext[r];
    p *= g.pot_ext[r];
  }
  PP_REQUIRE(s < (1ll << 31) && p < (1ll << 31), "outer fibre count exceeds int32");
  long long total = 1;
  for (auto& v : per) total *= (long long)v.size();
  PP_REQUIRE(total < (1ll << 31), "tuple count exceeds int32");
  out.reserve((size_t)total);
  std::vector<size_t> idx(R - 1, 0);
  // iterate the nested loops (rank 0 outermost)
  while (true) {
    long long d = 0, sc = 0, pp_ = 0;
    int cj = 0;
    for (int r = 0; r < R - 1; ++r) {
      const RankEntry& e = per[r][idx[r]];
      d += e.row * sstride[r];
      sc += e.col * sstride[r];
      pp_ += e.pidx * pstride[r];
      cj ^= e.toggle;
    }
    out.push_back({(int)d, (int)sc, (int)pp_, cj});
    int r = R - 2;
    while (r >= 0) {
      if (++idx[r] < per[r].size()) break;
      idx[r] = 0;
      --r;
    }
    if (r < 0) break;
  }
  return out;
}

static void build_inner_csr(const TPGeometry& g, std::vector<int>& row_ptr, std::vector<int4>& entries) {
  const int R = g.rank;
  const int id = g.ids[R - 1];
  const int n = g.src_ext[R - 1];
  const int pin = g.pot_ext[R - 1];
  std::vector<std::vector<int4>> rows(n);
  if (id == PP_STORAGE_BAND) {
    PP_REQUIRE(pin % n == 0, "Band potential extent must be a multiple of N");
    const int k = pin / n;
    for (int i = 0; i < n; ++i) {
      for (int j = std::max(0, i - k + 1); j < i; ++j) rows[i].push_back(make_int4(j, j * k + i - j, 4, 0));
      rows[i].push_back(make_int4(i, i * k, 2 | 4, 0));
      for (int j = i + 1; j < std::min(n, i + k); ++j) rows[i].push_back(make_int4(j, i * k + j - i, 1 | 4, 0));
    }
  } else {
    auto e = enumerate_rank(id, pin, n, g.pairs[R - 1].empty() ? nullptr : g.pairs[R - 1].data(),
                            (int)(g.pairs[R - 1].size() / 2));
    for (auto& x : e) rows[x.row].push_back(make_int4(x.col, x.pidx, x.toggle, 0));
  }
  row_ptr.assign(n + 1, 0);
  for (int i = 0; i < n; ++i) row_ptr[i + 1] = row_ptr[i] + (int)rows[i].size();
  entries.clear();
  for (auto& r : rows) entries.insert(entries.end(), r.begin(), r.end());
}

static unsigned symmetric_terms(const std::vector<const TPTerm*>& terms) {
  unsigned m = 0;
  for (size_t t = 0; t < terms.size(); ++t) m |= (terms[t]->sym ? 1u : 0u) << t;
  return m;
}
static bool any_compact(const std::vector<const TPTerm*>& terms) {
  for (auto* t : terms)
    if (t->sym || !t->canon.empty()) return true;
  return false;
}

// Launch order of a compact plan: workgroup b runs on XCD b % 8, and the destination fibres (.., i) and
// (.., j) of one group (equal indices but the last outer one) read the same stored fibres at about
// the same time.  Each XCD therefore takes a contiguous range of fibres of about an eighth of the
// tuples, heaviest groups first, so that a stored fibre comes into its L2 once; ranges that are
// shorter in number are filled up with -1.  Helium's full H: longest fibres first 203 us, this order
// 181 us.
static void xcd_order(TPPlanData& pd, int group) {
  constexpr int kXcds = 8;
  auto count = [&](long long f) { return pd.fib_ptr[f + 1] - pd.fib_ptr[f]; };
  std::vector<int> weight((pd.n_fibres + group - 1) / group, 0);
  for (long long f = 0; f < pd.n_fibres; ++f) weight[f / group] = std::max(weight[f / group], count(f));
  std::vector<int> part[kXcds];
  const long long total = pd.fib_ptr[pd.n_fibres] + pd.n_fibres;  // an empty fibre is some work too
  long long done = 0;
  for (long long f = 0; f < pd.n_fibres; ++f) {
    part[std::min<long long>(kXcds - 1, done * kXcds / total)].push_back((int)f);
    done += count(f) + 1;
  }
  size_t most = 0;
  for (auto& p : part) {
    std::stable_sort(p.begin(), p.end(), [&](int a, int b) { return weight[a / group] > weight[b / group]; });
    most = std::max(most, p.size());
  }
  // (tuples gathered in few fibres: the other XCDs' ranges hold most fibres and the filling most
  // workgroups; the order by length is kept)
  if (most * kXcds > 2 * (size_t)pd.n_fibres + 64) return;
  pd.fib_order.assign(most * kXcds, -1);
  for (int x = 0; x < kXcds; ++x)
    for (size_t k = 0; k < part[x].size(); ++k) pd.fib_order[k * kXcds + x] = part[x][k];
}

TPPlanData build_plan_host(const std::vector<const TPTerm*>& terms) {
  PP_REQUIRE(!terms.empty() && terms.size() <= (size_t)kMaxTerms, "1..8 terms per plan");
  const TPGeometry& g0 = terms[0]->geom;
  TPPlanData pd;
  const int R = g0.rank;
  pd.n = g0.src_ext[R - 1];
  long long nf = 1;
  for (int r = 0; r + 1 < R; ++r) nf *= g0.src_ext[r];
  pd.n_fibres = nf;
  std::vector<std::vector<int4>> byfib(nf);
  for (size_t t = 0; t < terms.size(); ++t) {
    const TPGeometry& g = terms[t]->geom;
    PP_REQUIRE(g.rank == R, "terms must share the rank");
    for (int r = 0; r < R; ++r) PP_REQUIRE(g.src_ext[r] == g0.src_ext[r], "terms must share the source shape");
    const bool ignore_conj = g.ids[R - 1] == PP_STORAGE_BAND;  // zhbmv takes no conjugate flag
    const std::vector<int>& canon = terms[t]->canon;
    for (const Tuple& tp : outer_tuples(g))
      byfib[tp.dst].push_back(make_int4(tp.src, canon.empty() ? tp.pot : canon[tp.pot], (int)(t << 1) | (ignore_conj ? 0 : tp.conj), 0));
  }
  pd.fib_ptr.assign(nf + 1, 0);
  for (long long f = 0; f < nf; ++f) pd.fib_ptr[f + 1] = pd.fib_ptr[f] + (int)byfib[f].size();
  pd.tuples.reserve(pd.fib_ptr[nf]);
  for (auto& v : byfib) pd.tuples.insert(pd.tuples.end(), v.begin(), v.end());
  pd.fib_order.resize(nf);
  std::iota(pd.fib_order.begin(), pd.fib_order.end(), 0);
  std::stable_sort(pd.fib_order.begin(), pd.fib_order.end(), [&](int a, int b) {
    return (pd.fib_ptr[a + 1] - pd.fib_ptr[a]) > (pd.fib_ptr[b + 1] - pd.fib_ptr[b]);
  });
  pd.non_empty = 0;
  for (long long f = 0; f < nf; ++f)
    if (pd.fib_ptr[f + 1] > pd.fib_ptr[f]) ++pd.non_empty;
  if (any_compact(terms)) xcd_order(pd, R > 1 ? g0.src_ext[R - 2] : 1);
  return pd;
}

void upload_plan(const TPPlanData& pd, TPPlanDevice& dv, hipStream_t s) {
  dv.tuples.upload(pd.tuples.data(), pd.tuples.size(), s);
  dv.fib_ptr.upload(pd.fib_ptr.data(), pd.fib_ptr.size(), s);
  dv.fib_order.upload(pd.fib_order.data(), pd.fib_order.size(), s);
  dv.n = pd.n;
  dv.n_fibres = pd.n_fibres;
  dv.non_empty = pd.non_empty;
  dv.order_count = (int)pd.fib_order.size();
  dv.tuple_count = (long long)pd.tuples.size();
}

// flag |= some element (i, i + d - hb) below the diagonal differs in its bits from its mirror image
__global__ void asymmetric_kernel(const double* __restrict__ dia, long long fibres, int n, int bw,
                                  unsigned long long* flag) {
  const int hb = (bw - 1) / 2;
  const long long total = fibres * hb * (long long)n;
  bool differs = false;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(idx % n), d = (int)(idx / n % hb), j = i + d - hb;
    const double* f = dia + idx / ((long long)n * hb) * bw * n;
    if (j >= 0) differs |= __double_as_longlong(f[d * n + i]) != __double_as_longlong(f[(2 * hb - d) * n + j]);
  }
  if (__any(differs) && (threadIdx.x & 63) == 0) atomicOr(flag, 1ull);
}

// Enters fibre f into a hash table (keys zero where empty, at least twice as many slots as fibres) under
// the bits of its rows [first, first + len): slot[f] is its slot, owner[slot] the smallest fibre there.
// One wave per fibre; the hash is a sum over its values of SplitMix64's finaliser (G. L. Steele, D. Lea,
// C. H. Flood, OOPSLA 2014) of (bits, position).
__global__ __launch_bounds__(256) void fibre_hash_kernel(const double* __restrict__ dia, long long fibres, int stride,
                                                         int first, int len, unsigned long long mask,
                                                         unsigned long long* keys, int* owner, int* __restrict__ slot) {
  const long long f = blockIdx.x * 4LL + (threadIdx.x >> 6);
  if (f >= fibres) return;
  const double* v = dia + f * stride + first;
  unsigned long long h = 0;
  for (int k = threadIdx.x & 63; k < len; k += 64) {
    unsigned long long w = (unsigned long long)__double_as_longlong(v[k]) + 0x9E3779B97F4A7C15ull * (k + 1);
    w = (w ^ (w >> 30)) * 0xBF58476D1CE4E5B9ull;
    w = (w ^ (w >> 27)) * 0x94D049BB133111EBull;
    h += w ^ (w >> 31);
  }
  for (int off = 32; off > 0; off >>= 1) h += __shfl_down(h, off, 64);
  if ((threadIdx.x & 63) != 0) return;
  if (h == 0) h = 1;
  unsigned long long i = h & mask;
  for (unsigned long long old; (old = atomicCAS(&keys[i], 0ull, h)) != 0 && old != h;) i = (i + 1) & mask;
  atomicMin(&owner[i], (int)f);
  slot[f] = (int)i;
}

// rep[f] (slot[f] on entry) = the first fibre of f's slot; flag |= they differ in their bits
__global__ __launch_bounds__(256) void fibre_differs_kernel(const double* __restrict__ dia, long long fibres, int stride,
                                                            int first, int len, const int* __restrict__ owner, int* rep,
                                                            unsigned long long* flag) {
  const long long f = blockIdx.x * 4LL + (threadIdx.x >> 6);
  if (f >= fibres) return;
  const int r = owner[rep[f]];
  const double *a = dia + f * stride + first, *b = dia + (long long)r * stride + first;
  bool differs = false;
  if (r != f)
    for (int k = threadIdx.x & 63; k < len; k += 64)
      differs |= __double_as_longlong(a[k]) != __double_as_longlong(b[k]);
  if (__any(differs) && (threadIdx.x & 63) == 0) atomicOr(flag, 1ull);
  if ((threadIdx.x & 63) == 0) rep[f] = r;
}

// out[u] = rows [first, first + len) of fibre kept[u]
__global__ __launch_bounds__(256) void gather_fibres_kernel(const double* __restrict__ dia, long long kept_count,
                                                            int stride, int first, int len,
                                                            const int* __restrict__ kept, double* __restrict__ out) {
  const long long u = blockIdx.x * 4LL + (threadIdx.x >> 6);
  if (u >= kept_count) return;
  const double* v = dia + (long long)kept[u] * stride + first;
  for (int k = threadIdx.x & 63; k < len; k += 64) out[u * len + k] = v[k];
}

// Values of a term from which compact storage is looked for: the search costs 0.1 ms a term, and a
// smaller term is read from L2 in any case (hydrogen, 8 x 120: set-up 0.25 ms without it, 0.42 with; the
// same product).  5 x 12 x 12 helium, of 40000 values and more a term, gains: 10 us of a product's 23.
constexpr long long kCompactFrom = 1 << 15;

// Stores a real banded term compactly where that saves at least a quarter (a hash collision keeps it
// as it is: equality is checked value by value).  The table is built on the device: setting up helium's
// three terms (425000 fibres, 2.65 GB) takes 16.9 ms, 16.0 without the search and 24.7 with the table on
// the host.
static void compact_term(TPTerm& term, long long pfib, int n, hipStream_t s) {
  if (pfib >= (1ll << 26)) return;  // a wave per fibre: a launch holds fewer than 2^32 threads
  const int bw = term.bw, hb = (bw - 1) / 2, stride = bw * n;
  const int wave_blocks = ceil_div(pfib, 4);
  // one allocation for the search: a flag, the table's keys and owners, and an index per fibre
  size_t slots = 64;
  while (slots < 2 * (size_t)pfib) slots *= 2;
  DeviceBuffer<unsigned long long> scratch(1 + slots + (slots + pfib + 1) / 2);
  unsigned long long *flag = scratch.ptr, *keys = flag + 1;
  int *owner = reinterpret_cast<int*>(keys + slots), *index = owner + slots;
  PP_HIP(hipMemsetAsync(flag, 0, (1 + slots) * sizeof(unsigned long long), s));
  PP_HIP(hipMemsetAsync(owner, 0x7f, slots * sizeof(int), s));
  auto read_flag = [&]() {
    unsigned long long h = 0;
    PP_HIP(hipMemcpyAsync(&h, flag, sizeof(h), hipMemcpyDeviceToHost, s));
    PP_HIP(hipStreamSynchronize(s));
    return h != 0;
  };
  bool sym = hb > 0;
  if (sym) {
    const long long total = pfib * hb * (long long)n;
    hipLaunchKernelGGL(asymmetric_kernel, dim3((int)std::min<long long>(65536, (total + 255) / 256)), dim3(256), 0, s,
                       term.dia_real.ptr, pfib, n, bw, flag);
    PP_HIP(hipGetLastError());
    sym = !read_flag();
    if (!sym) PP_HIP(hipMemsetAsync(flag, 0, sizeof(unsigned long long), s));
  }
  const int first = sym ? hb * n : 0, len = sym ? (hb + 1) * n : stride;
  hipLaunchKernelGGL(fibre_hash_kernel, dim3(wave_blocks), dim3(256), 0, s, term.dia_real.ptr, pfib, stride, first, len,
                     (unsigned long long)(slots - 1), keys, owner, index);
  hipLaunchKernelGGL(fibre_differs_kernel, dim3(wave_blocks), dim3(256), 0, s, term.dia_real.ptr, pfib, stride, first,
                     len, owner, index, flag);
  PP_HIP(hipGetLastError());
  std::vector<int> canon(pfib), rep(pfib), kept;
  PP_HIP(hipMemcpyAsync(rep.data(), index, pfib * sizeof(int), hipMemcpyDeviceToHost, s));
  bool merged = !read_flag();
  for (long long f = 0; merged && f < pfib; ++f) {  // rep[f] <= f
    canon[f] = rep[f] == f ? (int)kept.size() : canon[rep[f]];
    if (rep[f] == f) kept.push_back((int)f);
  }
  merged = merged && kept.size() < (size_t)pfib;
  if (!merged) {
    kept.resize(pfib);
    std::iota(kept.begin(), kept.end(), 0);
  }
  const long long size = (long long)kept.size() * len;
  if (size * 4 > pfib * (long long)stride * 3) return;
  DeviceBuffer<double> out(size);
  PP_HIP(hipMemcpyAsync(index, kept.data(), kept.size() * sizeof(int), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(gather_fibres_kernel, dim3(ceil_div((long long)kept.size(), 4)), dim3(256), 0, s,
                     term.dia_real.ptr, (long long)kept.size(), stride, first, len, index, out.ptr);
  PP_HIP(hipGetLastError());
  PP_HIP(hipStreamSynchronize(s));  // before what the copy reads is released
  std::swap(term.dia_real.ptr, out.ptr);
  std::swap(term.dia_real.count, out.count);
  term.sym = sym;
  if (merged) term.canon = std::move(canon);
  term.stream_bytes = size * (long long)sizeof(double);
}

static bool is_band(int id) { return id == PP_STORAGE_BANDNH || id == PP_STORAGE_BAND; }

void tp_create_impl(int rank, const int* ids, const double2* potential, const int* pot_ext,
                    const int* src_ext, const int32_t* const* pairs, const int* pair_counts,
                    hipStream_t s, TPTerm& term, bool compact) {
  PP_REQUIRE(rank >= 1 && rank <= kMaxRank, "rank must be 1..4");
  PP_REQUIRE(potential != nullptr, "potential is NULL");
  TPGeometry& g = term.geom;
  g.rank = rank;
  long long pcount = 1;
  for (int r = 0; r < rank; ++r) {
    g.ids[r] = ids[r];
    g.pot_ext[r] = pot_ext[r];
    g.src_ext[r] = src_ext[r];
    PP_REQUIRE(pot_ext[r] > 0 && src_ext[r] > 0, "extents must be positive");
    pcount *= pot_ext[r];
    if (ids[r] == PP_STORAGE_SIMP || ids[r] == PP_STORAGE_HERM) {
      PP_REQUIRE(pairs && pairs[r] && pair_counts && pair_counts[r] == pot_ext[r],
                 "Simp/Herm rank needs a pair list of the potential extent");
      g.pairs[r].assign(pairs[r], pairs[r] + 2 * (size_t)pair_counts[r]);
    } else {
      g.pairs[r].clear();
    }
    if (ids[r] == PP_STORAGE_DIAG) PP_REQUIRE(pot_ext[r] <= src_ext[r], "Diag extent exceeds source extent");
    if (ids[r] == PP_STORAGE_IDENT) PP_REQUIRE(pot_ext[r] == 1, "Ident potential extent must be 1");
    if (ids[r] == PP_STORAGE_DENSE) PP_REQUIRE(pot_ext[r] == src_ext[r] * src_ext[r], "Dense potential extent must be N*N");
  }
  const int inner = ids[rank - 1];
  const int n = src_ext[rank - 1];
  const long long pin = pot_ext[rank - 1];
  const long long pfib = pcount / pin;
  term.pot_elements = pcount;
  term.pot_fibres = pfib;

  // realness of the potential
  {
    DeviceBuffer<unsigned long long> flag(1);
    PP_HIP(hipMemsetAsync(flag.ptr, 0, sizeof(unsigned long long), s));
    int blocks = (int)std::min<long long>(4096, (pcount + 255) / 256);
    hipLaunchKernelGGL(max_abs_imag_kernel, dim3(blocks), dim3(256), 0, s, potential, pcount, flag.ptr);
    PP_HIP(hipGetLastError());
    unsigned long long h = 0;
    PP_HIP(hipMemcpyAsync(&h, flag.ptr, sizeof(h), hipMemcpyDeviceToHost, s));
    PP_HIP(hipStreamSynchronize(s));
    term.is_real = (h == 0);
  }

  term.inner_kind = inner;
  if (is_band(inner) && n <= kMaxDiaRows) {
    PP_REQUIRE(pin % n == 0, "band potential extent must be a multiple of the source extent");
    int bw = (inner == PP_STORAGE_BANDNH) ? (int)(pin / n) : (int)(2 * (pin / n) - 1);
    PP_REQUIRE(bw % 2 == 1 && bw >= 1, "band width must be odd");
    term.dia = true;
    term.bw = bw;
    const long long total = pfib * bw * (long long)n;
    int blocks = (int)std::min<long long>(65536, (total + 255) / 256);
    if (term.is_real) {
      term.dia_real.resize(total);
      hipLaunchKernelGGL(repack_band_kernel<double>, dim3(blocks), dim3(256), 0, s, potential,
                         term.dia_real.ptr, pfib, n, bw, inner, pin);
      term.stream_bytes = total * (long long)sizeof(double);
    } else {
      term.dia_cplx.resize(total);
      hipLaunchKernelGGL(repack_band_kernel<double2>, dim3(blocks), dim3(256), 0, s, potential,
                         term.dia_cplx.ptr, pfib, n, bw, inner, pin);
      term.stream_bytes = total * (long long)sizeof(double2);
    }
    PP_HIP(hipGetLastError());
    if (compact && term.is_real && total >= kCompactFrom) {
      // Without room for the search or the second copy the term is kept as it is (compact_term changes it
      // at its end only).
      try {
        compact_term(term, pfib, n, s);
      } catch (const Error& e) {
        if (e.code != PP_ERR_ALLOC) throw;
        (void)hipGetLastError();  // or the next launch's check would report the failed allocation
      } catch (const std::bad_alloc&) {
      }
    }
  } else {
    term.dia = false;
    term.vref.resize(pcount);
    PP_HIP(hipMemcpyAsync(term.vref.ptr, potential, pcount * sizeof(double2), hipMemcpyDeviceToDevice, s));
    std::vector<int> row_ptr;
    std::vector<int4> entries;
    build_inner_csr(g, row_ptr, entries);
    term.row_ptr.upload(row_ptr.data(), row_ptr.size(), s);
    term.entries.upload(entries.data(), entries.size(), s);
    term.stream_bytes = pcount * (long long)sizeof(double2);
  }
  TPPlanData pd = build_plan_host({&term});
  upload_plan(pd, term.plan, s);
  PP_HIP(hipStreamSynchronize(s));
}

void tp_ensure_f32(const TPTerm& t, hipStream_t s) {
  if (!t.dia) throw Error(PP_ERR_INVALID, "FP32 multiply needs a banded innermost storage");
  TPTerm& m = const_cast<TPTerm&>(t);
  const long long total = (long long)(t.is_real ? t.dia_real.count : t.dia_cplx.count);  // as stored
  if (t.is_real) {
    if (m.dia_real_f.count == (size_t)total) return;
    m.dia_real_f.resize(total);
    int blocks = (int)std::min<long long>(65536, (total + 255) / 256);
    hipLaunchKernelGGL(convert_f64_f32_kernel, dim3(blocks), dim3(256), 0, s, t.dia_real.ptr,
                       m.dia_real_f.ptr, total);
  } else {
    if (m.dia_cplx_f.count == (size_t)total) return;
    m.dia_cplx_f.resize(total);
    int blocks = (int)std::min<long long>(65536, (2 * total + 255) / 256);
    hipLaunchKernelGGL(convert_f64_f32_kernel, dim3(blocks), dim3(256), 0, s,
                       reinterpret_cast<const double*>(t.dia_cplx.ptr),
                       reinterpret_cast<float*>(m.dia_cplx_f.ptr), 2 * total);
  }
  PP_HIP(hipGetLastError());
}

// ----------------------------------------------------------------------------------
// launch
// ----------------------------------------------------------------------------------
template <class V, class C, int BW, int COMPACT>
static void launch_dia_bw(const DiaArgs<C>& a, int nr, int blocks, hipStream_t s) {
  // rows per lane rounded up to 1, 2, 4 or 8 (the kernel masks rows >= n)
  if (nr <= 1) hipLaunchKernelGGL((tp_dia_kernel<V, C, BW, 1, COMPACT>), dim3(blocks), dim3(256), 0, s, a);
  else if (nr <= 2) hipLaunchKernelGGL((tp_dia_kernel<V, C, BW, 2, COMPACT>), dim3(blocks), dim3(256), 0, s, a);
  else if (nr <= 4) hipLaunchKernelGGL((tp_dia_kernel<V, C, BW, 4, COMPACT>), dim3(blocks), dim3(256), 0, s, a);
  else if (nr <= 8) hipLaunchKernelGGL((tp_dia_kernel<V, C, BW, 8, COMPACT>), dim3(blocks), dim3(256), 0, s, a);
  else throw Error(PP_ERR_INVALID, "innermost extent too large for the banded kernel");
}

template <class V, class C, int COMPACT>
static void launch_dia(const DiaArgs<C>& a, int bw, int nr, int blocks, hipStream_t s) {
  switch (bw) {
    case 1: launch_dia_bw<V, C, 1, COMPACT>(a, nr, blocks, s); break;
    case 3: launch_dia_bw<V, C, 3, COMPACT>(a, nr, blocks, s); break;
    case 5: launch_dia_bw<V, C, 5, COMPACT>(a, nr, blocks, s); break;
    case 7: launch_dia_bw<V, C, 7, COMPACT>(a, nr, blocks, s); break;
    case 9: launch_dia_bw<V, C, 9, COMPACT>(a, nr, blocks, s); break;
    case 11: launch_dia_bw<V, C, 11, COMPACT>(a, nr, blocks, s); break;
    case 13: launch_dia_bw<V, C, 13, COMPACT>(a, nr, blocks, s); break;
    case 15: launch_dia_bw<V, C, 15, COMPACT>(a, nr, blocks, s); break;
    case 17: launch_dia_bw<V, C, 17, COMPACT>(a, nr, blocks, s); break;
    case 19: launch_dia_bw<V, C, 19, COMPACT>(a, nr, blocks, s); break;
    case 21: launch_dia_bw<V, C, 21, COMPACT>(a, nr, blocks, s); break;
    default: throw Error(PP_ERR_INVALID, "band width not instantiated (odd 1..21 supported)");
  }
}

bool terms_fusable(const std::vector<const TPTerm*>& terms) {
  if (terms.empty() || terms.size() > (size_t)kMaxTerms) return false;
  const TPTerm* t0 = terms[0];
  for (auto* t : terms) {
    if (t->dia != t0->dia || t->geom.rank != t0->geom.rank) return false;
    for (int r = 0; r < t0->geom.rank; ++r)
      if (t->geom.src_ext[r] != t0->geom.src_ext[r]) return false;
    if (t->dia && (t->bw != t0->bw || t->is_real != t0->is_real)) return false;
    if (!t->dia && t->geom.pot_ext[t->geom.rank - 1] != t0->geom.pot_ext[t0->geom.rank - 1]) return false;
    if (!t->dia && (t->geom.ids[t->geom.rank - 1] != t0->geom.ids[t0->geom.rank - 1])) return false;
    if (!t->dia && t->geom.pairs[t->geom.rank - 1] != t0->geom.pairs[t0->geom.rank - 1]) return false;
  }
  return true;
}

// Workgroups of a multiply; only the fibres with tuples need one where the others keep their value
// (a streaming plan has those first)
static int plan_blocks(const TPPlanDevice& plan, const std::vector<const TPTerm*>& terms, bool keeps_empty) {
  if (any_compact(terms)) return plan.tuple_count == 0 && keeps_empty ? 0 : plan.order_count;
  return keeps_empty ? plan.non_empty : (int)plan.n_fibres;
}

void tp_run_f64(const TPPlanDevice& plan, const std::vector<const TPTerm*>& terms,
                const double2* scales, const double2* src, double2* dst, const double2* addend,
                double2 alpha, bool accumulate, hipStream_t s) {
  const TPTerm* t0 = terms[0];
  const int blocks = plan_blocks(plan, terms, accumulate && !addend);
  if (blocks == 0) return;
  if (t0->dia) {
    DiaArgs<double2> a{};
    a.tuples = plan.tuples.ptr;
    a.fib_ptr = plan.fib_ptr.ptr;
    a.fib_order = plan.fib_order.ptr;
    for (size_t i = 0; i < terms.size(); ++i) {
      a.dia[i] = t0->is_real ? (const void*)terms[i]->dia_real.ptr : (const void*)terms[i]->dia_cplx.ptr;
      a.scale[i] = scales[i];
    }
    a.n = plan.n;
    a.src = src;
    a.dst = dst;
    a.addend = addend;
    a.alpha = alpha;
    a.accumulate = accumulate ? 1 : 0;
    const int nr = (plan.n + 63) / 64;
    a.sym = symmetric_terms(terms);
    if (!t0->is_real) launch_dia<double2, double2, kStreamed>(a, t0->bw, nr, blocks, s);
    else if (a.sym == (1u << terms.size()) - 1) launch_dia<double, double2, kSymmetric>(a, t0->bw, nr, blocks, s);
    else if (any_compact(terms)) launch_dia<double, double2, kMixed>(a, t0->bw, nr, blocks, s);
    else launch_dia<double, double2, kStreamed>(a, t0->bw, nr, blocks, s);
  } else {
    GenArgs<double2> a{};
    a.tuples = plan.tuples.ptr;
    a.fib_ptr = plan.fib_ptr.ptr;
    a.fib_order = plan.fib_order.ptr;
    a.row_ptr = t0->row_ptr.ptr;
    a.entries = t0->entries.ptr;
    for (size_t i = 0; i < terms.size(); ++i) {
      a.vref[i] = terms[i]->vref.ptr;
      a.scale[i] = scales[i];
    }
    a.pin = t0->geom.pot_ext[t0->geom.rank - 1];
    a.n = plan.n;
    a.src = src;
    a.dst = dst;
    a.addend = addend;
    a.alpha = alpha;
    a.accumulate = accumulate ? 1 : 0;
    hipLaunchKernelGGL(tp_generic_kernel<double2>, dim3(blocks), dim3(64), 0, s, a);
  }
  PP_HIP(hipGetLastError());
}

void tp_run_f32(const TPPlanDevice& plan, const std::vector<const TPTerm*>& terms,
                const float2* scales, const float2* src, float2* dst, const float2* addend,
                float2 alpha, bool accumulate, hipStream_t s) {
  const TPTerm* t0 = terms[0];
  PP_REQUIRE(t0->dia, "FP32 multiply needs a banded innermost storage");
  for (auto* t : terms) tp_ensure_f32(*t, s);
  const int blocks = plan_blocks(plan, terms, accumulate && !addend);
  if (blocks == 0) return;
  DiaArgs<float2> a{};
  a.tuples = plan.tuples.ptr;
  a.fib_ptr = plan.fib_ptr.ptr;
  a.fib_order = plan.fib_order.ptr;
  for (size_t i = 0; i < terms.size(); ++i) {
    a.dia[i] = t0->is_real ? (const void*)terms[i]->dia_real_f.ptr : (const void*)terms[i]->dia_cplx_f.ptr;
    a.scale[i] = scales[i];
  }
  a.n = plan.n;
  a.src = src;
  a.dst = dst;
  a.addend = addend;
  a.alpha = alpha;
  a.accumulate = accumulate ? 1 : 0;
  const int nr = (plan.n + 63) / 64;
  a.sym = symmetric_terms(terms);
  if (!t0->is_real) launch_dia<float2, float2, kStreamed>(a, t0->bw, nr, blocks, s);
  else if (a.sym == (1u << terms.size()) - 1) launch_dia<float, float2, kSymmetric>(a, t0->bw, nr, blocks, s);
  else if (any_compact(terms)) launch_dia<float, float2, kMixed>(a, t0->bw, nr, blocks, s);
  else launch_dia<float, float2, kStreamed>(a, t0->bw, nr, blocks, s);
  PP_HIP(hipGetLastError());
}

}  // namespace pp

// ----------------------------------------------------------------------------------
// C ABI
// ----------------------------------------------------------------------------------
using namespace pp;

extern "C" int pp_tp_create(int rank, const int* storage_ids, const pp_cplx* potential,
                            const int* potential_extents, const int* source_extents,
                            const int32_t* const* pairs, const int* pair_counts, pp_stream stream,
                            pp_tensor_potential** out) {
  return guarded([&] {
    PP_REQUIRE(out && storage_ids && potential_extents && source_extents, "NULL argument");
    auto* t = new pp_tensor_potential();
    try {
      tp_create_impl(rank, storage_ids, reinterpret_cast<const double2*>(potential), potential_extents,
                     source_extents, pairs, pair_counts, (hipStream_t)stream, t->term, true);
    } catch (...) {
      delete t;
      throw;
    }
    *out = t;
  });
}

extern "C" int pp_tp_multiply(const pp_tensor_potential* tp, double scaling, const pp_cplx* source,
                              pp_cplx* dest, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(tp && source && dest, "NULL argument");
    double2 sc = make_double2(scaling, 0.0);
    tp_run_f64(tp->term.plan, {&tp->term}, &sc, reinterpret_cast<const double2*>(source),
               reinterpret_cast<double2*>(dest), nullptr, make_double2(1.0, 0.0), true, (hipStream_t)stream);
  });
}

extern "C" int pp_tp_multiply_f32(const pp_tensor_potential* tp, float scaling, const pp_cplxf* source,
                                  pp_cplxf* dest, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(tp && source && dest, "NULL argument");
    float2 sc = make_float2(scaling, 0.f);
    tp_run_f32(tp->term.plan, {&tp->term}, &sc, reinterpret_cast<const float2*>(source),
               reinterpret_cast<float2*>(dest), nullptr, make_float2(1.f, 0.f), true, (hipStream_t)stream);
  });
}

extern "C" int pp_tp_info(const pp_tensor_potential* tp, int64_t* stream_bytes, int64_t* tuple_count,
                          int* is_real, int* inner_kind) {
  return guarded([&] {
    PP_REQUIRE(tp, "NULL plan");
    if (stream_bytes) *stream_bytes = tp->term.stream_bytes;
    if (tuple_count) *tuple_count = tp->term.plan.tuple_count;
    if (is_real) *is_real = tp->term.is_real ? 1 : 0;
    if (inner_kind) *inner_kind = tp->term.dia ? tp->term.inner_kind : -1 - tp->term.inner_kind;
  });
}

extern "C" int pp_tp_destroy(pp_tensor_potential* tp) {
  return guarded([&] { delete tp; });
}

extern "C" int pp_tensor_potential_multiply(int rank, const int* storage_ids, const pp_cplx* potential,
                                            const int* potential_extents, double scaling,
                                            const pp_cplx* source, const int* source_extents,
                                            pp_cplx* dest, const int* dest_extents,
                                            const int32_t* const* pairs, const int* pair_counts,
                                            pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(dest_extents && source_extents, "NULL extents");
    for (int r = 0; r < rank; ++r)
      PP_REQUIRE(dest_extents[r] == source_extents[r], "dest and source extents must match");
    pp_tensor_potential t;
    tp_create_impl(rank, storage_ids, reinterpret_cast<const double2*>(potential), potential_extents,
                   source_extents, pairs, pair_counts, (hipStream_t)stream, t.term, false);
    double2 sc = make_double2(scaling, 0.0);
    tp_run_f64(t.term.plan, {&t.term}, &sc, reinterpret_cast<const double2*>(source),
               reinterpret_cast<double2*>(dest), nullptr, make_double2(1.0, 0.0), true, (hipStream_t)stream);
    PP_HIP(hipStreamSynchronize((hipStream_t)stream));
  });
}

extern "C" int pp_expand_potential(int terms, int64_t p0, int64_t r_count, const double* coeffs, const double* radial,
                                   pp_cplx* out, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(coeffs && radial && out && terms > 0 && p0 > 0 && r_count > 0, "invalid expand arguments");
    expand_terms(terms, p0, r_count, coeffs, radial, reinterpret_cast<double2*>(out), 0, (hipStream_t)stream);
  });
}
