// Learned correction to the Kronecker preconditioner (no reference counterpart).
//
// Network, shared by all channel blocks c (in = 2 n^2 reals of one n x n complex block):
//   z1 = W1 x + b1 + e_c   h1 = GELU(z1)       W1: hidden x in, e: nchan x hidden
//   z2 = W2 h1 + b2        h2 = GELU(z2)       W2: hidden x hidden
//   y  = W3 h2 + b3                             W3: in x hidden
// GELU(z) = z Phi(z) (exact, erf form).  The matrix products run on BF16 MFMA
// (v_mfma_f32_16x16x32_bf16) with FP32 accumulation; x, h1, h2 and the backward signals
// enter them rounded to BF16 (round to nearest even), bias and embedding sums and the
// Adam update stay in FP32 on FP32 master weights.
//
// As a preconditioner: P(v)_c = K_c^-1 (v_c + sigma |v| y(v_c / |v|)) with the norm |v| of
// the whole vector (in flexible GMRES the first direction is r / |r|): the network
// corrects the right-hand side of the Kronecker solve, where A K^-1 is close to the
// identity, so its errors are not amplified by the stiff part of A.  Training pairs (r, d)
// with A d = r come from the plain FP64 Cayley solve; P(r) = d exactly when
// y_c = (K d - r)_c / (sigma |r|), which is the target of block c; the loss is
// sum |y - t / sigma|^2 / rows.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "pp_common.h"
#include "pp_internal.h"
#include "pp_krylov.h"
#include "pp_learned.h"
#include "pp_mixed.h"

namespace pp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes at byte offset off of the buffer behind r (range-checked: zeros past its end, so a
// masked-out lane passes kOff16 and its load needs no branch)
constexpr int kOff16 = 0x7ffffff0;  // beyond every buffer read this way (all under 2 GiB)
__device__ __forceinline__ u32x4 ld16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

static int grid_for_n(long long n) {
  long long b = (n + 255) / 256;
  return (int)std::max(1LL, std::min(b, 4096LL));
}

// ------------------------------------------------------------------------------------
// BF16 GEMM on MFMA: 64 x 64 tile per workgroup, four waves of 32 x 32, K step 64
// ------------------------------------------------------------------------------------
// The products here are small (256 x 512 x 7200 and its transposes): each workgroup runs 4 to 16
// K steps, so what bounds it is the latency of a step, not the matrix cores.  A step's operands
// are therefore loaded into registers two steps ahead (the loads of a whole step, 16 bytes each,
// in flight together) and stored into the other of two LDS buffers while the matrix cores work
// from the first: one barrier per step.
// LDS holds X(r, k) as 64 rows of 64 BF16 without padding; the 16-byte chunk c of row r sits at
// c ^ (r ^ r >> 3) & 7, so that the 16 rows of an operand read and the rows that a transposed
// store touches fall in different banks.  An operand stored with k as the slow index is
// transposed on the way: a thread loads the same 8 rows at k and k + 1 and stores 8 (k, k + 1)
// pairs.
// One K step of 32 at a time, loaded, stored and used in turn: 17.8 us per product over a training
// step's eight (256 rows, 7200 -> 512 -> 512 -> 7200); this form 8.0 us (the four long ones 17 -> 8.7 to
// 11.2, of which the 14.7 MB of FP32 gradients written take 3).  Loads behind a branch on the tile edge
// made the compiler wait for all of them at each step: 11.1 us.
constexpr int GBM = 64, GBN = 64, GBK = 64;

__device__ __forceinline__ int gswz(int r, int chunk) { return (chunk ^ r ^ (r >> 3)) & 7; }

struct GemmFrag {
  u32x4 v[2];
};

// How an operand is read (gemm_form): 16 bytes at a time; value by value through range-checked loads
// too, so that in neither form a load waits at a branch; or value by value from any address.
enum { kWide = 2, kSingle = 1, kAnyStride = 0 };

// Thread t's share of the tile rows r0..r0+63, k0..k0+63 of X(r, k) = p[r*sr + k*sk], zeros outside
// (in the range-checked forms by an offset past the range).
// KC (k contiguous): rows t / 8 and t / 8 + 32, k chunk t % 8.  Otherwise rows 8 (t % 8) .. + 7 at
// k = 2 (t / 8) and the next.
template <bool KC, int FORM>
__device__ __forceinline__ GemmFrag gemm_load(const uint16_t* __restrict__ p, long long sr, long long sk, int R, int r0,
                                              int k0, int ke, int t) {
  GemmFrag f;
  const __amdgpu_buffer_rsrc_t tile =
      rsrc(p + (FORM == kSingle ? r0 * sr + k0 * sk : KC ? (long long)r0 * sr : (long long)r0), kOff16 - 16);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = KC ? r0 + (t >> 3) + 32 * h : r0 + (t & 7) * 8;
    const int k = KC ? k0 + (t & 7) * 8 : k0 + (t >> 3) * 2 + h;
    if (FORM == kWide) {
      const int off = KC ? ((r - r0) * (int)sr + k) * 2 : (k * (int)sk + (r - r0)) * 2;
      f.v[h] = ld16(tile, r < R && k < ke ? off : kOff16);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        unsigned w[2] = {0, 0};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int rr = KC ? r : r + 2 * q + e, kk = KC ? k + 2 * q + e : k;
          const bool in = rr < R && kk < ke;
          if (FORM == kSingle) {
            const int off = ((rr - r0) * (int)sr + (kk - k0) * (int)sk) * 2;
            w[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(tile, in ? off : kOff16, 0, 0);
          } else if (in) {
            w[e] = p[(long long)rr * sr + (long long)kk * sk];
          }
        }
        f.v[h][q] = w[0] | (w[1] << 16);
      }
    }
  }
  return f;
}

// The form for an operand of R rows (k in [0, K)).  Wide where shares of eight lie inside or outside
// it as a whole and are 16-byte aligned; the range-checked forms where a tile's offsets fit the 31
// bits of a buffer offset.
static int gemm_form(const uint16_t* p, int R, int K, long long sr, long long sk) {
  if (sr < 0 || sk < 0) return kAnyStride;
  if ((reinterpret_cast<uintptr_t>(p) & 15) == 0) {
    if (sk == 1 && sr % 8 == 0 && K % 8 == 0 && 2 * (GBM * sr + K) < kOff16 - 16) return kWide;
    if (sk != 1 && sr == 1 && sk % 8 == 0 && R % 8 == 0 && 2 * (K * sk + GBM) < kOff16 - 16) return kWide;
  }
  return 2 * (GBM * sr + GBK * sk) < kOff16 - 16 ? kSingle : kAnyStride;
}

template <bool KC>
__device__ __forceinline__ void gemm_store(const GemmFrag& f, uint16_t* S, int t) {
  if (KC) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = (t >> 3) + 32 * h;
      *reinterpret_cast<u32x4*>(&S[r * GBK + gswz(r, t & 7) * 8]) = f.v[h];
    }
  } else {
    const int k = (t >> 3) * 2;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int r = (t & 7) * 8 + q;
      const unsigned lo = (q & 1) ? f.v[0][q >> 1] >> 16 : f.v[0][q >> 1] & 0xFFFFu;
      const unsigned hi = (q & 1) ? f.v[1][q >> 1] & 0xFFFF0000u : f.v[1][q >> 1] << 16;
      *reinterpret_cast<unsigned*>(&S[r * GBK + gswz(r, k >> 3) * 8 + (k & 7)]) = lo | hi;
    }
  }
}

template <bool AK, bool BK, int AF, int BF>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(int M, int N, int K, int kchunk, const uint16_t* __restrict__ a,
                                                        long long sam, long long sak, const uint16_t* __restrict__ b,
                                                        long long sbk, long long sbn, float* __restrict__ c) {
  __shared__ __align__(16) uint16_t As[2][GBM * GBK];
  __shared__ __align__(16) uint16_t Bs[2][GBN * GBK];
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous range of tiles (n fastest), so the
  // operand that a row of tiles shares comes into one L2 instead of eight
  const unsigned tiles = gridDim.x * gridDim.y, id = blockIdx.x + gridDim.x * blockIdx.y;
  const unsigned tile = (id & 7) * (tiles >> 3) + min(id & 7, tiles & 7) + (id >> 3);
  const int m0 = (int)(tile / gridDim.x) * GBM, n0 = (int)(tile % gridDim.x) * GBN;
  const int kb = blockIdx.z * kchunk;
  const int ke = min(K, kb + kchunk);
  float* cz = c + (long long)blockIdx.z * M * N;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (ke - kb + GBK - 1) / GBK;
  GemmFrag fa[2], fb[2];
  fa[0] = gemm_load<AK, AF>(a, sam, sak, M, m0, kb, ke, t);
  fb[0] = gemm_load<BK, BF>(b, sbn, sbk, N, n0, kb, ke, t);  // B viewed as (n, k)
  fa[1] = gemm_load<AK, AF>(a, sam, sak, M, m0, kb + GBK, ke, t);
  fb[1] = gemm_load<BK, BF>(b, sbn, sbk, N, n0, kb + GBK, ke, t);
  auto step = [&](int s, GemmFrag& ra, GemmFrag& rb) {
    // buffer s & 1 was last read in step s - 2; the barrier of step s - 1 lies in between
    gemm_store<AK>(ra, As[s & 1], t);
    gemm_store<BK>(rb, Bs[s & 1], t);
    // past the last step the loads are masked: issued all the same, so that the compiler knows
    // how many are in flight and waits for the older step's only
    ra = gemm_load<AK, AF>(a, sam, sak, M, m0, kb + (s + 2) * GBK, ke, t);
    rb = gemm_load<BK, BF>(b, sbn, sbk, N, n0, kb + (s + 2) * GBK, ke, t);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 av[2], bv[2];
      const int chunk = (lane >> 4) + 4 * h;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = wm * 32 + i * 16 + (lane & 15);
        av[i] = *reinterpret_cast<const bf16x8*>(&As[s & 1][r * GBK + gswz(r, chunk) * 8]);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = wn * 32 + j * 16 + (lane & 15);
        bv[j] = *reinterpret_cast<const bf16x8*>(&Bs[s & 1][r * GBK + gswz(r, chunk) * 8]);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
  };
  for (int s = 0;;) {
    step(s, fa[0], fb[0]);
    if (++s >= steps) break;
    step(s, fa[1], fb[1]);
    if (++s >= steps) break;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * 32 + i * 16 + (lane >> 4) * 4 + r;
        const int col = n0 + wn * 32 + j * 16 + (lane & 15);
        if (row < M && col < N) cz[(long long)row * N + col] = acc[i][j][r];
      }
}

int gemm_bf16(int M, int N, int K, const uint16_t* a, long long sam, long long sak, const uint16_t* b, long long sbk,
              long long sbn, float* c, int splits, hipStream_t s) {
  PP_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty operand");
  PP_REQUIRE((N + GBN - 1) / GBN < (1 << 30) && (M + GBM - 1) / GBM < 65536, "gemm: grid too large");
  splits = std::max(1, splits);
  const int kchunk = (int)ceil_div(ceil_div(K, splits), GBK) * GBK;
  const int z = (int)ceil_div(K, kchunk);
  const dim3 grid((N + GBN - 1) / GBN, (M + GBM - 1) / GBM, z);
  // Each operand by its own layout: the training of an odd number of B-splines multiplies matrices of
  // 2 n^2 columns, which cannot be read 16 bytes at a time, by matrices of the hidden width, which can:
  // 512 x 6962 x 256, A rows of 256 and B rows of 6962: 18.4 us (39.5 with both value by value behind
  // branches; 21.5 one K step of 32 at a time); 256 x 512 x 6962, rows of 6962 in both: 178 (448; 652).
  // Stored with aligned rows (6968): 177.  A training step at 59 B-splines: 184 us (266; 515).
  auto launch = [&](auto fa, auto fb) {
#define PP_GEMM(AK, BK)                                                                                           \
  hipLaunchKernelGGL((gemm_bf16_kernel<AK, BK, fa.value, fb.value>), grid, dim3(256), 0, s, M, N, K, kchunk, a, sam, \
                     sak, b, sbk, sbn, c)
    if (sak == 1 && sbk == 1) PP_GEMM(true, true);
    else if (sak == 1) PP_GEMM(true, false);
    else if (sbk == 1) PP_GEMM(false, true);
    else PP_GEMM(false, false);
#undef PP_GEMM
  };
  const int form_a = gemm_form(a, M, K, sam, sak), form_b = gemm_form(b, N, K, sbn, sbk);
  constexpr std::integral_constant<int, kWide> wide;
  constexpr std::integral_constant<int, kSingle> single;
  constexpr std::integral_constant<int, kAnyStride> any;
  if (form_a == kAnyStride || form_b == kAnyStride) launch(any, any);
  else if (form_a == kWide && form_b == kWide) launch(wide, wide);
  else if (form_a == kWide) launch(wide, single);
  else if (form_b == kWide) launch(single, wide);
  else launch(single, single);
  PP_HIP(hipGetLastError());
  return z;
}

// Split-K factor: enough workgroups for the chip (about 512), at most 32 splits and at
// least 128 of K per split (256 x 512 x 7200: 8 splits 12 us, 15 splits 10).  Skinny products (the
// inference of a few dozen channel rows)
// split most.
constexpr int kOutSplitsMax = 4;  // split-K of the output layer (its partials are rows x in)
static int pick_splits(int M, int N, int K) {
  const long long tiles = ceil_div(M, GBM) * ceil_div(N, GBN);
  int sp = (int)std::max(1LL, 512 / std::max(1LL, tiles));
  sp = std::min(sp, 32);
  sp = std::min(sp, std::max(1, K / 128));
  return sp;
}

// ------------------------------------------------------------------------------------
// elementwise pieces
// ------------------------------------------------------------------------------------
// v = sum_p parts + bias[n] (+ emb[chan[m]][n]); z_out = v; act = gelu ? GELU(v) : v;
// h_out = bf16(act); y_out = act
__global__ void bias_act_kernel(int M, int N, const float* __restrict__ parts, int nparts,
                                const float* __restrict__ bias, const float* __restrict__ emb,
                                const int* __restrict__ chan, int nchan, float* __restrict__ z_out,
                                uint16_t* __restrict__ h_out, float* __restrict__ y_out, int use_gelu) {
  const long long total = (long long)M * N;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    const int m = (int)(idx / N), n = (int)(idx % N);
    float v = 0.f;
    for (int p = 0; p < nparts; ++p) v += parts[p * total + idx];
    v += bias[n];
    if (emb) {
      const int c = chan[m];
      if (c >= 0 && c < nchan) v += emb[(long long)c * N + n];
    }
    if (z_out) z_out[idx] = v;
    const float act = use_gelu ? gelu(v) : v;
    if (h_out) h_out[idx] = f2bf(act);
    if (y_out) y_out[idx] = act;
  }
}

// d = y - t*inv_sigma ; g = 2 d / M (FP32 and BF16) ; block partials of sum d^2
__global__ __launch_bounds__(256) void loss_grad_kernel(int M, int N, const float* __restrict__ y,
                                                        const float* __restrict__ t, float inv_sigma,
                                                        float* __restrict__ gf, uint16_t* __restrict__ gh,
                                                        double2* __restrict__ partial) {
  __shared__ double sh[4];
  const long long total = (long long)M * N;
  const float sc = 2.0f / (float)M;
  double acc = 0;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    const float d = y[idx] - t[idx] * inv_sigma;
    acc += (double)d * d;
    const float g = sc * d;
    gf[idx] = g;
    gh[idx] = f2bf(g);
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(sh[0] + sh[1] + sh[2] + sh[3], 0.0);
}

// dz = (sum_p parts) * GELU'(z): FP32 and BF16
__global__ void gelu_back_kernel(int M, int N, const float* __restrict__ parts, int nparts, const float* __restrict__ z,
                                 float* __restrict__ dzf, uint16_t* __restrict__ dzh) {
  const long long total = (long long)M * N;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    float v = 0.f;
    for (int p = 0; p < nparts; ++p) v += parts[p * total + idx];
    const float d = v * gelu_grad(z[idx]);
    dzf[idx] = d;
    dzh[idx] = f2bf(d);
  }
}

// out[n] = sum_m x[m][n].  A workgroup takes 64 columns; its 16 waves share the rows (wave w:
// rows w, w + 16, ...) and their partial sums are added in wave order.  One thread per column
// over all rows was a chain of M dependent loads on 29 workgroups and fewer: 56.9 us on average over a
// training step's three (256 x 7200, which is 7.4 MB, and twice 256 x 512); this form 4.3 us.
constexpr int CSW = 16;
__global__ __launch_bounds__(64 * CSW) void colsum_kernel(int M, int N, const float* __restrict__ x,
                                                          float* __restrict__ out) {
  __shared__ float sh[CSW][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (n < N) {
#pragma unroll 8
    for (int m = wave; m < M; m += CSW) s += x[(long long)m * N + n];
  }
  sh[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && n < N) {
    for (int w = 1; w < CSW; ++w) s += sh[w][lane];
    out[n] = s;
  }
}

// out[c][n] = sum over rows m of channel c of x[m][n], in increasing m.  One wave per (64
// columns, channel): a ballot over 64 rows' channels gives the rows of c, whose values are
// loaded four at a time.  With a thread per (c, n) walking all rows the loop's branch per row
// cost 18.5 us at 256 rows x 512 columns x 42 channels; this form 3.5 us.
__global__ __launch_bounds__(64) void embgrad_kernel(int M, int N, const float* __restrict__ x,
                                                     const int* __restrict__ chan, float* __restrict__ out) {
  const int strips = (N + 63) / 64;
  const int c = blockIdx.x / strips, lane = threadIdx.x;
  const int n = (blockIdx.x - c * strips) * 64 + lane;
  const float* xn = x + min(n, N - 1);
  float s = 0.f;
  for (int m0 = 0; m0 < M; m0 += 64) {
    unsigned long long rows = __ballot(m0 + lane < M && chan[min(m0 + lane, M - 1)] == c);
    while (rows) {
      float v[4];
      bool on[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        on[q] = rows != 0;
        const int m = on[q] ? m0 + __builtin_ctzll(rows) : m0;
        rows &= rows - 1;  // stays 0 once empty
        v[q] = xn[(long long)m * N];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (on[q]) s += v[q];
    }
  }
  if (n < N) out[(long long)c * N + n] = s;
}

__global__ void to_bf16_kernel(long long n, const float* __restrict__ x, uint16_t* __restrict__ y) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

// One Adam step on n parameters (n a multiple of 2, the matrices' ranges multiples of 8), writing
// the BF16 copies of the three weight matrices as it goes.  HBM-bound: 28 bytes a parameter, four
// parameters to a thread in 16-byte accesses.  Measured on the 7.6 M parameters of 7200-512-512-7200:
// 33.4 us and 11.8 us of three conversion launches re-reading the weights, now 36.1 us in all (6.1 TB/s).
struct Bf16Copies {
  long long first[3], count[3];  // parameter ranges of W1, W2, W3
  uint16_t* to[3];
};
__global__ __launch_bounds__(256) void adam_kernel(long long n, float* __restrict__ p, const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                                   float b2, float eps, float c1, float c2, Bf16Copies w) {
  auto update = [&](float pi, float gi, float& mi, float& vi) {
    mi = b1 * mi + (1.f - b1) * gi;
    vi = b2 * vi + (1.f - b2) * gi * gi;
    return pi - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  };
  const long long quads = n / 4;
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < quads;
       q += (long long)gridDim.x * blockDim.x) {
    const long long i = 4 * q;
    const f32x4 gi = *reinterpret_cast<const f32x4*>(g + i);
    f32x4 pi = *reinterpret_cast<const f32x4*>(p + i), mi = *reinterpret_cast<const f32x4*>(m + i),
          vi = *reinterpret_cast<const f32x4*>(v + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float me = mi[e], ve = vi[e];
      pi[e] = update(pi[e], gi[e], me, ve);
      mi[e] = me;
      vi[e] = ve;
    }
    *reinterpret_cast<f32x4*>(m + i) = mi;
    *reinterpret_cast<f32x4*>(v + i) = vi;
    *reinterpret_cast<f32x4*>(p + i) = pi;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const long long o = i - w.first[k];
      if (o >= 0 && o < w.count[k])
        *reinterpret_cast<uint2*>(w.to[k] + o) = make_uint2(f2bf(pi[0]) | (unsigned)f2bf(pi[1]) << 16,
                                                            f2bf(pi[2]) | (unsigned)f2bf(pi[3]) << 16);
    }
  }
  // the last two (of the output bias)
  const long long i = 4 * quads + threadIdx.x;
  if (blockIdx.x == 0 && i < n) p[i] = update(p[i], g[i], m[i], v[i]);
}

// Norms.  One workgroup per channel block: nrm[c] = |v_c|.
template <class T2>
__global__ __launch_bounds__(256) void block_norm_kernel(int nb, const T2* __restrict__ v, double* __restrict__ nrm) {
  __shared__ double sh[4];
  const int c = blockIdx.x;
  const T2* vc = v + (long long)c * nb;
  double acc = 0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) acc += (double)vc[i].x * vc[i].x + (double)vc[i].y * vc[i].y;
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) nrm[c] = std::sqrt(sh[0] + sh[1] + sh[2] + sh[3]);
}

// nrm[nchan] = sqrt(sum_c nrm[c]^2)  (the global norm, one thread)
__global__ void global_norm_kernel(int nchan, double* __restrict__ nrm) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double s = 0;
  for (int c = 0; c < nchan; ++c) s += nrm[c] * nrm[c];
  nrm[nchan] = std::sqrt(s);
}

// x[c] = bf16(v_c / |v|) with the global norm |v| = sqrt(sum_c nrm[c]^2), summed by every
// block in the same order; block 0 also stores it in nrm[nchan] (zero vector -> 0)
__global__ void block_pack_kernel(int nchan, int nb, const float2* __restrict__ v, double* __restrict__ nrm,
                                  uint16_t* __restrict__ x) {
  double g2 = 0;
  for (int c = 0; c < nchan; ++c) g2 += nrm[c] * nrm[c];
  const double g = std::sqrt(g2);
  if (blockIdx.x == 0 && threadIdx.x == 0) nrm[nchan] = g;
  const float inv = g > 0 ? (float)(1.0 / g) : 0.f;
  const long long total = (long long)nchan * nb;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    x[2 * i] = f2bf(v[i].x * inv);
    x[2 * i + 1] = f2bf(v[i].y * inv);
  }
}


// training rows: x_c = r_c / |r|, t_c = (kd_c - r_c) / |r| (FP32) with the global |r| = nrm[nchan];
// nrm_out[c] = |r_c| / |r|
__global__ void prepare_kernel(int nchan, int nb, const double2* __restrict__ r, const double2* __restrict__ kd,
                               const double* __restrict__ nrm, float* __restrict__ x, float* __restrict__ t,
                               float* __restrict__ nrm_out) {
  const double g = nrm[nchan];
  const double inv = g > 0 ? 1.0 / g : 0.0;
  const long long total = (long long)nchan * nb;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    x[2 * i] = (float)(r[i].x * inv);
    x[2 * i + 1] = (float)(r[i].y * inv);
    t[2 * i] = (float)((kd[i].x - r[i].x) * inv);
    t[2 * i + 1] = (float)((kd[i].y - r[i].y) * inv);
    if (i < nchan) nrm_out[i] = (float)(nrm[i] * inv);
  }
}

// ------------------------------------------------------------------------------------
// Learned
// ------------------------------------------------------------------------------------
void Learned::ensure(int rows) {
  PP_REQUIRE(rows > 0, "learned: empty batch");
  if (rows <= cap) return;
  cap = rows;
  const size_t ri = (size_t)rows * in, rh = (size_t)rows * hidden;
  xh.resize(ri);
  h1h.resize(rh);
  h2h.resize(rh);
  gh.resize(ri);
  dz1h.resize(rh);
  dz2h.resize(rh);
  z1.resize(rh);
  z2.resize(rh);
  y.resize(ri);
  gf.resize(ri);
  dzf.resize(rh);
  part.resize(std::max((size_t)splits_max * rh, (size_t)kOutSplitsMax * ri));
  loss_part.resize(1024);
}

void Learned::refresh_bf16(hipStream_t s) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for_n((long long)hidden * in)), dim3(256), 0, s,
                     (long long)hidden * in, params.ptr + o_w1, w1h.ptr);
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for_n((long long)hidden * hidden)), dim3(256), 0, s,
                     (long long)hidden * hidden, params.ptr + o_w2, w2h.ptr);
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for_n((long long)in * hidden)), dim3(256), 0, s,
                     (long long)in * hidden, params.ptr + o_w3, w3h.ptr);
  PP_HIP(hipGetLastError());
}

void Learned::forward(int rows, const int* chan, hipStream_t s) {
  const long long rh = (long long)rows * hidden, ri = (long long)rows * in;
  int sp = gemm_bf16(rows, hidden, in, xh.ptr, in, 1, w1h.ptr, 1, in, part.ptr,
                     std::min(splits_max, pick_splits(rows, hidden, in)), s);
  hipLaunchKernelGGL(bias_act_kernel, dim3(grid_for_n(rh)), dim3(256), 0, s, rows, hidden, part.ptr, sp,
                     params.ptr + o_b1, params.ptr + o_emb, chan, nchan, z1.ptr, h1h.ptr, (float*)nullptr, 1);
  sp = gemm_bf16(rows, hidden, hidden, h1h.ptr, hidden, 1, w2h.ptr, 1, hidden, part.ptr,
                 std::min(splits_max, pick_splits(rows, hidden, hidden)), s);
  hipLaunchKernelGGL(bias_act_kernel, dim3(grid_for_n(rh)), dim3(256), 0, s, rows, hidden, part.ptr, sp,
                     params.ptr + o_b2, (const float*)nullptr, (const int*)nullptr, 0, z2.ptr, h2h.ptr, (float*)nullptr,
                     1);
  sp = gemm_bf16(rows, in, hidden, h2h.ptr, hidden, 1, w3h.ptr, 1, hidden, part.ptr,
                 std::min(kOutSplitsMax, pick_splits(rows, in, hidden)), s);
  hipLaunchKernelGGL(bias_act_kernel, dim3(grid_for_n(ri)), dim3(256), 0, s, rows, in, part.ptr, sp,
                     params.ptr + o_b3, (const float*)nullptr, (const int*)nullptr, 0, (float*)nullptr,
                     (uint16_t*)nullptr, y.ptr, 0);
  PP_HIP(hipGetLastError());
}

double Learned::backward(int rows, const int* chan, const float* t, hipStream_t s, bool want_loss) {
  const long long rh = (long long)rows * hidden, ri = (long long)rows * in;
  const int lb = (int)std::min<long long>(1024, std::max<long long>(1, ceil_div(ri, 256)));
  hipLaunchKernelGGL(loss_grad_kernel, dim3(lb), dim3(256), 0, s, rows, in, y.ptr, t, 1.0f / sigma, gf.ptr, gh.ptr,
                     loss_part.ptr);
  // layer 3
  gemm_bf16(in, hidden, rows, gh.ptr, 1, in, h2h.ptr, hidden, 1, grads.ptr + o_w3, 1, s);
  hipLaunchKernelGGL(colsum_kernel, dim3(ceil_div(in, 64)), dim3(64 * CSW), 0, s, rows, in, gf.ptr, grads.ptr + o_b3);
  int sp = gemm_bf16(rows, hidden, in, gh.ptr, in, 1, w3h.ptr, hidden, 1, part.ptr,
                     std::min(splits_max, pick_splits(rows, hidden, in)), s);
  hipLaunchKernelGGL(gelu_back_kernel, dim3(grid_for_n(rh)), dim3(256), 0, s, rows, hidden, part.ptr, sp, z2.ptr,
                     dzf.ptr, dz2h.ptr);
  // layer 2
  hipLaunchKernelGGL(colsum_kernel, dim3(ceil_div(hidden, 64)), dim3(64 * CSW), 0, s, rows, hidden, dzf.ptr,
                     grads.ptr + o_b2);
  gemm_bf16(hidden, hidden, rows, dz2h.ptr, 1, hidden, h1h.ptr, hidden, 1, grads.ptr + o_w2, 1, s);
  sp = gemm_bf16(rows, hidden, hidden, dz2h.ptr, hidden, 1, w2h.ptr, hidden, 1, part.ptr,
                 std::min(splits_max, pick_splits(rows, hidden, hidden)), s);
  hipLaunchKernelGGL(gelu_back_kernel, dim3(grid_for_n(rh)), dim3(256), 0, s, rows, hidden, part.ptr, sp, z1.ptr,
                     dzf.ptr, dz1h.ptr);
  // layer 1
  hipLaunchKernelGGL(colsum_kernel, dim3(ceil_div(hidden, 64)), dim3(64 * CSW), 0, s, rows, hidden, dzf.ptr,
                     grads.ptr + o_b1);
  hipLaunchKernelGGL(embgrad_kernel, dim3(ceil_div(hidden, 64) * nchan), dim3(64), 0, s, rows, hidden, dzf.ptr, chan,
                     grads.ptr + o_emb);
  gemm_bf16(hidden, in, rows, dz1h.ptr, 1, hidden, xh.ptr, in, 1, grads.ptr + o_w1, 1, s);
  PP_HIP(hipGetLastError());
  if (!want_loss) return 0.0;
  std::vector<double2> h(lb);
  PP_HIP(hipMemcpyAsync(h.data(), loss_part.ptr, lb * sizeof(double2), hipMemcpyDeviceToHost, s));
  PP_HIP(hipStreamSynchronize(s));
  double l = 0;
  for (auto& v : h) l += v.x;
  return l / rows;
}

void Learned::adam(float lr, float b1, float b2, float eps, hipStream_t s) {
  ++adam_t;
  const float c1 = 1.f - std::pow(b1, (float)adam_t), c2 = 1.f - std::pow(b2, (float)adam_t);
  const Bf16Copies w = {{o_w1, o_w2, o_w3},
                        {(long long)hidden * in, (long long)hidden * hidden, (long long)in * hidden},
                        {w1h.ptr, w2h.ptr, w3h.ptr}};
  hipLaunchKernelGGL(adam_kernel, dim3(grid_for_n((p_count + 3) / 4)), dim3(256), 0, s, p_count, params.ptr, grads.ptr,
                     adam_m.ptr, adam_v.ptr, lr, b1, b2, eps, c1, c2, w);
  PP_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// Inference: one row per channel block (rows <= 48), weights streamed once
// ------------------------------------------------------------------------------------
// The training GEMM tiles 64 x 64 outputs and splits K; with a few dozen rows most of its
// tile is padding and each weight tile is loaded for one row block.  Inference instead
// covers all rows (three 16-row MFMA tiles) in every wave, so every weight element is read
// from HBM once and used for all rows: the first layer gives each wave a 16-column strip of
// a 256-wide K slice (the normalised input staged in LDS as BF16), the two dense layers a
// quarter of K of a workgroup's strips, with the operands loaded straight into registers.
// Rounding points are those of the training forward pass: x = bf16(v_c / |v|), h1 and h2
// in BF16, y in FP32.
constexpr int IMR = 48;        // rows covered (3 x 16)
constexpr int IKC = 256;       // K range of one first-layer workgroup
constexpr int IKMAX = 640;     // K of the dense layers (hidden width) the streaming path takes

union BfPack {  // eight BF16 values as one MFMA operand
  bf16x8 v;
  uint16_t u[8];
};

constexpr int INP = 128;  // FP64 partial sums of squares behind the inference input's norm
// n2p[b] = sum of squares (FP64) over the b-th of INP equal contiguous ranges of the nf floats
// of v (nf < 2^29).  Each pass of a thread issues its four 16-byte loads before summing them in
// order; the range ends (nf, or v not 16-byte aligned) are summed value by value.
__global__ __launch_bounds__(256) void norm_part_kernel(long long nf, const float* __restrict__ v,
                                                        double* __restrict__ n2p) {
  __shared__ double sh[4];
  const int t = threadIdx.x;
  const int chunk = (int)(((nf + INP - 1) / INP + 3) / 4 * 4);
  const int lo = (int)blockIdx.x * chunk, hi = (int)min(nf, (long long)lo + chunk);
  double acc = 0;
  if ((reinterpret_cast<uintptr_t>(v) & 15) == 0) {
    const __amdgpu_buffer_rsrc_t vr = rsrc(v, nf * 4);
    const int hv = lo + max(0, hi - lo) / 4 * 4;  // end of the whole 16-byte groups
    for (int base = lo; base < hv; base += 4096) {
      u32x4 q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = base + (t + u * 256) * 4;
        q[u] = ld16(vr, i < hv ? i * 4 : kOff16);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 x = __builtin_bit_cast(float4, q[u]);
        acc += (double)x.x * x.x + (double)x.y * x.y + (double)x.z * x.z + (double)x.w * x.w;
      }
    }
    if (hv + t < hi) acc += (double)v[hv + t] * v[hv + t];
  } else {
    for (int i = lo + t; i < hi; i += 256) acc += (double)v[i] * v[i];
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((t & 63) == 0) sh[t >> 6] = acc;
  __syncthreads();
  if (t == 0) n2p[blockIdx.x] = ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

// part[slice][m][n] = sum_{k in slice} bf16(v[m][k] / |v|) W1[n][k]   (v: rows x K floats,
// K a multiple of 8, v 16-byte aligned, v and W1 under 2 GiB).  A wave issues its W1 operands first (they wait for
// nothing), then the norm partials and its share of v; |v| = sqrt(sum n2p) is summed by every
// wave in the same order, and workgroup (0, 0) stores it in gout[0].
__global__ __launch_bounds__(256) void infer_l1_kernel(int M, int N, int K, const float* __restrict__ v,
                                                       const double* __restrict__ n2p, double* __restrict__ gout,
                                                       const uint16_t* __restrict__ w, float* __restrict__ part) {
  __shared__ __align__(16) uint16_t As[IMR * (IKC + 8)];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int k0 = blockIdx.y * IKC;
  const int kn = min(IKC, K - k0);  // a multiple of 8
  const int col = (blockIdx.x * 4 + wave) * 16 + (lane & 15);
  constexpr int KS = IKC / 32;
  const __amdgpu_buffer_rsrc_t wr = rsrc(w, (long long)N * K * 2), vr = rsrc(v, (long long)M * K * 4);
  u32x4 b[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int kq = s * 32 + (lane >> 4) * 8;
    b[s] = ld16(wr, col < N && kq < kn ? (col * K + k0 + kq) * 2 : kOff16);
  }
  static_assert(INP == 128, "two norm partials per lane");
  const double p0 = n2p[lane], p1 = n2p[lane + 64];
  // v in groups of 8 consecutive values (two 16-byte loads), 6 groups per thread
  constexpr int GROUPS = IMR * IKC / 8 / 256;
  u32x4 vq[GROUPS][2];
#pragma unroll
  for (int q = 0; q < GROUPS; ++q) {
    const int gidx = t + q * 256, m = gidx / (IKC / 8), kk = (gidx % (IKC / 8)) * 8;
    const int off = m < M && kk < kn ? (m * K + k0 + kk) * 4 : kOff16;
    vq[q][0] = ld16(vr, off);
    vq[q][1] = ld16(vr, off == kOff16 ? kOff16 : off + 16);
  }
  __builtin_amdgcn_sched_barrier(0);  // every load above in flight before the norm is summed
  double g2 = p0 + p1;
  for (int off = 32; off > 0; off >>= 1) g2 += __shfl_down(g2, off, 64);
  const double g = std::sqrt(__shfl(g2, 0, 64));
  const float inv = g > 0 ? (float)(1.0 / g) : 0.f;
  if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) gout[0] = g;  // read by the Kronecker combination
#pragma unroll
  for (int q = 0; q < GROUPS; ++q) {
    const int gidx = t + q * 256, m = gidx / (IKC / 8), kk = (gidx % (IKC / 8)) * 8;
    const float4 lo = __builtin_bit_cast(float4, vq[q][0]), hi = __builtin_bit_cast(float4, vq[q][1]);
    BfPack pk;
    pk.u[0] = f2bf(lo.x * inv);
    pk.u[1] = f2bf(lo.y * inv);
    pk.u[2] = f2bf(lo.z * inv);
    pk.u[3] = f2bf(lo.w * inv);
    pk.u[4] = f2bf(hi.x * inv);
    pk.u[5] = f2bf(hi.y * inv);
    pk.u[6] = f2bf(hi.z * inv);
    pk.u[7] = f2bf(hi.w * inv);
    *reinterpret_cast<bf16x8*>(&As[m * (IKC + 8) + kk]) = pk.v;
  }
  __syncthreads();
  f32x4 acc[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (s * 32 >= kn) break;
    const int kq = s * 32 + (lane >> 4) * 8;
    const bf16x8 bv = __builtin_bit_cast(bf16x8, b[s]);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const bf16x8 av = *reinterpret_cast<const bf16x8*>(&As[(r * 16 + (lane & 15)) * (IKC + 8) + kq]);
      acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[r], 0, 0, 0);
    }
  }
  float* out = part + (long long)blockIdx.y * M * N;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = r * 16 + (lane >> 4) * 4 + q;
      if (row < M && col < N) out[(long long)row * N + col] = acc[r][q];
    }
}

// h[m][n] = bf16(GELU(sum_slices part + b[n] + emb[m][n]))  (the training bias_act order)
__global__ void infer_act1_kernel(int M, int N, int slices, const float* __restrict__ part,
                                  const float* __restrict__ bias, const float* __restrict__ emb,
                                  uint16_t* __restrict__ h) {
  const int total = M * N;
  for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += gridDim.x * blockDim.x) {
    const int n = idx % N;
    float v = 0.f;
#pragma unroll 8
    for (int p = 0; p < slices; ++p) v += part[(long long)p * total + idx];
    v += bias[n];
    v += emb[idx];  // row m is channel m
    h[idx] = f2bf(gelu(v));
  }
}

// out[m][n] = act(sum_k A[m][k] W[n][k] + b[n]) for rows <= 48 and K <= 128 S (a multiple of
// 8; A, W and out under 2 GiB).  A workgroup owns NS 16-column strips; its four waves split K, each over at most S
// 32-wide steps, and load their MFMA operands (A rows and W columns, 16 bytes per lane and
// step) straight from memory, all before the first MFMA.  The four partial tiles are added
// through LDS in wave order.  GELU_BF16: bf16(GELU(.)) into hout, else the FP32 value into fout.
constexpr int ISMAX = (IKMAX / 32 + 3) / 4;  // K steps of one wave at K = IKMAX
template <bool GELU_BF16, int NS, int S>
__global__ __launch_bounds__(256) void infer_layer_kernel(int M, int N, int K, const uint16_t* __restrict__ a,
                                                          const uint16_t* __restrict__ w,
                                                          const float* __restrict__ bias,
                                                          uint16_t* __restrict__ hout, float* __restrict__ fout) {
  __shared__ f32x4 red[3][3 * NS][64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int s0 = wave * S, nsteps = (K + 31) / 32;
  const int n0 = blockIdx.x * 16 * NS;
  u32x4 av[S][3], bv[S][NS];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int kq = (s0 + s) * 32 + (lane >> 4) * 8;
    const bool kok = kq < K;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int row = r * 16 + (lane & 15);
      const bool ok = kok && row < M;
      const u32x4 x = *reinterpret_cast<const u32x4*>(ok ? a + (long long)row * K + kq : a);
      av[s][r] = ok ? x : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int col = n0 + j * 16 + (lane & 15);
      const bool ok = kok && col < N;
      const u32x4 x = *reinterpret_cast<const u32x4*>(ok ? w + (long long)col * K + kq : w);
      bv[s][j] = ok ? x : u32x4{0u, 0u, 0u, 0u};
    }
  }
  f32x4 acc[3][NS];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int j = 0; j < NS; ++j) acc[r][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (s0 + s >= nsteps) break;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int j = 0; j < NS; ++j)
        acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[s][r]),
                                                            __builtin_bit_cast(bf16x8, bv[s][j]), acc[r][j], 0, 0, 0);
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int j = 0; j < NS; ++j) red[wave - 1][r * NS + j][lane] = acc[r][j];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int j = 0; j < NS; ++j) acc[r][j] += red[p][r * NS + j][lane];
  // range-checked buffer stores: a masked-out value goes to an offset past the end and is
  // dropped, so no store waits behind a branch
  constexpr int esz = GELU_BF16 ? 2 : 4;
  const __amdgpu_buffer_rsrc_t orr = rsrc(GELU_BF16 ? (const void*)hout : (const void*)fout, (long long)M * N * esz);
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int col = n0 + j * 16 + (lane & 15);
    const float bn = bias[min(col, N - 1)];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = r * 16 + (lane >> 4) * 4 + q;
        const int off = row < M && col < N ? (row * N + col) * esz : kOff16;
        const float v = acc[r][j][q] + bn;
        if (GELU_BF16) __builtin_amdgcn_raw_buffer_store_b16(f2bf(gelu(v)), orr, off, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), orr, off, 0, 0);
      }
  }
}

template <bool GELU_BF16, int NS>
static void launch_infer_layer(int M, int N, int K, const uint16_t* a, const uint16_t* w, const float* bias,
                               uint16_t* hout, float* fout, hipStream_t s) {
  const int steps = (int)ceil_div((K + 31) / 32, 4);
  const dim3 grid((unsigned)ceil_div(N, 16 * NS));
  switch (steps) {
#define PP_INFER_LAYER(S)                                                                                        \
  case S:                                                                                                        \
    hipLaunchKernelGGL((infer_layer_kernel<GELU_BF16, NS, S>), grid, dim3(256), 0, s, M, N, K, a, w, bias, hout, \
                       fout);                                                                                    \
    break;
    PP_INFER_LAYER(1)
    PP_INFER_LAYER(2)
    PP_INFER_LAYER(3)
    PP_INFER_LAYER(4)
    PP_INFER_LAYER(5)
#undef PP_INFER_LAYER
    default: PP_REQUIRE(false, "learned inference: hidden width above the streaming limit");
  }
  static_assert(ISMAX == 5, "the dispatch covers 1 .. ISMAX steps per wave");
}

// y (rows = channels) from v: the norm partials, then the streaming kernels above
static void infer_streaming(Learned& L, const float2* in, hipStream_t s) {
  const int M = L.nchan, H = L.hidden, I = L.in;
  const int slices = (int)ceil_div(I, IKC);
  PP_REQUIRE((size_t)slices * M * H <= L.part.count, "learned: partial buffer too small");
  hipLaunchKernelGGL(norm_part_kernel, dim3(INP), dim3(256), 0, s, (long long)M * I,
                     reinterpret_cast<const float*>(in), L.n2p.ptr);
  hipLaunchKernelGGL(infer_l1_kernel, dim3((unsigned)ceil_div(H, 64), slices), dim3(256), 0, s, M, H, I,
                     reinterpret_cast<const float*>(in), L.n2p.ptr, L.nrm.ptr + M, L.w1h.ptr, L.part.ptr);
  hipLaunchKernelGGL(infer_act1_kernel, dim3((unsigned)ceil_div((long long)M * H, 256)), dim3(256), 0, s, M, H, slices,
                     L.part.ptr, L.params.ptr + L.o_b1, L.params.ptr + L.o_emb, L.h1h.ptr);
  launch_infer_layer<true, 1>(M, H, H, L.h1h.ptr, L.w2h.ptr, L.params.ptr + L.o_b2, L.h2h.ptr, nullptr, s);
  launch_infer_layer<false, 2>(M, I, H, L.h2h.ptr, L.w3h.ptr, L.params.ptr + L.o_b3, nullptr, L.y.ptr, s);
  PP_HIP(hipGetLastError());
}

void learned_apply(Learned& L, const Kron& K, double2 a, const float2* in, float2* out, hipStream_t s, float2* sz) {
  PP_REQUIRE(K.nchan == L.nchan && K.n == L.n, "learned preconditioner and Kronecker shapes differ");
  const int nb = L.n * L.n;
  L.ensure(L.nchan);
  const long long n = (long long)L.nchan * nb;
  if (L.nchan <= IMR && L.hidden <= IKMAX && L.hidden % 8 == 0 && L.in % 8 == 0 &&
      (reinterpret_cast<uintptr_t>(in) & 15) == 0 && (long long)L.in * std::max(L.nchan, L.hidden) * 4 < (1LL << 31)) {
    infer_streaming(L, in, s);
  } else {
    hipLaunchKernelGGL((block_norm_kernel<float2>), dim3(L.nchan), dim3(256), 0, s, nb, in, L.nrm.ptr);
    hipLaunchKernelGGL(block_pack_kernel, dim3(grid_for_n(n)), dim3(256), 0, s, L.nchan, nb, in, L.nrm.ptr, L.xh.ptr);
    L.forward(L.nchan, L.iota.ptr, s);
  }
  // out = K^-1 (in + sigma |v| y): the combination is formed as the Kronecker solve loads its input
  K.apply32_add(a, in, reinterpret_cast<const float2*>(L.y.ptr), L.nrm.ptr + L.nchan, L.sigma, out, s, sz);
  PP_HIP(hipGetLastError());
}

}  // namespace pp

// ------------------------------------------------------------------------------------
// C-ABI
// ------------------------------------------------------------------------------------
using namespace pp;

extern "C" int pp_learned_create(int nchan, int n, int hidden, unsigned long long seed, pp_learned** out) {
  return guarded([&] {
    PP_REQUIRE(out && nchan > 0 && n > 0 && hidden > 0 && hidden % 8 == 0, "invalid learned-network shape");
    auto* p = new pp_learned();
    Learned& L = p->L;
    L.nchan = nchan;
    L.n = n;
    L.in = 2 * n * n;
    L.hidden = hidden;
    long long o = 0;
    L.o_w1 = o; o += (long long)hidden * L.in;
    L.o_b1 = o; o += hidden;
    L.o_emb = o; o += (long long)nchan * hidden;
    L.o_w2 = o; o += (long long)hidden * hidden;
    L.o_b2 = o; o += hidden;
    L.o_w3 = o; o += (long long)L.in * hidden;
    L.o_b3 = o; o += L.in;
    L.p_count = o;
    // deterministic initialisation: W1, W2 uniform in +-1/sqrt(fan_in); W3, biases, embedding zero
    std::vector<float> h(o, 0.f);
    unsigned long long st = seed ^ 0x9E3779B97F4A7C15ULL;
    auto uni = [&]() {
      st += 0x9E3779B97F4A7C15ULL;
      unsigned long long z = st;
      z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
      z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
      z ^= z >> 31;
      return (double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
    };
    const double s1 = 1.0 / std::sqrt((double)L.in), s2 = 1.0 / std::sqrt((double)hidden);
    for (long long i = 0; i < (long long)hidden * L.in; ++i) h[L.o_w1 + i] = (float)(s1 * uni());
    for (long long i = 0; i < (long long)hidden * hidden; ++i) h[L.o_w2 + i] = (float)(s2 * uni());
    hipStream_t s = nullptr;
    L.params.upload(h.data(), h.size(), s);
    std::vector<float> zero(o, 0.f);
    L.grads.upload(zero.data(), zero.size(), s);
    L.adam_m.upload(zero.data(), zero.size(), s);
    L.adam_v.upload(zero.data(), zero.size(), s);
    L.w1h.resize((size_t)hidden * L.in);
    L.w2h.resize((size_t)hidden * hidden);
    L.w3h.resize((size_t)L.in * hidden);
    std::vector<int> iota(nchan);
    for (int c = 0; c < nchan; ++c) iota[c] = c;
    L.iota.upload(iota.data(), iota.size(), s);
    L.nrm.resize(nchan + 1);
    L.n2p.resize(INP);
    L.refresh_bf16(s);
    PP_HIP(hipStreamSynchronize(s));
    *out = p;
  });
}

extern "C" int pp_learned_destroy(pp_learned* l) {
  return guarded([&] { delete l; });
}

extern "C" int pp_learned_param_count(const pp_learned* l, long long* count) {
  return guarded([&] {
    PP_REQUIRE(l && count, "null argument");
    *count = l->L.p_count;
  });
}

extern "C" int pp_learned_get_params(const pp_learned* l, float* host) {
  return guarded([&] {
    PP_REQUIRE(l && host, "null argument");
    PP_HIP(hipMemcpy(host, l->L.params.ptr, l->L.p_count * sizeof(float), hipMemcpyDeviceToHost));
  });
}

extern "C" int pp_learned_set_params(pp_learned* l, const float* host) {
  return guarded([&] {
    PP_REQUIRE(l && host, "null argument");
    PP_HIP(hipMemcpy(l->L.params.ptr, host, l->L.p_count * sizeof(float), hipMemcpyHostToDevice));
    l->L.refresh_bf16(nullptr);
    PP_HIP(hipDeviceSynchronize());
  });
}

extern "C" int pp_learned_get_grads(const pp_learned* l, float* host) {
  return guarded([&] {
    PP_REQUIRE(l && host, "null argument");
    PP_HIP(hipMemcpy(host, l->L.grads.ptr, l->L.p_count * sizeof(float), hipMemcpyDeviceToHost));
  });
}

extern "C" int pp_learned_set_scale(pp_learned* l, float sigma) {
  return guarded([&] {
    PP_REQUIRE(l && sigma > 0, "invalid output scale");
    l->L.sigma = sigma;
  });
}

static void load_rows(Learned& L, int rows, const float* x, hipStream_t s) {
  L.ensure(rows);
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for_n((long long)rows * L.in)), dim3(256), 0, s,
                     (long long)rows * L.in, x, L.xh.ptr);
}

extern "C" int pp_learned_forward(pp_learned* l, int rows, const float* x, const int* chan, float* y,
                                  pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(l && x && chan && y && rows > 0, "invalid argument");
    Learned& L = l->L;
    hipStream_t s = (hipStream_t)stream;
    load_rows(L, rows, x, s);
    L.forward(rows, chan, s);
    PP_HIP(hipMemcpyAsync(y, L.y.ptr, (size_t)rows * L.in * sizeof(float), hipMemcpyDeviceToDevice, s));
  });
}

extern "C" int pp_learned_gradient(pp_learned* l, int rows, const float* x, const int* chan, const float* t,
                                   double* loss, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(l && x && chan && t && rows > 0, "invalid argument");
    Learned& L = l->L;
    hipStream_t s = (hipStream_t)stream;
    load_rows(L, rows, x, s);
    L.forward(rows, chan, s);
    const double v = L.backward(rows, chan, t, s, loss != nullptr);
    if (loss) *loss = v;
  });
}

extern "C" int pp_learned_train_step(pp_learned* l, int rows, const float* x, const int* chan, const float* t,
                                     float lr, double* loss, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(l && x && chan && t && rows > 0 && lr > 0, "invalid argument");
    Learned& L = l->L;
    hipStream_t s = (hipStream_t)stream;
    load_rows(L, rows, x, s);
    L.forward(rows, chan, s);
    const double v = L.backward(rows, chan, t, s, loss != nullptr);
    L.adam(lr, 0.9f, 0.999f, 1e-8f, s);
    if (loss) *loss = v;
  });
}

extern "C" int pp_learned_prepare(pp_learned* l, const pp_kron* k, double dt, const pp_cplx* r, const pp_cplx* d,
                                  float* x_out, float* t_out, float* nrm_out, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(l && k && r && d && x_out && t_out && nrm_out, "null argument");
    Learned& L = l->L;
    PP_REQUIRE(k->k.nchan == L.nchan && k->k.n == L.n, "Kronecker and network shapes differ");
    hipStream_t s = (hipStream_t)stream;
    const long long n = (long long)L.nchan * L.n * L.n;
    if (L.tmp64.count < (size_t)n) L.tmp64.resize(n);
    PP_HIP(hipMemcpyAsync(L.tmp64.ptr, d, n * sizeof(double2), hipMemcpyDeviceToDevice, s));
    k->k.multiply64(make_double2(0.0, 0.5 * dt), L.tmp64.ptr, s);
    const double2* rr = reinterpret_cast<const double2*>(r);
    hipLaunchKernelGGL((block_norm_kernel<double2>), dim3(L.nchan), dim3(256), 0, s, L.n * L.n, rr, L.nrm.ptr);
    hipLaunchKernelGGL(global_norm_kernel, dim3(1), dim3(64), 0, s, L.nchan, L.nrm.ptr);
    hipLaunchKernelGGL(prepare_kernel, dim3(grid_for_n(n)), dim3(256), 0, s, L.nchan, L.n * L.n, rr, L.tmp64.ptr,
                       L.nrm.ptr, x_out, t_out, nrm_out);
    PP_HIP(hipGetLastError());
  });
}

extern "C" int pp_learned_apply(pp_learned* l, const pp_kron* k, double dt, const pp_cplxf* in, pp_cplxf* out,
                                pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(l && k && in && out, "null argument");
    learned_apply(l->L, k->k, make_double2(0.0, 0.5 * dt), reinterpret_cast<const float2*>(in),
                  reinterpret_cast<float2*>(out), (hipStream_t)stream);
  });
}

extern "C" int pp_gemm_bf16(int M, int N, int K, const uint16_t* a, long long sam, long long sak, const uint16_t* b,
                            long long sbk, long long sbn, float* c, pp_stream stream) {
  return guarded([&] {
    PP_REQUIRE(a && b && c, "null argument");
    gemm_bf16(M, N, K, a, sam, sak, b, sbk, sbn, c, 1, (hipStream_t)stream);
  });
}
