// MLX-affine quantize / dequantize of a [rows, cols] fp32 matrix
// (mlx_quantize / mlx_dequantize, mlx-rs/src/ops/quantization.rs:50-83,124-158; format
// statement :31-47,85-87; shapes pinned by the reference test :298-315).
//
// One thread takes eight consecutive values; the lanes that share a quantisation group (group_size / 8 of
// them) exchange the group's min and max.  Every step is a correctly rounded fp32 operation in the same order as
// the host-side checker, so codes, scales and biases agree with it bit for bit.
#include <type_traits>

#include "common.hpp"
#include "dense_rule.hpp"

namespace mi_moe {

// Element types of activations, scales and biases (mi_moe_dtype of the C ABI).  fp16 goes through the
// hardware's round-to-nearest-even conversion, bf16 through the integer rounding every other kernel
// here uses.
template <class T> struct Elem;
template <> struct Elem<uint16_t> {  // bfloat16, raw bits
  static __device__ __forceinline__ float load(const uint16_t *p) { return bf16_to_f32(*p); }
  static __device__ __forceinline__ void store(uint16_t *p, float v) { *p = f32_to_bf16(v); }
};
template <> struct Elem<_Float16> {
  static __device__ __forceinline__ float load(const _Float16 *p) { return (float)*p; }
  static __device__ __forceinline__ void store(_Float16 *p, float v) { *p = (_Float16)v; }
};
template <> struct Elem<float> {
  static __device__ __forceinline__ float load(const float *p) { return *p; }
  static __device__ __forceinline__ void store(float *p, float v) { *p = v; }
};

// Eight consecutive values of one element type: one 16-byte access (two for float).  No address needs more than the
// alignment of its elements: global memory takes such accesses anywhere, and the compiler is told nothing else.
template <class O>
__device__ __forceinline__ void store8(O *p, const float (&v)[8]) {
  O o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) Elem<O>::store(o + j, v[j]);
  __builtin_memcpy(p, o, sizeof o);
}
// The codes of eight consecutive values: half a word, one word or two.
template <int BITS> struct Codes8;
template <> struct Codes8<2> { typedef uint16_t type; };
template <> struct Codes8<4> { typedef uint32_t type; };
template <> struct Codes8<8> { typedef uint64_t type; };
// the codes of octet i: q is aligned for its words
template <int BITS>
__device__ __forceinline__ typename Codes8<BITS>::type load_codes(const uint32_t *q, int64_t i) {
  typename Codes8<BITS>::type c;
  __builtin_memcpy(&c, reinterpret_cast<const unsigned char *>(q) + i * BITS, BITS);
  return c;
}
template <int BITS>
__device__ __forceinline__ void store_codes(uint32_t *q, int64_t i, typename Codes8<BITS>::type c) {
  __builtin_memcpy(reinterpret_cast<unsigned char *>(q) + i * BITS, &c, BITS);
}

// Groups are runs of the flat array (columns are a multiple of the group), so the matrix is one stream of
// values.  A thread takes eight of them: two 16-byte loads, and the 4, 8 or 16 lanes of a group sit in one
// row of 16 lanes, where the minimum and maximum come through DPP.  Bound by memory.  Measured at 98304 x 2048,
// 4-bit groups of 64 to bfloat16 (918 MB): 203 us by the profiler = 4.5 TB/s (a thread per packed word, eight 4-byte loads 32
// bytes apart: 474 us); quantised and dequantised in the time of the calls 287 us = 5.0 TB/s, where a large copy reaches 5.2.
template <class T, int BITS, int GROUP>
__global__ __launch_bounds__(256) void quantize_kernel(const float *__restrict__ w, int64_t n_octets,
                                                       uint32_t *__restrict__ q,
                                                       T *__restrict__ scales, T *__restrict__ biases) {
#pragma clang fp contract(off)
  constexpr int LANES = GROUP / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool on = i < n_octets;
  float v[8];
  __builtin_memcpy(v, w + 8 * (on ? i : n_octets - 1), sizeof v);  // (keep every lane in the exchanges)
  float w_min = INFINITY, w_max = -INFINITY;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    w_min = fminf(w_min, v[j]);
    w_max = fmaxf(w_max, v[j]);
  }
  auto join = [&](auto ctrl) __attribute__((always_inline)) {
    constexpr int CTRL = decltype(ctrl)::value;
    w_min = fminf(w_min, __uint_as_float(dpp_u32<CTRL>(__float_as_uint(w_min))));
    w_max = fmaxf(w_max, __uint_as_float(dpp_u32<CTRL>(__float_as_uint(w_max))));
  };
  join(std::integral_constant<int, kDppXor1>{});
  join(std::integral_constant<int, kDppXor2>{});
  if constexpr (LANES >= 8) join(std::integral_constant<int, kDppHalfMirror>{});
  if constexpr (LANES == 16) join(std::integral_constant<int, kDppMirror>{});
  constexpr float n_bins = (float)((1 << BITS) - 1);
  const bool mask = fabsf(w_min) > fabsf(w_max);
  float scale = fmaxf((w_max - w_min) / n_bins, 1e-7f);
  scale = mask ? scale : -scale;
  const float edge = mask ? w_min : w_max;
  const float q0 = __builtin_rintf(edge / scale);
  float bias = 0.0f;
  if (q0 != 0.0f) {
    scale = edge / q0;
    bias = edge;
  }
  typename Codes8<BITS>::type codes = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float c = __builtin_rintf((v[j] - bias) / scale);
    c = fminf(fmaxf(c, 0.0f), n_bins);
    codes |= (typename Codes8<BITS>::type)((typename Codes8<BITS>::type)(uint32_t)c << (j * BITS));
  }
  if (on) {
    store_codes<BITS>(q, i, codes);
    if (i % LANES == 0) {  // the codes come from the fp32 scale and bias; these are cast afterwards
      Elem<T>::store(scales + i / LANES, scale);
      Elem<T>::store(biases + i / LANES, bias);
    }
  }
}

// O: element type of the result (float, or the type of scales and biases: what mlx_dequantize returns).  A
// thread writes eight values with one or two 16-byte stores; bound by the bytes written.  Measured at
// 98304 x 2048, 4-bit groups of 64 to bfloat16 (516 MB): 114 us = 4.5 TB/s (eight 2-byte stores a thread: 245 us).
template <class T, class O, int BITS>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint32_t *__restrict__ q,
                                                         const T *__restrict__ scales,
                                                         const T *__restrict__ biases, int64_t n_octets,
                                                         int lanes_log2, O *__restrict__ out) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_octets) return;
  const int64_t g = i >> lanes_log2;
  const typename Codes8<BITS>::type codes = load_codes<BITS>(q, i);
  const float s = Elem<T>::load(scales + g), b = Elem<T>::load(biases + g);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = s * (float)(uint32_t)((codes >> (j * BITS)) & ((1u << BITS) - 1u)) + b;  // two fp32 roundings (contraction is off), then O's
  store8(out + i * 8, v);
}

constexpr int64_t kOctetsMost = (int64_t)1 << 31;  // of one launch, which takes fewer than 2^32 threads: a whole number of groups

template <class T, int BITS>
static void start_quantize(const float *w, int64_t n_octets, int group, uint32_t *q, void *s, void *b, hipStream_t st) {
  T *sc = static_cast<T *>(s), *bi = static_cast<T *>(b);
  for (int64_t n; n_octets > 0; n_octets -= n, w += 8 * n, q += n * BITS / 4, sc += 8 * n / group, bi += 8 * n / group) {
    n = n_octets < kOctetsMost ? n_octets : kOctetsMost;
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (group == 32) quantize_kernel<T, BITS, 32><<<grid, 256, 0, st>>>(w, n, q, sc, bi);
    else if (group == 64) quantize_kernel<T, BITS, 64><<<grid, 256, 0, st>>>(w, n, q, sc, bi);
    else quantize_kernel<T, BITS, 128><<<grid, 256, 0, st>>>(w, n, q, sc, bi);
  }
}

template <class T, class O>
static void start_dequantize(const uint32_t *q, const void *s, const void *b, int64_t n_octets, int group, int bits,
                             void *out, hipStream_t st) {
  const int lanes_log2 = group == 32 ? 2 : (group == 64 ? 3 : 4);
  const T *sc = static_cast<const T *>(s), *bi = static_cast<const T *>(b);
  O *o = static_cast<O *>(out);
  for (int64_t n; n_octets > 0; n_octets -= n, q += n * bits / 4, sc += 8 * n / group, bi += 8 * n / group, o += 8 * n) {
    n = n_octets < kOctetsMost ? n_octets : kOctetsMost;
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (bits == 2) dequantize_kernel<T, O, 2><<<grid, 256, 0, st>>>(q, sc, bi, n, lanes_log2, o);
    else if (bits == 4) dequantize_kernel<T, O, 4><<<grid, 256, 0, st>>>(q, sc, bi, n, lanes_log2, o);
    else dequantize_kernel<T, O, 8><<<grid, 256, 0, st>>>(q, sc, bi, n, lanes_log2, o);
  }
}

// dt: 0 bf16, 1 fp16, 2 fp32 (mi_moe_dtype)
hipError_t launch_quantize(const float *w, int64_t rows, int64_t cols, int group, int bits,
                           uint32_t *q, void *s, void *b, int dt, hipStream_t st) {
  const int64_t n = rows * cols / 8;  // columns are a multiple of the group
  if (n == 0) return hipSuccess;
  auto start = [&](auto elem) {
    typedef decltype(elem) T;
    if (bits == 2) start_quantize<T, 2>(w, n, group, q, s, b, st);
    else if (bits == 4) start_quantize<T, 4>(w, n, group, q, s, b, st);
    else start_quantize<T, 8>(w, n, group, q, s, b, st);
  };
  if (dt == 0) start(uint16_t{});
  else if (dt == 1) start(_Float16{});
  else start(float{});
  return hipGetLastError();
}

// native_out: the result has the element type of scales and biases (dt); otherwise float
hipError_t launch_dequantize(const uint32_t *q, const void *s, const void *b,
                             int64_t rows, int64_t cols, int group, int bits, void *out, int dt, bool native_out,
                             hipStream_t st) {
  const int64_t n = rows * cols / 8;
  if (n == 0) return hipSuccess;
  if (dt == 0 && native_out) start_dequantize<uint16_t, uint16_t>(q, s, b, n, group, bits, out, st);
  else if (dt == 0) start_dequantize<uint16_t, float>(q, s, b, n, group, bits, out, st);
  else if (dt == 1 && native_out) start_dequantize<_Float16, _Float16>(q, s, b, n, group, bits, out, st);
  else if (dt == 1) start_dequantize<_Float16, float>(q, s, b, n, group, bits, out, st);
  else start_dequantize<float, float>(q, s, b, n, group, bits, out, st);
  return hipGetLastError();
}

// y[m][n] += bias[n], one rounding to T: the add that follows the product in a linear layer with a bias
// (mlx-rs/src/nn/quantized.rs:363-386: quantized_matmul, then add, each rounded to the element type)
template <class T>
__global__ __launch_bounds__(256) void add_row_bias_kernel(T *__restrict__ y, const T *__restrict__ bias, int64_t n, int N) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  Elem<T>::store(y + i, Elem<T>::load(y + i) + Elem<T>::load(bias + i % N));
}

hipError_t launch_add_row_bias(void *y, const void *bias, int64_t M, int N, int dt, hipStream_t st) {
  const int64_t n = M * N;
  if (n == 0) return hipSuccess;
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (dt == 0) add_row_bias_kernel<uint16_t><<<grid, 256, 0, st>>>((uint16_t *)y, (const uint16_t *)bias, n, N);
  else if (dt == 1) add_row_bias_kernel<_Float16><<<grid, 256, 0, st>>>((_Float16 *)y, (const _Float16 *)bias, n, N);
  else add_row_bias_kernel<float><<<grid, 256, 0, st>>>((float *)y, (const float *)bias, n, N);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Plain quantized products: every combination the tuned kernels do not take -- activations, scales
// and biases in fp32 or fp16 (mlx_quantized_matmul and mlx_gather_qmm accept any floating type; the
// reference's own tests run them in fp32, mlx-rs/src/ops/quantization.rs:318-423), group sizes 32 and
// 128, 2-bit codes, and the untransposed weight layout (transpose = false, the default of
// ops::quantized_matmul, :91-122).  Correct and simple, not tuned: fp32 accumulation, weights
// dequantised as fma(scale, q, bias) in fp32, one rounding to the output type.
//
// Output row r = j * M + m (j: index pair, m: row of the M x K matrix):
//   expert e = rhs[rhs_map ? rhs_map[j] : j] (0 without rhs), x row = (lhs ? lhs[j] : j) * M + m,
//   destination row = dst_map ? dst_map[r] : r.
struct PlainMaps {
  const uint32_t *lhs, *rhs, *rhs_map, *dst_map;
  uint32_t n_lhs, n_rhs;  // matrices behind lhs / rhs (0 = unknown): indices beyond are clamped, never followed
};

__device__ __forceinline__ int64_t clamped_index(uint32_t v, uint32_t n) { return n && v >= n ? n - 1u : v; }

// transpose = true: w [E, N, K*bits/32], scales / biases [E, N, K/group].  One wave per output
// element, lanes over the packed words of the weight row, sum over the lanes in a fixed order.
template <class T, int BITS>
__global__ __launch_bounds__(256) void qmm_plain_t_kernel(const T *__restrict__ x, const uint32_t *__restrict__ w,
                                                          const T *__restrict__ scales, const T *__restrict__ biases,
                                                          PlainMaps mp, int M, int N, int K, int group,
                                                          T *__restrict__ y) {
  constexpr int CPW = 32 / BITS;
  const int64_t r = blockIdx.x;
  const int n = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int lane = lane_id();
  const int64_t j = r / M;
  const int m = (int)(r % M);
  const int64_t e = mp.rhs ? clamped_index(mp.rhs[mp.rhs_map ? mp.rhs_map[j] : j], mp.n_rhs) : 0;
  const int64_t xb = mp.lhs ? clamped_index(mp.lhs[j], mp.n_lhs) : j;
  const T *xr = x + (xb * M + m) * K;
  const int wpr = K / CPW, gpr = K / group;
  const uint32_t *wp = w + (e * N + n) * wpr;
  const T *sp = scales + (e * N + n) * gpr, *bp = biases + (e * N + n) * gpr;
  float acc = 0.f;
  for (int wi = lane; wi < wpr; wi += kWave) {
    const uint32_t word = wp[wi];
    const int k0 = wi * CPW;
    const float sc = Elem<T>::load(sp + k0 / group), bi = Elem<T>::load(bp + k0 / group);  // a word never straddles groups
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      const float qv = (float)((word >> (c * BITS)) & ((1u << BITS) - 1u));
      acc = __builtin_fmaf(Elem<T>::load(xr + k0 + c), __builtin_fmaf(sc, qv, bi), acc);
    }
  }
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) acc += __shfl_xor(acc, d, kWave);
  const int64_t dr = mp.dst_map ? (int64_t)mp.dst_map[r] : r;
  if (lane == 0) Elem<T>::store(y + dr * N + n, acc);
}

// The same product of dense float32 rows, 4- and 8-bit codes, R rows by C columns a wave: a word of codes is read and
// dequantised once for R rows, a value of x once for C columns.  Every sum runs over the same lanes in the same order as
// in qmm_plain_t_kernel, so the bits are the same.  (The matrix cores on raw codes lose two bits: see qmm_codes.hip; many rows and columns: qmm_f32.hip.)
// Sums meet by halving: at lane distance d each lane hands the half of its sums that its partner keeps; an addition
// commutes, so the tree of a sum does not depend on the lane that holds it.
// What bounds it: the vector unit, an fma per value and sum (430 us of it at 1000 x 4096 x 4096) beside the loads of x.
// (Figures: at the rule that picks R and C.)
template <int BITS, int R, int C>
__global__ __launch_bounds__(256) void qmm_plain_f32_kernel(const float *__restrict__ x, const uint32_t *__restrict__ w,
                                                            const float *__restrict__ scales, const float *__restrict__ biases,
                                                            int64_t rows, int N, int K, int group, float *__restrict__ y) {
  constexpr int CPW = 32 / BITS, V = R * C;
  const int64_t r0 = (int64_t)blockIdx.x * R;
  const int n0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * C;
  if (n0 >= N) return;
  const int lane = lane_id(), wpr = K / CPW, gpr = K / group;
  const float *xr[R];
#pragma unroll
  for (int i = 0; i < R; ++i) xr[i] = x + (r0 + i < rows ? r0 + i : rows - 1) * K;  // (rows and columns outside: the last one again, not stored)
  float acc[V] = {};
  for (int wi = lane; wi < wpr; wi += kWave) {
    const int k0 = wi * CPW, g = k0 / group;
    float4 xv[R][CPW / 4];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int p = 0; p < CPW / 4; ++p) xv[i][p] = reinterpret_cast<const float4 *>(xr[i] + k0)[p];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int64_t n = n0 + j < N ? n0 + j : N - 1;
      const uint32_t word = w[n * wpr + wi];
      const float sc = scales[n * gpr + g], bi = biases[n * gpr + g];
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        const float wv = __builtin_fmaf(sc, (float)((word >> (c * BITS)) & ((1u << BITS) - 1u)), bi);
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const float4 q = xv[i][c / 4];
          acc[i * C + j] = __builtin_fmaf(c % 4 == 0 ? q.x : c % 4 == 1 ? q.y : c % 4 == 2 ? q.z : q.w, wv, acc[i * C + j]);
        }
      }
    }
  }
  int held = V, first = 0;  // this lane holds sums first .. first + held - 1
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    if (held > 1) {
      held /= 2;
      const bool upper = lane & d;
      if (upper) first += held;
#pragma unroll
      for (int i = 0; i < V / 2; ++i) {
        if (i < held) {
          const float lo = acc[i], hi = acc[i + held], away = upper ? lo : hi;
          acc[i] = (upper ? hi : lo) + __shfl_xor(away, d, kWave);
        }
      }
    } else {
      acc[0] += __shfl_xor(acc[0], d, kWave);
    }
  }
  const int64_t row = r0 + first / C;
  const int n = n0 + first % C;
  if (lane < V && row < rows && n < N) y[row * N + n] = acc[0];
}

// transpose = false: w [E, K, N*bits/32], scales / biases [E, K, N/group] (K x N matrices quantised
// along N).  One thread per packed word of an output row, fp32 accumulation in k order.
template <class T, int BITS>
__global__ __launch_bounds__(256) void qmm_plain_n_kernel(const T *__restrict__ x, const uint32_t *__restrict__ w,
                                                          const T *__restrict__ scales, const T *__restrict__ biases,
                                                          PlainMaps mp, int M, int N, int K, int group,
                                                          T *__restrict__ y) {
  constexpr int CPW = 32 / BITS;  // codes per word
  const int64_t r = blockIdx.x;   // output row = j * M + m
  const int wi = blockIdx.y * 256 + threadIdx.x;
  const int wpr = N / CPW;
  if (wi >= wpr) return;
  const int64_t j = r / M;
  const int m = (int)(r % M);
  const int64_t e = mp.rhs ? clamped_index(mp.rhs[mp.rhs_map ? mp.rhs_map[j] : j], mp.n_rhs) : 0;
  const int64_t xb = mp.lhs ? clamped_index(mp.lhs[j], mp.n_lhs) : j;
  const T *xr = x + (xb * M + m) * K;
  const int gpr = N / group, g = wi * CPW / group;
  const uint32_t *wp = w + e * K * wpr + wi;
  const T *sp = scales + e * K * gpr + g, *bp = biases + e * K * gpr + g;
  float acc[CPW];
#pragma unroll
  for (int c = 0; c < CPW; ++c) acc[c] = 0.f;
  for (int k = 0; k < K; ++k) {
    const uint32_t word = wp[(int64_t)k * wpr];
    const float sc = Elem<T>::load(sp + (int64_t)k * gpr), bi = Elem<T>::load(bp + (int64_t)k * gpr);
    const float xv = Elem<T>::load(xr + k);
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      const float qv = (float)((word >> (c * BITS)) & ((1u << BITS) - 1u));
      acc[c] = __builtin_fmaf(xv, __builtin_fmaf(sc, qv, bi), acc[c]);
    }
  }
  const int64_t dr = mp.dst_map ? (int64_t)mp.dst_map[r] : r;
  T *yo = y + dr * N + (int64_t)wi * CPW;
#pragma unroll
  for (int c = 0; c < CPW; ++c) Elem<T>::store(yo + c, acc[c]);
}

template <class T>
static hipError_t launch_plain_t(const void *x, const uint32_t *w, const void *s, const void *b, const PlainMaps &mp,
                                 int64_t rows, int M, int N, int K, int group, int bits, void *y, bool transpose,
                                 hipStream_t st) {
  const T *xs = static_cast<const T *>(x), *ss = static_cast<const T *>(s), *bs = static_cast<const T *>(b);
  T *ys = static_cast<T *>(y);
  if (transpose) {
    dim3 grid((unsigned)rows, (unsigned)((N + 3) / 4));
    if (bits == 2) qmm_plain_t_kernel<T, 2><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
    else if (bits == 4) qmm_plain_t_kernel<T, 4><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
    else qmm_plain_t_kernel<T, 8><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
  } else {
    const int wpr = N * bits / 32;
    dim3 grid((unsigned)rows, (unsigned)((wpr + 255) / 256));
    if (bits == 2) qmm_plain_n_kernel<T, 2><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
    else if (bits == 4) qmm_plain_n_kernel<T, 4><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
    else qmm_plain_n_kernel<T, 8><<<grid, 256, 0, st>>>(xs, w, ss, bs, mp, M, N, K, group, ys);
  }
  return hipGetLastError();
}

// Which tile: the largest that leaves the launch two waves a SIMD (8 x 4 with 4-bit codes and 4 x 4; the 8-bit 4 x 4 tile
// holds twice the values of x and wants four; 4 x 2 one), if half of its rows are there: fewer waves do not hide the loads.
// Measured, us of the kernel with a wave per output element / 2 x 1 / 4 x 2 / 4 x 4 / 8 x 4 (rows, N, K):
//   4-bit (8, 256, 1024) 2.9 / 2.8 / 3.4 / 4.6 / 6.7, (8, 1024, 4096) 9.1 / 7.4 / 6.1 / 10.9 / 17.4, (12, 2080, 3968) 23.9 / 20.0 / 12.0 /
//   12.1 / 17.7, (17, 4096, 4096) 54.7 / 51.1 / 36.6 / 23.9 / 26.2, (32, 4096, 4096) 96.5 / 82.6 / 57.7 / 40.4 / 31.7,
//   (1000, 4096, 4096) 2754 / 2379 / 1670 / 1063 / 1005;
//   8-bit (8, 256, 1024) 3.2 / 3.1 / 3.7 / 5.6 / 10.4, (12, 2080, 3968) 33.0 / 22.1 / 14.7 / 26.1 / 30.9, (24, 4096, 4096) 106 / 68.8 /
//   37.9 / 35.4 / 61.6, (1000, 4096, 4096) 3601 / 2488 / 1497 / 1079 / 1387.
// (8 rows by one column from five rows on, whatever the waves: 3.9, 7.9, 23.7, 60.2 in the first four, slower than a wave per
// output element in three of them.)
template <int BITS>
static hipError_t launch_plain_f32(const float *x, const uint32_t *w, const float *s, const float *b, int64_t rows, int N, int K,
                                   int group, float *y, hipStream_t st) {
  auto run = [&](auto r, auto c) {
    constexpr int R = decltype(r)::value, C = decltype(c)::value;
    const dim3 grid((unsigned)((rows + R - 1) / R), (unsigned)((N + 4 * C - 1) / (4 * C)));
    qmm_plain_f32_kernel<BITS, R, C><<<grid, 256, 0, st>>>(x, w, s, b, rows, N, K, group, y);
    return hipGetLastError();
  };
  const std::integral_constant<int, 2> two{};
  const std::integral_constant<int, 4> four{};
  const auto waves = [&](int r, int c) { return (rows + r - 1) / r * ((N + c - 1) / c); };
  if constexpr (BITS == 4)
    if (rows > 4 && waves(8, 4) >= 2048) return run(std::integral_constant<int, 8>{}, four);
  if (rows > 2 && waves(4, 4) >= (BITS == 4 ? 2048 : 4096)) return run(four, four);
  if (rows > 2 && waves(4, 2) >= 1024) return run(four, two);
  return run(two, std::integral_constant<int, 1>{});
}

// dt: 0 bf16, 1 fp16, 2 fp32.  rows = n_idx * M output rows (at most 2^31 - 1: they are the grid's x extent).
hipError_t launch_qmm_plain(const void *x, const uint32_t *w, const void *scales, const void *biases,
                            const uint32_t *lhs, const uint32_t *rhs, const uint32_t *rhs_map,
                            const uint32_t *dst_map, uint32_t n_lhs, uint32_t n_rhs, int64_t rows, int M, int N,
                            int K, int group, int bits, bool transpose, int dt, void *y, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (transpose && (N + 3) / 4 > 65535) return hipErrorInvalidValue;  // the grid's y extent
  const PlainMaps mp{lhs, rhs, rhs_map, dst_map, n_lhs, n_rhs};
  if (dt == 2 && transpose && bits != 2 && rows > 1 && !lhs && !rhs && !dst_map && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
    const float *xs = static_cast<const float *>(x), *ss = static_cast<const float *>(scales), *bs = static_cast<const float *>(biases);
    if (float32_tiles(rows, N, K, bits)) return launch_qmm_f32(xs, w, ss, bs, rows, N, K, group, bits, static_cast<float *>(y), st);
    if (bits == 4) return launch_plain_f32<4>(xs, w, ss, bs, rows, N, K, group, static_cast<float *>(y), st);
    return launch_plain_f32<8>(xs, w, ss, bs, rows, N, K, group, static_cast<float *>(y), st);
  }
  if (dt == 0) return launch_plain_t<uint16_t>(x, w, scales, biases, mp, rows, M, N, K, group, bits, y, transpose, st);
  if (dt == 1) return launch_plain_t<_Float16>(x, w, scales, biases, mp, rows, M, N, K, group, bits, y, transpose, st);
  return launch_plain_t<float>(x, w, scales, biases, mp, rows, M, N, K, group, bits, y, transpose, st);
}

}  // namespace mi_moe
