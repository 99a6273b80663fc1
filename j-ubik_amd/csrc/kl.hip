// Positions, prior energy and mean gradient of the sampled KL (kl.hpp).
//
// Both kernels stream: they read and write each array once and are bound by
// that traffic.  As separate array operations (broadcast add, conversion to
// double, squares, sums and means) the same results took about 750 us of a
// 2048^2 x 2-field, 4-sample KL evaluation; fused they take 114 us (18 passes over
// a field of 33.6 MB, 0.60 GB).
#include <algorithm>

#include "kl.hpp"

namespace jubik {

namespace {

constexpr int KNT = 256;
constexpr int kKlBlocks = 2048;

// W values of T: 16 bytes where the arrays allow it, else one value.
template <typename T, int W>
struct Pack {
  T v[W];
};
template <typename T, int W>
__device__ __forceinline__ Pack<T, W> load_pack(const void* p, int64_t i) {
  using V = T __attribute__((ext_vector_type(W)));
  Pack<T, W> r;
  if constexpr (W == 1) {
    r.v[0] = static_cast<const T*>(p)[i];
  } else {
    const V x = static_cast<const V*>(p)[i];
#pragma unroll
    for (int k = 0; k < W; ++k) r.v[k] = x[k];
  }
  return r;
}
template <typename T, int W>
__device__ __forceinline__ void store_pack(void* p, int64_t i, const Pack<T, W>& a) {
  using V = T __attribute__((ext_vector_type(W)));
  if constexpr (W == 1) {
    static_cast<T*>(p)[i] = a.v[0];
  } else {
    V x;
#pragma unroll
    for (int k = 0; k < W; ++k) x[k] = a.v[k];
    static_cast<V*>(p)[i] = x;
  }
}

// grid (blocks, fields); np packs per field and sample.
template <typename T, int W>
__global__ __launch_bounds__(KNT) void k_kl_positions(int S, int64_t np, KlFields f,
                                                      double* __restrict__ partial) {
  __shared__ double red[KNT / 64];
  const int fi = blockIdx.y;
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)KNT + threadIdx.x; i < np;
       i += (int64_t)gridDim.x * KNT) {
    const Pack<T, W> x = load_pack<T, W>(f.xbar[fi], i);
    for (int s = 0; s < S; ++s) {
      Pack<T, W> p = load_pack<T, W>(f.delta[fi], s * np + i);
#pragma unroll
      for (int k = 0; k < W; ++k) {
        p.v[k] = x.v[k] + p.v[k];
        acc += (double)p.v[k] * (double)p.v[k];
      }
      store_pack<T, W>(f.pos[fi], s * np + i, p);
    }
  }
  acc = block_sum<KNT>(acc, red);
  if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = acc;
}

__global__ __launch_bounds__(KNT) void k_kl_prior(const double* __restrict__ partial, int n,
                                                  double* __restrict__ prior) {
  __shared__ double red[KNT / 64];
  double acc = 0.0;
  for (int k = threadIdx.x; k < n; k += KNT) acc += partial[k];
  acc = block_sum<KNT>(acc, red);
  if (threadIdx.x == 0) prior[0] = acc;
}

template <typename T, int W>
__global__ __launch_bounds__(KNT) void k_kl_mean(int S, int64_t np, KlFields f) {
  const int fi = blockIdx.y;
  const double inv = 1.0 / S;
  for (int64_t i = blockIdx.x * (int64_t)KNT + threadIdx.x; i < np;
       i += (int64_t)gridDim.x * KNT) {
    double g[W], p[W];
#pragma unroll
    for (int k = 0; k < W; ++k) g[k] = p[k] = 0.0;
    for (int s = 0; s < S; ++s) {
      const Pack<T, W> a = load_pack<T, W>(f.grad[fi], s * np + i);
      const Pack<T, W> b = load_pack<T, W>(f.pos[fi], s * np + i);
#pragma unroll
      for (int k = 0; k < W; ++k) {
        g[k] += (double)a.v[k];
        p[k] += (double)b.v[k];
      }
    }
    Pack<T, W> o;
#pragma unroll
    for (int k = 0; k < W; ++k) o.v[k] = (T)(g[k] * inv + p[k] * inv);
    store_pack<T, W>(f.out[fi], i, o);
  }
}

// 16-byte accesses need every sample's base on that boundary.
bool packed(int dtype, int64_t n, std::initializer_list<const void* const*> arrays, int nf) {
  const int w = dtype == 0 ? 4 : 2;
  if (n % w) return false;
  for (const void* const* a : arrays)
    for (int k = 0; k < nf; ++k)
      if (reinterpret_cast<uintptr_t>(a[k]) % 16) return false;
  return true;
}

// f(T tag, pack width) for the element type and alignment.
template <class F>
void with_pack(int dtype, bool wide, F&& f) {
  if (dtype == 0) {
    if (wide) f(float{}, std::integral_constant<int, 4>{});
    else f(float{}, std::integral_constant<int, 1>{});
  } else {
    if (wide) f(double{}, std::integral_constant<int, 2>{});
    else f(double{}, std::integral_constant<int, 1>{});
  }
}

}  // namespace

int kl_positions(int dtype, int S, int64_t n, const KlFields& f, double* work,
                 int64_t max_partial, double* prior, hipStream_t s) {
  const int nf = f.xbar[1] ? 2 : 1;
  const bool wide =
      packed(dtype, n, {f.xbar, f.delta, (const void* const*)f.pos}, nf);
  with_pack(dtype, wide, [&](auto tag, auto width) {
    using T = decltype(tag);
    constexpr int W = decltype(width)::value;
    const int64_t np = n / W;
    const int nb = (int)std::max<int64_t>(
        1, std::min({(np + KNT - 1) / KNT, (int64_t)kKlBlocks, max_partial / nf}));
    k_kl_positions<T, W><<<dim3(nb, nf), KNT, 0, s>>>(S, np, f, work);
    k_kl_prior<<<1, KNT, 0, s>>>(work, nb * nf, prior);
  });
  return check_hip(hipGetLastError(), "kl_positions");
}

int kl_mean(int dtype, int S, int64_t n, const KlFields& f, hipStream_t s) {
  const int nf = f.xbar[1] ? 2 : 1;
  const bool wide = packed(
      dtype, n, {f.grad, (const void* const*)f.pos, (const void* const*)f.out}, nf);
  with_pack(dtype, wide, [&](auto tag, auto width) {
    using T = decltype(tag);
    constexpr int W = decltype(width)::value;
    const int64_t np = n / W;
    const int nb = (int)std::min<int64_t>((np + KNT - 1) / KNT, 2 * kKlBlocks);
    k_kl_mean<T, W><<<dim3(nb, nf), KNT, 0, s>>>(S, np, f);
  });
  return check_hip(hipGetLastError(), "kl_mean");
}

}  // namespace jubik
