// Symmetric-power monomial contractions (the reference's symmetric_power_*
// ops; CPU core ye3t_runtime_core.cpp:5279-5540, CUDA execution_plan_cuda.cu:
// 5229, 5931-6000): the grouped table S[b, o] = sum_{t in o} v_t prod_c
// x[b, c]^e[t, c], its adjoint, the shared form in which outputs are sparse
// combinations of unique monomials, and that form with sparse monomial supports
// (with its second order).  These are the reference's stand-alone ops;
// the ACE product plan evaluates its symmetric blocks inside its own kernels.
//
// Forward and adjoint run on tiles of 64 rows (monomial_tile_*_kernel: lane =
// row); rows too wide for a tile, and the second order, on one thread per
// (row, output) or per row.  No atomics, fixed order.  The tables are validated
// by the caller (ye3t_amd.runtime checks them on the host).
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace ye3t {
namespace {

// Complex scalar of the sparse kernels (YE3T_C64 / YE3T_C128: interleaved
// (re, im) pairs, as torch stores complex tensors), with the arithmetic the
// kernels use.  Division is Smith's algorithm (R. L. Smith, "Algorithm 116:
// Complex division", CACM 5(8), 1962): the larger of |c| and |d| scales the
// denominator, so no intermediate overflows for finite operands.
template <typename R>
struct cplx {
  R re, im;
  cplx() = default;
  __device__ constexpr cplx(R r, R i) : re(r), im(i) {}
  __device__ constexpr cplx(int v) : re(R(v)), im(R(0)) {}
  __device__ constexpr cplx(int64_t v) : re(R(v)), im(R(0)) {}
};
template <typename R>
__device__ inline cplx<R> operator+(cplx<R> a, cplx<R> b) { return {a.re + b.re, a.im + b.im}; }
template <typename R>
__device__ inline cplx<R> operator-(cplx<R> a, cplx<R> b) { return {a.re - b.re, a.im - b.im}; }
template <typename R>
__device__ inline cplx<R> operator*(cplx<R> a, cplx<R> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename R>
__device__ inline cplx<R> operator/(cplx<R> a, cplx<R> b) {
  if (fabs(b.re) >= fabs(b.im)) {
    const R t = b.im / b.re, s = R(1) / (b.re + b.im * t);
    return {(a.re + a.im * t) * s, (a.im - a.re * t) * s};
  }
  const R t = b.re / b.im, s = R(1) / (b.im + b.re * t);
  return {(a.re * t + a.im) * s, (a.im * t - a.re) * s};
}
template <typename R>
__device__ inline cplx<R>& operator+=(cplx<R>& a, cplx<R> b) { return a = a + b; }
template <typename R>
__device__ inline cplx<R>& operator*=(cplx<R>& a, cplx<R> b) { return a = a * b; }
template <typename R>
__device__ inline bool operator==(cplx<R> a, cplx<R> b) { return a.re == b.re && a.im == b.im; }

// conjugate (the identity for real scalars): the adjoints multiply by the
// conjugates of coefficients and derivatives, as the reference's complex
// kernels do (execution_plan_cuda.cu:5757-5955, 6002-6033)
template <typename Real>
__device__ inline Real conjv(Real a) { return a; }
template <typename R>
__device__ inline cplx<R> conjv(cplx<R> a) { return {a.re, -a.im}; }

// integer_power of the reference core (ye3t_runtime_core.cpp:98-110): square and multiply
template <typename Real>
__device__ inline Real ipow(Real b, int64_t e) {
  Real v = Real(1);
  while (e > 0) {
    if (e & 1) v *= b;
    e >>= 1;
    if (e > 0) b *= b;
  }
  return v;
}

inline unsigned grid_for(int64_t work, int threads) {
  int64_t g = (work + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > (1 << 20)) g = 1 << 20;
  return unsigned(g);
}

template <typename Real>
__global__ __launch_bounds__(256) void sym_monomial_kernel(const Real* __restrict__ x, int64_t batch, int64_t D,
                                                           const int64_t* __restrict__ counts,
                                                           const int64_t* __restrict__ offsets,
                                                           const Real* __restrict__ values, int64_t O,
                                                           Real* __restrict__ out) {
  const int64_t total = batch * O;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t b = idx / O, o = idx - (idx / O) * O;
    const Real* row = x + b * D;
    Real acc = Real(0);
    for (int64_t t = offsets[o]; t < offsets[o + 1]; ++t) {
      Real m = values[t];
      for (int64_t c = 0; c < D; ++c) m *= ipow(row[c], counts[t * D + c]);
      acc += m;
    }
    out[idx] = acc;
  }
}

// The adjoint rule of one monomial m = scale * prod x_c^e_c (ye3t_runtime_core.cpp:
// 5331-5388): zero factors are left out of the product; two or more of them
// give no gradient, one of exponent 1 gives the cofactor, otherwise factor c
// gets e_c m / x_c.  `g` multiplies every contribution.
template <typename Real>
__device__ inline void monomial_gradient(const Real* __restrict__ row, const int64_t* __restrict__ e, int64_t D,
                                         Real scale, Real g, Real* __restrict__ grad) {
  Real mono = scale;
  int zeros = 0;
  int64_t zc = -1;
  for (int64_t c = 0; c < D; ++c) {
    if (e[c] == 0) continue;
    if (row[c] == Real(0)) {
      ++zeros;
      zc = c;
      continue;
    }
    mono *= ipow(row[c], e[c]);
  }
  if (zeros >= 2) return;
  if (zeros == 1) {
    if (e[zc] == 1) grad[zc] += g * mono;
    return;
  }
  for (int64_t c = 0; c < D; ++c) {
    if (e[c] == 0) continue;
    grad[c] += g * (Real(e[c]) * mono / row[c]);
  }
}

template <typename Real>
__global__ __launch_bounds__(256) void sym_monomial_adjoint_kernel(
    const Real* __restrict__ gout, const Real* __restrict__ x, int64_t batch, int64_t D,
    const int64_t* __restrict__ counts, const int64_t* __restrict__ out_index, const Real* __restrict__ values,
    int64_t T, int64_t O, Real* __restrict__ gin) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < batch; b += int64_t(gridDim.x) * blockDim.x) {
    const Real* row = x + b * D;
    Real* grad = gin + b * D;
    for (int64_t c = 0; c < D; ++c) grad[c] = Real(0);
    for (int64_t t = 0; t < T; ++t)
      monomial_gradient(row, counts + t * D, D, values[t], gout[b * O + out_index[t]], grad);
  }
}

template <typename Real>
__global__ __launch_bounds__(256) void shared_monomial_kernel(const Real* __restrict__ x, int64_t batch, int64_t D,
                                                              const int64_t* __restrict__ counts,
                                                              const int64_t* __restrict__ offsets,
                                                              const int64_t* __restrict__ terms,
                                                              const Real* __restrict__ values, int64_t O,
                                                              Real* __restrict__ out) {
  const int64_t total = batch * O;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t b = idx / O, o = idx - (idx / O) * O;
    const Real* row = x + b * D;
    Real acc = Real(0);
    for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k) {
      const int64_t* e = counts + terms[k] * D;
      Real m = Real(1);
      for (int64_t c = 0; c < D; ++c) m *= ipow(row[c], e[c]);
      acc += values[k] * m;
    }
    out[idx] = acc;
  }
}

// Shared monomials' adjoint: coefficient k of output o contributes
// g[b, o] v_k d(monomial terms[k]) -- the reference's per-monomial adjoint
// (ye3t_runtime_core.cpp:5442-5540) with its sum over coefficients taken
// term by term.
template <typename Real>
__global__ __launch_bounds__(256) void shared_monomial_adjoint_kernel(
    const Real* __restrict__ gout, const Real* __restrict__ x, int64_t batch, int64_t D,
    const int64_t* __restrict__ counts, const int64_t* __restrict__ offsets, const int64_t* __restrict__ terms,
    const Real* __restrict__ values, int64_t O, Real* __restrict__ gin) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < batch; b += int64_t(gridDim.x) * blockDim.x) {
    const Real* row = x + b * D;
    Real* grad = gin + b * D;
    for (int64_t c = 0; c < D; ++c) grad[c] = Real(0);
    for (int64_t o = 0; o < O; ++o) {
      const Real g = gout[b * O + o];
      for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k)
        monomial_gradient(row, counts + terms[k] * D, D, Real(1), g * values[k], grad);
    }
  }
}

// Sparse shared monomials (the reference's symmetric_power_shared_sparse_*
// ops, execution_plan_cuda.cu:5720-5955 and host :11012-11330): monomial t is
// prod_{q in [toff[t], toff[t+1])} x[comp[q]]^ex[q], stored as a support list
// instead of a dense exponent row.  Zero factors add their exponents to a
// "zero degree" that selects the derivative rule.
template <typename Real>
__device__ inline Real sparse_monomial(const Real* __restrict__ row, const int64_t* __restrict__ toff,
                                       const int64_t* __restrict__ comp, const int64_t* __restrict__ ex, int64_t t) {
  Real v = Real(1);
  for (int64_t q = toff[t]; q < toff[t + 1]; ++q) v *= ipow(row[comp[q]], ex[q]);
  return v;
}

// Product of the nonzero factors, the zero degree and the first two zero
// components of monomial t.
template <typename Real>
struct SparseFactors {
  Real mono;
  int64_t zdeg, z1, z2;
};

template <typename Real>
__device__ inline SparseFactors<Real> sparse_factors(const Real* __restrict__ row, const int64_t* __restrict__ toff,
                                                     const int64_t* __restrict__ comp,
                                                     const int64_t* __restrict__ ex, int64_t t) {
  SparseFactors<Real> f{Real(1), 0, -1, -1};
  for (int64_t q = toff[t]; q < toff[t + 1]; ++q) {
    const Real xv = row[comp[q]];
    if (xv == Real(0)) {
      f.zdeg += ex[q];
      if (f.z1 < 0) f.z1 = comp[q];
      else if (f.z2 < 0) f.z2 = comp[q];
    } else {
      f.mono *= ipow(xv, ex[q]);
    }
  }
  return f;
}

template <typename Real>
__global__ __launch_bounds__(256) void sparse_monomial_kernel(const Real* __restrict__ x, int64_t batch, int64_t D,
                                                              const int64_t* __restrict__ toff,
                                                              const int64_t* __restrict__ comp,
                                                              const int64_t* __restrict__ ex,
                                                              const int64_t* __restrict__ offsets,
                                                              const int64_t* __restrict__ terms,
                                                              const Real* __restrict__ values, int64_t O,
                                                              Real* __restrict__ out) {
  const int64_t total = batch * O;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t b = idx / O, o = idx - (idx / O) * O;
    const Real* row = x + b * D;
    Real acc = Real(0);
    for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k) acc += values[k] * sparse_monomial(row, toff, comp, ex, terms[k]);
    out[idx] = acc;
  }
}

// One thread per row owns its input-gradient row: coefficient k of output o
// adds g[b, o] v_k times the gradient of monomial terms[k] (zero degree one:
// the cofactor to the zero component; zero degree zero: e m / x per entry).
template <typename Real>
__global__ __launch_bounds__(256) void sparse_monomial_adjoint_kernel(
    const Real* __restrict__ gout, const Real* __restrict__ x, int64_t batch, int64_t D,
    const int64_t* __restrict__ toff, const int64_t* __restrict__ comp, const int64_t* __restrict__ ex,
    const int64_t* __restrict__ offsets, const int64_t* __restrict__ terms, const Real* __restrict__ values,
    int64_t O, Real* __restrict__ gin) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < batch; b += int64_t(gridDim.x) * blockDim.x) {
    const Real* row = x + b * D;
    Real* grad = gin + b * D;
    for (int64_t c = 0; c < D; ++c) grad[c] = Real(0);
    for (int64_t o = 0; o < O; ++o) {
      const Real g = gout[b * O + o];
      for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k) {
        const int64_t t = terms[k];
        const Real w = g * conjv(values[k]);
        const SparseFactors<Real> f = sparse_factors(row, toff, comp, ex, t);
        if (f.zdeg == 1) {
          grad[f.z1] += w * conjv(f.mono);
        } else if (f.zdeg == 0) {
          for (int64_t q = toff[t]; q < toff[t + 1]; ++q)
            grad[comp[q]] += w * conjv(Real(ex[q]) * f.mono / row[comp[q]]);
        }
      }
    }
  }
}

// ---- tiles of 64 rows -------------------------------------------------------
//
// Lane = row, so that the table, the same for every row, is wave-uniform: no
// lane waits for another's term.  The rows' components are in LDS (component-major), and so is
// the table where it fits; the waves of a workgroup share the outputs
// (forward) or the coefficients (adjoint, each wave with its own gradient rows
// in LDS, summed in wave order).  Small exponents of few components are packed
// into one word a monomial.  Bound by the latency of those short dependent
// steps, hence as many waves a tile as its gradients leave room for.  70
// monomials of degree 4 over 5 components, 315 coefficients, 20 000 rows, fp64:
// forward 68 -> 46 us, adjoint 473 -> 61 us (one thread a row, its gradient read
// and written in memory for every factor; 65 and 82 us with the exponents unpacked).

// One table for the three forms.  Monomial t has factors [begin(t), end(t)),
// factor q is x[component(q)]^exponent(q); coefficient k combines monomial
// term(k).
struct MonomialTable {
  const int64_t* counts;  // dense: exponents [M, D]; NULL: sparse supports
  const int64_t* toff;
  const int64_t* comp;
  const int64_t* ex;
  const int64_t* terms;    // NULL: coefficient k is monomial k, which starts from its value
  const int64_t* outputs;  // output of coefficient k; NULL: by the output offsets
  int64_t D, M, S, C, O;
};

constexpr int kTileRows = 64;
constexpr size_t kTileLds = 64 * 1024;    // rows and gradients of a tile
constexpr size_t kTableLds = 32 * 1024;   // table held beside them
constexpr int64_t kPackedComponents = 16;

__device__ inline int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v))));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v) >> 32)));
  return int64_t((uint64_t(hi) << 32) | lo);
}

template <typename Real>
__device__ inline Real uniform_value(Real v) {
  if constexpr (sizeof(Real) == 4) {
    return __builtin_bit_cast(Real, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
  } else if constexpr (sizeof(Real) == 8) {
    return __builtin_bit_cast(Real, uniform64(__builtin_bit_cast(int64_t, v)));
  } else {
    return {uniform_value(v.re), uniform_value(v.im)};
  }
}

// The table's arrays in LDS (copied by the whole workgroup) or in memory.
struct HeldTable {
  const uint64_t* packed;  // dense, held, at most kPackedComponents components, exponents below 16: four bits each
  const int64_t *exps, *comp, *toff, *terms, *outputs, *offsets;
  const void* values;
};

inline size_t held_bytes(const MonomialTable& t, size_t elem) {
  const int64_t words = (t.counts ? t.M * t.D + (t.D <= kPackedComponents ? t.M + 1 : 0) : t.M + 1 + 2 * t.S) + (t.terms ? t.C : 0) + (t.outputs ? t.C : t.O + 1);
  return size_t(words) * 8 + size_t(t.C) * elem;
}

template <bool HELD, typename Real>
__device__ inline HeldTable hold_table(const MonomialTable& t, const int64_t* offsets, const Real* values,
                                       unsigned char* lds) {
  if (!HELD) return {nullptr, t.counts ? t.counts : t.ex, t.comp, t.toff, t.terms, t.outputs, offsets, values};
  auto copy = [&](const auto* from, int64_t n) {
    using T = std::remove_cv_t<std::remove_reference_t<decltype(*from)>>;
    T* to = reinterpret_cast<T*>(lds);
    lds += size_t(n) * sizeof(T);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) to[i] = from[i];
    return static_cast<const T*>(to);
  };
  HeldTable h = {};
  h.exps = t.counts ? copy(t.counts, t.M * t.D) : copy(t.ex, t.S);
  if (!t.counts) {
    h.comp = copy(t.comp, t.S);
    h.toff = copy(t.toff, t.M + 1);
  }
  if (t.terms) h.terms = copy(t.terms, t.C);
  if (t.counts && t.D <= kPackedComponents) {
    // word M counts the monomials that do not fit, and the table is read as it is if any does not
    uint64_t* const packed = reinterpret_cast<uint64_t*>(lds);
    lds += size_t(t.M + 1) * 8;
    if (threadIdx.x == 0) packed[t.M] = 0;
    __syncthreads();
    for (int64_t m = threadIdx.x; m < t.M; m += blockDim.x) {
      uint64_t bits = 0;
      bool fits = true;
      for (int64_t c = 0; c < t.D; ++c) {
        const int64_t e = t.counts[m * t.D + c];
        fits = fits && e < 16;
        bits |= uint64_t(e & 15) << (4 * c);
      }
      packed[m] = bits;
      if (!fits) packed[t.M] = 1;
    }
    __syncthreads();
    h.packed = packed[t.M] == 0 ? packed : nullptr;
  }
  if (t.outputs) h.outputs = copy(t.outputs, t.C);
  if (offsets) h.offsets = copy(offsets, t.O + 1);
  h.values = copy(values, t.C);  // last: an odd number of 4-byte values would misalign what follows
  return h;
}

// body(component, exponent) for each factor of monomial m that is not to the
// power of zero.  A packed row is one read, and its zeros cost nothing.
template <bool DENSE, typename Body>
__device__ inline void for_factors(const MonomialTable& t, const HeldTable& h, int64_t m, Body body) {
  if (DENSE && h.packed != nullptr) {
    for (uint64_t bits = uint64_t(uniform64(int64_t(h.packed[m]))); bits != 0;) {
      const int c = __builtin_ctzll(bits) >> 2;
      body(c, int64_t(bits >> (4 * c)) & 15);
      bits &= ~(uint64_t(15) << (4 * c));
    }
    return;
  }
  const int64_t q0 = DENSE ? m * t.D : uniform64(h.toff[m]), q1 = DENSE ? q0 + t.D : uniform64(h.toff[m + 1]);
  for (int64_t q = q0; q < q1; ++q) {
    const int64_t e = uniform64(h.exps[q]);
    if (e != 0) body(int(DENSE ? q - q0 : uniform64(h.comp[q])), e);
  }
}

// rows of x into xs[component][row]; rows past the batch hold ones
template <typename Real>
__device__ inline void load_rows(const Real* __restrict__ x, int64_t b0, int64_t batch, int64_t D, Real* xs) {
  for (int64_t i = threadIdx.x; i < kTileRows * D; i += blockDim.x) {
    const int64_t r = i / D, c = i - r * D;
    xs[c * kTileRows + r] = b0 + r < batch ? x[(b0 + r) * D + c] : Real(1);
  }
}

template <bool DENSE, bool HELD, typename Real>
__global__ __launch_bounds__(512) void monomial_tile_kernel(const Real* __restrict__ x, int64_t batch, MonomialTable t,
                                                            const int64_t* __restrict__ offsets,
                                                            const Real* __restrict__ values, Real* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char tile_smem[];
  Real* const xs = reinterpret_cast<Real*>(tile_smem);
  const int64_t b0 = int64_t(blockIdx.x) * kTileRows;
  const int lane = threadIdx.x & 63;
  const int waves = int(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const HeldTable h =
      hold_table<HELD>(t, offsets, values, tile_smem + size_t(t.D) * kTileRows * sizeof(Real));
  const Real* const hv = static_cast<const Real*>(h.values);
  load_rows(x, b0, batch, t.D, xs);
  __syncthreads();
  // a launch of few tiles shares the outputs among several workgroups a tile (blockIdx.y)
  for (int64_t o = wave + int64_t(waves) * blockIdx.y; o < t.O; o += int64_t(waves) * gridDim.y) {
    const int64_t k1 = uniform64(h.offsets[o + 1]);
    Real acc = Real(0);
    for (int64_t k = uniform64(h.offsets[o]); k < k1; ++k) {
      const Real v = uniform_value(hv[k]);
      const int64_t m = t.terms ? uniform64(h.terms[k]) : k;
      Real p = t.terms ? Real(1) : v;
      for_factors<DENSE>(t, h, m, [&](int c, int64_t e) { p *= ipow(xs[c * kTileRows + lane], e); });
      if (t.terms) acc += v * p;
      else acc += p;
    }
    if (b0 + lane < batch) out[(b0 + lane) * t.O + o] = acc;
  }
}

// Input gradient, with the zero-factor rules of monomial_gradient (dense: a
// single zero factor of exponent one takes the cofactor) and of
// sparse_monomial_adjoint_kernel, which are one: a zero degree of one.  SHARED:
// coefficients name their monomials.
template <bool DENSE, bool HELD, bool SHARED, typename Real>
__global__ __launch_bounds__(512) void monomial_tile_adjoint_kernel(
    const Real* __restrict__ gout, const Real* __restrict__ x, int64_t batch, MonomialTable t,
    const int64_t* __restrict__ offsets, const Real* __restrict__ values, Real* __restrict__ gin) {
  extern __shared__ __align__(16) unsigned char tile_smem[];
  const int64_t size = t.D * kTileRows;
  Real* const xs = reinterpret_cast<Real*>(tile_smem);
  const int64_t b0 = int64_t(blockIdx.x) * kTileRows;
  const int lane = threadIdx.x & 63;
  const int waves = int(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  Real* const grads = xs + size;
  Real* const grad = grads + wave * size;
  const HeldTable h =
      hold_table<HELD>(t, offsets, values, tile_smem + size_t(size) * size_t(1 + waves) * sizeof(Real));
  const Real* const hv = static_cast<const Real*>(h.values);
  load_rows(x, b0, batch, t.D, xs);
  for (int64_t i = threadIdx.x; i < size * waves; i += blockDim.x) grads[i] = Real(0);
  __syncthreads();
  const int64_t b = b0 + lane < batch ? b0 + lane : batch - 1;
  const int64_t k0 = t.C * wave / waves, k1 = t.C * (wave + 1) / waves;
  // the output before the wave's first coefficient's, and where it ends
  int64_t o = -1, end = k0;
  if (!t.outputs && k0 < k1) {
    int64_t lo = 0, hi = t.O;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (uniform64(h.offsets[mid]) <= k0) lo = mid;
      else hi = mid;
    }
    o = lo - 1;
  }
  Real g = Real(0);
  for (int64_t k = k0; k < k1; ++k) {
    const int64_t before = o;
    if (t.outputs) {
      o = uniform64(h.outputs[k]);
    } else {
      while (k >= end) end = uniform64(h.offsets[++o + 1]);
    }
    if (o != before) g = gout[b * t.O + o];
    const Real v = uniform_value(hv[k]);
    const int64_t m = SHARED ? uniform64(h.terms[k]) : k;
    // a grouped table's monomial starts from its value (as forward: the product may fit where it alone does not)
    const Real w = SHARED ? g * conjv(v) : g;
    Real mono = SHARED ? Real(1) : v;
    int64_t zdeg = 0;  // exponents of the zero factors (dense: those past one factor make it two or more)
    int zc = 0;
    for_factors<DENSE>(t, h, m, [&](int c, int64_t e) {
      const Real xv = xs[c * kTileRows + lane];
      if (xv == Real(0)) {
        zdeg += e;
        zc = c;
      } else {
        mono *= ipow(xv, e);
      }
    });
    if (zdeg == 0) {
      for_factors<DENSE>(t, h, m, [&](int c, int64_t e) {
        grad[c * kTileRows + lane] += w * conjv(Real(e) * mono / xs[c * kTileRows + lane]);
      });
    } else if (zdeg == 1) {
      grad[zc * kTileRows + lane] += w * conjv(mono);
    }
  }
  __syncthreads();
  for (int64_t i = threadIdx.x; i < size; i += blockDim.x) {
    const int64_t r = i / t.D, c = i - r * t.D;
    if (b0 + r >= batch) break;
    Real sum = grads[c * kTileRows + r];
    for (int k = 1; k < waves; ++k) sum += grads[k * size + c * kTileRows + r];
    gin[(b0 + r) * t.D + c] = sum;
  }
}

// Launches a tile kernel; YE3T_EUNSUPPORTED, with nothing launched, where a
// tile of rows (and one wave's gradients) does not fit in kTileLds, or the tiles
// not in one grid.
template <typename Real>
int launch_tiles(const Real* gout, const Real* x, int64_t batch, const MonomialTable& t, const int64_t* offsets,
                 const Real* values, Real* out, hipStream_t s) {
  const size_t rows = size_t(t.D) * kTileRows * sizeof(Real);
  const int64_t tiles = (batch + kTileRows - 1) / kTileRows;
  if (t.D < 1 || t.O < 1 || t.D > 1024) return YE3T_EUNSUPPORTED;
  int waves = 8;
  while (waves > 0 && rows * size_t(1 + (gout ? waves : 0)) > kTileLds) waves /= 2;
  if (waves == 0) return YE3T_EUNSUPPORTED;
  if (!gout && t.O < waves) waves = int(t.O);
  if (!fits_grid(tiles, 64 * waves)) return YE3T_EUNSUPPORTED;  // the kernels of one thread a row take any batch
  // one gradient copy only: a wave a tile, no faster than a thread a row unless the tile is full (one row of 100
  // fp32 components, 1000 coefficients: 1136 us by the thread, 1458 here)
  if (gout && waves == 1 && batch < kTileRows) return YE3T_EUNSUPPORTED;
  const size_t held = held_bytes(t, sizeof(Real));
  const bool hold = held <= kTableLds;
  const size_t lds = rows * size_t(1 + (gout ? waves : 0)) + (hold ? held : 0);
  // forward: up to two workgroups a compute unit, each with its share of a tile's outputs
  int64_t split = gout ? 1 : std::min<int64_t>((t.O + waves - 1) / waves, 512 / tiles);
  if (split < 1) split = 1;
  const dim3 grid{unsigned(tiles), unsigned(split)}, block{unsigned(64 * waves)};
  auto launch = [&](auto dense, auto keep, auto shared) {
    auto start = [&](auto* kernel, const char* name, auto... args) {
      if (lds > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)) != hipSuccess) {
        (void)hipGetLastError();
        return int(YE3T_EUNSUPPORTED);
      }
      hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
      return check_launch(name);
    };
    if (gout)
      return start(&monomial_tile_adjoint_kernel<dense.value, keep.value, shared.value, Real>,
                   "monomial_tile_adjoint_kernel", gout, x, batch, t, offsets, values, out);
    return start(&monomial_tile_kernel<dense.value, keep.value, Real>, "monomial_tile_kernel", x, batch, t, offsets,
                 values, out);
  };
  const std::true_type yes;
  const std::false_type no;
  if (!t.counts) return hold ? launch(no, yes, yes) : launch(no, no, yes);
  if (t.terms) return hold ? launch(yes, yes, yes) : launch(yes, no, yes);
  return hold ? launch(yes, yes, no) : launch(yes, no, no);
}

int launch_tiles(int dtype, const void* gout, const void* x, int64_t batch, const MonomialTable& t,
                 const int64_t* offsets, const void* values, void* out, hipStream_t s) {
  auto as = [&](auto zero) {
    using Real = decltype(zero);
    return launch_tiles<Real>(static_cast<const Real*>(gout), static_cast<const Real*>(x), batch, t, offsets,
                              static_cast<const Real*>(values), static_cast<Real*>(out), s);
  };
  switch (dtype) {
    case YE3T_F64: return as(double{});
    case YE3T_F32: return as(float{});
    case YE3T_C128: return as(cplx<double>{});
    case YE3T_C64: return as(cplx<float>{});
    default: return YE3T_EUNSUPPORTED;
  }
}

// Directional derivative of monomial t along v.
template <typename Real>
__device__ inline Real sparse_directional(const Real* __restrict__ row, const Real* __restrict__ v,
                                          const int64_t* __restrict__ toff, const int64_t* __restrict__ comp,
                                          const int64_t* __restrict__ ex, int64_t t) {
  const SparseFactors<Real> f = sparse_factors(row, toff, comp, ex, t);
  if (f.zdeg == 1) return v[f.z1] * f.mono;
  if (f.zdeg != 0) return Real(0);
  Real logdir = Real(0);
  for (int64_t q = toff[t]; q < toff[t + 1]; ++q) logdir += Real(ex[q]) * v[comp[q]] / row[comp[q]];
  return f.mono * logdir;
}

// Output tangent of the double backward: the forward's linearisation along v.
template <typename Real>
__global__ __launch_bounds__(256) void sparse_monomial_tangent_kernel(
    const Real* __restrict__ tangent, const Real* __restrict__ x, int64_t batch, int64_t D,
    const int64_t* __restrict__ toff, const int64_t* __restrict__ comp, const int64_t* __restrict__ ex,
    const int64_t* __restrict__ offsets, const int64_t* __restrict__ terms, const Real* __restrict__ values,
    int64_t O, Real* __restrict__ out_tangent) {
  const int64_t total = batch * O;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t b = idx / O, o = idx - (idx / O) * O;
    const Real* row = x + b * D;
    const Real* v = tangent + b * D;
    Real acc = Real(0);
    for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k)
      acc += values[k] * sparse_directional(row, v, toff, comp, ex, terms[k]);
    out_tangent[idx] = acc;
  }
}

// Input tangent of the double backward: sum over coefficients of
// g[b, o] v_k (Hessian of monomial terms[k]) v, one thread per row.
template <typename Real>
__global__ __launch_bounds__(256) void sparse_monomial_hessian_kernel(
    const Real* __restrict__ tangent, const Real* __restrict__ gout, const Real* __restrict__ x, int64_t batch,
    int64_t D, const int64_t* __restrict__ toff, const int64_t* __restrict__ comp, const int64_t* __restrict__ ex,
    const int64_t* __restrict__ offsets, const int64_t* __restrict__ terms, const Real* __restrict__ values,
    int64_t O, Real* __restrict__ in_tangent) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < batch; b += int64_t(gridDim.x) * blockDim.x) {
    const Real* row = x + b * D;
    const Real* v = tangent + b * D;
    Real* it = in_tangent + b * D;
    for (int64_t c = 0; c < D; ++c) it[c] = Real(0);
    for (int64_t o = 0; o < O; ++o) {
      const Real g = gout[b * O + o];
      for (int64_t k = offsets[o]; k < offsets[o + 1]; ++k) {
        const int64_t t = terms[k];
        const Real w = g * conjv(values[k]);
        const SparseFactors<Real> f = sparse_factors(row, toff, comp, ex, t);
        if (f.zdeg == 0) {
          Real logdir = Real(0);
          for (int64_t q = toff[t]; q < toff[t + 1]; ++q) logdir += Real(ex[q]) * v[comp[q]] / row[comp[q]];
          for (int64_t q = toff[t]; q < toff[t + 1]; ++q) {
            const int64_t c = comp[q];
            it[c] += w * conjv(Real(ex[q]) * f.mono / row[c] * (logdir - v[c] / row[c]));
          }
        } else if (f.zdeg == 1) {
          Real zdir = Real(0);
          for (int64_t q = toff[t]; q < toff[t + 1]; ++q) {
            const int64_t c = comp[q];
            if (c == f.z1) continue;
            const Real d = Real(ex[q]) * f.mono / row[c];
            zdir += v[c] * d;
            it[c] += w * conjv(v[f.z1] * d);
          }
          it[f.z1] += w * conjv(zdir);
        } else if (f.zdeg == 2) {
          if (f.z2 < 0) {
            it[f.z1] += w * conjv(Real(2) * f.mono * v[f.z1]);
          } else {
            it[f.z1] += w * conjv(f.mono * v[f.z2]);
            it[f.z2] += w * conjv(f.mono * v[f.z1]);
          }
        }
      }
    }
  }
}

}  // namespace
}  // namespace ye3t

using namespace ye3t;

extern "C" {

int ye3t_hip_symmetric_power_monomial(int dtype, const void* x, int64_t batch, int64_t D, const int64_t* counts,
                                      const int64_t* offsets, const int64_t* output_indices, const void* values,
                                      int64_t T, int64_t O, void* out, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && O >= 0 && T >= 0, "negative size");
  if (batch * O == 0) return YE3T_OK;
  YE3T_REQUIRE(x && offsets && out && (T == 0 || (counts && values && output_indices)), "NULL argument");
  if ((dtype == YE3T_F64 || dtype == YE3T_F32) && T > 0) {
    const MonomialTable t = {counts, nullptr, nullptr, nullptr, nullptr, nullptr, D, T, 0, T, O};
    const int rc = launch_tiles(dtype, nullptr, x, batch, t, offsets, values, out, as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  const unsigned grid = grid_for(batch * O, 256);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(sym_monomial_kernel<double>, dim3(grid), dim3(256), 0, as_stream(stream), (const double*)x,
                       batch, D, counts, offsets, (const double*)values, O, (double*)out);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(sym_monomial_kernel<float>, dim3(grid), dim3(256), 0, as_stream(stream), (const float*)x,
                       batch, D, counts, offsets, (const float*)values, O, (float*)out);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  return check_launch("sym_monomial_kernel");
}

int ye3t_hip_symmetric_power_monomial_adjoint(int dtype, const void* output_adjoint, const void* x, int64_t batch,
                                              int64_t D, const int64_t* counts, const int64_t* output_indices,
                                              const void* values, int64_t T, int64_t O, void* input_adjoint,
                                              ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && O >= 0 && T >= 0, "negative size");
  if (batch * D == 0) return YE3T_OK;
  YE3T_REQUIRE(x && input_adjoint && (T == 0 || (output_adjoint && counts && values && output_indices)),
               "NULL argument");
  if ((dtype == YE3T_F64 || dtype == YE3T_F32) && T > 0) {
    const MonomialTable t = {counts, nullptr, nullptr, nullptr, nullptr, output_indices, D, T, 0, T, O};
    const int rc = launch_tiles(dtype, output_adjoint, x, batch, t, nullptr, values, input_adjoint, as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  const unsigned grid = grid_for(batch, 256);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(sym_monomial_adjoint_kernel<double>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const double*)output_adjoint, (const double*)x, batch, D, counts, output_indices,
                       (const double*)values, T, O, (double*)input_adjoint);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(sym_monomial_adjoint_kernel<float>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const float*)output_adjoint, (const float*)x, batch, D, counts, output_indices,
                       (const float*)values, T, O, (float*)input_adjoint);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  return check_launch("sym_monomial_adjoint_kernel");
}

int ye3t_hip_symmetric_power_shared_monomial(int dtype, const void* x, int64_t batch, int64_t D,
                                             const int64_t* counts, int64_t M, const int64_t* output_offsets,
                                             const int64_t* coefficient_terms, const void* coefficient_values,
                                             int64_t C, int64_t O, void* out, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && O >= 0 && M >= 0 && C >= 0, "negative size");
  if (batch * O == 0) return YE3T_OK;
  YE3T_REQUIRE(x && output_offsets && out && (C == 0 || (counts && coefficient_terms && coefficient_values)),
               "NULL argument");
  if ((dtype == YE3T_F64 || dtype == YE3T_F32) && C > 0) {
    const MonomialTable t = {counts, nullptr, nullptr, nullptr, coefficient_terms, nullptr, D, M, 0, C, O};
    const int rc = launch_tiles(dtype, nullptr, x, batch, t, output_offsets, coefficient_values, out, as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  const unsigned grid = grid_for(batch * O, 256);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(shared_monomial_kernel<double>, dim3(grid), dim3(256), 0, as_stream(stream), (const double*)x,
                       batch, D, counts, output_offsets, coefficient_terms, (const double*)coefficient_values, O,
                       (double*)out);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(shared_monomial_kernel<float>, dim3(grid), dim3(256), 0, as_stream(stream), (const float*)x,
                       batch, D, counts, output_offsets, coefficient_terms, (const float*)coefficient_values, O,
                       (float*)out);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  (void)M;
  return check_launch("shared_monomial_kernel");
}

int ye3t_hip_symmetric_power_shared_monomial_adjoint(int dtype, const void* output_adjoint, const void* x,
                                                     int64_t batch, int64_t D, const int64_t* counts, int64_t M,
                                                     const int64_t* output_offsets, const int64_t* coefficient_terms,
                                                     const void* coefficient_values, int64_t C, int64_t O,
                                                     void* input_adjoint, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && O >= 0 && M >= 0 && C >= 0, "negative size");
  if (batch * D == 0) return YE3T_OK;
  YE3T_REQUIRE(x && input_adjoint && output_offsets &&
                   (C == 0 || (output_adjoint && counts && coefficient_terms && coefficient_values)),
               "NULL argument");
  if ((dtype == YE3T_F64 || dtype == YE3T_F32) && C > 0) {
    const MonomialTable t = {counts, nullptr, nullptr, nullptr, coefficient_terms, nullptr, D, M, 0, C, O};
    const int rc = launch_tiles(dtype, output_adjoint, x, batch, t, output_offsets, coefficient_values, input_adjoint,
                                as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  const unsigned grid = grid_for(batch, 256);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(shared_monomial_adjoint_kernel<double>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const double*)output_adjoint, (const double*)x, batch, D, counts, output_offsets,
                       coefficient_terms, (const double*)coefficient_values, O, (double*)input_adjoint);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(shared_monomial_adjoint_kernel<float>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const float*)output_adjoint, (const float*)x, batch, D, counts, output_offsets,
                       coefficient_terms, (const float*)coefficient_values, O, (float*)input_adjoint);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  (void)M;
  return check_launch("shared_monomial_adjoint_kernel");
}

#define SPARSE_DISPATCH(KERNEL, GRID, ...)                                                                 \
  do {                                                                                                     \
    if (dtype == YE3T_F64) {                                                                               \
      using Real = double;                                                                                 \
      hipLaunchKernelGGL(KERNEL<double>, dim3(GRID), dim3(256), 0, as_stream(stream), __VA_ARGS__);        \
    } else if (dtype == YE3T_F32) {                                                                        \
      using Real = float;                                                                                  \
      hipLaunchKernelGGL(KERNEL<float>, dim3(GRID), dim3(256), 0, as_stream(stream), __VA_ARGS__);         \
    } else if (dtype == YE3T_C128) {                                                                       \
      using Real = cplx<double>;                                                                           \
      hipLaunchKernelGGL(KERNEL<Real>, dim3(GRID), dim3(256), 0, as_stream(stream), __VA_ARGS__);          \
    } else if (dtype == YE3T_C64) {                                                                        \
      using Real = cplx<float>;                                                                            \
      hipLaunchKernelGGL(KERNEL<Real>, dim3(GRID), dim3(256), 0, as_stream(stream), __VA_ARGS__);          \
    } else {                                                                                               \
      return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);                                        \
    }                                                                                                      \
  } while (0)

int ye3t_hip_symmetric_power_shared_sparse_monomial(int dtype, const void* x, int64_t batch, int64_t D,
                                                    const int64_t* term_offsets, const int64_t* term_components,
                                                    const int64_t* term_exponents, int64_t M, int64_t S,
                                                    const int64_t* output_offsets, const int64_t* coefficient_terms,
                                                    const void* coefficient_values, int64_t C, int64_t O, void* out,
                                                    ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && M >= 0 && S >= 0 && C >= 0 && O >= 0, "negative size");
  if (batch * O == 0) return YE3T_OK;
  YE3T_REQUIRE(x && output_offsets && out && term_offsets &&
                   (C == 0 || (coefficient_terms && coefficient_values)) && (S == 0 || (term_components && term_exponents)),
               "NULL argument");
  if (C > 0) {
    const MonomialTable t = {nullptr, term_offsets, term_components, term_exponents, coefficient_terms, nullptr, D, M, S, C, O};
    const int rc = launch_tiles(dtype, nullptr, x, batch, t, output_offsets, coefficient_values, out, as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  SPARSE_DISPATCH(sparse_monomial_kernel, grid_for(batch * O, 256), (const Real*)x, batch, D, term_offsets,
                  term_components, term_exponents, output_offsets, coefficient_terms, (const Real*)coefficient_values,
                  O, (Real*)out);
  (void)M;
  return check_launch("sparse_monomial_kernel");
}

int ye3t_hip_symmetric_power_shared_sparse_monomial_adjoint(
    int dtype, const void* output_adjoint, const void* x, int64_t batch, int64_t D, const int64_t* term_offsets,
    const int64_t* term_components, const int64_t* term_exponents, int64_t M, int64_t S,
    const int64_t* output_offsets, const int64_t* coefficient_terms, const void* coefficient_values, int64_t C,
    int64_t O, void* input_adjoint, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && M >= 0 && S >= 0 && C >= 0 && O >= 0, "negative size");
  if (batch * D == 0) return YE3T_OK;
  YE3T_REQUIRE(x && input_adjoint && output_offsets && term_offsets &&
                   (C == 0 || (output_adjoint && coefficient_terms && coefficient_values)) &&
                   (S == 0 || (term_components && term_exponents)),
               "NULL argument");
  if (C > 0) {
    const MonomialTable t = {nullptr, term_offsets, term_components, term_exponents, coefficient_terms, nullptr, D, M, S, C, O};
    const int rc = launch_tiles(dtype, output_adjoint, x, batch, t, output_offsets, coefficient_values, input_adjoint,
                                as_stream(stream));
    if (rc != YE3T_EUNSUPPORTED) return rc;
  }
  SPARSE_DISPATCH(sparse_monomial_adjoint_kernel, grid_for(batch, 256), (const Real*)output_adjoint, (const Real*)x,
                  batch, D, term_offsets, term_components, term_exponents, output_offsets, coefficient_terms,
                  (const Real*)coefficient_values, O, (Real*)input_adjoint);
  (void)M;
  return check_launch("sparse_monomial_adjoint_kernel");
}

int ye3t_hip_symmetric_power_shared_sparse_monomial_double_backward(
    int dtype, const void* input_adjoint_tangent, const void* output_adjoint, const void* x, int64_t batch,
    int64_t D, const int64_t* term_offsets, const int64_t* term_components, const int64_t* term_exponents, int64_t M,
    int64_t S, const int64_t* output_offsets, const int64_t* coefficient_terms, const void* coefficient_values,
    int64_t C, int64_t O, void* output_tangent, void* input_tangent, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(batch >= 0 && D >= 0 && M >= 0 && S >= 0 && C >= 0 && O >= 0, "negative size");
  YE3T_REQUIRE((batch * O == 0 || output_tangent) && (batch * D == 0 || input_tangent), "NULL argument");
  if (batch == 0) return YE3T_OK;
  YE3T_REQUIRE(x && output_offsets && term_offsets && (D == 0 || input_adjoint_tangent) &&
                   (C == 0 || (output_adjoint && coefficient_terms && coefficient_values)) &&
                   (S == 0 || (term_components && term_exponents)),
               "NULL argument");
  if (O > 0) {
    SPARSE_DISPATCH(sparse_monomial_tangent_kernel, grid_for(batch * O, 256), (const Real*)input_adjoint_tangent,
                    (const Real*)x, batch, D, term_offsets, term_components, term_exponents, output_offsets,
                    coefficient_terms, (const Real*)coefficient_values, O, (Real*)output_tangent);
    const int rc = check_launch("sparse_monomial_tangent_kernel");
    if (rc != YE3T_OK) return rc;
  }
  if (D > 0) {
    SPARSE_DISPATCH(sparse_monomial_hessian_kernel, grid_for(batch, 256), (const Real*)input_adjoint_tangent,
                    (const Real*)output_adjoint, (const Real*)x, batch, D, term_offsets, term_components,
                    term_exponents, output_offsets, coefficient_terms, (const Real*)coefficient_values, O,
                    (Real*)input_tangent);
    return check_launch("sparse_monomial_hessian_kernel");
  }
  (void)M;
  return YE3T_OK;
}

}  // extern "C"
