// ye3t_hip: library bookkeeping (errors, ABI, device caps, SH normalisation)
// and the standalone per-edge tables (radial, real SH) and CSR density scatter.
#include <cmath>
#include <mutex>

#include "common.h"
#include "sph.h"

namespace ye3t {

namespace {
thread_local std::string g_last_error;
thread_local const char* g_last_density_kernel = "";
thread_local const char* g_last_kernel = "";
}

void set_density_kernel(const char* name) { g_last_density_kernel = name; }
void set_last_kernel(const char* name) { g_last_kernel = name; }

int set_error(int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

void clear_error() { g_last_error.clear(); }

const NormTable& norm_table() {
  static NormTable table;
  static std::once_flag once;
  std::call_once(once, [] {
    for (int l = 0; l <= kMaxL; ++l) {
      for (int m = 0; m <= kMaxL; ++m) {
        double v = 0.0;
        if (m <= l) {
          // (2l+1)/(4 pi) * (l-m)!/(l+m)!  computed as a product of reciprocals
          double ratio = 1.0;
          for (int k = l - m + 1; k <= l + m; ++k) ratio /= double(k);
          v = std::sqrt((2.0 * l + 1.0) / (4.0 * M_PI) * ratio);
        }
        table.v[l * (kMaxL + 1) + m] = v;
      }
    }
    table.inv[0] = 0.0;
    for (int k = 1; k < 2 * kMaxL + 2; ++k) table.inv[k] = 1.0 / double(k);
  });
  return table;
}

// ---------------------------------------------------------------------------
inline unsigned grid_for(int64_t work, int threads) {
  int64_t g = (work + threads - 1) / threads;
  if (g < 1) g = 1;
  if (g > (1 << 20)) g = 1 << 20;
  return unsigned(g);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// The per-edge tables.  An edge's row is 25 to 200 values, so a lane that
// stores its own row puts 64 lines under every store; both kernels write their
// rows to an LDS tile instead and copy the tile out, which is contiguous in the
// table, 16 bytes a lane.  Bound by those writes: 640 000 edges with n_max 10,
// l_max 4 and gradients in fp64 are 640 MB.  Kernel trace there: radial
// 78 -> 28 us, harmonics 519 -> 94 us (lane-wise stores, the harmonics' recurrences in
// 1.5 KB of scratch a lane).

// Copies a tile of `rows` x W values (row pitch P in LDS) to `out`: 16 bytes a
// lane, single values where `out` is not aligned for that and past the last
// whole vector.
template <int W, int P, typename Real>
__device__ inline void copy_rows(const Real* __restrict__ tile, int rows, Real* __restrict__ out) {
  constexpr int V = 16 / int(sizeof(Real));
  typedef Real vec __attribute__((ext_vector_type(V)));
  const int n = rows * W;
  int done = 0;
  if (reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    done = n / V * V;
    for (int i = int(threadIdx.x) * V; i < done; i += int(blockDim.x) * V) {
      vec v;
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const unsigned r = unsigned(i + q) / unsigned(W);
        v[q] = tile[r * P + (unsigned(i + q) - r * W)];
      }
      *reinterpret_cast<vec*>(out + i) = v;
    }
  }
  for (int i = done + int(threadIdx.x); i < n; i += int(blockDim.x)) {
    const unsigned r = unsigned(i) / unsigned(W);
    out[i] = tile[r * P + (unsigned(i) - r * W)];
  }
}

// Radial table: lane = edge, one Chebyshev pass over n.  128 edges a
// workgroup: 34 KB of tile at 16 fp64 values and derivatives, four workgroups
// in a compute unit.
constexpr int kRadialRows = 128;

template <int NR, bool DERIVS, typename Real>
__global__ __launch_bounds__(kRadialRows) void radial_table_kernel(const Real* __restrict__ radii,
                                                                   const Real* __restrict__ cutoffs,
                                                                   const Real* __restrict__ lambdas, int64_t E,
                                                                   Real* __restrict__ values,
                                                                   Real* __restrict__ derivs) {
  constexpr int P = NR | 1;  // odd: consecutive rows start in different banks
  __shared__ Real vt[kRadialRows * P];
  __shared__ Real dt[DERIVS ? kRadialRows * P : 1];
  const int t = threadIdx.x;
  for (int64_t e0 = int64_t(blockIdx.x) * kRadialRows; e0 < E; e0 += int64_t(gridDim.x) * kRadialRows) {
    const int rows = E - e0 < kRadialRows ? int(E - e0) : kRadialRows;
    if (t < rows) {
      // The basis is evaluated in fp64 for both storage types: the Chebyshev
      // recurrence amplifies rounding of the warped variable by ~n^2.
      double v[NR], d[NR];
      cheb_exp_cos_row<double, DERIVS>(double(radii[e0 + t]), double(cutoffs[e0 + t]), double(lambdas[e0 + t]), NR - 1,
                                       v, d);
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        vt[t * P + n] = Real(v[n]);
        if (DERIVS) dt[t * P + n] = Real(d[n]);
      }
    }
    __syncthreads();
    copy_rows<NR, P>(vt, rows, values + e0 * NR);
    if (DERIVS) copy_rows<NR, P>(dt, rows, derivs + e0 * NR);
    __syncthreads();  // the tile is read before the next one is written
  }
}

template <int NR, typename Real>
int launch_radial(int nr, const Real* radii, const Real* cutoffs, const Real* lambdas, int64_t E, Real* values,
                  Real* derivs, hipStream_t s) {
  if constexpr (NR < 16) {
    if (nr > NR) return launch_radial<NR + 1>(nr, radii, cutoffs, lambdas, E, values, derivs, s);
  }
  const dim3 grid{grid_for(E, kRadialRows)};
  if (derivs) {
    hipLaunchKernelGGL((radial_table_kernel<NR, true, Real>), grid, dim3(kRadialRows), 0, s, radii, cutoffs, lambdas, E,
                       values, derivs);
  } else {
    hipLaunchKernelGGL((radial_table_kernel<NR, false, Real>), grid, dim3(kRadialRows), 0, s, radii, cutoffs, lambdas, E,
                       values, derivs);
  }
  return check_launch("radial_table_kernel");
}

// Scheduled radial-angular edge channels: output (e, k) is
// scale_k R[e, ri_k] Y[e, ai_k] when channel k takes every edge type
// (type -1) or edge e's type, zero otherwise, with its Cartesian derivative
// scale_k (dR[e, ri_k] dir[e] Y[e, ai_k] + R[e, ri_k] dY[e, ai_k]).  The
// products are rounded in the reference core's order
// (ye3t_runtime_core.cpp:1550-1604) with no fused multiply-adds, so the
// results are the core's bit for bit.  Indices are validated by the caller;
// the kernel clamps them into the tables rather than faulting.
//
// Four values are written for each of E K outputs; those writes bound it.  A
// workgroup takes whole edges, up to about 4 096 outputs, with their table rows
// and the schedule in LDS (an output reads ten values, each of them shared by a
// row of others) and lane = output; the three components of a wave's 64 outputs
// go through LDS too, so that every store is contiguous.  240 000 edges x 144
// channels in fp64 (1.1 GB written): 425 -> 250 us (one thread an output with
// a 64-bit division and 24-byte strided stores before; 354 us with the rows
// read from memory).  Fewer outputs a workgroup where that leaves compute units
// without one: 1 000 edges x 144 11.5 -> 5.3 us (one thread an output: 5.3).
// Rows are held only where the channels read most of them: 100 channels of
// 1 000 harmonics, fp32, 100 000 edges, 907 us held, 223 from memory; 12
// channels of 3 and 4, 200 000 edges, 22 and 24.
constexpr int kChannelThreads = 256;
constexpr int64_t kChannelTable = 1024;     // channels whose schedule is held in LDS (24 KB)
constexpr int64_t kChannelRows = 16 * 1024;  // bytes of edge rows held in LDS: six workgroups a compute unit

template <typename Real>
struct ChannelSchedule {
  int64_t type;
  Real scale;
  int32_t ri, ai;
};

// HELD: the schedule and the edges' rows are in LDS.
template <bool HELD, typename Real>
__global__ __launch_bounds__(kChannelThreads) void scheduled_channels_kernel(
    const Real* __restrict__ rv, const Real* __restrict__ rd, const Real* __restrict__ av,
    const Real* __restrict__ ad, const Real* __restrict__ dir, const int64_t* __restrict__ edge_types,
    const int64_t* __restrict__ cri, const int64_t* __restrict__ cai, const int64_t* __restrict__ ctype,
    const Real* __restrict__ cscale, int64_t E, int64_t NR, int64_t NA, int64_t K, int64_t tile, int64_t part,
    Real* __restrict__ values, Real* __restrict__ derivs) {
#pragma clang fp contract(off)
  constexpr int V = 16 / int(sizeof(Real));
  typedef Real vec __attribute__((ext_vector_type(V)));
  extern __shared__ __align__(16) unsigned char channel_smem[];
  __shared__ __align__(16) Real stage[kChannelThreads / 64][192];
  auto schedule = [&](int64_t k) {
    ChannelSchedule<Real> c;
    const int64_t ri = cri[k], ai = cai[k];
    c.type = ctype[k];
    c.scale = cscale[k];
    c.ri = int32_t(ri < 0 ? 0 : (ri >= NR ? NR - 1 : ri));
    c.ai = int32_t(ai < 0 ? 0 : (ai >= NA ? NA - 1 : ai));
    return c;
  };
  const int64_t e0 = int64_t(blockIdx.x) * tile;
  const int64_t edges = E - e0 < tile ? E - e0 : tile;
  ChannelSchedule<Real>* const table = reinterpret_cast<ChannelSchedule<Real>*>(channel_smem);
  int64_t* const type = reinterpret_cast<int64_t*>(table + (HELD ? K : 0));
  Real* const srv = reinterpret_cast<Real*>(type + (HELD ? tile : 0));
  Real* const srd = srv + (HELD ? tile * NR : 0);
  Real* const sav = srd + (HELD ? tile * NR : 0);
  Real* const sad = sav + (HELD ? tile * NA : 0);
  Real* const sdir = sad + (HELD ? tile * NA * 3 : 0);
  if (HELD) {
    auto hold = [&](Real* to, const Real* from, int64_t n) {
      for (int64_t i = threadIdx.x; i < n; i += kChannelThreads) to[i] = from[i];
    };
    for (int64_t k = threadIdx.x; k < K; k += kChannelThreads) table[k] = schedule(k);
    for (int64_t i = threadIdx.x; i < edges; i += kChannelThreads) type[i] = edge_types[e0 + i];
    hold(srv, rv + e0 * NR, edges * NR);
    hold(srd, rd + e0 * NR, edges * NR);
    hold(sav, av + e0 * NA, edges * NA);
    hold(sad, ad + e0 * NA * 3, edges * NA * 3);
    hold(sdir, dir + e0 * 3, edges * 3);
    __syncthreads();
  }
  const int64_t first = int64_t(blockIdx.y) * part;  // this workgroup's part of the tile's outputs
  const int64_t outputs = edges * K < first + part ? edges * K : first + part;
  const int64_t o0 = e0 * K;
  const int lane = threadIdx.x & 63;
  Real* const mine = stage[threadIdx.x >> 6];
  const bool aligned = reinterpret_cast<uintptr_t>(derivs + 3 * o0) % 16 == 0;
  // the lane's channel and edge (of the tile) advance by 256 outputs a step
  const int dk = int(kChannelThreads % K), de = int(kChannelThreads / K);
  int64_t e = (first + threadIdx.x) / K, k = first + threadIdx.x - e * K;
  for (int64_t w = first + threadIdx.x - lane; w < outputs; w += kChannelThreads) {
    const int left = outputs - w < 64 ? int(outputs - w) : 64;  // outputs of this wave's step
    if (lane < left) {
      const ChannelSchedule<Real> c = HELD ? table[k] : schedule(k);
      Real v = Real(0), d0 = Real(0), d1 = Real(0), d2 = Real(0);
      if (!(c.type >= 0 && (HELD ? type[e] : edge_types[e0 + e]) != c.type)) {
        const int64_t row = HELD ? e : e0 + e;
        const Real r = (HELD ? srv : rv)[row * NR + c.ri], dr = (HELD ? srd : rd)[row * NR + c.ri];
        const Real a = (HELD ? sav : av)[row * NA + c.ai], sc = c.scale;
        const Real* const ya = (HELD ? sad : ad) + 3 * (row * NA + c.ai);
        const Real* const u = (HELD ? sdir : dir) + 3 * row;
        v = sc * r * a;
        d0 = sc * (dr * u[0] * a + r * ya[0]);
        d1 = sc * (dr * u[1] * a + r * ya[1]);
        d2 = sc * (dr * u[2] * a + r * ya[2]);
      }
      values[o0 + w + lane] = v;
      mine[3 * lane] = d0;
      mine[3 * lane + 1] = d1;
      mine[3 * lane + 2] = d2;
    }
    // the wave's own 192 components: written by its lanes, read by others of them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    Real* const out = derivs + 3 * (o0 + w);
    const int n = 3 * left;
    const int whole = aligned ? n / V * V : 0;
    for (int i = lane * V; i < whole; i += 64 * V)
      *reinterpret_cast<vec*>(out + i) = *reinterpret_cast<const vec*>(mine + i);
    for (int i = whole + lane; i < n; i += 64) out[i] = mine[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    e += de;
    k += dk;
    if (k >= K) {
      k -= K;
      ++e;
    }
  }
}

template <typename Real>
int launch_channels(const Real* rv, const Real* rd, const Real* av, const Real* ad, const Real* dir,
                    const int64_t* types, const int64_t* cri, const int64_t* cai, const int64_t* ctype,
                    const Real* cscale, int64_t E, int64_t NR, int64_t NA, int64_t K, Real* values, Real* derivs,
                    hipStream_t s) {
  // outputs of a workgroup: 4 096, or fewer where that leaves compute units
  // without one; edges: as many as have those, an even number (rows of three
  // fp64 values start on 16 bytes every second output), as far as their rows
  // fit; a tile of two edges with more outputs than that is shared by several
  int64_t part = (E * K / 1024 + kChannelThreads - 1) / kChannelThreads * kChannelThreads;
  part = part < kChannelThreads ? kChannelThreads : (part > 4096 ? 4096 : part);
  int64_t tile = part / K;
  tile = tile < 2 ? 2 : tile / 2 * 2;
  while (tile * K > part * 65535) part *= 2;  // the second grid axis' limit
  const int64_t parts = tile * K <= part + part / 2 ? 1 : (tile * K + part - 1) / part;
  if (parts == 1) part = tile * K;
  // held: whole edges, and rows of which the channels read most
  const int64_t row = (2 * NR + 4 * NA + 3) * int64_t(sizeof(Real)) + 8;
  const int64_t fit = kChannelRows / row / 2 * 2;
  const bool held = parts == 1 && K <= kChannelTable && fit >= 2 && 2 * NR + 4 * NA <= 8 * K;
  if (held && tile > fit) {
    tile = fit;
    part = tile * K;
  }
  const int64_t groups = (E + tile - 1) / tile;
  YE3T_REQUIRE(fits_grid(groups, kChannelThreads), "too many edges for one launch");  // from 500 GB of rows on
  const dim3 grid{unsigned(groups), unsigned(parts)};
  if (held) {
    hipLaunchKernelGGL((scheduled_channels_kernel<true, Real>), grid, dim3(kChannelThreads),
                       size_t(K) * sizeof(ChannelSchedule<Real>) + size_t(tile * row), s, rv, rd, av, ad, dir, types,
                       cri, cai, ctype, cscale, E, NR, NA, K, tile, part, values, derivs);
  } else {
    hipLaunchKernelGGL((scheduled_channels_kernel<false, Real>), grid, dim3(kChannelThreads), 0, s, rv, rd, av, ad, dir,
                       types, cri, cai, ctype, cscale, E, NR, NA, K, tile, part, values, derivs);
  }
  return check_launch("scheduled_channels_kernel");
}

// Real SH table with optional Cartesian gradient for a compile-time LMAX: lane
// = edge of a tile of T, and each of four waves takes the orders m of MASK
// (about a quarter of the components), all in registers.  The tile holds whole
// rows, up to 100 KB at l_max 6 in fp64, so it is the four waves on one tile that
// keep a compute unit busy; above that (l_max 7 and 8 in fp64) a tile has 32
// edges.  Gradients w.r.t. the unit vector use d/dz Q_l^m = Q_l^{m+1},
// projected with (I - u u^T) / |r| (reference ye3t_runtime_core.cpp:226-286,
// 808-843).
template <int LMAX>
constexpr unsigned sph_orders(int wave) {
  return wave == 0 ? 0x02u | (LMAX == 7 ? 0x80u : 0x100u)
         : wave == 1 ? 0x04u | (LMAX == 5 ? 0x20u : 0x40u)
         : wave == 2 ? 0x08u | (LMAX <= 5 ? 0x10u : 0x20u)
                     : 0x01u | (LMAX <= 5 ? 0u : 0x10u) | (LMAX == 8 ? 0x80u : 0u);
}

template <int LMAX, unsigned MASK, bool GRAD, typename Real>
__device__ inline void sph_tile_rows(const double (&u)[3], double sr, bool project, const NormTable& nt,
                                     Real* __restrict__ row, Real* __restrict__ grow) {
  const double sqrt2 = 1.4142135623730950488016887242096981;
  double cr = 1.0, ci = 0.0, pr = 1.0, pi = 0.0;  // (x + i y)^m and ^(m-1)
  double qmm = 1.0;                               // Q_m^m
  const double inv = 1.0 / sr;
  const double rem = sr == HUGE_VAL ? 0.0 : sr;  // a length that overflows has gradient zero
  // the gradient (gx, gy, gz) w.r.t. u of component k, taken to the vector and stored
  auto put = [&](int k, double gx, double gy, double gz) {
    if (project) {
      const double ug = u[0] * gx + u[1] * gy + u[2] * gz;
      gx -= u[0] * ug;
      gy -= u[1] * ug;
      gz -= u[2] * ug;
    }
    // g / sr, the reciprocal's product corrected by its remainder
    auto over = [&](double g) {
      const double q = g * inv;
      return fma(fma(-q, rem, g), inv, q);
    };
    grow[3 * k] = Real(over(gx));
    grow[3 * k + 1] = Real(over(gy));
    grow[3 * k + 2] = Real(over(gz));
  };
#pragma unroll
  for (int m = 0; m <= LMAX; ++m) {
    if (m > 0) {
      qmm *= double(2 * m - 1);
      pr = cr;
      pi = ci;
      const double nr = cr * u[0] - ci * u[1];
      const double ni = cr * u[1] + ci * u[0];
      cr = nr;
      ci = ni;
    }
    if (((MASK >> m) & 1) == 0) continue;
    // q: Q_l^m, d: Q_l^{m+1}, by their recurrences in l
    const double dmm = qmm * double(2 * m + 1);
    double q2 = 0.0, q1 = 0.0, d2 = 0.0, d1 = 0.0;
#pragma unroll
    for (int l = m; l <= LMAX; ++l) {
      double q, d = 0.0;
      if (l == m) {
        q = qmm;
      } else if (l == m + 1) {
        q = double(2 * m + 1) * u[2] * qmm;
        d = dmm;
      } else {
        q = (double(2 * l - 1) * u[2] * q1 - double(l + m - 1) * q2) / double(l - m);
        d = l == m + 2 ? double(2 * m + 3) * u[2] * dmm
                       : (double(2 * l - 1) * u[2] * d1 - double(l + m) * d2) / double(l - m - 1);
      }
      q2 = q1;
      q1 = q;
      d2 = d1;
      d1 = d;
      const double n = nt.v[l * (kMaxL + 1) + m];
      const int base = l * l + l;
      if (m == 0) {
        row[base] = Real(n * q);
        if (GRAD) put(base, 0.0, 0.0, n * d);
      } else {
        const double s = sqrt2 * n;
        row[base + m] = Real(s * q * cr);
        row[base - m] = Real(-s * q * ci);
        if (GRAD) {
          const double mq = s * q * double(m), sd = s * d;
          put(base + m, mq * pr, -mq * pi, sd * cr);
          put(base - m, -mq * pi, -mq * pr, -sd * ci);
        }
      }
    }
  }
}

template <int LMAX, bool GRAD, int T, typename Real>
__global__ __launch_bounds__(256) void sph_tile_kernel(const Real* __restrict__ vec, int64_t E, double eps,
                                                       NormTable nt, Real* __restrict__ values,
                                                       Real* __restrict__ grads) {
  constexpr int W = (LMAX + 1) * (LMAX + 1);
  constexpr int P = W | 1, GP = 3 * W | 1;  // odd: consecutive rows start in different banks
  __shared__ Real vt[T * P];
  __shared__ Real gt[GRAD ? T * GP : 1];
  const int64_t e0 = int64_t(blockIdx.x) * T;
  const int rows = E - e0 < T ? int(E - e0) : T;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (lane < rows) {
    const int64_t e = e0 + lane;
    const double x0 = double(vec[3 * e]), y0 = double(vec[3 * e + 1]), z0 = double(vec[3 * e + 2]);
    const double r = d_sqrt(x0 * x0 + y0 * y0 + z0 * z0);
    const double sr = r > eps ? r : eps;
    const double u[3] = {x0 / sr, y0 / sr, z0 / sr};
    Real* const row = vt + lane * P;
    Real* const grow = gt + (GRAD ? lane * GP : 0);
    const bool project = r > eps;
    if (wave == 0) sph_tile_rows<LMAX, sph_orders<LMAX>(0), GRAD>(u, sr, project, nt, row, grow);
    else if (wave == 1) sph_tile_rows<LMAX, sph_orders<LMAX>(1), GRAD>(u, sr, project, nt, row, grow);
    else if (wave == 2) sph_tile_rows<LMAX, sph_orders<LMAX>(2), GRAD>(u, sr, project, nt, row, grow);
    else sph_tile_rows<LMAX, sph_orders<LMAX>(3), GRAD>(u, sr, project, nt, row, grow);
  }
  __syncthreads();
  copy_rows<W, P>(vt, rows, values + e0 * W);
  if (GRAD) copy_rows<3 * W, GP>(gt, rows, grads + e0 * 3 * W);
}

// edges of a tile
constexpr int sph_tile_edges(int lmax, size_t elem) { return lmax > 6 && elem == 8 ? 32 : 64; }

template <int LMAX, typename Real>
int launch_sph_tile(int lmax, const Real* vec, int64_t E, double eps, Real* values, Real* grads, hipStream_t s) {
  if constexpr (LMAX < 8) {
    if (lmax > LMAX) return launch_sph_tile<LMAX + 1>(lmax, vec, E, eps, values, grads, s);
  }
  constexpr int T = sph_tile_edges(LMAX, sizeof(Real));
  const dim3 grid{unsigned((E + T - 1) / T)};
  if (grads) {
    hipLaunchKernelGGL((sph_tile_kernel<LMAX, true, T, Real>), grid, dim3(256), 0, s, vec, E, eps, norm_table(), values,
                       grads);
  } else {
    hipLaunchKernelGGL((sph_tile_kernel<LMAX, false, T, Real>), grid, dim3(256), 0, s, vec, E, eps, norm_table(),
                       values, grads);
  }
  return check_launch("sph_tile_kernel");
}

// The same table for any l_max and edge count (l_max 9 and above, and more edges
// than one grid has tiles): one lane per edge, the recurrences in scratch.
template <typename Real>
__global__ __launch_bounds__(128) void real_sph_table_kernel(const Real* __restrict__ vec, int64_t E, int lmax,
                                                             double eps, NormTable nt, Real* __restrict__ values,
                                                             Real* __restrict__ grads) {
  const int width = (lmax + 1) * (lmax + 1);
  const double sqrt2 = double(1.4142135623730950488016887242096981);
  for (int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < E; e += int64_t(gridDim.x) * blockDim.x) {
    const double x0 = double(vec[3 * e]), y0 = double(vec[3 * e + 1]), z0 = double(vec[3 * e + 2]);
    const double r = d_sqrt(x0 * x0 + y0 * y0 + z0 * z0);
    const double sr = r > eps ? r : eps;
    const double u[3] = {x0 / sr, y0 / sr, z0 / sr};
    Real* row = values + e * width;
    if (!grads) {
      double yrow[(kMaxL + 1) * (kMaxL + 1)];
      real_sph_row<double>(u[0], u[1], u[2], lmax, nt, yrow, 1);
      for (int k = 0; k < width; ++k) row[k] = Real(yrow[k]);
      continue;
    }
    // Q[l][m] for m <= l+1 (Q_l^{l+1} = 0)
    double Q[kMaxL + 2][kMaxL + 2];
    double qmm = double(1);
    for (int m = 0; m <= lmax + 1; ++m) {
      if (m > 0) qmm *= double(2 * m - 1);
      double q2 = double(0), q1 = double(0);
      for (int l = 0; l <= lmax; ++l) {
        double q;
        if (l < m) {
          q = double(0);
        } else if (l == m) {
          q = qmm;
        } else if (l == m + 1) {
          q = double(2 * m + 1) * u[2] * qmm;
        } else {
          q = (double(2 * l - 1) * u[2] * q1 - double(l + m - 1) * q2) / double(l - m);
        }
        if (l >= m) {
          q2 = q1;
          q1 = q;
        }
        Q[l][m] = q;
      }
    }
    double cr = double(1), ci = double(0), pr = double(1), pi = double(0);
    for (int m = 0; m <= lmax; ++m) {
      if (m > 0) {
        pr = cr;
        pi = ci;
        const double nr = cr * u[0] - ci * u[1];
        const double ni = cr * u[1] + ci * u[0];
        cr = nr;
        ci = ni;
      }
      for (int l = m; l <= lmax; ++l) {
        const double n = double(nt.v[l * (kMaxL + 1) + m]);
        const int base = l * l + l;
        double ug[2][3];
        int idx[2];
        int count;
        if (m == 0) {
          row[base] = Real(n * Q[l][0]);
          ug[0][0] = double(0);
          ug[0][1] = double(0);
          ug[0][2] = n * Q[l][1];
          idx[0] = base;
          count = 1;
        } else {
          const double s = sqrt2 * n;
          const double q = Q[l][m], qz = Q[l][m + 1];
          row[base + m] = Real(s * q * cr);
          row[base - m] = Real(-s * q * ci);
          ug[0][0] = s * q * (double(m) * pr);
          ug[0][1] = s * q * (-double(m) * pi);
          ug[0][2] = s * qz * cr;
          ug[1][0] = -s * q * (double(m) * pi);
          ug[1][1] = -s * q * (double(m) * pr);
          ug[1][2] = -s * qz * ci;
          idx[0] = base + m;
          idx[1] = base - m;
          count = 2;
        }
        for (int c = 0; c < count; ++c) {
          for (int a = 0; a < 3; ++a) {
            double g = double(0);
            for (int b = 0; b < 3; ++b) {
              double jac;
              if (r > eps) {
                jac = ((a == b ? double(1) : double(0)) - u[a] * u[b]) / sr;
              } else {
                jac = (a == b) ? double(1) / sr : double(0);
              }
              g += ug[c][b] * jac;
            }
            grads[(e * width + idx[c]) * 3 + a] = Real(g);
          }
        }
      }
    }
  }
}

// CSR segment reduction: thread per (atom, channel), edges summed in order.
template <typename Real>
__global__ __launch_bounds__(256) void density_csr_kernel(const Real* __restrict__ ev,
                                                          const int64_t* __restrict__ offsets, int64_t N,
                                                          int64_t C, Real* __restrict__ out) {
  const int64_t total = N * C;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t i = idx / C, c = idx - (idx / C) * C;
    Real acc = Real(0);
    for (int64_t e = offsets[i]; e < offsets[i + 1]; ++e) acc += ev[e * C + c];
    out[idx] = acc;
  }
}

// Row offsets of centre-sorted edges: lane = row, a bisection for the first
// edge whose centre is not below it (any run of empty rows costs the same).
__global__ __launch_bounds__(256) void csr_offsets_kernel(const int64_t* __restrict__ centers, int64_t E, int64_t N,
                                                          int64_t* __restrict__ offsets) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i <= N; i += int64_t(gridDim.x) * blockDim.x) {
    int64_t lo = 0, hi = E;  // centers[lo - 1] < i <= centers[hi]
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (centers[mid] < i) lo = mid + 1;
      else hi = mid;
    }
    offsets[i] = lo;
  }
}

// Gather of centre-row adjoints to edge rows.  A workgroup copies 256 vectors
// at a time (V = 16 bytes when the rows allow it), STEPS steps over consecutive
// vectors of the edge rows with every step's read requested before the first
// write; the output is streamed with non-temporal stores (written once, not
// re-read here).  Centres are validated by the caller; an index outside [0, N)
// is clamped so that no access leaves the array.  Eight steps where the copies
// do not fit the caches any more, one where more workgroups count: fp64, 144
// channels, 240 000 edges (17 million vectors) after the sums of the same call
// 92 us by one step, 70 by four, 67 by eight; by itself 20 000 edges (1.4
// million) 5.5 by one and 7.5 by eight, 225 channels (single values) of 100 000
// edges (23 million) 53 and 40.
constexpr int64_t kGatherLarge = 5000000;  // vectors

template <int STEPS, typename Index, typename V>
__global__ __launch_bounds__(256) void density_adjoint_kernel(const V* __restrict__ adj,
                                                              const int64_t* __restrict__ centers, int64_t E,
                                                              int64_t CV, int64_t N, V* __restrict__ out) {
  const int64_t total = E * CV;
  const int64_t dc = 256 % CV, de = 256 / CV;
  for (int64_t x0 = int64_t(blockIdx.x) * (256 * STEPS); x0 < total; x0 += int64_t(gridDim.x) * (256 * STEPS)) {
    const int64_t x = x0 + threadIdx.x;
    int64_t e = Index(x) / Index(CV), c = x - e * CV;
    V v[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
      if (x + 256 * k < total) {
        int64_t i = centers[e];
        i = i < 0 ? 0 : (i >= N ? N - 1 : i);
        v[k] = adj[i * CV + c];
      }
      e += de;
      c += dc;
      if (c >= CV) {
        c -= CV;
        ++e;
      }
    }
#pragma unroll
    for (int k = 0; k < STEPS; ++k)
      if (x + 256 * k < total) __builtin_nontemporal_store(v[k], out + x + 256 * k);
  }
}

template <typename V>
int launch_gather(const void* adj, const int64_t* centers, int64_t E, int64_t CV, int64_t N, void* out, hipStream_t s) {
  if (E * CV >= kGatherLarge) {
    hipLaunchKernelGGL((density_adjoint_kernel<8, int64_t, V>), dim3(grid_for(E * CV, 256 * 8)), dim3(256), 0, s,
                       static_cast<const V*>(adj), centers, E, CV, N, static_cast<V*>(out));
  } else {
    hipLaunchKernelGGL((density_adjoint_kernel<1, uint32_t, V>), dim3(grid_for(E * CV, 256)), dim3(256), 0, s,
                       static_cast<const V*>(adj), centers, E, CV, N, static_cast<V*>(out));
  }
  return check_launch("density_adjoint_kernel");
}

// Range checks of index inputs in one pass over them, one grid row an array:
// nothing is reduced, a lane that sees a violation stores its word of `status`
// (host memory the device can write, zeroed by the host), and the first and
// last values are copied there.  A structure of 50 000 atoms and 1.2 M edges is
// 10 MB, about 4 us of reads; taken as torch reductions with a read-back each
// (minimum and maximum of the neighbours, first and last offset, monotony) the
// same checks are six kernels and five synchronisations: a 16-channel density
// and product of 50 000 atoms took 260 us with those, 169 us with this, and
// one of 128 atoms 110 and 40 us.
struct IndexChecks {
  ye3t_index_check c[YE3T_MAX_CHECKS];
};

template <typename T>
__device__ inline void check_one(const ye3t_index_check& c, int64_t* __restrict__ status) {
  const T* __restrict__ v = static_cast<const T*>(c.data);
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t == 0) {
    status[0] = int64_t(v[0]);
    status[1] = int64_t(v[c.count - 1]);
  }
  for (int64_t k = t; k < c.count; k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t x = int64_t(v[k]);
    if (x < c.first || x >= c.limit) status[2] = 1;
    if (c.ordered && k > 0 && int64_t(v[k - 1]) > x) status[3] = 1;
  }
}

__global__ __launch_bounds__(256) void check_indices_kernel(IndexChecks checks, int64_t* __restrict__ status) {
  const ye3t_index_check& c = checks.c[blockIdx.y];
  if (c.count == 0) return;
  if (c.width == 8) check_one<int64_t>(c, status + 4 * blockIdx.y);
  else check_one<int32_t>(c, status + 4 * blockIdx.y);
}

// The status words of the calling thread: pinned host memory, made at the
// thread's first check and freed when the thread ends.  A check waits for its
// kernel before it returns, so one set per thread is enough for any number of
// streams.
struct CheckStatus {
  int64_t* words = nullptr;
  ~CheckStatus() {
    if (words != nullptr) (void)hipHostFree(words);
  }
};
constexpr int kCheckWords = 4 * YE3T_MAX_CHECKS;


}  // namespace ye3t

using namespace ye3t;

extern "C" {

int ye3t_hip_abi_version(void) { return YE3T_HIP_ABI_VERSION; }

int ye3t_hip_has_hip(void) {
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return count > 0 ? 1 : 0;
}

int ye3t_hip_has_cpu(void) { return 0; }

const char* ye3t_hip_last_error(void) { return g_last_error.c_str(); }

const char* ye3t_hip_last_density_kernel(void) { return g_last_density_kernel; }

const char* ye3t_hip_last_kernel(void) { return g_last_kernel; }

int ye3t_hip_device_caps(int device, ye3t_hip_caps* out) {
  YE3T_REQUIRE(out != nullptr, "caps output is NULL");
  hipDeviceProp_t prop;
  YE3T_CHECK_HIP(hipGetDeviceProperties(&prop, device));
  std::snprintf(out->arch, sizeof out->arch, "%s", prop.gcnArchName);
  out->device = device;
  out->cu_count = prop.multiProcessorCount;
  out->wavefront_size = prop.warpSize;
  out->lds_bytes_per_block = int(prop.sharedMemPerBlock);
  out->clock_khz = prop.clockRate;
  out->hbm_bytes = int64_t(prop.totalGlobalMem);
  out->hbm_peak_gbs = 8000.0;  // MI355X nominal HBM3E peak
  return YE3T_OK;
}

int ye3t_hip_radial_table(int dtype, const void* radii, const void* cutoffs, const void* lambdas, int64_t E,
                          int64_t n_max, void* values, void* derivs, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(E >= 0, "edge_count must be non-negative");
  YE3T_REQUIRE(n_max >= 0 && n_max < 16, "max_radial_index must be in [0, 15], got %lld", (long long)n_max);
  if (E == 0) return YE3T_OK;
  YE3T_REQUIRE(radii && cutoffs && lambdas && values, "NULL input or output");
  if (dtype == YE3T_F64)
    return launch_radial<1>(int(n_max) + 1, (const double*)radii, (const double*)cutoffs, (const double*)lambdas, E,
                            (double*)values, (double*)derivs, as_stream(stream));
  if (dtype == YE3T_F32)
    return launch_radial<1>(int(n_max) + 1, (const float*)radii, (const float*)cutoffs, (const float*)lambdas, E,
                            (float*)values, (float*)derivs, as_stream(stream));
  return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
}

int ye3t_hip_scheduled_radial_angular_channels(int dtype, int64_t edge_count, int64_t radial_width,
                                               int64_t angular_width, int64_t channel_count,
                                               const void* radial_values, const void* radial_derivatives,
                                               const void* angular_values, const void* angular_derivatives,
                                               const void* radial_directions, const int64_t* edge_types,
                                               const int64_t* channel_radial_indices,
                                               const int64_t* channel_angular_indices,
                                               const int64_t* channel_types, const void* channel_scales,
                                               void* edge_values, void* edge_derivatives, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(edge_count >= 0 && channel_count >= 0, "edge and channel counts must be non-negative");
  if (edge_count == 0 || channel_count == 0) return YE3T_OK;
  YE3T_REQUIRE(radial_width > 0 && angular_width > 0, "radial and angular tables must not be empty");
  YE3T_REQUIRE(edge_count <= INT64_MAX / channel_count / 3, "edge_count * channel_count overflows");
  YE3T_REQUIRE(radial_values && radial_derivatives && angular_values && angular_derivatives && radial_directions &&
                   edge_types && channel_radial_indices && channel_angular_indices && channel_types &&
                   channel_scales && edge_values && edge_derivatives,
               "NULL input or output");
  YE3T_REQUIRE(radial_width <= INT32_MAX && angular_width <= INT32_MAX, "tables too wide");
  if (dtype == YE3T_F64)
    return launch_channels((const double*)radial_values, (const double*)radial_derivatives,
                           (const double*)angular_values, (const double*)angular_derivatives,
                           (const double*)radial_directions, edge_types, channel_radial_indices,
                           channel_angular_indices, channel_types, (const double*)channel_scales, edge_count,
                           radial_width, angular_width, channel_count, (double*)edge_values,
                           (double*)edge_derivatives, as_stream(stream));
  if (dtype == YE3T_F32)
    return launch_channels((const float*)radial_values, (const float*)radial_derivatives, (const float*)angular_values,
                           (const float*)angular_derivatives, (const float*)radial_directions, edge_types,
                           channel_radial_indices, channel_angular_indices, channel_types,
                           (const float*)channel_scales, edge_count, radial_width, angular_width, channel_count,
                           (float*)edge_values, (float*)edge_derivatives, as_stream(stream));
  return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
}

int ye3t_hip_real_sph_table(int dtype, const void* vec, int64_t E, int64_t lmax, double eps, void* values,
                            void* grads, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(E >= 0, "edge_count must be non-negative");
  YE3T_REQUIRE(lmax >= 0 && lmax <= kMaxL, "maximum_angular_momentum must be in [0, %d]", kMaxL);
  if (E == 0) return YE3T_OK;
  YE3T_REQUIRE(vec && values, "NULL input or output");
  const int tile = sph_tile_edges(int(lmax), dtype == YE3T_F64 ? 8 : 4);
  if (lmax <= 8 && fits_grid((E + tile - 1) / tile, 256)) {
    if (dtype == YE3T_F64)
      return launch_sph_tile<0>(int(lmax), (const double*)vec, E, eps, (double*)values, (double*)grads, as_stream(stream));
    if (dtype == YE3T_F32)
      return launch_sph_tile<0>(int(lmax), (const float*)vec, E, eps, (float*)values, (float*)grads, as_stream(stream));
  }
  const unsigned grid = grid_for(E, 128);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(real_sph_table_kernel<double>, dim3(grid), dim3(128), 0, as_stream(stream),
                       (const double*)vec, E, int(lmax), eps, norm_table(), (double*)values, (double*)grads);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(real_sph_table_kernel<float>, dim3(grid), dim3(128), 0, as_stream(stream),
                       (const float*)vec, E, int(lmax), eps, norm_table(), (float*)values, (float*)grads);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  return check_launch("real_sph_table_kernel");
}

int ye3t_hip_density_accumulate_csr(int dtype, const void* ev, const int64_t* offsets, int64_t N, int64_t C,
                                    void* out, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(N >= 0 && C >= 0, "negative size");
  if (N * C == 0) return YE3T_OK;
  YE3T_REQUIRE(offsets && out, "NULL offsets or output");
  const unsigned grid = grid_for(N * C, 256);
  if (dtype == YE3T_F64) {
    hipLaunchKernelGGL(density_csr_kernel<double>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const double*)ev, offsets, N, C, (double*)out);
  } else if (dtype == YE3T_F32) {
    hipLaunchKernelGGL(density_csr_kernel<float>, dim3(grid), dim3(256), 0, as_stream(stream),
                       (const float*)ev, offsets, N, C, (float*)out);
  } else {
    return set_error(YE3T_EDTYPE, "unsupported dtype %d", dtype);
  }
  return check_launch("density_csr_kernel");
}

int ye3t_hip_check_indices(const ye3t_index_check* checks, int check_count, int64_t* result, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(check_count >= 1 && check_count <= YE3T_MAX_CHECKS, "between 1 and %d checks", YE3T_MAX_CHECKS);
  YE3T_REQUIRE(checks != nullptr && result != nullptr, "NULL checks or result");
  IndexChecks all = {};
  int64_t most = 0;
  for (int k = 0; k < check_count; ++k) {
    YE3T_REQUIRE(checks[k].count >= 0 && (checks[k].width == 4 || checks[k].width == 8), "bad index check");
    YE3T_REQUIRE(checks[k].count == 0 || checks[k].data != nullptr, "NULL indices");
    all.c[k] = checks[k];
    if (checks[k].count > most) most = checks[k].count;
  }
  const hipStream_t s = as_stream(stream);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  YE3T_CHECK_HIP(hipStreamIsCapturing(s, &capture));
  if (capture != hipStreamCaptureStatusNone)
    return set_error(YE3T_EUNSUPPORTED, "indices cannot be checked while the stream is captured");
  for (int k = 0; k < 4 * check_count; ++k) result[k] = 0;
  if (most == 0) return YE3T_OK;
  static thread_local CheckStatus status;
  if (status.words == nullptr) {
    void* words = nullptr;
    YE3T_CHECK_HIP(hipHostMalloc(&words, kCheckWords * sizeof(int64_t), hipHostMallocPortable | hipHostMallocMapped));
    status.words = static_cast<int64_t*>(words);
  }
  for (int k = 0; k < kCheckWords; ++k) status.words[k] = 0;
  // eight indices per lane: enough wavefronts to cover the latency of a short
  // read, and few enough workgroups for the smallest calls to start at once
  hipLaunchKernelGGL(check_indices_kernel, dim3(grid_for((most + 7) / 8, 256), unsigned(check_count)), dim3(256), 0, s,
                     all, status.words);
  const int rc = check_launch("check_indices_kernel");
  if (rc != YE3T_OK) return rc;
  YE3T_CHECK_HIP(hipStreamSynchronize(s));
  for (int k = 0; k < 4 * check_count; ++k) result[k] = status.words[k];
  return YE3T_OK;
}

int ye3t_hip_csr_offsets(const int64_t* centers, int64_t edge_count, int64_t atom_count, int64_t* row_offsets,
                         ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(edge_count >= 0 && atom_count >= 0, "negative size");
  YE3T_REQUIRE(row_offsets != nullptr && (edge_count == 0 || centers != nullptr), "NULL centres or output");
  hipLaunchKernelGGL(csr_offsets_kernel, dim3(grid_for(atom_count + 1, 256)), dim3(256), 0, as_stream(stream), centers,
                     edge_count, atom_count, row_offsets);
  return check_launch("csr_offsets_kernel");
}

int ye3t_hip_density_accumulate_adjoint(int dtype, const void* adj, const int64_t* centers, int64_t E, int64_t C,
                                        int64_t N, void* out, ye3t_stream_t stream) {
  clear_error();
  YE3T_REQUIRE(E >= 0 && C >= 0 && N >= 0, "negative size");
  if (E * C == 0) return YE3T_OK;
  YE3T_REQUIRE(N >= 1, "edges need at least one atom");
  YE3T_REQUIRE(adj && centers && out, "NULL input or output");
  const size_t elem = dtype == YE3T_F64 ? 8 : 4;
  YE3T_REQUIRE(dtype == YE3T_F64 || dtype == YE3T_F32, "unsupported dtype %d", dtype);
  const bool vec = (size_t(C) * elem) % 16 == 0 && reinterpret_cast<uintptr_t>(adj) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const hipStream_t s = as_stream(stream);
  const int64_t CV = vec ? int64_t(size_t(C) * elem / 16) : C;
  if (vec) return launch_gather<f32x4>(adj, centers, E, CV, N, out, s);
  if (dtype == YE3T_F64) return launch_gather<double>(adj, centers, E, CV, N, out, s);
  return launch_gather<float>(adj, centers, E, CV, N, out, s);
}

}  // extern "C"
