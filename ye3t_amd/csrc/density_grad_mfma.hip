// Edge-vector gradient of the stage-1 density (forces) on the fp64 matrix
// cores, for species (and single-channel) densities.  With the adjoint block
// g[n][k] of edge e's centre and channel (density_grad.hip states the whole
// formula), the per-edge sums
//
//   t_k = sum_n R_n g[n][k],   u_k = sum_n R'_n g[n][k],   a = sum_k u_k Y_k
//
// are products of an [edges x n] by an [n x k] matrix that all edges of one
// (atom, channel) group share.  The lane-per-edge kernel gathers the block once
// per edge: 637 loads an edge at n_max 12, l_max 6, from as many cache lines as
// a wave has groups.  Here one wave walks an equal share of the edges in chunks
// of whole atoms with at most 64 edges together (a share or an atom of more
// edges may end a chunk within an atom, whose groups are then read twice):
//   basis    lane = edge: radial values and derivatives and harmonics, to LDS
//            at the edge's column, columns grouped by (atom, channel);
//   product  per group; the block comes straight from global memory in the
//            B-operand layout, once, as full lines, requested four groups
//            ahead; each four edges take one v_mfma_f64_4x4x4 per four radial
//            rows and 16 components, so a group is padded to four edges and not
//            to the sixteen of the larger shape (its average is six at eight
//            species and 48 neighbours); t replaces Y in LDS;
//   chain    lane = edge: the gradient of the harmonics contracted with t.
// Measured (events): 8 species, n_max 12, l_max 6, 30 000 atoms x 48: 691 us for
// the lane-per-edge kernel, 465 us here; 4 species, n_max 10, l_max 4,
// 20 000 x 32: 121 and 97 us.  It is bound by one wave per SIMD
// (two at l_max 4) working through dependent fp64 instructions: the tile, 40 KB
// at l_max 6, limits how many are resident.  Without the block loads it takes
// 469 us, without the products 161.  Four waves sharing a tile, each with a
// part of the basis, the groups and the harmonics' orders, took 520-570 us
// (barriers, and the prologue four times); with 168 or 128 registers, for three
// or four of them per SIMD, they spilled and took 540-670 us.
// Lane layout of the 4x4x4 product (l = lane): A[i][k] in lanes i + 4 b + 16 k
// for every b, B[k][j] in lane j + 16 k, D[i][j] in lane j + 16 i, j < 16.
#include <cmath>

#include "common.h"
#include "density_grad.h"

namespace ye3t {
namespace {

constexpr int kGmPitch = 68;  // pitch (doubles) of the radial rows: operand reads of 4 rows x 4 columns meet no bank twice

__device__ inline uint64_t gm_ballot(bool v) { return __builtin_amdgcn_ballot_w64(v); }

// LDS written by some lanes of the wave is read by others
__device__ inline void gm_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL>
__device__ inline double gm_dpp(double x) {
  const long long v = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_update_dpp(0, int(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(v >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (long long)((uint64_t(uint32_t(hi)) << 32) | uint32_t(lo)));
}

// sum over each 16 lanes, in every one of them
__device__ inline double gm_sum16(double x) {
  x += gm_dpp<0xB1>(x);   // quad_perm [1, 0, 3, 2]
  x += gm_dpp<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  x += gm_dpp<0x141>(x);  // row_half_mirror
  x += gm_dpp<0x140>(x);  // row_mirror
  return x;
}

template <typename G>
__device__ inline G gm_load(__amdgpu_buffer_rsrc_t rb, unsigned voff, unsigned soff) {
  if constexpr (sizeof(G) == 8) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, voff, soff, 0));
  } else {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, voff, soff, 0));
  }
}

// Clamps, applied where a loaded index is used and not where it is loaded (a
// use waits for the load): out-of-range input is never dereferenced.
__device__ inline int64_t gm_clamp(int64_t i, int64_t n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }

// Up to 64 whole atoms with at most 64 edges together from edge e of atom a on,
// or 64 edges of an atom that has more of them left, of the edges before the
// wave's end.  `end` of lane j is the end of atom a + j relative to e.
struct GmChunk {
  int64_t a, e;
  int na, cnt;
  int end;
};

// offsets of the atoms after a, one per lane
template <typename In, typename G>
__device__ inline int64_t gm_window(const GradParams<In, G>& p, int64_t a, int lane) {
  return p.row_offsets[a + 1 + lane < p.N ? a + 1 + lane : p.N];
}

// lane 0's value
__device__ inline int64_t gm_first(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v))));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v) >> 32)));
  return int64_t((uint64_t(hi) << 32) | lo);
}

// For each of `key`, the last atom i with row_offsets[i] + per_atom * i <= key
// (atom 0 if there is none): 64 probes a step for all of them, three steps up
// to 262 144 atoms.
template <int K, typename In, typename G>
__device__ inline void gm_atoms(const GradParams<In, G>& p, const int64_t (&key)[K], int64_t per_atom, int lane,
                                int64_t (&lo)[K]) {
  int64_t n[K];
  bool more = false;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    lo[k] = 0;
    n[k] = p.N;
    more = more || n[k] > 1;
  }
  while (more) {
    more = false;
    int64_t at[K], off[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      at[k] = lane * ((n[k] + 63) >> 6);
      at[k] = at[k] < n[k] ? at[k] : 0;
      off[k] = p.row_offsets[lo[k] + at[k]];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t step = (n[k] + 63) >> 6;
      const uint64_t m = gm_ballot(lane == 0 || (at[k] > 0 && off[k] + per_atom * (lo[k] + at[k]) <= key[k]));
      const int hit = ~m == 0 ? 63 : __builtin_ctzll(~m) - 1;  // the keys rise: the probes that pass are a prefix
      lo[k] += hit * step;
      n[k] -= hit * step;
      n[k] = n[k] < step ? n[k] : step;
      more = more || n[k] > 1;
    }
  }
}

// A share of the work ends, and the next begins, at `key` in atom a (whose
// edges start at `first` and end at `last`): an atom's work is its edges and,
// for the quads that its groups fill in part, `per_atom` edges more.  Atoms of at
// most 64 edges are not cut: their chunks would be more, not shorter.
__device__ inline int64_t gm_bound(int64_t key, int64_t per_atom, int64_t a, int64_t first, int64_t last, int64_t edges) {
  first = gm_clamp(first, edges + 1);
  last = gm_clamp(last, edges + 1);
  const int64_t in = key - per_atom * (a + 1) - first;
  return last - first <= 64 || in < 0 ? first : first + (in & ~int64_t(3));
}

// The chunk at (a, e), from the offsets `window` after a.  The wave's last
// edge ends its last atom, and the last atom ends the edges.
template <typename In, typename G>
__device__ inline GmChunk gm_take(const GradParams<In, G>& p, int64_t a, int64_t e, int64_t e_end, int64_t window,
                                  int lane) {
  GmChunk c;
  c.a = a;
  c.e = e;
  const int most = e_end - e < 65 ? int(e_end - e) : 65;
  const int64_t rel = window - e;
  c.end = rel < 0 ? 0 : (rel > most || a + 1 + lane >= p.N ? most : int(rel));
  const uint64_t before = gm_ballot(c.end < most);
  // a prefix (the offsets rise): the atoms that fit a chunk, or, where the wave
  // ends in this one, those before its last
  const int n = ~before == 0 ? 64 : __builtin_ctzll(~before);
  c.na = most == 65 ? n : (most <= 0 ? 0 : (n < 64 ? n + 1 : 64));
  c.cnt = c.na > 0 ? __builtin_amdgcn_readlane(c.end, c.na - 1) : (most <= 0 ? 0 : 64);
  return c;
}

template <typename In, typename G>
__device__ inline GmChunk gm_form(const GradParams<In, G>& p, int64_t a, int64_t e, int64_t e_end, int64_t window,
                                  int lane) {
  GmChunk c = gm_take(p, a < p.N ? a : p.N - 1, e, e_end, window, lane);
  if (c.cnt == 0 && e < e_end) {  // empty atoms only: on to the atom that holds edge e
    int64_t to[1];
    gm_atoms<1>(p, {e}, 0, lane, to);
    a = to[0];
    c = gm_take(p, a, e, e_end, gm_window(p, a, lane), lane);
    if (c.cnt == 0) {  // offsets that fall: the edges are this atom's, so that the wave ends
      c.na = 0;
      c.cnt = e_end - e < 64 ? int(e_end - e) : 64;
    }
  }
  return c;
}

template <typename In>
struct GmEdge {
  In x, y, z;
  int64_t j;
};

template <typename In, typename G>
__device__ inline GmEdge<In> gm_edge(const GradParams<In, G>& p, const GmChunk& c, int lane) {
  // lanes past the chunk read edge 0 (no branch: their loads need no wait before the join)
  const int64_t e = lane < c.cnt ? c.e + lane : 0;
  GmEdge<In> r;
  r.x = p.vec[3 * e];
  r.y = p.vec[3 * e + 1];
  r.z = p.vec[3 * e + 2];
  r.j = p.neighbors ? p.neighbors[e] : 0;
  return r;
}


// sum_k t_k grad_u Y_k(u) (sph_gradient_dot's sum, t read from a row of the tile).
template <int LMAX>
__device__ inline void gm_gradient(double x, double y, double z, const NormTable& nt, const double* __restrict__ t,
                                   double& gx, double& gy, double& gz) {
  const double sqrt2 = 1.4142135623730950488016887242096981;
  gx = gy = gz = 0.0;
  double cr = 1.0, ci = 0.0, pr = 1.0, pi = 0.0;  // (x + i y)^m and ^(m-1)
  double qmm = 1.0;
#pragma unroll
  for (int m = 0; m <= LMAX; ++m) {
    if (m > 0) {
      qmm *= double(2 * m - 1);
      pr = cr;
      pi = ci;
      const double nr = cr * x - ci * y;
      const double ni = cr * y + ci * x;
      cr = nr;
      ci = ni;
    }
    // q: Q_l^m, d: Q_l^{m+1} = dQ_l^m / dz, both by their recurrences in l
    double q2 = 0.0, q1 = 0.0, d2 = 0.0, d1 = 0.0;
    const double dmm = qmm * double(2 * m + 1);
#pragma unroll
    for (int l = m; l <= LMAX; ++l) {
      double q, d = 0.0;
      if (l == m) {
        q = qmm;
      } else if (l == m + 1) {
        q = double(2 * m + 1) * z * qmm;
        d = dmm;
      } else {
        q = (double(2 * l - 1) * z * q1 - double(l + m - 1) * q2) * nt.inv[l - m];
        if (l == m + 2) {
          d = double(2 * m + 3) * z * dmm;
        } else {
          d = (double(2 * l - 1) * z * d1 - double(l + m) * d2) * nt.inv[l - m - 1];
        }
      }
      q2 = q1;
      q1 = q;
      d2 = d1;
      d1 = d;
      const double n = nt.v[l * (kMaxL + 1) + m];
      const int base = l * l + l;
      if (m == 0) {
        gz += t[base] * (n * d);
      } else {
        const double s = sqrt2 * n;
        const double tp = t[base + m], tm = t[base - m];
        // grad Y_{l,+m} = s (m q pr, -m q pi, d cr); grad Y_{l,-m} = -s (m q pi, m q pr, d ci)
        const double sq = s * double(m) * q;
        gx += sq * (tp * pr - tm * pi);
        gy -= sq * (tp * pi + tm * pr);
        gz += s * d * (tp * cr - tm * ci);
      }
    }
  }
}

// Radial constants of a launch, from the host.
struct GmRadial {
  double rc, lambda, den;  // cutoff, lambda, expm1(lambda)
};

// The radial values and derivatives of cheb_exp_cos_row for a fixed count,
// with one sincospi and one expm1, in fewer instructions.
template <int NRC>
__device__ inline void gm_radial(double r, const GmRadial& c, double (&R)[NRC], double (&dR)[NRC]) {
  const double pi = 3.141592653589793238462643383279502884;
  const double s = r / c.rc;
  const bool live = !(s > 1.0);
  double sn, cs;
  sincospi(s, &sn, &cs);
  const double env = 1.0 + cs;
  const double denv = -pi * sn / c.rc;
  R[0] = live ? 1.0 : 0.0;
  dR[0] = 0.0;
  R[1] = live ? 0.5 * env : 0.0;
  dR[1] = live ? 0.5 * denv : 0.0;
  const double arg = -c.lambda * (s - 1.0);
  const double em1 = expm1(arg);
  // e^x = 1 + expm1(x) keeps its last bit while the sum does not cancel
  const double ex = arg > -0.5 ? 1.0 + em1 : exp(arg);
  const double x = 1.0 - 2.0 * em1 / c.den;
  const double dx = 2.0 * c.lambda * ex / (c.den * c.rc);
  double t0 = 1.0, t1 = x, u0 = 1.0, u1 = 2.0 * x;
#pragma unroll
  for (int n = 2; n < NRC; ++n) {
    const double t2 = 2.0 * x * t1 - t0;
    R[n] = live ? 0.25 * (1.0 - t2) * env : 0.0;
    dR[n] = live ? 0.25 * ((1.0 - t2) * denv - (double(n) * u1) * dx * env) : 0.0;
    t0 = t1;
    t1 = t2;
    const double u2 = 2.0 * x * u1 - u0;
    u0 = u1;
    u1 = u2;
  }
}

// Shares of a launch: the work is the edges and `per_atom` for each atom (a
// group leaves one and a half of a quad's four places empty on average), the
// first `larger` waves have size + 1 of it and the others size.
struct GmShares {
  int64_t size, larger, per_atom;
};

// waves a SIMD that a kernel is compiled for
constexpr int kGmSimdWaves(int lmax) { return lmax >= 6 ? 1 : 2; }

// groups whose adjoint blocks are on their way at once
constexpr int kGmAhead = 4;

// NRC: radial rows compiled (>= p.nr; rows from p.nr on are not read).
template <int LMAX, int NRC, typename In, typename G>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, kGmSimdWaves(LMAX)))) void
density_edge_gradient_mfma_kernel(GradParams<In, G> p, GmRadial radial, GmShares shares) {
  constexpr int LW = (LMAX + 1) * (LMAX + 1);
  constexpr int CT = (LW + 15) / 16;
  constexpr int KS = (NRC + 3) / 4;        // k-steps of four
  constexpr int YP = LW | 1;               // odd: rows of consecutive edges start in different banks
  __shared__ double At[2 * NRC][kGmPitch];  // R rows, then R' rows
  __shared__ double Yt[64][YP];            // Y, then t
  __shared__ double Al[64];
  __shared__ int4 gt[64];                  // groups: block, first column, size
  const int lane = threadIdx.x;
  const int kq = lane >> 4, cc = lane & 15;
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  const int64_t share = int64_t(blockIdx.x);
  const int64_t keys[2] = {shares.size * share + (share < shares.larger ? share : shares.larger),
                           shares.size * (share + 1) + (share + 1 < shares.larger ? share + 1 : shares.larger)};
  int64_t atoms[2];
  gm_atoms<2>(p, keys, shares.per_atom, lane, atoms);
  const int64_t first = p.row_offsets[atoms[0]], first_after = p.row_offsets[atoms[1]];
  const int64_t last_after = p.row_offsets[atoms[1] + 1];
  int64_t window = gm_window(p, atoms[0], lane);
  const int64_t e_begin = share == 0 ? 0 : gm_bound(keys[0], shares.per_atom, atoms[0], first, gm_first(window), p.E);
  const int64_t e_end = share + 1 == int64_t(gridDim.x)
                            ? p.E
                            : gm_bound(keys[1], shares.per_atom, atoms[1], first_after, last_after, p.E);
  if (e_begin >= e_end) return;
  // the lane's row in the last step (the steps before it are full, launch_shape).  Rows past the
  // model's last meet a zero adjoint, but may hold no number themselves (0 / 0 at lambda 0): its last stands in
  const int last = 4 * (KS - 1) + kq < p.nr ? 4 * (KS - 1) + kq : p.nr - 1;
  const int64_t block = int64_t(p.nr) * LW;
  const unsigned voff = unsigned(kq * LW + cc) * unsigned(sizeof(G));
  auto channel = [&](const GmEdge<In>& edge) {
    if (!p.species) return 0;
    return p.species[gm_clamp(edge.j, p.N)];
  };
  // Groups of a chunk: each edge's column, and the list of groups.
  auto group = [&](const GmChunk& c, int kind, int& col, int& ng) {
    const bool valid = lane < c.cnt;
    const int sp = kind < 0 ? 0 : (kind >= p.C ? p.C - 1 : kind);
    int la = 0;
    for (int j = 0; j < c.na; ++j) la += lane >= __builtin_amdgcn_readlane(c.end, j) ? 1 : 0;
    col = lane;
    ng = 0;
    int base = 0;
    uint64_t left = gm_ballot(valid);
    while (left != 0) {
      const int f = __builtin_ctzll(left);
      const int fa = __builtin_amdgcn_readlane(la, f);
      const int fs = __builtin_amdgcn_readlane(sp, f);
      const bool in = valid && la == fa && sp == fs;
      const uint64_t m = gm_ballot(in);
      const int n = __builtin_popcountll(m);
      if (in) col = base + __builtin_popcountll(m & lt);
      if (lane == f) gt[ng] = int4{fa * p.C + fs, base, n, 0};
      ++ng;
      base += n;
      left &= ~m;
    }
    gm_wave_sync();
  };
  auto entry = [&](int k) {
    const int4 v = gt[k];
    return int3{__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y),
                __builtin_amdgcn_readfirstlane(v.z)};
  };
  // The adjoint block of a group in the B-operand layout; rows past it read
  // zero, components past a row are not used.  Without a group the loads are
  // made all the same, over no bytes, so that the number of loads in flight is
  // known where the older ones are waited for.
  auto fetch = [&](int64_t a, bool any, const int3& g, G (&b)[KS][CT]) {
    const G* src = p.gA + (a * p.C + (any ? g.x : 0)) * block;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<G*>(src), (short)0, any ? int(block * int64_t(sizeof(G))) : 0, 0x00020000);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) b[s][ct] = gm_load<G>(rb, voff, unsigned(4 * s * LW + 16 * ct) * sizeof(G));
  };
  // t and a of a group's edges
  auto product = [&](const int3& g, const G (&b)[KS][CT]) {
    const int pos = g.y, c = g.z;
#pragma unroll 1
    for (int m = 0; m < c; m += 4) {
      const int i = m + (lane & 3);
      const int ci = pos + (i < c ? i : c - 1);
      double t[CT], u[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) t[ct] = u[ct] = 0.0;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int n = s + 1 < KS ? 4 * s + kq : last;
        const double ar = At[n][ci], ad = At[NRC + n][ci];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          t[ct] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, double(b[s][ct]), t[ct], 0, 0, 0);
          u[ct] = __builtin_amdgcn_mfma_f64_4x4x4f64(ad, double(b[s][ct]), u[ct], 0, 0, 0);
        }
      }
      const int q = m + kq;
      const int ce = pos + (q < c ? q : c - 1);
      double part = 0.0;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        if (16 * ct + 15 < LW || 16 * ct + cc < LW) part += u[ct] * Yt[ce][16 * ct + cc];
      part = gm_sum16(part);
      if (q < c) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
          if (16 * ct + 15 < LW || 16 * ct + cc < LW) Yt[ce][16 * ct + cc] = t[ct];
        if (cc == 0) Al[ce] = part;
      }
    }
  };

  // Software pipeline.  Loads return in order, so each is issued before those
  // that are waited for after it: behind the products of chunk i come the edges
  // of chunk i + 2 and the offsets after it, and last the first blocks of
  // chunk i + 1, which then have the chain of chunk i and the basis of chunk
  // i + 1 to arrive in.  The species of chunk i + 1 are gathered during the
  // basis and products of chunk i.
  GmChunk cur = gm_form(p, atoms[0], e_begin, e_end, window, lane);
  GmEdge<In> E = gm_edge(p, cur, lane);
  GmChunk nxt = gm_form(p, cur.a + cur.na, cur.e + cur.cnt, e_end, gm_window(p, cur.a + cur.na, lane), lane);
  GmEdge<In> NE = gm_edge(p, nxt, lane);
  window = gm_window(p, nxt.a + nxt.na, lane);
  int col = 0, ng = 0;
  int3 g[kGmAhead];
  G b[kGmAhead][KS][CT];
  group(cur, channel(E), col, ng);
#pragma unroll
  for (int d = 0; d < kGmAhead; ++d) {
    g[d] = entry(d);
    fetch(cur.a, d < ng, g[d], b[d]);
  }
  while (cur.e < e_end) {
    const bool valid = lane < cur.cnt;
    const int nsp = channel(NE);
    const double vx = double(E.x), vy = double(E.y), vz = double(E.z);
    const double r = d_sqrt(vx * vx + vy * vy + vz * vz);
    const double sr = r > p.eps ? r : p.eps;
    const double ux = vx / sr, uy = vy / sr, uz = vz / sr;
    // ---- basis
    {
      double R[NRC], dR[NRC];
      gm_radial<NRC>(r, radial, R, dR);
      if (valid) {
#pragma unroll
        for (int n = 0; n < NRC; ++n) {
          At[n][col] = R[n];
          At[NRC + n][col] = dR[n];
        }
      }
    }
    if (valid) sph_values<LMAX>(ux, uy, uz, p.nt, Yt[col]);
    gm_wave_sync();

    // ---- products, group by group
    for (int k = 0; k < ng; k += kGmAhead) {
#pragma unroll
      for (int d = 0; d < kGmAhead; ++d) {
        if (k + d >= ng) break;
        product(g[d], b[d]);
        if (k + d + kGmAhead < ng) {
          g[d] = entry(k + d + kGmAhead);
          fetch(cur.a, true, g[d], b[d]);
        }
      }
    }
    gm_wave_sync();

    // ---- the chunk after next, and the next one's groups and first blocks
    const int tcol = col;
    group(nxt, nsp, col, ng);
    const GmChunk nn = gm_form(p, nxt.a + nxt.na, nxt.e + nxt.cnt, e_end, window, lane);
    const GmEdge<In> NNE = gm_edge(p, nn, lane);
    window = gm_window(p, nn.a + nn.na, lane);
#pragma unroll
    for (int d = 0; d < kGmAhead; ++d) {
      g[d] = entry(d);
      fetch(nxt.a, d < ng, g[d], b[d]);
    }

    // ---- chain: the contracted gradient of the harmonics
    if (valid) {
      double gx, gy, gz;
      gm_gradient<LMAX>(ux, uy, uz, p.nt, Yt[tcol], gx, gy, gz);
      const double a = Al[tcol];
      if (r > p.eps) {  // J^T G with J = (I - u u^T) / r
        const double ug = ux * gx + uy * gy + uz * gz;
        gx -= ux * ug;
        gy -= uy * ug;
        gz -= uz * ug;
      }  // else u = v / eps: J = I / eps
      const int64_t e = cur.e + lane;
      p.out[3 * e] = In(a * ux + gx / sr);
      p.out[3 * e + 1] = In(a * uy + gy / sr);
      p.out[3 * e + 2] = In(a * uz + gz / sr);
    }
    gm_wave_sync();  // the tile is read before the next chunk writes it
    cur = nxt;
    E = NE;
    nxt = nn;
    NE = NNE;
  }
}

// Waves of a compute unit: as many as its LDS holds tiles (allocated in steps of
// 1 280 bytes) and its SIMDs waves of the kernel, but not five, of which two
// share a SIMD while three have their own: the launch ends with that pair (l_max
// 5, n_max 7: 92 us, with four 88).
template <int LMAX, int NRC, typename In, typename G>
int gm_waves() {
  int regs = 0, lds = 0;
  hipFuncAttributes at;
  if (hipFuncGetAttributes(&at, reinterpret_cast<const void*>(&density_edge_gradient_mfma_kernel<LMAX, NRC, In, G>)) ==
      hipSuccess) {
    regs = at.numRegs;
    lds = int(at.sharedSizeBytes);
  } else {
    (void)hipGetLastError();
  }
  if (lds <= 0) return 4;
  const int tiles = 160 * 1024 / ((lds + 1279) / 1280 * 1280);
  const int simd = regs > 256 ? 1 : kGmSimdWaves(LMAX);
  const int waves = tiles < 4 * simd ? tiles : 4 * simd;
  return waves == 5 ? 4 : waves;
}

template <int LMAX, int NRC, typename In, typename G>
int launch_shape(const GradParams<In, G>& p, hipStream_t s) {
  if (p.nr > NRC || p.nr <= (NRC - 1) / 4 * 4) return YE3T_EUNSUPPORTED;  // all but the last step full
  static const int per_cu = gm_waves<LMAX, NRC, In, G>();  // the kernel's own, the same on every gfx950
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  GmRadial radial;
  radial.rc = p.cutoff > 2.220446049250313e-16 ? p.cutoff : 2.220446049250313e-16;
  radial.lambda = p.lambda;
  radial.den = std::expm1(p.lambda);
  int64_t waves = int64_t(cus) * per_cu;  // as many as the device holds at once
  if (waves > (p.E + 63) / 64) waves = (p.E + 63) / 64;
  GmShares shares;
  shares.per_atom = (3 * int64_t(p.C) + 1) / 2;
  shares.size = (p.E + shares.per_atom * p.N) / waves;
  shares.larger = (p.E + shares.per_atom * p.N) % waves;
  hipLaunchKernelGGL((density_edge_gradient_mfma_kernel<LMAX, NRC, In, G>), dim3(unsigned(waves)),
                     dim3(64), 0, s, p, radial, shares);
  return check_launch("density_edge_gradient_mfma_kernel");
}

// Rows compiled: whole steps of four (8, 12, 16), and below 12 and 16 the most
// whose tile leaves room for another wave in a compute unit (11: six rather than
// five at l_max 4; 13: four rather than three at l_max 6).
template <int LMAX, typename In, typename G>
int launch_lmax(const GradParams<In, G>& p, hipStream_t s) {
  if (p.nr <= 8) return launch_shape<LMAX, 8>(p, s);
  if (p.nr <= 11) return launch_shape<LMAX, 11>(p, s);
  if (p.nr <= 12) return launch_shape<LMAX, 12>(p, s);
  if (p.nr <= 13) return launch_shape<LMAX, 13>(p, s);
  return launch_shape<LMAX, 16>(p, s);
}

}  // namespace

// Taken where a group fills its four rows on average, where the radial rows
// fill two steps of four, and where the other kernel's gathers (E nr (l_max +
// 1)^2 values) cost more than the start of a wave here: 2.5e7 of them, three
// times as many with one channel, whose edges gather the same block together.
// Both sides measured (lane-per-edge / here, us):
//   edges a group   5 000 x 16, 8 species, l_max 4 (two): 28 / 35; 20 000 x 32,
//                   l_max 4, 4 species (eight), n_max 10: 121 / 98
//   radial rows     400 000 edges, 4 species, n_max 1, 3, 5, 7, 10, 15:
//                   l_max 4: 38 / 43, 47 / 44, 58 / 52, 67 / 51, 82 / 68, 133 / 84
//                   l_max 5: 45 / 60, 67 / 60, 70 / 79, 102 / 80, 98 / 88, 175 / 101
//                   l_max 6: 60 / 76, 77 / 76, 93 / 87, 113 / 88, 142 / 104, 267 / 169
//   gathers         n_max 7, 4 species, l_max 4, 66 000 and 132 000 edges (1.3e7,
//                   2.6e7): 16 / 17, 28 / 26; l_max 6 (2.6e7, 5.2e7): 31 / 26,
//                   49 / 39; one channel, n_max 10, l_max 4, 132 000, 264 000,
//                   400 000 edges (3.6e7, 7.3e7, 1.1e8): 24 / 24, 45 / 38, 66 / 55
//   l_max           below 4 the blocks are small enough for the lane-per-edge
//                   kernel (l_max 2: 33 / 71; l_max 3: 62 / 51 to 111 / 116)
// Uneven structures at n_max 10, l_max 4, four species: all edges in a tenth of
// 20 000 atoms 141 / 98, degrees rising from 0 to 64 147 / 117 (551 and 132 with
// equal shares of the atoms).
template <typename In, typename G>
int launch_edge_gradient_mfma(const GradParams<In, G>& p, int lmax, hipStream_t s) {
  if (p.mix || p.feats || p.C > (1 << 24)) return YE3T_EUNSUPPORTED;  // a group's block is 32-bit within its chunk
  if (p.E < 65536 || p.E / 4 < p.N * int64_t(p.C) || p.nr < 7) return YE3T_EUNSUPPORTED;
  if (double(p.E) * (p.nr * (lmax + 1) * (lmax + 1)) < (p.C > 1 ? 2.5e7 : 7.5e7)) return YE3T_EUNSUPPORTED;
  switch (lmax) {
    case 4: return launch_lmax<4>(p, s);
    case 5: return launch_lmax<5>(p, s);
    case 6: return launch_lmax<6>(p, s);
    default: return YE3T_EUNSUPPORTED;
  }
}

template int launch_edge_gradient_mfma<double, double>(const GradParams<double, double>&, int, hipStream_t);
template int launch_edge_gradient_mfma<float, float>(const GradParams<float, float>&, int, hipStream_t);
template int launch_edge_gradient_mfma<float, double>(const GradParams<float, double>&, int, hipStream_t);

}  // namespace ye3t
