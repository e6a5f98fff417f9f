// What the edge-gradient kernels of the stage-1 density share: their
// parameters and the harmonics with compile-time bounds; and the harmonics'
// contracted gradient of the lane-per-edge kernel (the grouped one reads its
// factors from a tile).
#pragma once

#include "common.h"

namespace ye3t {

constexpr int kGradMaxRadial = 16;  // n_max + 1 <= 16

template <typename In, typename G>
struct GradParams {
  const In* vec;             // [E, 3]
  const int64_t* row_offsets;  // [N + 1]
  const int64_t* neighbors;  // [E] or NULL
  const int32_t* species;    // [N] or NULL
  const In* feats;           // [N, C] or NULL
  const In* mix;             // [C, nr] or NULL
  const G* gA;               // [N, C, rows, lw]
  In* out;                   // [E, 3]
  int64_t N, E;
  int C, nr, rows;
  double cutoff, lambda, eps;
  NormTable nt;
};

// Y_k(u) for k < (LMAX + 1)^2 (the reference's real SH, same recurrence as
// real_sph_row) with compile-time bounds, so Y stays in registers, or goes to a
// row of a tile.
template <int LMAX>
__device__ inline void sph_values(double x, double y, double z, const NormTable& nt, double* __restrict__ Y) {
  const double sqrt2 = 1.4142135623730950488016887242096981;
  double cr = 1.0, ci = 0.0, qmm = 1.0;
#pragma unroll
  for (int m = 0; m <= LMAX; ++m) {
    if (m > 0) {
      qmm *= double(2 * m - 1);
      const double nr = cr * x - ci * y;
      const double ni = cr * y + ci * x;
      cr = nr;
      ci = ni;
    }
    double q2 = 0.0, q1 = 0.0;
#pragma unroll
    for (int l = m; l <= LMAX; ++l) {
      double q;
      if (l == m) {
        q = qmm;
      } else if (l == m + 1) {
        q = double(2 * m + 1) * z * qmm;
      } else {
        q = (double(2 * l - 1) * z * q1 - double(l + m - 1) * q2) * nt.inv[l - m];
      }
      q2 = q1;
      q1 = q;
      const double n = nt.v[l * (kMaxL + 1) + m];
      const int base = l * l + l;
      if (m == 0) {
        Y[base] = n * q;
      } else {
        const double s = sqrt2 * n * q;
        Y[base + m] = s * cr;
        Y[base - m] = -s * ci;
      }
    }
  }
}

// G = sum_k t_k grad_u Y_k(u), the harmonics taken as polynomials in u:
// Y_{l,0} = N Q_l^0(z), Y_{l,+-m} = sqrt2 N Q_l^m(z) (Re, -Im) (x + i y)^m with
// Q_l^m = d^m P_l / dz^m, so d/dz brings Q_l^{m+1} and d/dx, d/dy bring
// m (x + i y)^{m-1}.
template <int LMAX>
__device__ inline void sph_gradient_dot(double x, double y, double z, const NormTable& nt, const double* t,
                                        double& gx, double& gy, double& gz) {
  const double sqrt2 = 1.4142135623730950488016887242096981;
  double Q[LMAX + 2][LMAX + 1];  // Q[m][l] = Q_l^m for l <= LMAX, m <= LMAX + 1
  double qmm = 1.0;
#pragma unroll
  for (int m = 0; m <= LMAX + 1; ++m) {
    if (m > 0) qmm *= double(2 * m - 1);
    double q2 = 0.0, q1 = 0.0;
#pragma unroll
    for (int l = 0; l <= LMAX; ++l) {
      double q = 0.0;
      if (l == m) {
        q = qmm;
      } else if (l == m + 1) {
        q = double(2 * m + 1) * z * qmm;
      } else if (l > m + 1) {
        q = (double(2 * l - 1) * z * q1 - double(l + m - 1) * q2) * nt.inv[l - m];
      }
      if (l >= m) {
        q2 = q1;
        q1 = q;
      }
      Q[m][l] = q;
    }
  }
  gx = gy = gz = 0.0;
  double cr = 1.0, ci = 0.0, pr = 1.0, pi = 0.0;  // (x + i y)^m and ^(m-1)
#pragma unroll
  for (int m = 0; m <= LMAX; ++m) {
    if (m > 0) {
      pr = cr;
      pi = ci;
      const double nr = cr * x - ci * y;
      const double ni = cr * y + ci * x;
      cr = nr;
      ci = ni;
    }
#pragma unroll
    for (int l = m; l <= LMAX; ++l) {
      const double n = nt.v[l * (kMaxL + 1) + m];
      const int base = l * l + l;
      if (m == 0) {
        gz += t[base] * (n * Q[1][l]);
      } else {
        const double s = sqrt2 * n;
        const double q = Q[m][l], qz = Q[m + 1][l];
        const double tp = t[base + m], tm = t[base - m];
        // grad Y_{l,+m} = s (m q pr, -m q pi, qz cr); grad Y_{l,-m} = -s (m q pi, m q pr, qz ci)
        gx += s * double(m) * q * (tp * pr - tm * pi);
        gy += -s * double(m) * q * (tp * pi + tm * pr);
        gz += s * qz * (tp * cr - tm * ci);
      }
    }
  }
}

// The gradient on the fp64 matrix cores (density_grad_mfma.hip);
// YE3T_EUNSUPPORTED, with nothing launched, for shapes it is not built for.
template <typename In, typename G>
int launch_edge_gradient_mfma(const GradParams<In, G>& p, int lmax, hipStream_t s);

}  // namespace ye3t
