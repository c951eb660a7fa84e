// diff_kernels.hpp -- kernels of the differentiable periodic-box bispectrum
// (B_000 diag form): real-mesh assignment and its adjoint, the fused
// loaders of the adjoint transforms, and the shell accumulations.
//
// Forward (the reference chain of compute_bispec_in_gpp_box,
// threept.cpp:1473-2188, restricted to l1 = l2 = L = 0):
//   D(k)   = V_cell FFT[delta](k)
//   G(x)   = IFFT[D / (W V)](x)
//   F_b(x) = IFFT[shell_b D / W](x)
//   B_b    = norm V_cell / n_b^2  sum_x F_b(x)^2 G(x)
// Adjoint, with a_b = dL/dB_b norm V_cell / n_b^2 and both k-space masks
// even in k:
//   dL/ddelta = V_cell IFFT[ sum_b shell_b / W  FFT[2 a_b F_b G]
//                            + 1 / (W V)        FFT[sum_b a_b F_b^2] ].
#pragma once

#include "kernels.hpp"

namespace trvg {

// Assignment stencil of one axis (the index and weight rules of k_assign,
// field.cpp:569-1112) with dW/ds, s the in-cell offset in cell units.
template <int ORDER>
__device__ __forceinline__ void stencil_1d(double pos, int ng, double L,
                                           int idx_out[ORDER],
                                           double win[ORDER],
                                           double dwin[ORDER]) {
  const double loc = __ddiv_rn(__dmul_rn(double(ng), pos), L);
  int idx = int(loc);
  const double s = __dadd_rn(loc, -double(idx));
  auto nxt = [ng](int i) { return (i == ng - 1) ? 0 : i + 1; };
  auto prv = [ng](int i) { return (i == 0) ? ng - 1 : i - 1; };
  if (ORDER == 1) {
    if (s >= 0.5) idx = nxt(idx);
    idx_out[0] = idx;
    win[0] = 1.;
    dwin[0] = 0.;
  } else if (ORDER == 2) {
    idx_out[0] = idx;
    idx_out[1] = nxt(idx);
    win[0] = 1. - s;
    win[1] = s;
    dwin[0] = -1.;
    dwin[1] = 1.;
  } else if (ORDER == 3) {
    if (s < 0.5) {
      idx_out[0] = prv(idx);
      idx_out[1] = idx;
      idx_out[2] = nxt(idx);
      win[0] = 0.5 * (0.5 - s) * (0.5 - s);
      win[1] = 0.75 - s * s;
      win[2] = 0.5 * (0.5 + s) * (0.5 + s);
      dwin[0] = -(0.5 - s);
      dwin[1] = -2. * s;
      dwin[2] = 0.5 + s;
    } else {
      idx_out[0] = idx;
      idx_out[1] = nxt(idx);
      idx_out[2] = nxt(idx_out[1]);
      const double sp = 1. - s;
      win[0] = 0.5 * (0.5 + sp) * (0.5 + sp);
      win[1] = 0.75 - sp * sp;
      win[2] = 0.5 * (0.5 - sp) * (0.5 - sp);
      dwin[0] = -(0.5 + sp);
      dwin[1] = 2. * sp;
      dwin[2] = 0.5 - sp;
    }
  } else {
    idx_out[0] = prv(idx);
    idx_out[1] = idx;
    idx_out[2] = nxt(idx);
    idx_out[3] = nxt(idx_out[2]);
    const double sm = 1. - s;
    win[0] = 1. / 6 * sm * sm * sm;
    win[1] = 1. / 6 * (4. - 6. * s * s + 3. * s * s * s);
    win[2] = 1. / 6 * (4. - 6. * sm * sm + 3. * sm * sm * sm);
    win[3] = 1. / 6 * s * s * s;
    dwin[0] = -0.5 * sm * sm;
    dwin[1] = -2. * s + 1.5 * s * s;
    dwin[2] = 2. * sm - 1.5 * sm * sm;
    dwin[3] = 0.5 * s * s;
  }
}

// n(x) += w_p W(x - x_p) / V_cell on a real mesh (positions n x 3,
// row-major; weights may be null for unit weights).
template <typename T, int ORDER>
__global__ void __launch_bounds__(256)
k_assign_real(T* __restrict__ mesh, const double* __restrict__ pos,
              const double* __restrict__ w, long long n, Geom g) {
  const double inv_vol_cell = 1 / g.vol_cell;
  for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < n;
       p += (long long)gridDim.x * blockDim.x) {
    int ix[3][ORDER];
    double wn[3][ORDER], dw[3][ORDER];
#pragma unroll
    for (int a = 0; a < 3; a++)
      stencil_1d<ORDER>(pos[3 * p + a], g.n[a], g.L[a], ix[a], wn[a], dw[a]);
    const double wp = (w ? w[p] : 1.) * inv_vol_cell;
#pragma unroll
    for (int il = 0; il < ORDER; il++)
#pragma unroll
      for (int jl = 0; jl < ORDER; jl++) {
        const long long row = ((long long)ix[0][il] * g.n[1] + ix[1][jl]) * g.n[2];
        const double wij = wp * wn[0][il] * wn[1][jl];
#pragma unroll
        for (int kl = 0; kl < ORDER; kl++) {
          const long long gid = row + ix[2][kl];
          if (gid < 0 || gid >= g.nmesh) continue;
          unsafeAtomicAdd(mesh + gid, T(wij * wn[2][kl]));
        }
      }
  }
}

// Adjoint of k_assign_real: for each particle, gather the mesh cotangent
// through the stencil (grad_w = sum gm W / V_cell) and its derivative
// (grad_pos = w / V_cell sum gm dW/dx).  Either output may be null.
template <typename T, int ORDER>
__global__ void __launch_bounds__(256)
k_assign_real_adjoint(const T* __restrict__ gmesh, const double* __restrict__ pos,
                      const double* __restrict__ w, long long n, Geom g,
                      double* __restrict__ gpos, double* __restrict__ gw) {
  const double inv_vol_cell = 1 / g.vol_cell;
  for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < n;
       p += (long long)gridDim.x * blockDim.x) {
    int ix[3][ORDER];
    double wn[3][ORDER], dw[3][ORDER];
#pragma unroll
    for (int a = 0; a < 3; a++)
      stencil_1d<ORDER>(pos[3 * p + a], g.n[a], g.L[a], ix[a], wn[a], dw[a]);
    double val = 0., dx = 0., dy = 0., dz = 0.;
#pragma unroll
    for (int il = 0; il < ORDER; il++)
#pragma unroll
      for (int jl = 0; jl < ORDER; jl++) {
        const long long row = ((long long)ix[0][il] * g.n[1] + ix[1][jl]) * g.n[2];
#pragma unroll
        for (int kl = 0; kl < ORDER; kl++) {
          const long long gid = row + ix[2][kl];
          if (gid < 0 || gid >= g.nmesh) continue;
          const double v = double(gmesh[gid]);
          val += v * wn[0][il] * wn[1][jl] * wn[2][kl];
          dx += v * dw[0][il] * wn[1][jl] * wn[2][kl];
          dy += v * wn[0][il] * dw[1][jl] * wn[2][kl];
          dz += v * wn[0][il] * wn[1][jl] * dw[2][kl];
        }
      }
    const double wp = (w ? w[p] : 1.) * inv_vol_cell;
    if (gw) gw[p] = val * inv_vol_cell;
    if (gpos) {
      gpos[3 * p] = wp * dx * (double(g.n[0]) / g.L[0]);
      gpos[3 * p + 1] = wp * dy * (double(g.n[1]) / g.L[1]);
      gpos[3 * p + 2] = wp * dz * (double(g.n[2]) / g.L[2]);
    }
  }
}

// Real mesh -> complex transform input (v scale, 0).
template <typename T>
struct LoadReal {
  const T* src;
  T scale;
  __device__ c2<T> operator()(long long g, int, int, int) const {
    return mk<T>(src[g] * scale, T(0));
  }
};

// sum_x Re F(x)^2 Re G(x), per-block FP64 partials.
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_f2g_partials(const c2<T>* __restrict__ F, const c2<T>* __restrict__ G,
               long long n, double* __restrict__ part, int stride) {
  __shared__ double red[RED_THREADS];
  double s = 0.;
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    const double f = double(F[c].x);
    s += f * f * double(G[c].x);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = RED_THREADS / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(long long)blockIdx.x * stride] = red[0];
}

// sum_x F_b(x)^2 Re G(x) of the two real fields of mesh blockIdx.y of a
// packed slab: per-block FP64 partials part[blockIdx.x][2 gridDim.y].
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_f2g_packed(const c2<T>* __restrict__ F, const c2<T>* __restrict__ G, long long n,
             double* __restrict__ part) {
  __shared__ double red[2][RED_THREADS];
  const c2<T>* f = F + blockIdx.y * n;
  double s0 = 0., s1 = 0.;
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    const c2<T> v = f[c];
    const double g = double(G[c].x), x = double(v.x), y = double(v.y);
    s0 += x * x * g;
    s1 += y * y * g;
  }
  red[0][threadIdx.x] = s0;
  red[1][threadIdx.x] = s1;
  __syncthreads();
  for (int h = RED_THREADS / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) {
      red[0][threadIdx.x] += red[0][threadIdx.x + h];
      red[1][threadIdx.x] += red[1][threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x < 2)
    part[((long long)blockIdx.x * gridDim.y + blockIdx.y) * 2 + threadIdx.x] =
        red[threadIdx.x][0];
}

// Cotangents of the shell fields and of G: mesh p of the packed slab F
// becomes 2 (a_2p F_2p + i a_2p+1 F_2p+1) G; sum_b a_b F_b^2 goes to the complex
// mesh gk if there is one, else is added to the real mesh gG.
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_cotangents(c2<T>* __restrict__ F, const c2<T>* __restrict__ G, long long n, int nt,
             const double* __restrict__ a, c2<T>* __restrict__ gk, T* __restrict__ gG) {
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    const double g = double(G[c].x);
    double s = 0.;
    for (int p = 0; p < nt; p++) {
      const c2<T> f = F[(long long)p * n + c];
      const double x = double(f.x), y = double(f.y), a0 = a[2 * p], a1 = a[2 * p + 1];
      s += a0 * x * x + a1 * y * y;
      F[(long long)p * n + c] = mk<T>(T(2. * a0 * x * g), T(2. * a1 * y * g));
    }
    if (gk) gk[c] = mk<T>(T(s), T(0));
    else gG[c] = T(double(gG[c]) + s);
  }
}

// acc(k) += [the spectrum of the cotangent of the bin holding k, + scale
// times that of G's cotangent, gk (may be null)] / W(k), from the transformed
// slab of k_cotangents on the mesh `c` to the full mesh `g` (window tables of
// g).  Bin b of the batch is real field slot[b] of the slab (-1: not in it):
// with P = FFT[u + i v], u(k) = (P(k) + P(-k)^*) / 2 and v(k) = (P(k) -
// P(-k)^*) / 2i.  Each cell of c is one cell of g, so the update is
// race-free.
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_adj_acc(c2<T>* __restrict__ acc, const c2<T>* __restrict__ P,
          const c2<T>* __restrict__ gk, Geom g, Geom c,
          AxisTables tab, const double* __restrict__ edge, int nb,
          const int* __restrict__ slot, double scale) {
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < c.nmesh;
       q += (long long)gridDim.x * blockDim.x) {
    const long long ij = q / c.n[2];
    const int ix[3] = {int(ij / c.n[1]), int(ij % c.n[1]), int(q % c.n[2])};
    int f[3], r[3];
    double k[3];
    bool edge_mode = false;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int m = shifted(ix[a], c.n[a]);
      edge_mode |= c.n[a] < g.n[a] && ix[a] == c.n[a] / 2;
      f[a] = m < 0 ? m + g.n[a] : m;
      r[a] = ix[a] == 0 ? 0 : c.n[a] - ix[a];
      k[a] = grid_coord(ix[a], c.n[a], c.dk[a]);
    }
    if (edge_mode) continue;   // beyond the products of any bin
    double re = 0., im = 0.;
    if (gk) {
      const c2<T> t = gk[q];
      re = scale * double(t.x);
      im = scale * double(t.y);
    }
    const int b = find_bin(edge, nb, mag2_exact(k[0], k[1], k[2]));
    const int s = b < 0 ? -1 : slot[b];
    if (s >= 0) {
      const c2<T>* p = P + (long long)(s / 2) * c.nmesh;
      const c2<T> u = p[q];
      const c2<T> v = p[((long long)r[0] * c.n[1] + r[1]) * c.n[2] + r[2]];
      if (s % 2 == 0) {
        re += 0.5 * (double(u.x) + double(v.x));
        im += 0.5 * (double(u.y) - double(v.y));
      } else {
        re += 0.5 * (double(u.y) + double(v.y));
        im -= 0.5 * (double(u.x) - double(v.x));
      }
    }
    const double iw = 1. / window_at(tab, f[0], f[1], f[2]);
    c2<T>* o = acc + ((long long)f[0] * g.n[1] + f[1]) * g.n[2] + f[2];
    *o = mk<T>(T(double(o->x) + re * iw), T(double(o->y) + im * iw));
  }
}

// Zero a real mesh.
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_zero_real(T* __restrict__ f, long long n) {
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x)
    f[c] = T(0);
}

// out(x) = scale Re src(x).
template <typename T>
__global__ void __launch_bounds__(RED_THREADS)
k_real_part(T* __restrict__ out, const c2<T>* __restrict__ src, long long n,
            double scale) {
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x)
    out[c] = T(double(src[c].x) * scale);
}

}  // namespace trvg
