// Adjoint (reverse mode) of the plain MLS-MPM substep on gfx950.
//
// The reference differentiates p2g / grid_op / g2p with Taichi's autodiff
// (mpm_exps/engine/mpm_solver.py:800-858, nlogn_loop_forward_grad
// :1167-1188) and accumulates the squared state adjoints per component
// (accu_grad :1232-1271).  Here the three adjoint phases are hand-written:
//   k_adj_g2p   per particle: adjoints of x and J/F through G2P, and the
//               grid-velocity adjoint scattered with float atomics;
//   k_adj_grid  per node: adjoint of the grid update, (m v, m) adjoints;
//   k_adj_p2g   per particle: adjoints of x, v, C, J/F through P2G (gathered),
//               plus the squared adjoints summed per component in f64.
// The stencil base is piecewise constant; quadratic B-spline weights are C1,
// so this is the derivative almost everywhere.  Wall conditions that zero a
// velocity component zero its adjoint.
// On a sorted state the particle phases run over work items with LDS tiles
// (k_adj_g2p_tiled, k_adj_p2g_tiled) and the grid phase is part of the
// gather of the scattered tiles (AdjEmit); k_adj_g2p and k_adj_p2g are the
// same phases on an unsorted state (grid in global memory, float atomics).
#pragma once

#include "aq_gather.hpp"  // collider_probe
#include "aq_mpm_kernels.hpp"

namespace aq {

template <class T> struct AdjStencil {
  int base[3];
  T fx[3], w[3][3], dw[3][3];
};

template <int DIM, class T>
__device__ __forceinline__ AdjStencil<T> adj_stencil(const T *x, const ParamsT<T> &P) {
  AdjStencil<T> S;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    S.base[a] = 0;
    S.fx[a] = (T)0;
#pragma unroll
    for (int i = 0; i < 3; ++i) S.w[a][i] = S.dw[a][i] = (T)0;
  }
#pragma unroll
  for (int a = 0; a < DIM; ++a) {
    S.base[a] = stencil_1d<T>(x[a], P, S.fx[a], S.w[a]);
    const T f = S.fx[a];
    S.dw[a][0] = f - (T)1.5;
    S.dw[a][1] = (T)-2 * (f - (T)1);
    S.dw[a][2] = f - (T)0.5;
  }
  return S;
}

// weight of stencil node off and its gradient in fx
template <int DIM, class T>
__device__ __forceinline__ T adj_weight(const AdjStencil<T> &S, const int (&off)[3], T (&g)[3]) {
  T w = (T)1;
#pragma unroll
  for (int a = 0; a < DIM; ++a) w *= S.w[a][off[a]];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    g[c] = (T)0;
    if (c < DIM) {
      T v = S.dw[c][off[c]];
#pragma unroll
      for (int a = 0; a < DIM; ++a)
        if (a != c) v *= S.w[a][off[a]];
      g[c] = v;
    }
  }
  return w;
}

template <int DIM>
__device__ __forceinline__ int64_t adj_node(const int (&base)[3], const int (&off)[3], int nb) {
  constexpr int LG = BlockShape<DIM>::LOG, E = BlockShape<DIM>::E;
  const int i = base[0] + off[0], j = base[1] + off[1], k = base[2] + off[2];
  if constexpr (DIM == 3) {
    const int64_t blk = ((int64_t)(i >> LG) * nb + (j >> LG)) * nb + (k >> LG);
    return blk * 64 + (((i & (E - 1)) << 4) | ((j & (E - 1)) << 2) | (k & (E - 1)));
  } else {
    const int64_t blk = (int64_t)(i >> LG) * nb + (j >> LG);
    return blk * 64 + (((i & (E - 1)) << 3) | (j & (E - 1)));
  }
}

// The f32 phases sum node by node, each product and sum rounded on its own
// in the order of the reference's loops: the gradients of an f32 run then
// differ from one way of accumulating the grid to another by that
// accumulation alone (6e-6 of grad x, as two runs do; 7e-6 to 2e-5 with the
// separable sums, which are 7 % faster).  The f64 phases, where the order
// changes 1e-13, take the separable form: over the 3^DIM stencil nodes with
// a node field f and the particle's affine function u_n = c + A (off_n - 1),
//   S_a    = sum_n w_n f_n,a
//   M_ab   = sum_n w_n f_n,a (off_n,b - 1)
//   X_c    = sum_n (dw_n / dfx_c) (f_n . u_n + extra_n)
// axis by axis (innermost axis first, fused multiply-adds: about half the
// arithmetic).  The three dw of an axis sum to zero, so the derivative sums
// take differences from the middle node: exact for nearly equal values,
// where summing dw times the values themselves would cancel.  fetch(off)
// returns the node's record, extra(record) what is added to f . u; add(off,
// w, u) sees every node's weight and u_n.
template <class T> struct AdjSums {
  T S[3], M[3][3], X[3];
};

template <int DIM, class T, class Fetch, class Extra, class Add>
__device__ __forceinline__ void adj_sums(const AdjStencil<T> &St, const T (&c)[3], const T (&A)[3][3], Fetch &&fetch,
                                         Extra &&extra, Add &&add, AdjSums<T> &R) {
  constexpr int NK = DIM == 3 ? 3 : 1;
  const auto ddw = [&](int a, const T (&y)[3]) {  // sum_i dw_i y_i
    return tfma<T>(St.dw[a][0], y[0] - y[1], St.dw[a][2] * (y[2] - y[1]));
  };
  T qi[3];  // f . u summed over (j, k)
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    R.S[a] = R.X[a] = (T)0;
#pragma unroll
    for (int b = 0; b < 3; ++b) R.M[a][b] = (T)0;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    T ci[3] = {(T)0, (T)0, (T)0}, Sj[3] = {(T)0, (T)0, (T)0}, Mj[3] = {(T)0, (T)0, (T)0}, Mk[3] = {(T)0, (T)0, (T)0};
    T qj[3], q = (T)0, qk = (T)0;  // f . u summed over k; over (j, k) with weights w w, w dw
#pragma unroll
    for (int a = 0; a < DIM; ++a) ci[a] = i == 0 ? c[a] - A[a][0] : (i == 2 ? c[a] + A[a][0] : c[a]);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      T cj[3] = {(T)0, (T)0, (T)0}, Sk[3] = {(T)0, (T)0, (T)0}, Dk[3] = {(T)0, (T)0, (T)0}, dots[3], s0 = (T)0;
#pragma unroll
      for (int a = 0; a < DIM; ++a) cj[a] = j == 0 ? ci[a] - A[a][1] : (j == 2 ? ci[a] + A[a][1] : ci[a]);
      const T wij = St.w[0][i] * St.w[1][j];
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const int off[3] = {i, j, k};
        const vec4_t<T> nd = fetch(off);
        const T f[3] = {nd.x, nd.y, nd.z};
        T u[3] = {(T)0, (T)0, (T)0}, dot = extra(nd);
#pragma unroll
        for (int a = 0; a < DIM; ++a) {
          u[a] = cj[a];
          if constexpr (DIM == 3) {
            if (k == 0) u[a] = cj[a] - A[a][2];
            if (k == 2) u[a] = cj[a] + A[a][2];
            Sk[a] = tfma<T>(St.w[2][k], f[a], Sk[a]);
            if (k == 0) Dk[a] = tfma<T>(-St.w[2][0], f[a], Dk[a]);
            if (k == 2) Dk[a] = tfma<T>(St.w[2][2], f[a], Dk[a]);
          } else {
            Sk[a] = f[a];
          }
          dot = tfma<T>(f[a], u[a], dot);
        }
        if constexpr (DIM == 3) {
          s0 = tfma<T>(St.w[2][k], dot, s0);
          dots[k] = dot;
          add(off, wij * St.w[2][k], u);
        } else {
          s0 = dot;
          add(off, wij, u);
        }
      }
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        Sj[a] = tfma<T>(St.w[1][j], Sk[a], Sj[a]);
        if (j == 0) Mj[a] = tfma<T>(-St.w[1][0], Sk[a], Mj[a]);
        if (j == 2) Mj[a] = tfma<T>(St.w[1][2], Sk[a], Mj[a]);
        if constexpr (DIM == 3) Mk[a] = tfma<T>(St.w[1][j], Dk[a], Mk[a]);
      }
      qj[j] = s0;
      q = tfma<T>(St.w[1][j], s0, q);
      if constexpr (DIM == 3) qk = tfma<T>(St.w[1][j], ddw(2, dots), qk);
    }
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      R.S[a] = tfma<T>(St.w[0][i], Sj[a], R.S[a]);
      if (i == 0) R.M[a][0] = tfma<T>(-St.w[0][0], Sj[a], R.M[a][0]);
      if (i == 2) R.M[a][0] = tfma<T>(St.w[0][2], Sj[a], R.M[a][0]);
      R.M[a][1] = tfma<T>(St.w[0][i], Mj[a], R.M[a][1]);
      if constexpr (DIM == 3) R.M[a][2] = tfma<T>(St.w[0][i], Mk[a], R.M[a][2]);
    }
    qi[i] = q;
    R.X[1] = tfma<T>(St.w[0][i], ddw(1, qj), R.X[1]);
    if constexpr (DIM == 3) R.X[2] = tfma<T>(St.w[0][i], qk, R.X[2]);
  }
  R.X[0] = ddw(0, qi);
}

// The values are computed here: the compiler may not move their sums down.
template <class T, int N, int M>
__device__ __forceinline__ void hold_all(T (&a)[N], T (&b)[M]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
  for (int i = 0; i < M; ++i) asm volatile("" : "+v"(b[i]));
}

// G2P adjoint of one particle, shared by the tiled and untiled kernels:
// from its stencil, its J/F and the adjoint of its next values (begin), the
// adjoints of x and J/F (sums: xo, jo).  The velocity adjoint of stencil
// node off, w_n u_n with u_n = vb + 4 inv_dx C_b (off - fx), goes to add(off,
// w, u); fetch(off) returns the node's velocity.
template <int DIM, int MAT, class T> struct AdjG2P {
  using CI = Comps<DIM, MAT>;
  static constexpr int NJF = CI::NC - CI::CJ;
  T xb[3], vb[3], Cb[DIM * DIM], jf[NJF], jn[NJF];
  T c[3], A[3][3];  // u_n = c + A (off - 1)
  // adj_next's x, v, C, J/F in xb, vb, Cb, jn and the state's J/F in jf:
  // completes vb and C_b (the update of J/F reads C), then c and A
  __device__ __forceinline__ void begin(const ParamsT<T> &P, const AdjStencil<T> &S) {
#pragma unroll
    for (int a = 0; a < DIM; ++a) vb[a] = vb[a] + P.dt * xb[a];
    if constexpr (MAT == AQ_FLUID) {
#pragma unroll
      for (int a = 0; a < DIM; ++a) Cb[a * DIM + a] += jn[0] * P.dt * jf[0];
    } else {
#pragma unroll
      for (int a = 0; a < DIM; ++a)
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
          T acc2 = (T)0;
#pragma unroll
          for (int k = 0; k < DIM; ++k) acc2 += jn[a * DIM + k] * jf[b * DIM + k];
          Cb[a * DIM + b] += P.dt * acc2;
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) c[a] = (T)0;
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      c[a] = vb[a];
#pragma unroll
      for (int b = 0; b < DIM; ++b) {
        A[a][b] = P.c4 * Cb[a * DIM + b];
        c[a] = tfma<T>(-A[a][b], S.fx[b] - (T)1, c[a]);
      }
    }
  }
  template <class Fetch, class Add>
  __device__ __forceinline__ void sums(const ParamsT<T> &P, const AdjStencil<T> &S, Fetch &&fetch, Add &&add,
                                       T (&xo)[3], T (&jo)[NJF]) const {
    T nC[DIM * DIM];
    if constexpr (IsF64<T>::value) {
      AdjSums<T> R;
      adj_sums<DIM, T>(S, c, A, fetch, [](const vec4_t<T> &) { return (T)0; }, add, R);
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        T f = R.X[a];
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
          f = tfma<T>(-A[b][a], R.S[b], f);
          nC[a * DIM + b] = P.c4 * tfma<T>(-R.S[a], S.fx[b] - (T)1, R.M[a][b]);
        }
        xo[a] = xb[a] + P.inv_dx * f;
      }
    } else {
      T fxb[3] = {(T)0, (T)0, (T)0};
#pragma unroll
      for (int i = 0; i < DIM * DIM; ++i) nC[i] = (T)0;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int k = 0; k < (DIM == 3 ? 3 : 1); ++k) {
            const int off[3] = {i, j, k};
            T gw[3];
            const T w = adj_weight<DIM, T>(S, off, gw);
            const vec4_t<T> nd = fetch(off);
            const T g[3] = {nd.x, nd.y, nd.z};
            T u[3] = {(T)0, (T)0, (T)0}, gu = (T)0;
#pragma unroll
            for (int a = 0; a < DIM; ++a) {
              u[a] = vb[a];
#pragma unroll
              for (int b = 0; b < DIM; ++b) {
                nC[a * DIM + b] += P.c4 * w * g[a] * ((T)off[b] - S.fx[b]);
                u[a] += P.c4 * Cb[a * DIM + b] * ((T)off[b] - S.fx[b]);
              }
              gu += g[a] * u[a];
            }
            add(off, w, u);
#pragma unroll
            for (int q = 0; q < DIM; ++q) {
              T t = (T)0;
#pragma unroll
              for (int a = 0; a < DIM; ++a) t += Cb[a * DIM + q] * g[a];
              fxb[q] += gw[q] * gu - P.c4 * w * t;
            }
          }
        // a slice's sums end here, as in g2p_apply: 256 VGPRs and 36 spills ->
        // 163, 38 -> 32 us (262,144 particles of a 3D fluid)
        if constexpr (DIM == 3) hold_all(nC, fxb);
      }
#pragma unroll
      for (int a = 0; a < DIM; ++a) xo[a] = xb[a] + P.inv_dx * fxb[a];
    }
    if constexpr (MAT == AQ_FLUID) {
      T tr = (T)0;
#pragma unroll
      for (int a = 0; a < DIM; ++a) tr += nC[a * DIM + a];
      jo[0] = jn[0] * ((T)1 + P.dt * tr);
    } else {
      T M[DIM * DIM];
#pragma unroll
      for (int a = 0; a < DIM; ++a)
#pragma unroll
        for (int b = 0; b < DIM; ++b) M[a * DIM + b] = (a == b ? (T)1 : (T)0) + P.dt * nC[a * DIM + b];
#pragma unroll
      for (int a = 0; a < DIM; ++a)
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
          T acc = (T)0;
#pragma unroll
          for (int k = 0; k < DIM; ++k) acc += M[k * DIM + a] * jn[k * DIM + b];
          jo[a * DIM + b] = acc;
        }
    }
  }
};

template <int DIM, int MAT, class T>
__device__ __forceinline__ void adj_g2p_load(const T *__restrict__ st, const T *__restrict__ adj_next, int64_t cap,
                                             int64_t p, T (&x)[3], AdjG2P<DIM, MAT, T> &A) {
  using CI = Comps<DIM, MAT>;
#pragma unroll
  for (int a = 0; a < DIM; ++a) {
    x[a] = st[(int64_t)(CI::CX + a) * cap + p];
    A.xb[a] = adj_next[(int64_t)(CI::CX + a) * cap + p];
    A.vb[a] = adj_next[(int64_t)(CI::CV + a) * cap + p];
  }
#pragma unroll
  for (int i = 0; i < DIM * DIM; ++i) A.Cb[i] = adj_next[(int64_t)(CI::CC + i) * cap + p];
#pragma unroll
  for (int i = 0; i < A.NJF; ++i) {
    A.jf[i] = st[(int64_t)(CI::CJ + i) * cap + p];
    A.jn[i] = adj_next[(int64_t)(CI::CJ + i) * cap + p];
  }
}

template <int DIM, int MAT, class T>
__device__ __forceinline__ void adj_g2p_store(T *__restrict__ adj_out, int64_t cap, int64_t p, const T (&xo)[3],
                                              const T (&jo)[AdjG2P<DIM, MAT, T>::NJF]) {
  using CI = Comps<DIM, MAT>;
#pragma unroll
  for (int a = 0; a < DIM; ++a) adj_out[(int64_t)(CI::CX + a) * cap + p] = xo[a];
#pragma unroll
  for (int i = 0; i < CI::NC - CI::CJ; ++i) adj_out[(int64_t)(CI::CJ + i) * cap + p] = jo[i];
}

// G2P adjoint on an unsorted state.  st, adj_next, adj_out: value planes
// [NC][cap]; grid_v: velocities.
template <int DIM, int MAT, class T>
__global__ void __launch_bounds__(256) k_adj_g2p(const T *__restrict__ st, const T *__restrict__ adj_next,
                                                 T *__restrict__ adj_out, int64_t cap, int64_t n, ParamsT<T> P,
                                                 const vec4_t<T> *__restrict__ grid_v, T *__restrict__ gbar) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  T x[3] = {(T)0, (T)0, (T)0}, xo[3], jo[AdjG2P<DIM, MAT, T>::NJF];
  AdjG2P<DIM, MAT, T> A;
  adj_g2p_load<DIM, MAT, T>(st, adj_next, cap, p, x, A);
  const AdjStencil<T> S = adj_stencil<DIM, T>(x, P);
  A.begin(P, S);
  A.sums(
      P, S, [&](const int (&off)[3]) { return grid_v[adj_node<DIM>(S.base, off, P.nb)]; },
      [&](const int (&off)[3], T w, const T (&u)[3]) {
        const int64_t node = adj_node<DIM>(S.base, off, P.nb);
#pragma unroll
        for (int a = 0; a < DIM; ++a) atomic_add<T>(gbar + node * 4 + a, w * u[a]);
      },
      xo, jo);
  adj_g2p_store<DIM, MAT, T>(adj_out, cap, p, xo, jo);
}

// Adjoint of the grid update at node I: from the adjoint gb of the updated
// velocity and the P2G result pre = (m v, m), the adjoint of (m v, m).  With
// the collider (3D), first its adjoint: where the node is inside and the
// velocity after the walls moves into the collider (v_rel . n < 0), the
// update v - (v_rel . n) n has Jacobian I - n n^T.
template <int DIM, class T>
__device__ __forceinline__ vec4_t<T> adj_grid_node(const ParamsT<T> &P, const ColliderK &K, const int (&I)[3],
                                                   const vec4_t<T> &pre, T (&gb)[3]) {
  const T mv[3] = {pre.x, pre.y, pre.z};
  const T inv_m = (T)1 / (pre.w + P.eps_m);
  T v[3] = {inv_m * mv[0], inv_m * mv[1], inv_m * mv[2]};
  v[1] = v[1] - P.g_dt;
  if constexpr (DIM == 3) {
    T n[3], cv[3];
    if (K.on && collider_probe<T>(P, K, I, n, cv)) {
      T vw[3] = {v[0], v[1], v[2]};  // the velocity after the walls, as the forward collides it
      if (P.boundary == AQ_STICKY) {
        bool wall = false;
#pragma unroll
        for (int d = 0; d < 3; ++d) wall = wall || I[d] < P.lb[d] || I[d] > P.ub[d];
        if (wall) vw[0] = vw[1] = vw[2] = (T)0;
      } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (I[d] < P.lb[d] && vw[d] < (T)0) vw[d] = (T)0;
          if (I[d] > P.ub[d] && vw[d] > (T)0) vw[d] = (T)0;
        }
      }
      const T dn = (vw[0] - cv[0]) * n[0] + (vw[1] - cv[1]) * n[1] + (vw[2] - cv[2]) * n[2];
      if (dn < (T)0) {
        const T ng = gb[0] * n[0] + gb[1] * n[1] + gb[2] * n[2];
#pragma unroll
        for (int a = 0; a < 3; ++a) gb[a] -= ng * n[a];
      }
    }
  }
  if (P.boundary == AQ_STICKY) {
    bool wall = false;
#pragma unroll
    for (int d = 0; d < DIM; ++d) wall = wall || I[d] < P.lb[d] || I[d] > P.ub[d];
    if (wall) gb[0] = gb[1] = gb[2] = (T)0;
  } else {
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      if (I[d] < P.lb[d] && v[d] < (T)0) gb[d] = (T)0;
      if (I[d] > P.ub[d] && v[d] > (T)0) gb[d] = (T)0;
    }
  }
  vec4_t<T> r;
  r.x = r.y = r.z = (T)0;
  T mb = (T)0;
#pragma unroll
  for (int a = 0; a < DIM; ++a) mb -= gb[a] * mv[a] * inv_m * inv_m;
  r.x = gb[0] * inv_m;
  r.y = gb[1] * inv_m;
  if constexpr (DIM == 3) r.z = gb[2] * inv_m;
  r.w = mb;
  return r;
}

// Grid-update adjoint on the active blocks: gbar (adjoint of the velocity)
// becomes the adjoint of (m v, m) in place; pre holds the P2G result.
template <int DIM, class T>
__global__ void __launch_bounds__(256) k_adj_grid(ParamsT<T> P, ColliderK K, int32_t nblocks,
                                                  const uint32_t *__restrict__ act,
                                                  const vec4_t<T> *__restrict__ pre, vec4_t<T> *__restrict__ gbar) {
  const int32_t b = (int32_t)(blockIdx.x * 4u + (threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  if (b >= nblocks || !act[b]) return;
  int bc[3], loc[3], I[3];
  block_coords<DIM>(b, P.nb, bc);
  lane_coords<DIM>(lane, loc);
#pragma unroll
  for (int a = 0; a < 3; ++a) I[a] = bc[a] * BlockShape<DIM>::E + loc[a];
  const int64_t node = (int64_t)b * 64 + lane;
  const vec4_t<T> g = gbar[node];
  T gb[3] = {g.x, g.y, g.z};
  gbar[node] = adj_grid_node<DIM, T>(P, K, I, pre[node], gb);
}

// Gather of s_t's P2G for the adjoint: (m v, m) kept in pre, velocities in
// grid_v.
template <int DIM, class T> struct PreEmit {
  const ParamsT<T> &P;
  const ColliderK &K;
  vec4_t<T> *__restrict__ grid_v;
  vec4_t<T> *__restrict__ pre;
  __device__ __forceinline__ void operator()(const int (&I)[3], int64_t node, const vec4_t<T> &sum) const {
    pre[node] = sum;
    grid_v[node] = grid_op_node<DIM, T>(P, K, I, sum);
  }
};

// Gather of the scattered velocity adjoints with the grid update's adjoint.
// The scatter reaches the nodes that the P2G of the same state reached, so
// pre holds this substep's (m v, m) wherever a node has a contribution.
template <int DIM, class T> struct AdjEmit {
  const ParamsT<T> &P;
  const ColliderK &K;
  const vec4_t<T> *__restrict__ pre;
  vec4_t<T> *__restrict__ gbar;
  __device__ __forceinline__ void operator()(const int (&I)[3], int64_t node, const vec4_t<T> &sum) const {
    T gb[3] = {sum.x, sum.y, sum.z};
    gbar[node] = adj_grid_node<DIM, T>(P, K, I, pre[node], gb);
  }
};

template <int DIM, class T>
__global__ void __launch_bounds__(256) k_adj_pre(ParamsT<T> P, ColliderK K, ListArgs L,
                                                 const int32_t *__restrict__ item_off,
                                                 const uint32_t *__restrict__ near,
                                                 const vec4_t<T> *__restrict__ tiles, vec4_t<T> *__restrict__ grid_f,
                                                 uint32_t *__restrict__ fflags, vec4_t<T> *__restrict__ grid_v,
                                                 uint32_t *__restrict__ act, vec4_t<T> *__restrict__ pre) {
  gather_list<DIM, T>(blockIdx.x, gridDim.x, P, PreEmit<DIM, T>{P, K, grid_v, pre}, L, item_off, near, tiles, grid_f, fflags, grid_v, act);
}

template <int DIM, class T>
__global__ void __launch_bounds__(256) k_adj_gather(ParamsT<T> P, ColliderK K, ListArgs L,
                                                    const int32_t *__restrict__ item_off,
                                                    const uint32_t *__restrict__ near,
                                                    const vec4_t<T> *__restrict__ tiles,
                                                    vec4_t<T> *__restrict__ grid_f, uint32_t *__restrict__ fflags,
                                                    const vec4_t<T> *__restrict__ pre, vec4_t<T> *__restrict__ gbar) {
  gather_list<DIM, T>(blockIdx.x, gridDim.x, P, AdjEmit<DIM, T>{P, K, pre, gbar}, L, item_off, near, tiles, grid_f, fflags, gbar,
                      (uint32_t *)nullptr);
}

// 2D fixed-corotated stress adjoint: sigma_bar -> F_bar (added).
template <class T>
__device__ __forceinline__ void adj_corotated(const ParamsT<T> &P, const T (&F)[4], const T (&sb)[4], T (&Fb)[4]) {
  const T J = F[0] * F[3] - F[1] * F[2];
  const T x = F[0] + F[3], y = F[2] - F[1];
  const T r = tsqrt<T>(x * x + y * y);
  const T c = x / r, sn = y / r;
  const T R[4] = {c, -sn, sn, c};
  T A[4], Ab[4], Rb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) A[i] = P.two_mu * (F[i] - R[i]);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      Ab[i * 2 + k] = sb[i * 2 + 0] * F[0 * 2 + k] + sb[i * 2 + 1] * F[1 * 2 + k];
      Fb[i * 2 + k] += sb[0 * 2 + i] * A[0 * 2 + k] + sb[1 * 2 + i] * A[1 * 2 + k];
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    Fb[i] += P.two_mu * Ab[i];
    Rb[i] = -P.two_mu * Ab[i];
  }
  const T cb = Rb[0] + Rb[3], sbb = Rb[2] - Rb[1];
  const T r3 = r * r * r;
  const T xb = cb * (y * y / r3) - sbb * (x * y / r3);
  const T yb = -cb * (x * y / r3) + sbb * (x * x / r3);
  Fb[0] += xb;
  Fb[3] += xb;
  Fb[2] += yb;
  Fb[1] -= yb;
  const T Jb = P.la_0 * ((T)2 * J - (T)1) * (sb[0] + sb[3]);
  Fb[0] += Jb * F[3];
  Fb[3] += Jb * F[0];
  Fb[1] -= Jb * F[2];
  Fb[2] -= Jb * F[1];
}

// 3D elastic stress adjoint (sigma = mu_0 (F F^T - I) + la_0 log(J) on
// every entry): F_bar += mu_0 (sigma_bar + sigma_bar^T) F
//                      + la_0 (sum_ij sigma_bar_ij) F^-T,  F^-T = cof(F) / J.
template <class T>
__device__ __forceinline__ void adj_elastic3(const ParamsT<T> &P, const T (&F)[9], const T (&sb)[9], T (&Fb)[9]) {
  const T mu = P.two_mu * (T)0.5;
  T ssum = (T)0;
#pragma unroll
  for (int i = 0; i < 9; ++i) ssum += sb[i];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      T acc = (T)0;
#pragma unroll
      for (int j = 0; j < 3; ++j) acc += (sb[a * 3 + j] + sb[j * 3 + a]) * F[j * 3 + b];
      Fb[a * 3 + b] += mu * acc;
    }
  // cofactors: cof_ab = (-1)^(a+b) minor_ab; F^-T = cof / det
  const T c00 = F[4] * F[8] - F[5] * F[7], c01 = F[5] * F[6] - F[3] * F[8], c02 = F[3] * F[7] - F[4] * F[6];
  const T c10 = F[2] * F[7] - F[1] * F[8], c11 = F[0] * F[8] - F[2] * F[6], c12 = F[1] * F[6] - F[0] * F[7];
  const T c20 = F[1] * F[5] - F[2] * F[4], c21 = F[2] * F[3] - F[0] * F[5], c22 = F[0] * F[4] - F[1] * F[3];
  const T J = F[0] * c00 + F[1] * c01 + F[2] * c02;
  const T k = P.la_0 * ssum / J;
  const T cof[9] = {c00, c01, c02, c10, c11, c12, c20, c21, c22};
#pragma unroll
  for (int i = 0; i < 9; ++i) Fb[i] += k * cof[i];
}

// P2G adjoint of one particle, shared by the tiled and untiled kernels: out
// from its values v, the adjoints that G2P left (x in xg, J/F in jfb) and
// the node adjoints of (m v, m), fetch(off).
template <int DIM, int MAT, class T, class Fetch>
__device__ __forceinline__ void adj_p2g_particle(const ParamsT<T> &P, const AdjStencil<T> &S,
                                                 const T (&v)[Comps<DIM, MAT>::NC], const T (&xg)[3],
                                                 const T (&jg)[Comps<DIM, MAT>::NC - Comps<DIM, MAT>::CJ],
                                                 Fetch &&fetch, T (&out)[Comps<DIM, MAT>::NC]) {
  using CI = Comps<DIM, MAT>;
  constexpr int NJF = CI::NC - CI::CJ;
  T aff[DIM * DIM], affb[DIM * DIM];
  affine_of<DIM, MAT, T>(v, P, aff);  // stress_k sigma + m C
  if constexpr (IsF64<T>::value) {
    T c[3] = {(T)0, (T)0, (T)0}, A[3][3];
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      c[a] = P.p_mass * v[CI::CV + a];
#pragma unroll
      for (int b = 0; b < DIM; ++b) {
        A[a][b] = aff[a * DIM + b] * P.dx;
        c[a] = tfma<T>(-A[a][b], S.fx[b] - (T)1, c[a]);
      }
    }
    AdjSums<T> R;
    adj_sums<DIM, T>(
        S, c, A, fetch, [&](const vec4_t<T> &nd) { return nd.w * P.p_mass; },
        [](const int (&)[3], T, const T (&)[3]) {}, R);
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      T f = R.X[a];
#pragma unroll
      for (int b = 0; b < DIM; ++b) {
        f = tfma<T>(-A[b][a], R.S[b], f);
        affb[a * DIM + b] = P.dx * tfma<T>(-R.S[a], S.fx[b] - (T)1, R.M[a][b]);
      }
      out[CI::CX + a] = xg[a] + P.inv_dx * f;
      out[CI::CV + a] = P.p_mass * R.S[a];
    }
  } else {
    T vb[3] = {(T)0, (T)0, (T)0}, fxb[3] = {(T)0, (T)0, (T)0};
#pragma unroll
    for (int i = 0; i < DIM * DIM; ++i) affb[i] = (T)0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < (DIM == 3 ? 3 : 1); ++k) {
          const int off[3] = {i, j, k};
          T gw[3];
          const T w = adj_weight<DIM, T>(S, off, gw);
          const vec4_t<T> nd = fetch(off);
          const T mvb[3] = {nd.x, nd.y, nd.z};
          T dp[3] = {(T)0, (T)0, (T)0};
#pragma unroll
          for (int a = 0; a < DIM; ++a) dp[a] = ((T)off[a] - S.fx[a]) * P.dx;
          T contrib = nd.w * P.p_mass;
#pragma unroll
          for (int a = 0; a < DIM; ++a) {
            T q = P.p_mass * v[CI::CV + a];
#pragma unroll
            for (int b = 0; b < DIM; ++b) q += aff[a * DIM + b] * dp[b];
            contrib += mvb[a] * q;
            vb[a] += P.p_mass * w * mvb[a];
#pragma unroll
            for (int b = 0; b < DIM; ++b) affb[a * DIM + b] += w * mvb[a] * dp[b];
          }
#pragma unroll
          for (int q = 0; q < DIM; ++q) {
            T t = (T)0;
#pragma unroll
            for (int a = 0; a < DIM; ++a) t += aff[a * DIM + q] * mvb[a];
            fxb[q] += gw[q] * contrib - P.dx * w * t;
          }
        }
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      out[CI::CX + a] = xg[a] + P.inv_dx * fxb[a];
      out[CI::CV + a] = vb[a];
    }
  }
#pragma unroll
  for (int i = 0; i < DIM * DIM; ++i) out[CI::CC + i] = P.p_mass * affb[i];
  T jfb[NJF];
#pragma unroll
  for (int i = 0; i < NJF; ++i) jfb[i] = jg[i];
  if constexpr (MAT == AQ_FLUID) {
    T tr = (T)0;
#pragma unroll
    for (int a = 0; a < DIM; ++a) tr += affb[a * DIM + a];
    jfb[0] += P.la * (P.stress_k * tr);
  } else {
    T F[DIM * DIM], sb[DIM * DIM], Fb[DIM * DIM];
#pragma unroll
    for (int i = 0; i < DIM * DIM; ++i) {
      F[i] = v[CI::CJ + i];
      sb[i] = P.stress_k * affb[i];
      Fb[i] = (T)0;
    }
    if constexpr (DIM == 3)
      adj_elastic3<T>(P, F, sb, Fb);
    else
      adj_corotated<T>(P, F, sb, Fb);
#pragma unroll
    for (int i = 0; i < DIM * DIM; ++i) jfb[i] += Fb[i];
  }
#pragma unroll
  for (int i = 0; i < NJF; ++i) out[CI::CJ + i] = jfb[i];
}

// P2G adjoint on an unsorted state: completes adj_out and adds sum_p
// adj_out[c][p]^2 to gsum[c].
template <int DIM, int MAT, class T>
__global__ void __launch_bounds__(256) k_adj_p2g(const T *__restrict__ st, T *__restrict__ adj_out, int64_t cap,
                                                 int64_t n, ParamsT<T> P, const vec4_t<T> *__restrict__ gbar,
                                                 double *__restrict__ gsum) {
  using CI = Comps<DIM, MAT>;
  constexpr int NC = CI::NC, NJF = NC - CI::CJ;
  __shared__ double part[4][NC];
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  T out[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) out[c] = (T)0;
  if (p < n) {
    T v[NC], xg[3], jg[NJF];
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = st[(int64_t)c * cap + p];
#pragma unroll
    for (int a = 0; a < DIM; ++a) xg[a] = adj_out[(int64_t)(CI::CX + a) * cap + p];
#pragma unroll
    for (int i = 0; i < NJF; ++i) jg[i] = adj_out[(int64_t)(CI::CJ + i) * cap + p];
    const AdjStencil<T> S = adj_stencil<DIM, T>(v, P);
    adj_p2g_particle<DIM, MAT, T>(
        P, S, v, xg, jg, [&](const int (&off)[3]) { return gbar[adj_node<DIM>(S.base, off, P.nb)]; }, out);
#pragma unroll
    for (int c = 0; c < NC; ++c) adj_out[(int64_t)c * cap + p] = out[c];
  }
  if (gsum) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      double q = (double)out[c] * (double)out[c];
      for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o);
      if (lane == 0) part[wave][c] = q;
    }
    __syncthreads();
    if (threadIdx.x < NC) {
      const int c = threadIdx.x;
      atomic_add<double>(gsum + c, ((part[0][c] + part[1][c]) + part[2][c]) + part[3][c]);
    }
  }
}

// ---- tiled particle phases ---------------------------------------------------
// Wavefronts per SIMD that the tiled adjoint kernels' registers are kept for:
// 3D f64 keeps one (292 to 488 VGPRs).  3D f32 elastic bodies spill 2 (G2P) and
// 13 (P2G) of 168 VGPRs.
template <int DIM, class T> struct AdjWaves {
  static constexpr int W = IsF64<T>::value ? (DIM == 3 ? 1 : 2) : (DIM == 3 ? 3 : 4);
};

// G2P adjoint over work items: the velocity tile staged in LDS is read by
// every particle, and its velocity adjoints w_n u_n (u_n = vb + 4 inv_dx C_b
// (off_n - fx)) are summed in an LDS tile: with global float atomics
// (k_adj_g2p) the 81 (3D) atomics a particle bound the phase.
// The sums are doubles, for f32 adjoints too.  The node adjoints are divided
// by the node's mass afterwards, so a node that little mass reaches, or that
// lies next to far larger adjoints, needs a sum that is accurate relative to
// itself.  In fixed point relative to the item's largest adjoints a
// contribution of 2^-40 of them keeps 22 of its bits (62-bit sums), and the
// bound, the scale and the rounding cost more than the f64 atomics: 262,144
// particles of a 3D fluid, f32: 31 us in fixed point, 27 so (1630 with global
// atomics), of a 3D elastic body 36 and 30; 80,000 of a 2D elastic body, f64:
// 7.2 both ways (101).
template <int DIM, int MAT, class T>
__global__ void __launch_bounds__(kItem) __attribute__((amdgpu_waves_per_eu(AdjWaves<DIM, T>::W)))
k_adj_g2p_tiled(const T *__restrict__ st, const T *__restrict__ adj_next,
                                                         T *__restrict__ adj_out, int64_t cap, int64_t n,
                                                         ParamsT<T> P, const int4 *__restrict__ items,
                                                         const int32_t *__restrict__ nitems,
                                                         const vec4_t<T> *__restrict__ grid_v,
                                                         vec4_t<T> *__restrict__ tiles, vec4_t<T> *__restrict__ grid_f,
                                                         uint32_t *__restrict__ fflags, int32_t *flist, uint32_t *gcnt,
                                                         uint32_t ctl, uint32_t *bmargin) {
  using TL = Tile<DIM>;
  constexpr int TS = TL::TS, TN = TL::TN, TE = TL::TE, NW = kItem / 64;
  __shared__ vec4_t<T> tv[TS];
  __shared__ double ts[DIM][TS];
  __shared__ uint32_t bdrift[NW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // commit of the last list gather's appends, as tiled_body does
  const uint32_t commit = (ctl >> 2) & 3u;
  if (commit && blockIdx.x == 0 && tid == 0) {
    gcnt[0] = gcnt[3];
    gcnt[commit] = 0u;
  }
  const FlagSink sink{fflags, flist, gcnt + (ctl & 3u)};
  const int32_t nblocks = DIM == 3 ? P.nb * P.nb * P.nb : P.nb * P.nb;
  const int32_t *item_off = nitems - nblocks;
  const int ni = *nitems;
  const int xcd = (int)(blockIdx.x & 7u), per = (int)(gridDim.x >> 3);
  const int lo = (int)((int64_t)ni * xcd / 8), hi = (int)((int64_t)ni * (xcd + 1) / 8);
  int it = lo + (int)(blockIdx.x >> 3);
  if (it >= hi) return;  // uniform over the workgroup
  TileShare<DIM> share;
  share.init(tid, P.nb);
  for (int q = tid; q < TS; q += kItem)
#pragma unroll
    for (int a = 0; a < DIM; ++a) ts[a][q] = 0.0;
  for (; it < hi; it += per) {
    const int4 item = items[it];
    int o[3];
    tile_origin<DIM>(item, o);
    const int64_t p = (int64_t)item.y + tid;
    const bool has = tid < item.z && p < n;
    T x[3] = {(T)0, (T)0, (T)0};
    AdjG2P<DIM, MAT, T> A;
    if (has) adj_g2p_load<DIM, MAT, T>(st, adj_next, cap, p, x, A);
    share.template copy<T>(item, tid, grid_v, tv);
    AdjStencil<T> S;
    int rel[3] = {0, 0, 0};
    bool inside = false, drift = false;
    if (has) {
      S = adj_stencil<DIM, T>(x, P);
      A.begin(P, S);
      inside = true;
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        rel[a] = S.base[a] - o[a];
        inside = inside && rel[a] >= 0 && rel[a] + 2 < TE;
        drift = drift || rel[a] == 0 || rel[a] == TE - 3;
      }
      drift = drift && inside;
    }
    const bool wdrift = __ballot(drift) != 0ull;
    if (lane == 0) bdrift[wave] = wdrift ? 1u : 0u;
    __syncthreads();  // tile staged, the previous item's sums written out
    uint32_t d = 0u;
#pragma unroll
    for (int w = 0; w < NW; ++w) d |= bdrift[w];
    const int ib = it - item_off[item.x];
    const bool margin = d != 0u || ib >= 31;
    if (margin && tid == 0) atomicOr(bmargin + item.x, 1u << (ib < 31 ? ib : 31));
    if (has) {
      T xo[3], jo[AdjG2P<DIM, MAT, T>::NJF];
      if (inside) {
        const int q0 = TL::slot(rel[0], rel[1], rel[2]);
        A.sums(
            P, S, [&](const int (&off)[3]) { return tv[q0 + TL::slot(off[0], off[1], off[2])]; },
            [&](const int (&off)[3], T w, const T (&u)[3]) {
              const int q = q0 + TL::slot(off[0], off[1], off[2]);
#pragma unroll
              for (int a = 0; a < DIM; ++a)
                __hip_atomic_fetch_add(&ts[a][q], (double)(w * u[a]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            },
            xo, jo);
      } else {
        A.sums(
            P, S, [&](const int (&off)[3]) { return grid_v[adj_node<DIM>(S.base, off, P.nb)]; },
            [&](const int (&off)[3], T w, const T (&u)[3]) {
              T *node = (T *)(grid_f + adj_node<DIM>(S.base, off, P.nb));
#pragma unroll
              for (int a = 0; a < DIM; ++a) atomic_add<T>(node + a, w * u[a]);
            },
            xo, jo);
        mark_stencil_blocks<DIM>(S.base, P.nb, sink);
      }
      adj_g2p_store<DIM, MAT, T>(adj_out, cap, p, xo, jo);
    }
    __syncthreads();  // tile sums complete
    vec4_t<T> *dst = tiles + (int64_t)it * TN;
#pragma unroll
    for (int r = 0; r < TileShare<DIM>::R; ++r) {
      const int nd = tid + r * kItem;  // position in the buffer
      if (nd >= TN) continue;
      if (!margin && share.margin(r)) continue;
      const int q = share.slot(r);
      vec4_t<T> val;
      val.z = val.w = (T)0;
      val.x = (T)ts[0][q];
      val.y = (T)ts[1][q];
      if constexpr (DIM == 3) val.z = (T)ts[DIM - 1][q];
      dst[nd] = val;
#pragma unroll
      for (int a = 0; a < DIM; ++a) ts[a][q] = 0.0;
    }
    // the next item's copy writes tv only after every thread passed the
    // barrier above (its last reads of tv), and its sums start after the
    // next barrier
  }
}

// P2G adjoint over work items: the node adjoints staged in LDS, completing
// adj_out; sum_p adj_out^2 is carried per lane over the workgroup's items
// and added to gsum once per workgroup by f64 atomics on one or two cache
// lines (262,144 particles of a 3D fluid, f32: 29 us, 22 without sums; 80,000
// of a 2D elastic body, f64: 9.6 and 7.2).
template <int DIM, int MAT, class T>
__global__ void __launch_bounds__(kItem) __attribute__((amdgpu_waves_per_eu(AdjWaves<DIM, T>::W)))
k_adj_p2g_tiled(const T *__restrict__ st, T *__restrict__ adj_out,
                                                         int64_t cap, int64_t n, ParamsT<T> P,
                                                         const int4 *__restrict__ items,
                                                         const int32_t *__restrict__ nitems,
                                                         const vec4_t<T> *__restrict__ gbar,
                                                         double *__restrict__ gsum, uint32_t *gcnt, uint32_t ctl) {
  using CI = Comps<DIM, MAT>;
  using TL = Tile<DIM>;
  constexpr int NC = CI::NC, NJF = NC - CI::CJ, TS = TL::TS, TE = TL::TE, NW = kItem / 64;
  constexpr int NS = NC <= 16 ? 16 : 32;  // components, padded
  using Fold = LaneFold<NS>;
  __shared__ vec4_t<T> tv[TS];
  __shared__ double part[NW][NS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint32_t commit = (ctl >> 2) & 3u;
  if (commit && blockIdx.x == 0 && tid == 0) {
    gcnt[0] = gcnt[3];
    gcnt[commit] = 0u;
  }
  const int ni = *nitems;
  const int xcd = (int)(blockIdx.x & 7u), per = (int)(gridDim.x >> 3);
  const int lo = (int)((int64_t)ni * xcd / 8), hi = (int)((int64_t)ni * (xcd + 1) / 8);
  int it = lo + (int)(blockIdx.x >> 3);
  if (it >= hi) return;  // uniform over the workgroup
  double total = 0.0;    // of the lane's component
  TileShare<DIM> share;
  share.init(tid, P.nb);
  for (; it < hi; it += per) {
    const int4 item = items[it];
    int o[3];
    tile_origin<DIM>(item, o);
    const int64_t p = (int64_t)item.y + tid;
    const bool has = tid < item.z && p < n;
    T v[NC], xg[3], jg[NJF];
    if (has) {
#pragma unroll
      for (int i = 0; i < NC; ++i) v[i] = st[(int64_t)i * cap + p];
#pragma unroll
      for (int a = 0; a < DIM; ++a) xg[a] = adj_out[(int64_t)(CI::CX + a) * cap + p];
#pragma unroll
      for (int i = 0; i < NJF; ++i) jg[i] = adj_out[(int64_t)(CI::CJ + i) * cap + p];
    }
    __syncthreads();  // the previous item's reads of the tile are over
    share.template copy<T>(item, tid, gbar, tv);
    __syncthreads();
    double sq[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) sq[i] = 0.0;
    if (has) {
      const AdjStencil<T> S = adj_stencil<DIM, T>(v, P);
      int rel[3] = {0, 0, 0};
      bool inside = true;
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        rel[a] = S.base[a] - o[a];
        inside = inside && rel[a] >= 0 && rel[a] + 2 < TE;
      }
      T out[NC];
      if (inside) {
        const int q0 = TL::slot(rel[0], rel[1], rel[2]);
        adj_p2g_particle<DIM, MAT, T>(
            P, S, v, xg, jg, [&](const int (&off)[3]) { return tv[q0 + TL::slot(off[0], off[1], off[2])]; }, out);
      } else {
        adj_p2g_particle<DIM, MAT, T>(
            P, S, v, xg, jg, [&](const int (&off)[3]) { return gbar[adj_node<DIM>(S.base, off, P.nb)]; }, out);
      }
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        adj_out[(int64_t)i * cap + p] = out[i];
        sq[i] = (double)out[i] * (double)out[i];
      }
    }
    if (gsum) total += Fold::fold(sq, lane, [](double a, double b) { return a + b; });
  }
  if (gsum) {
    part[wave][Fold::value(lane)] = total;  // the lanes of a component store the same sum
    __syncthreads();
    if (tid < NC) {
      double t = part[0][tid];
#pragma unroll
      for (int w = 1; w < NW; ++w) t += part[w][tid];
      atomic_add<double>(gsum + tid, t);
    }
  }
}

}  // namespace aq
