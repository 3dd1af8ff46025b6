// AMR projections between a cell of level l and its 3^D children
// (reference: ExaHyPE/kernels/aderdg/generic/c/{2d,3d}/amrRoutines.cpph):
//   prolongation  fine[m] = sum_n coarse[n] prod_k fgp[s_k][n_k][m_k]               (:23-41)
//   restriction   coarse[m] += sum_n prod_k (w[n_k] fgp[s_k][m_k][n_k] / w[m_k]) fine[n] / 3^K
//                                                                                    (:145-170)
// with K = D-1 axes for face data and K = D for volume data, node index
// first axis fastest, fgp[s][n][m] = phi_n((s + x_m) / 3).
//
// On the static two-level mesh (amr_host.cpp) a coarse leaf next to a
// refined cell owns 3^(D-1) virtual children per such face: their face data
// are the coarse face prolongated (face_prolong_kernel, the reference's
// prolongateFaceDataToVirtualCell), the Riemann solver runs on the fine
// subfaces, and face_restrict_kernel sums the children's restricted
// fluctuations into the coarse face (restrictToTopMostParent + the
// faceIntegral glue with levelDelta = 1), which the corrector then
// integrates with the coarse cell size.
#include <hip/hip_runtime.h>

#include "engine.h"

namespace exa {
namespace {

template <int K, int B>
__device__ __forceinline__ double restrict_weight(const double* __restrict__ fgp, const double* __restrict__ w, int s0,
                                                  int s1, int s2, int n, int m) {
  // prod_k w[n_k] fgp[s_k][m_k][n_k] / w[m_k]
  double r = 1.0;
  const int sk[3] = {s0, s1, s2};
  int nn = n, mm = m;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int a = nn % B, b = mm % B;
    r *= w[a] * fgp[(sk[k] * B + b) * B + a] / w[b];
    nn /= B;
    mm /= B;
  }
  return r;
}

// Both face kernels contract one face axis after the other (2 B or 6 B products
// per value where the tensor product takes B^2 or 9 B^2) from LDS, one workgroup
// per face, so that a few hundred faces fill the chip; the weights of an axis
// are formed once.  They are bound by launch and latency, not bytes: a
// two-level mesh of order 4 with 124 coarse and 1136 fine faces 135 -> 8 us
// (restriction) and 23 -> 6 us (prolongation).
constexpr int kProlongThreads = 64, kRestrictThreads = 256;

// LDS: the coarse face's states and fluxes [B^2][ND], [B^2][V], the same
// contracted along the fast axis, and the weights of both axes.
template <int B>
__global__ __launch_bounds__(kProlongThreads) void face_prolong_kernel(const int4* __restrict__ ent,
                                                                       double* __restrict__ qb, double* __restrict__ fb,
                                                                       const DevTables* __restrict__ T, int V, int ND) {
  constexpr int NF = B * B;
  extern __shared__ double sm[];
  double* c = sm;
  double* t = c + NF * (ND + V);
  double* p0 = t + NF * (ND + V);  // [n][m] of the fast axis
  double* p1 = p0 + NF;            // [n][m] of the slow axis
  const int4 q = ent[blockIdx.x];
  const int f = q.y, s0 = q.z % 3, s1 = q.z / 3;
  const double* cq = qb + (long(q.x) * 6 + f) * NF * ND;
  const double* cf = fb + (long(q.x) * 6 + f) * NF * V;
  for (int o = threadIdx.x; o < NF * ND; o += kProlongThreads) c[o] = cq[o];
  for (int o = threadIdx.x; o < NF * V; o += kProlongThreads) c[NF * ND + o] = cf[o];
  for (int o = threadIdx.x; o < NF; o += kProlongThreads) {
    p0[o] = T->fgp[s0 * NF + o];
    p1[o] = T->fgp[s1 * NF + o];
  }
  __syncthreads();
  for (int a = 0; a < 2; a++) {  // states, then fluxes
    const int nv = a ? V : ND, at = a ? NF * ND : 0;
    for (int o = threadIdx.x; o < NF * nv; o += kProlongThreads) {
      const int m = o / nv, v = o - m * nv, m1 = m % B, n2 = m / B;
      double acc = 0.0;
#pragma unroll
      for (int n1 = 0; n1 < B; n1++) acc += p0[n1 * B + m1] * c[at + (n2 * B + n1) * nv + v];
      t[at + o] = acc;
    }
  }
  __syncthreads();
  for (int a = 0; a < 2; a++) {
    const int nv = a ? V : ND, at = a ? NF * ND : 0;
    double* dst = (a ? fb : qb) + (long(q.w) * 6 + f) * NF * nv;
    for (int o = threadIdx.x; o < NF * nv; o += kProlongThreads) {
      const int m = o / nv, v = o - m * nv, m1 = m % B, m2 = m / B;
      double acc = 0.0;
#pragma unroll
      for (int n2 = 0; n2 < B; n2++) acc += p1[n2 * B + m2] * t[at + (n2 * B + m1) * nv + v];
      dst[o] = acc;
    }
  }
}

// LDS: the nine subfaces' fluxes [9][B^2][V], the same contracted along the fast
// axis and its subfaces [3][B][B][V], and the weights of an axis [3][m][n].
template <int B>
__global__ __launch_bounds__(kRestrictThreads) void face_restrict_kernel(const int4* __restrict__ ent,
                                                                         double* __restrict__ fb,
                                                                         const DevTables* __restrict__ T, int V) {
  constexpr int NF = B * B;
  extern __shared__ double sm[];
  double* c = sm;
  double* t = c + 9 * NF * V;
  double* r = t + 3 * NF * V;
  const int4 q = ent[blockIdx.x];
  const int f = q.y, per = NF * V;
  for (int o = threadIdx.x; o < 9 * per; o += kRestrictThreads) {
    const int sub = o / per;
    c[o] = fb[((long(q.z) + sub) * 6 + f) * per + (o - sub * per)];
  }
  for (int o = threadIdx.x; o < 3 * NF; o += kRestrictThreads)  // w[n] fgp[s][m][n] / w[m] / 3
    r[o] = T->w[o % B] * T->fgp[o] / T->w[o / B % B] / 3.0;
  __syncthreads();
  for (int o = threadIdx.x; o < 3 * per; o += kRestrictThreads) {
    const int m = o / V, v = o - m * V, m1 = m % B, n2 = m / B % B, s1 = m / NF;
    double acc = 0.0;
#pragma unroll
    for (int s0 = 0; s0 < 3; s0++)
#pragma unroll
      for (int n1 = 0; n1 < B; n1++)
        acc += r[(s0 * B + m1) * B + n1] * c[((s0 + 3 * s1) * NF + n2 * B + n1) * V + v];
    t[o] = acc;
  }
  __syncthreads();
  double* cf = fb + (long(q.x) * 6 + f) * per;
  for (int o = threadIdx.x; o < per; o += kRestrictThreads) {
    const int m = o / V, v = o - m * V, m1 = m % B, m2 = m / B;
    double acc = 0.0;
#pragma unroll
    for (int s1 = 0; s1 < 3; s1++)
#pragma unroll
      for (int n2 = 0; n2 < B; n2++) acc += r[(s1 * B + m2) * B + n2] * t[(s1 * NF + n2 * B + m1) * V + v];
    cf[o] = acc;
  }
}

template <int K, int B>
__global__ __launch_bounds__(256) void project_kernel(int nv, const double* __restrict__ in, double* __restrict__ out,
                                                      int s0, int s1, int s2, int mode,
                                                      const DevTables* __restrict__ T) {
  int NK = 1;
#pragma unroll
  for (int k = 0; k < K; k++) NK *= B;
  const double scale = (K == 1) ? 3.0 : (K == 2 ? 9.0 : 27.0);
  for (int o = threadIdx.x; o < NK * nv; o += blockDim.x) {
    const int m = o / nv, v = o - m * nv;
    double acc = 0.0;
    for (int nn = 0; nn < NK; nn++) {
      double wgt;
      if (mode == 0) {
        wgt = 1.0;
        int a = nn, b = m;
        const int sk[3] = {s0, s1, s2};
        for (int k = 0; k < K; k++) {
          wgt *= T->fgp[(sk[k] * B + a % B) * B + b % B];
          a /= B;
          b /= B;
        }
      } else {
        wgt = restrict_weight<K, B>(T->fgp, T->w, s0, s1, s2, nn, m);
      }
      acc += wgt * in[nn * nv + v];
    }
    if (mode == 0)
      out[o] = acc;
    else
      out[o] += acc / scale;
  }
}

template <int B>
int dispatch_faces(const KernelCfg& k, hipStream_t s, long n, const int* ent, double* qb, double* fb, bool prolong) {
  const int V = k.nvar, ND = k.nvar + k.npar;
  if (prolong)
    face_prolong_kernel<B><<<unsigned(n), kProlongThreads, sizeof(double) * B * B * (2 * (ND + V) + 2), s>>>(
        reinterpret_cast<const int4*>(ent), qb, fb, k.tab, V, ND);
  else
    face_restrict_kernel<B><<<unsigned(n), kRestrictThreads, sizeof(double) * B * B * (12 * V + 3), s>>>(
        reinterpret_cast<const int4*>(ent), fb, k.tab, V);
  return static_cast<int>(hipGetLastError());
}

int faces(const KernelCfg& k, hipStream_t s, long n, const int* ent, double* qb, double* fb, bool prolong) {
  if (n <= 0) return 0;
  if (k.dim != 3) return -1;  // the two-level mesh is 3D
  switch (k.order + 1) {
    case 2: return dispatch_faces<2>(k, s, n, ent, qb, fb, prolong);
    case 3: return dispatch_faces<3>(k, s, n, ent, qb, fb, prolong);
    case 4: return dispatch_faces<4>(k, s, n, ent, qb, fb, prolong);
    case 5: return dispatch_faces<5>(k, s, n, ent, qb, fb, prolong);
    case 6: return dispatch_faces<6>(k, s, n, ent, qb, fb, prolong);
    case 7: return dispatch_faces<7>(k, s, n, ent, qb, fb, prolong);
    default: return -1;
  }
}

template <int K>
int project_k(const KernelCfg& k, hipStream_t s, int nv, const double* in, double* out, int s0, int s1, int s2,
              int mode) {
  switch (k.order + 1) {
    case 2: project_kernel<K, 2><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    case 3: project_kernel<K, 3><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    case 4: project_kernel<K, 4><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    case 5: project_kernel<K, 5><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    case 6: project_kernel<K, 6><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    case 7: project_kernel<K, 7><<<1, 256, 0, s>>>(nv, in, out, s0, s1, s2, mode, k.tab); break;
    default: return -1;
  }
  return static_cast<int>(hipGetLastError());
}

}  // namespace

int launch_face_prolong(const KernelCfg& k, hipStream_t s, long n, const int* entries, double* qb, double* fb) {
  return faces(k, s, n, entries, qb, fb, true);
}

int launch_face_restrict(const KernelCfg& k, hipStream_t s, long n, const int* entries, double* fb) {
  return faces(k, s, n, entries, nullptr, fb, false);
}

int launch_face_project(const KernelCfg& k, hipStream_t s, int nv, const double* in, double* out, int s0, int s1,
                        int mode) {
  return k.dim == 3 ? project_k<2>(k, s, nv, in, out, s0, s1, 0, mode) : project_k<1>(k, s, nv, in, out, s0, 0, 0, mode);
}

int launch_volume_project(const KernelCfg& k, hipStream_t s, int nv, const double* in, double* out, int s0, int s1,
                          int s2, int mode) {
  return k.dim == 3 ? project_k<3>(k, s, nv, in, out, s0, s1, s2, mode) : project_k<2>(k, s, nv, in, out, s0, s1, 0, mode);
}

}  // namespace exa
