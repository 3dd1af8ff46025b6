// Space-time predictor + volume integral, column / line form (2D and 3D, all
// compiled shapes, FP64 and FP32; conservative PDEs).
//
// Reference path (ExaHyPE/kernels/aderdg/generic/c/{2d,3d}):
// spaceTimePredictorNonlinear.cpph (Picard loop :39-433, time averaging
// :441-515, extrapolation :517-687) and volumeIntegralNonlinear.cpph
// (time-averaged branch :133-223), with the update written as
//   g[t]    = dt sum_d (1/dx_d) dudx (x)_d F_d(lQi[t])     (flux divergence)
//   lQi'[t] = luh - sum_t' P[t][t'] g[t'],   P = iK1 diag(w)
// (Kxi[n][l] / w_l = dudx[l][n] and iK1 F0 = 1, so it equals the reference's
// W^-1 iK1 (W F0 luh - stiffness terms) up to rounding).
//
// Decomposition: a lane owns one spatial node and its whole time column
// lQi[0..B)[V] in registers, so flux evaluation and the time solve need no
// exchange.  A spatial derivative is taken line by line: the owners write
// their fluxes into LDS with the B values of each (variable, direction, line)
// contiguous, then the workgroup's lanes take those lines one each, contract
// them with the operator (uniform coefficients in scalar registers) and write
// the B results back in place, and the owners read their values.  An LDS value
// is read once per direction: 4 LDS accesses per value and slice where a node
// that reads the B-point lines through itself needs 1 + B, plus its column of
// the operator.  What bounds it: LDS (a 64-lane write of 8 bytes takes 6 cycles
// of a CU, a read 2.4 to 4) and FP64 issue, which overlap only between
// workgroups: in 3D order 5 both are busy about half of the time.  Against the
// node-column form before it (each lane reading the lines through its node;
// MI355X, predictor alone): 3D order 5 FP64 at 81^3 36.3 -> 23.9 ms (20 TF/s of
// executed contraction work, 78.6 peak), with the CERK guess at 40^3 2.60 ->
// 1.86 ms, 2D order 4 at 243^2 0.284 -> 0.212 ms.
#pragma once

#include <hip/hip_runtime.h>

#include "engine.h"

namespace exa {
namespace columns {

constexpr int cpow(int b, int e) { return e == 0 ? 1 : b * cpow(b, e - 1); }
constexpr int ceil64(int n) { return (n + 63) / 64 * 64; }

template <int D, int B, int V, int NP, typename R>
struct Shape {
  static constexpr int ND = V + NP;
  static constexpr int NS = cpow(B, D);      // spatial nodes per cell
  static constexpr int NF = cpow(B, D - 1);  // nodes per face
  static constexpr int NL = D * NF;          // lines per cell
  // The smallest workgroup whose lanes own nodes for at least 93 %: one
  // wavefront needs no barrier waits (orders 2 and 3 in 2D, 3 in 3D).  Two
  // exceptions, predictor alone, Euler:
  // - order 1, bound by HBM alone and in FP32 slower in 64 lanes than with the
  //   node-column form before it: 256 (375,000 3D cells, three FP32 iterations,
  //   237 -> 211 us; node-column 218).
  // - 3D order 2 in FP64: 54 of 64 lanes, because the barriers of 243 of 256
  //   weigh more than the idle lanes (8,000 cells 33.5 -> 29.4 us, 64 cells 13.1
  //   -> 9.5, node-column 12.3; 111,111 cells equal).
  static constexpr int threads() {
    if (B == 2) return 256;
    if (D == 3 && B == 3 && sizeof(R) == 8) return 64;
    for (int t : {64, 128, 256})
      if (t / NS * NS * 100 >= 93 * t) return t;
    return 256;
  }
  static constexpr int THREADS = threads();
  static constexpr int CPB = THREADS / NS;  // cells per workgroup
  static constexpr int SLICE = CPB * NL * V * B;  // values of one time slice
  // Time slices between two barriers.  Two fill the rounds of line tasks better
  // and halve the barriers where the registers allow two workgroups per CU
  // anyway (3D order 5 in FP64 at 81^3: 26.4 -> 23.9 ms; three leave LDS for one
  // workgroup: 38.3 ms); smaller 3D cells gain as much from the workgroups that
  // the LDS of a second slice would cost (batched 3D order 4: equal).
  static constexpr int TS = D == 3 && B <= 5 ? 1 : 2;
  static constexpr int NROW = NS / B;
  // orders 1 and 3 exchange their lines between lanes and need the buffer at the end only
  static constexpr bool LANES = B == 2 || B == 4;
  // 3D order 2 in FP32: a node reads the three lines through itself (three values
  // each, as many LDS accesses as a line task's four, and one phase less), from two
  // slices in turn; 64 cells, three iterations 12.2 -> 9.9 us (node-column 11.3),
  // 111,111 cells 264 -> 223 (233)
  static constexpr bool NODES = D == 3 && B == 3 && sizeof(R) == 4;
  static constexpr int LINE_BYTES = LANES ? 0 : (NODES ? 2 : TS) * SLICE * int(sizeof(R));
  static constexpr int END_BYTES = (SLICE + CPB * NS * ND) * 8;
  static constexpr int BUF_BYTES = LINE_BYTES > END_BYTES ? LINE_BYTES : END_BYTES;
  static constexpr int RED = CPB * (NS + NROW);
};

template <typename R>
__device__ __forceinline__ const R* tab_dudx(const DevTables* T) {
  if constexpr (sizeof(R) == 8) return T->dudx_eo; else return T->dudx_eof;
}
template <typename R>
__device__ __forceinline__ const R* tab_P(const DevTables* T) {
  if constexpr (sizeof(R) == 8) return T->Pt; else return T->Ptf;
}

// The operator tables are constant during a launch: in the constant address
// space uniform reads of them are scalar loads.  The pointer is also hidden
// from loop-invariant code motion, so a phase reads its entries through the
// scalar cache instead of all phases' entries being held in scalar registers
// (whose spills cost a vector instruction each).
template <typename X>
using Const = const __attribute__((address_space(4))) X;
template <typename X>
__device__ __forceinline__ Const<X>* opaque(const X* p) {
  unsigned long long a = reinterpret_cast<unsigned long long>(p);
  asm volatile("" : "+s"(a));
  return reinterpret_cast<Const<X>*>(a);
}

// Line of B values at p (16-byte pieces where the line start allows them).
template <typename R, int B>
__device__ __forceinline__ void load_line(const R* p, R (&f)[B]) {
  if constexpr (sizeof(R) == 8 && B % 2 == 0) {
#pragma unroll
    for (int i = 0; i < B / 2; i++) {
      const double2 v = reinterpret_cast<const double2*>(p)[i];
      f[2 * i] = v.x;
      f[2 * i + 1] = v.y;
    }
  } else if constexpr (sizeof(R) == 4 && B % 4 == 0) {
#pragma unroll
    for (int i = 0; i < B / 4; i++) {
      const float4 v = reinterpret_cast<const float4*>(p)[i];
      f[4 * i] = v.x;
      f[4 * i + 1] = v.y;
      f[4 * i + 2] = v.z;
      f[4 * i + 3] = v.w;
    }
  } else if constexpr (sizeof(R) == 4 && B % 2 == 0) {
#pragma unroll
    for (int i = 0; i < B / 2; i++) {
      const float2 v = reinterpret_cast<const float2*>(p)[i];
      f[2 * i] = v.x;
      f[2 * i + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < B; i++) f[i] = p[i];
  }
}
template <typename R, int B>
__device__ __forceinline__ void store_line(R* p, const R (&f)[B]) {
  if constexpr (sizeof(R) == 8 && B % 2 == 0) {
#pragma unroll
    for (int i = 0; i < B / 2; i++) reinterpret_cast<double2*>(p)[i] = make_double2(f[2 * i], f[2 * i + 1]);
  } else if constexpr (sizeof(R) == 4 && B % 4 == 0) {
#pragma unroll
    for (int i = 0; i < B / 4; i++)
      reinterpret_cast<float4*>(p)[i] = make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
  } else if constexpr (sizeof(R) == 4 && B % 2 == 0) {
#pragma unroll
    for (int i = 0; i < B / 2; i++) reinterpret_cast<float2*>(p)[i] = make_float2(f[2 * i], f[2 * i + 1]);
  } else {
#pragma unroll
    for (int i = 0; i < B; i++) p[i] = f[i];
  }
}

// Operator M with M[B-1-i][B-1-j] = -M[i][j] (dudx and Kxi on the symmetric
// Gauss-Legendre nodes) in the halves fill_even_odd (capi.cpp) stores.
template <typename R, int B>
struct EvenOdd {
  static constexpr int H = B / 2, N = 2 * H * H + (B % 2 ? 2 * H : 0);
  R m[N];
  __device__ __forceinline__ explicit EvenOdd(Const<R>* t) {
#pragma unroll
    for (int i = 0; i < N; i++) m[i] = t[i];
  }
  // out = M f: the sums out[i] + out[B-1-i] need only the differences of the
  // line's mirrored values, their differences only the sums (30 operations
  // instead of 36 at B = 6, half the coefficients)
  __device__ __forceinline__ void apply(const R (&f)[B], R (&out)[B]) const {
    R e[H], o[H];
#pragma unroll
    for (int j = 0; j < H; j++) {
      e[j] = f[j] + f[B - 1 - j];
      o[j] = f[j] - f[B - 1 - j];
    }
#pragma unroll
    for (int i = 0; i < H; i++) {
      R s = m[i * H] * o[0], a = m[H * H + i * H] * e[0];
#pragma unroll
      for (int j = 1; j < H; j++) {
        s += m[i * H + j] * o[j];
        a += m[H * H + i * H + j] * e[j];
      }
      if constexpr (B % 2 == 1) a += m[2 * H * H + i] * f[H];
      out[i] = s + a;
      out[B - 1 - i] = s - a;
    }
    if constexpr (B % 2 == 1) {
      R c = m[2 * H * H + H] * o[0];
#pragma unroll
      for (int j = 1; j < H; j++) c += m[2 * H * H + H + j] * o[j];
      out[H] = c;
    }
  }
};

// Lines of two nodes (order 1) lie in eight consecutive lanes, the bits of a lane
// its x, y and z: a partner's value comes by one exchange (x, y) or two (z).
// Four-node lines (order 3) stay in one wavefront: 16 consecutive lanes hold a
// plane (x fastest) and, in 3D, the wave's four rows the planes.  The other
// values of a line come by lane exchange instead of LDS: rotations of the quad
// (x) and of the row by four lanes (y), and the swaps of half waves and of rows
// for z.  A cell's lanes are all active or none.  Costs 6 to 12 register moves a
// value where LDS takes 4 accesses and their waits: bound by FP64 issue instead
// of LDS; predictor in FP64 at 35^3 0.398 (0.573 node-column) -> 0.375 ms and
// in 2D at 27^2, where the waits dominate, 15.8 -> 12.1 us, in FP32 at 45^3
// 0.480 -> 0.447 ms.
template <int CTRL, typename R>
__device__ __forceinline__ R dpp(R v) {
  if constexpr (sizeof(R) == 8) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(R, (static_cast<unsigned long long>(hi) << 32) | lo);
  } else {
    return __builtin_bit_cast(R, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
  }
}
constexpr int quad_rotate(int k) {  // lane i of a quad takes lane (i + k) % 4
  return (k & 3) | ((1 + k) & 3) << 2 | ((2 + k) & 3) << 4 | ((3 + k) & 3) << 6;
}
// lane i of a quad takes lane i ^ 1, i ^ 2, i ^ 3; lane i of eight takes lane i ^ 7
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kQuadXor3 = 0x1b, kHalfRowXor7 = 0x141;
constexpr int row_take(int n) { return 0x120 + 16 - n; }  // lane i of a row takes lane (i + n) % 16

// The values of the four rows at this lane's place in its row, in every row.
__device__ __forceinline__ void all_rows(unsigned v, unsigned (&r)[4]) {
  const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // rows 0 1 0 1 and 2 3 2 3
  const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
  r[0] = a[0];
  r[1] = a[1];
  r[2] = b[0];
  r[3] = b[1];
}
template <typename R>
__device__ __forceinline__ void all_rows(R v, R (&r)[4]) {
  if constexpr (sizeof(R) == 8) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    unsigned lo[4], hi[4];
    all_rows(static_cast<unsigned>(b), lo);
    all_rows(static_cast<unsigned>(b >> 32), hi);
#pragma unroll
    for (int i = 0; i < 4; i++)
      r[i] = __builtin_bit_cast(R, (static_cast<unsigned long long>(hi[i]) << 32) | lo[i]);
  } else {
    unsigned w[4];
    all_rows(__builtin_bit_cast(unsigned, v), w);
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = __builtin_bit_cast(R, w[i]);
  }
}

// Component of the Euler flux that F_d[v] shares with an earlier direction
// (the momentum fluxes are symmetric: F_d[1+e] = F_e[1+d]).
__host__ __device__ constexpr bool euler_canonical(int D, int d, int v) { return !(v >= 1 && v <= D && v < d + 1); }

// Flux of one state: the Euler fluxes from the velocities (each momentum flux
// once), other equations by their hook.
template <int D, int V, typename R, bool EU>
__device__ __forceinline__ void flux(const PdeParams& P, const R* __restrict__ Q, R (&F)[D][V]) {
  if constexpr (EU) {
    R irho;
    if constexpr (sizeof(R) == 8) {
      // hardware reciprocal and two Newton steps (error <= 1 ulp)
      irho = __builtin_amdgcn_rcp(Q[0]);
      R e = __builtin_fma(-Q[0], irho, R(1));
      irho = __builtin_fma(irho, e, irho);
      e = __builtin_fma(-Q[0], irho, R(1));
      irho = __builtin_fma(irho, e, irho);
    } else {
      irho = R(1) / Q[0];
    }
    R u[D];
    R j2 = R(0);
#pragma unroll
    for (int d = 0; d < D; d++) {
      u[d] = irho * Q[1 + d];
      j2 += u[d] * Q[1 + d];
    }
    const R p = static_cast<R>(1.4 - 1) * (Q[4] - R(0.5) * j2);
    const R h = Q[4] + p;
#pragma unroll
    for (int d = 0; d < D; d++) {
      F[d][0] = Q[1 + d];
#pragma unroll
      for (int e = 0; e < 3; e++)
        F[d][1 + e] = e == d ? u[d] * Q[1 + d] + p : (e < d ? F[e < d ? e : 0][1 + d] : u[d] * Q[1 + e]);
      F[d][4] = u[d] * h;
    }
  } else {
    pde_flux<D, R>(P, Q, F);
  }
}

// EU: the Euler equations (the symmetric momentum fluxes' time averages are
// kept once); CG: the CERK initial guess of the optimised kernels
// (KernelGenerator/kernelgenerator/templates/aderdg/fusedSPTVI_nonlinear_cpp.template:121-173).
template <int D, int B, int V, int NP, typename R, bool CG, bool EU>
struct Tile {
  using S = Shape<D, B, V, NP, R>;
  static constexpr int ND = S::ND, NS = S::NS, NF = S::NF, NL = S::NL, CPB = S::CPB, THREADS = S::THREADS,
                       SLICE = S::SLICE, TS = S::TS, VS = CPB * NL * B;

  // Two waves per SIMD leave the registers for the average in the loop (CERK at
  // 40^3, order 5: 2.02 -> 1.86 ms); order 3, in FP64 at two waves too, needs them for
  // the rows of its exchange.  The other shapes run at three or four (min_waves), order
  // 4 with a few spilled registers, and gain more from the third wave (batched 3D
  // order 4 at 23^3, whole step: 518 us at two waves, 539 at three with the
  // average in the loop, 481 this way; 2D at 243^2 0.220, 0.249 and 0.200 ms).
  static constexpr bool FHL = sizeof(R) == 8 && B >= 6;

  static constexpr bool LANES = S::LANES, NODES = S::NODES;

  // The node's solution stays in registers where the column leaves them (orders 1
  // and 2, bound by HBM: a second read of luh per iteration misses the L1; 375,000
  // 3D cells of order 1, three FP32 iterations in 64 lanes 266 -> 237 us)
  static constexpr bool HOLD = B <= 3;

  static __device__ __forceinline__ bool keep(int d, int v) { return !EU || euler_canonical(D, d, v); }

  // The line tasks of n slices: contract every line of the buffer in place,
  // the next line of a lane on its way while this one is contracted.
  static __device__ __forceinline__ void lines(R* buf, int n, const DevTables* __restrict__ T) {
    const int last = n * (SLICE / B);
    const EvenOdd<R, B> M(opaque(tab_dudx<R>(T)));
    int id = threadIdx.x;
    R f[B], o[B];
    if (id < last) load_line<R, B>(buf + id * B, f);
#pragma unroll 1
    while (id < last) {
      M.apply(f, o);
      const int next = id + THREADS;
      if (next < last) load_line<R, B>(buf + next * B, f);
      store_line<R, B>(buf + id * B, o);
      id = next;
    }
  }

  static __device__ void run(long blk, long ncells, const double* luh, const double* __restrict__ hcell,
                             const double* __restrict__ dtp, const int* __restrict__ cinst,
                             double* __restrict__ lduh, double* __restrict__ lQhbnd, double* __restrict__ lFhbnd,
                             int* __restrict__ picard, const DevTables* __restrict__ T, const PdeParams& P,
                             int mostIter, int adaptive, double* luh_upd, int dialect, int hdim, unsigned char* buf,
                             double* red) {
    const int tid = threadIdx.x;
    const int cib = tid / NS;
    const int s = tid - cib * NS;
    const bool inslot = cib < CPB;  // the lane owns a node of one of the workgroup's cell slots
    const long cell = blk * CPB + cib;
    const bool valid = inslot && cell < ncells;
    const int cs = inslot ? cib : 0;
    const int x = s % B, y = (s / B) % B, z = D == 3 ? s / (B * B) : 0;
    // position of the node's value (d, v = 0) in the buffer of one slice:
    // line (z, y), (z, x), (y, x) of direction x, y, z (2D: y, x), entry x, y, z
    int off[D], line[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
      line[d] = cs * NL + d * NF + (D == 3 ? (d == 0 ? z * B + y : (d == 1 ? z * B + x : y * B + x)) : (d == 0 ? y : x));
      off[d] = line[d] * B + (d == 0 ? x : (d == 1 ? y : z));
    }
    R* slab = reinterpret_cast<R*>(buf);
    const double dt = dtp[(cinst && valid) ? cinst[cell] : 0];
    R cd[D];  // dt / dx_d: hcell[cell] (cubic cells, hdim = 0) or hcell[cell][d] (hdim = D)
#pragma unroll
    for (int d = 0; d < D; d++)
      cd[d] = static_cast<R>(dt / (valid ? hcell[hdim ? cell * hdim + d : cell] : 1.0));

    // the node's solution: held, or read again where it is needed
    R held[ND];
    auto solution = [&](R(&u)[ND], bool first = false) {
#pragma unroll
      for (int v = 0; v < ND; v++) {
        if (HOLD && !first)
          u[v] = held[v];
        else
          u[v] = valid ? static_cast<R>(luh[(cell * NS + s) * ND + v]) : (v == 0 ? R(1) : R(0));
      }
    };
    if constexpr (HOLD) solution(held, true);

    auto publish = [&](int slice, const R(&F)[D][V]) {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) slab[slice * SLICE + off[d] + v * VS] = F[d][v];
    };
    auto gather = [&](int slice, R(&g)[V]) {
#pragma unroll
      for (int v = 0; v < V; v++) {
        R a = cd[0] * slab[slice * SLICE + off[0] + v * VS];
#pragma unroll
        for (int d = 1; d < D; d++) a += cd[d] * slab[slice * SLICE + off[d] + v * VS];
        g[v] = a;
      }
    };
    // LANES, NODES: row c_d of dt / dx_d dudx; LANES: from the node's own entry on
    // round the line (order 3 along z: from plane 0)
    R cl[LANES || NODES ? D : 1][B];
    if constexpr (LANES || NODES) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        const int c = d == 0 ? x : (d == 1 ? y : z);
#pragma unroll
        for (int k = 0; k < B; k++) {
          const int n = NODES || (B == 4 && d == 2) ? k : (c + k) % B;
          cl[d][k] = cd[d] * (sizeof(R) == 8 ? static_cast<R>(T->dudx[c * B + n]) : static_cast<R>(T->dudxf[c * B + n]));
        }
      }
    }
    // dt times the divergence of the flux F by lane exchange
    auto exchange = [&](const R(&F)[D][V], R(&g)[V]) __attribute__((always_inline)) {
      if constexpr (B == 2) {
#pragma unroll
        for (int v = 0; v < V; v++) {
          R a = cl[0][0] * F[0][v];
          a += cl[0][1] * dpp<kQuadXor1>(F[0][v]);
          a += cl[1][0] * F[1][v];
          a += cl[1][1] * dpp<kQuadXor2>(F[1][v]);
          if constexpr (D == 3) {
            a += cl[D - 1][0] * F[D - 1][v];
            a += cl[D - 1][1] * dpp<kQuadXor3>(dpp<kHalfRowXor7>(F[D - 1][v]));
          }
          asm volatile("" : "+v"(a));  // as below
          g[v] = a;
        }
      }
      if constexpr (B == 4) {
#pragma unroll
        for (int v = 0; v < V; v++) {
          R a = cl[0][0] * F[0][v];
          a += cl[0][1] * dpp<quad_rotate(1)>(F[0][v]);
          a += cl[0][2] * dpp<quad_rotate(2)>(F[0][v]);
          a += cl[0][3] * dpp<quad_rotate(3)>(F[0][v]);
          a += cl[1][0] * F[1][v];
          a += cl[1][1] * dpp<row_take(4)>(F[1][v]);
          a += cl[1][2] * dpp<row_take(8)>(F[1][v]);
          a += cl[1][3] * dpp<row_take(12)>(F[1][v]);
          if constexpr (D == 3) {
            R r[4];
            all_rows(F[D - 1][v], r);
#pragma unroll
            for (int k = 0; k < 4; k++) a += cl[D - 1][k] * r[k];
          }
          asm volatile("" : "+v"(a));  // formed here: sunk to its use, it would keep the exchanged values alive
          g[v] = a;
        }
      }
    };
    // NODES: the same from the lines of a published slice
    auto through = [&](int slice, R(&g)[V]) __attribute__((always_inline)) {
#pragma unroll
      for (int v = 0; v < V; v++) {
        R a = R(0);
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
          for (int n = 0; n < B; n++) a += cl[d][n] * slab[slice * SLICE + line[d] * B + n + v * VS];
        g[v] = a;
      }
    };
    // dt times the flux divergence of the one state Q at the node
    auto divergence = [&](const R* Q, R(&F)[D][V], R(&g)[V]) __attribute__((always_inline)) {
      if constexpr (LANES) {
        if (valid) {
          flux<D, V, R, EU>(P, Q, F);
          exchange(F, g);
        }
        return;
      }
      if (valid) {
        flux<D, V, R, EU>(P, Q, F);
        publish(0, F);
      }
      __syncthreads();
      if constexpr (NODES) {
        if (valid) through(0, g);
        __syncthreads();  // read before the slice is written again
      } else {
        lines(slab, 1, T);
        __syncthreads();
        if (valid) gather(0, g);
      }
    };

    // FHL: the time-averaged flux of the running iteration accumulates in
    // registers and q is the current iterate; otherwise q is the iterate an
    // iteration starts from, g becomes the one it gives, and the flux average is
    // formed from q after the loop
    R q[B][ND], g[B][V], fh[D][V];
    auto average = [&](int t, const R(&F)[D][V]) {
      const R wt = static_cast<R>(T->w[t]);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++)
          if (keep(d, v)) {
            if (t == 0)
              fh[d][v] = F[d][v] * wt;
            else
              fh[d][v] += F[d][v] * wt;
          }
    };
    bool active = valid;
    int maxIter = mostIter;
    int iters = maxIter;

    // Sum of the squared update of iteration iter over the cell and the adaptive
    // rule (stop below 1e-7); true when no cell of the workgroup iterates further.
    auto finished = [&](int iter, double sq) -> bool {
      if (!adaptive) return false;
      double res;
      if constexpr (CPB == 1 || (64 % NS == 0)) {
        // butterfly over the cell's lanes of the wave (every lane ends with the
        // same bits), then, in a cell of several waves, the wave sums in order
        constexpr int W = NS < 64 ? NS : 64;
        res = sq;  // 0 on lanes past the cell
#pragma unroll
        for (int m = W / 2; m >= 1; m >>= 1) res += __shfl_xor(res, m, 64);
        if constexpr (NS > 64) {
          if ((tid & 63) == 0) red[tid >> 6] = res;
          __syncthreads();
          res = 0.0;
#pragma unroll
          for (int i = 0; i < THREADS / 64; i++) res += red[i];
        }
      } else {
        // rows of B nodes, then the rows, in a fixed order
        if (inslot) red[cib * NS + s] = sq;
        __syncthreads();
        double* part = red + CPB * NS;
        if (inslot && s < S::NROW) {
          double a = 0.0;
#pragma unroll
          for (int i = 0; i < B; i++) a += red[cib * NS + s * B + i];
          part[cib * S::NROW + s] = a;
        }
        __syncthreads();
        res = 0.0;
#pragma unroll
        for (int i = 0; i < S::NROW; i++) res += part[cs * S::NROW + i];
      }
      const double tol = 1e-7;
      if (active && res < tol * tol) {
        active = false;
        // reference return conventions; optimised kernels: min(iter + 1, MaxIterations)
        iters = dialect ? (iter + 1 < maxIter ? iter + 1 : maxIter) : ((D == 3) ? iter : maxIter + 2);
      }
      if constexpr (CPB == 1) return !(valid_block(blk, ncells) && res >= tol * tol);
      if constexpr (THREADS == 64)
        return __ballot(active) == 0;
      else
        return !__syncthreads_or(active);
    };

    {
      R u[ND];
      solution(u);
      if constexpr (CG) {
        // K1 = sum_d dudx_d F_d(luh) / dx, lwh = luh - dt K1, K2 of lwh,
        // lQi(t) = luh - dt xi_t K1 - dt xi_t^2 (K2 - K1) / 2 (k1, k2 hold dt K)
        R k1[V], k2[V], lw[ND];
        divergence(u, fh, k1);
#pragma unroll
        for (int v = 0; v < ND; v++) lw[v] = v < V ? u[v] - k1[v < V ? v : 0] : u[v];
        divergence(lw, fh, k2);
#pragma unroll
        for (int t = 0; t < B; t++) {
          const R xt = static_cast<R>(T->x[t]);
#pragma unroll
          for (int v = 0; v < ND; v++)
            q[t][v] = v < V ? u[v] - xt * k1[v < V ? v : 0] - (R(0.5) * xt * xt) * (k2[v < V ? v : 0] - k1[v < V ? v : 0])
                            : u[v];
        }
      } else {
        // Trivial guess: the time slices of the first iterate all equal luh, so
        // iteration 0 takes one divergence k and its rows sum_t' P[t][t'] k = xi_t k
        R k[V];
        divergence(u, fh, k);  // the average of equal slices is the flux
        double sq = 0.0;
#pragma unroll
        for (int t = 0; t < B; t++) {
          const R xt = static_cast<R>(T->x[t]);
#pragma unroll
          for (int v = 0; v < ND; v++) {
            q[t][v] = u[v];
            if (v < V && valid) {
              const R a = u[v] - xt * k[v < V ? v : 0];
              const double dq = static_cast<double>(a) - static_cast<double>(u[v]);
              sq += dq * dq;
              if constexpr (FHL)
                q[t][v] = a;
              else
                g[t][v < V ? v : 0] = a;
            }
          }
        }
        if (finished(0, sq)) maxIter = 0;
      }
    }

#pragma unroll 1
    for (int iter = CG ? 0 : 1; iter < maxIter; iter++) {
      if (!FHL && active && (!CG || iter > 0)) {
#pragma unroll
        for (int t = 0; t < B; t++)
#pragma unroll
          for (int v = 0; v < V; v++) q[t][v] = g[t][v];
      }
      if constexpr (LANES) {
        if (active) {
#pragma unroll
          for (int t = 0; t < B; t++) {
            R F[D][V];
            flux<D, V, R, EU>(P, q[t], F);
            exchange(F, g[t]);
            __builtin_amdgcn_sched_barrier(0);  // slices one after the other: interleaved, they spill
          }
        }
      } else if constexpr (NODES) {
#pragma unroll
        for (int t = 0; t < B; t++) {
          if (active) {
            R F[D][V];
            flux<D, V, R, EU>(P, q[t], F);
            publish(t & 1, F);
          }
          __syncthreads();
          if (active) through(t & 1, g[t]);
        }
        __syncthreads();  // the last slice is read before the next iteration writes it
      } else {
#pragma unroll
        for (int t0 = 0; t0 < B; t0 += TS) {
          if (active) {
#pragma unroll
            for (int t = t0; t < t0 + TS && t < B; t++) {
              R F[D][V];
              flux<D, V, R, EU>(P, q[t], F);
              if constexpr (FHL) average(t, F);
              publish(t - t0, F);
            }
          }
          __syncthreads();
          lines(slab, t0 + TS <= B ? TS : B - t0, T);
          __syncthreads();
          if (active) {
#pragma unroll
            for (int t = t0; t < t0 + TS && t < B; t++) gather(t - t0, g[t]);
          }
        }
      }
      // time solve in place and squared update (variables only; parameters are carried)
      double sq = 0.0;
      if (active) {
        R u[ND];
        solution(u);
        auto update = [&](R a, const R& old) {
          const double dq = static_cast<double>(a) - static_cast<double>(old);
          sq += dq * dq;
        };
        if constexpr (FHL) {
#pragma unroll
          for (int t = 0; t < B; t++) {
            Const<R>* Pt = opaque(tab_P<R>(T) + t * B);
#pragma unroll
            for (int v = 0; v < V; v++) {
              R a = u[v];
#pragma unroll
              for (int k = 0; k < B; k++) a -= Pt[k] * g[k][v];
              update(a, q[t][v]);
              q[t][v] = a;
            }
          }
        } else {
          Const<R>* Pt = opaque(tab_P<R>(T));
#pragma unroll
          for (int v = 0; v < V; v++) {
            R a[B];
#pragma unroll
            for (int t = 0; t < B; t++) {
              a[t] = u[v];
#pragma unroll
              for (int k = 0; k < B; k++) a[t] -= Pt[t * B + k] * g[k][v];
            }
#pragma unroll
            for (int t = 0; t < B; t++) {
              update(a[t], q[t][v]);
              g[t][v] = a[t];
            }
          }
        }
      }
      if (finished(iter, sq)) break;
    }

    // ---- time averages -> LDS (FP64): the fluxes as lines, the states by node ----
    double* Fl = reinterpret_cast<double*>(buf);
    double* Qh = Fl + SLICE + cs * NS * ND;
    int end[D];
#pragma unroll
    for (int d = 0; d < D; d++) end[d] = line[d] * V * B + (d == 0 ? x : (d == 1 ? y : z));
    __syncthreads();  // the last slices are read
    if (valid) {
#pragma unroll
      for (int v = 0; v < ND; v++) {
        double a = 0.0;
#pragma unroll
        for (int t = 0; t < B; t++) a += static_cast<double>(!FHL && v < V ? g[t][v < V ? v : 0] : q[t][v]) * T->w[t];
        Qh[s * ND + v] = a;
      }
      if constexpr (!FHL) {
#pragma unroll
        for (int t = 0; t < B; t++) {
          R F[D][V];
          flux<D, V, R, EU>(P, q[t], F);
          average(t, F);
        }
      }
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) {
          // EU: the component stored once is read from its canonical (d, v)
          const int dd = keep(d, v) ? d : v - 1, vv = keep(d, v) ? v : d + 1;
          Fl[end[d] + v * B] = static_cast<double>(fh[dd][vv]);
        }
    }
    __syncthreads();

    // ---- flux lines: extrapolation to the two faces (spaceTimePredictorNonlinear.cpph:517-687)
    // and the volume integral along the line, in place ----
    {
      constexpr int NLV = NL * V, NFV = NF * V;
      const EvenOdd<double, B> M(opaque(T->Kxi_eo));
#pragma unroll 1
      for (int id = tid; id < CPB * NLV; id += THREADS) {
        double f[B], o[B];
        load_line<double, B>(Fl + id * B, f);
        double f0 = 0.0, f1 = 0.0;
#pragma unroll
        for (int l = 0; l < B; l++) {
          f0 += f[l] * T->F0[l];
          f1 += f[l] * T->F1[l];
        }
        M.apply(f, o);
        store_line<double, B>(Fl + id * B, o);
        const int c = CPB == 1 ? 0 : id / NLV;
        const int r = id - c * NLV;
        const int d = r / NFV;
        const long cl = blk * CPB + c;
        if (cl < ncells) {
          double* fb = lFhbnd + cl * (2 * D * NFV) + d * NFV + r;  // face 2d, entry r - d NFV
          fb[0] = f0;
          fb[NFV] = f1;
        }
      }
    }
    // ---- states on the faces: one (face node, value) pair per lane and direction ----
    if (valid) {
      constexpr int NPAIR = NF * ND;
      double* qb = lQhbnd + cell * (2 * D * NPAIR);
      for (int pr = s; pr < NPAIR; pr += NS) {
        const int v = pr % ND, fn = pr / ND;
        const int a = fn / B, b = fn % B;
#pragma unroll
        for (int d = 0; d < D; d++) {
          // the line through the face node along d: node n0 + l stride
          const int n0 = D == 3 ? (d == 0 ? fn * B : (d == 1 ? a * B * B + b : fn)) : (d == 0 ? fn * B : fn);
          constexpr int st[3] = {1, B, B * B};
          double q0 = 0.0, q1 = 0.0;
#pragma unroll
          for (int l = 0; l < B; l++) {
            const double qv = Qh[(n0 + l * st[d]) * ND + v];
            q0 += qv * T->F0[l];
            q1 += qv * T->F1[l];
          }
          if (D == 2 && d == 0 && v >= V) q0 = q1 = 0.0;  // 2D x-faces carry no parameters
          qb[(2 * d) * NPAIR + pr] = q0;
          qb[(2 * d + 1) * NPAIR + pr] = q1;
        }
      }
    }
    if (picard && valid && s == 0) picard[cell] = iters;
    __syncthreads();

    // ---- volume integral at the node (volumeIntegralNonlinear.cpph:133-223) ----
    if (valid) {
      const double* w = T->w;
      const double W = D == 3 ? w[z] * w[y] * w[x] : w[y] * w[x];
      double du[V];
#pragma unroll
      for (int v = 0; v < V; v++) du[v] = 0.0;
#pragma unroll
      for (int d = 0; d < D; d++) {
        const double tw = D == 3 ? (d == 0 ? w[z] * w[y] : (d == 1 ? w[z] * w[x] : w[y] * w[x])) : (d == 0 ? w[y] : w[x]);
        const double upd = tw / hcell[hdim ? cell * hdim + d : cell];
#pragma unroll
        for (int v = 0; v < V; v++) du[v] += upd * Fl[end[d] + v * B];
      }
      if (luh_upd) {
        // volume part of the solution update in place (solutionUpdate.cpph:28-67: dt / w)
        const double upd = dt / W;
#pragma unroll
        for (int v = 0; v < V; v++) luh_upd[(cell * NS + s) * ND + v] += du[v] * upd;
      } else {
#pragma unroll
        for (int v = 0; v < V; v++) lduh[(cell * NS + s) * V + v] = du[v];
      }
    }
  }

  static __device__ __forceinline__ bool valid_block(long blk, long ncells) { return blk * CPB < ncells; }
};

// Waves per SIMD the register allocation aims at: the two columns (2 B V values)
// and a line's working set; one wave more spills (FP64 order 5 at three: 52
// registers, 24 -> 30 ms at 81^3; order 3 at three: 27, 0.375 -> 0.390 ms at 35^3).
// Order 4 spills at three, 10 to 16 registers for Euler and 41 to 44 for the other
// equations, and still gains from the third wave once the cells fill it.
template <int D, int B, int V, int NP, typename R>
constexpr int min_waves() {
  if (D == 3 && B <= 3) return 3;  // as many as LDS takes
  if (sizeof(R) == 4) return 4;
  return B == 4 || B >= 6 ? 2 : 3;
}
// 3D order 4 in FP64 exists at two waves as well, for meshes that two waves per SIMD
// hold at once (node form before / three / two waves: Euler, one CERK iteration, 500
// cells 15.4 / 16.5 / 15.5 us; advection, three iterations, 1,000 cells 30.8 / 30.5 /
// 24.8; 1,500 cells 50.0 / 38.5 / 42.8) and for one CERK iteration of the other
// equations (24,000 cells 389 / 389 / 338; two iterations 602 / 488 / 495).
template <int D, int B, typename R>
constexpr bool kTwoWaves = D == 3 && B == 5 && sizeof(R) == 8;

// One workgroup per tile of CPB cells, or a smaller grid that loops over the tiles.
template <int D, int B, int V, int NP, typename R, bool CG, bool EU, int WAVES = min_waves<D, B, V, NP, R>()>
__global__ __launch_bounds__((Shape<D, B, V, NP, R>::THREADS), WAVES) void
column_predictor_kernel(long ncells, long ntiles, const double* luh, const double* __restrict__ hcell,
                        const double* __restrict__ dtp, const int* __restrict__ cinst, double* __restrict__ lduh,
                        double* __restrict__ lQhbnd, double* __restrict__ lFhbnd, int* __restrict__ picard,
                        const DevTables* __restrict__ T, PdeParams P, int maxIter, int adaptive, double* luh_upd,
                        int dialect, int hdim) {
  using S = Shape<D, B, V, NP, R>;
  __shared__ __align__(16) unsigned char buf[S::BUF_BYTES];
  __shared__ double red[S::RED];
  if constexpr (EU) P.id = kPdeEuler;  // the flux needs no run-time choice
#pragma unroll 1
  for (long blk = blockIdx.x; blk < ntiles; blk += gridDim.x) {
    Tile<D, B, V, NP, R, CG, EU>::run(blk, ncells, luh, hcell, dtp, cinst, lduh, lQhbnd, lFhbnd, picard, T, P, maxIter,
                                      adaptive, luh_upd, dialect, hdim, buf, red);
    __syncthreads();  // LDS of this tile fully consumed before the next one
  }
}

template <int D, int B, int V, int NP>
struct Launch {
  template <typename R, bool CG, bool EU>
  static void form(const KernelCfg& k, hipStream_t st, long n, const double* luh, const double* h, const double* dt,
                   double* lduh, double* qb, double* fb, int* pic, int maxIter, int adaptive, const LaunchOpts& o) {
    using S = Shape<D, B, V, NP, R>;
    const long tiles = (n + S::CPB - 1) / S::CPB;
    const long grid = (o.grid > 0 && o.grid < tiles) ? o.grid : tiles;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(unsigned(grid)), dim3(S::THREADS), 0, st, n, tiles, luh, h, dt, o.cinst, lduh, qb, fb,
                         pic, k.tab, k.pde, maxIter, adaptive, o.luh_update, k.dialect, o.hdim);
    };
    if constexpr (kTwoWaves<D, B, R>) {
      if (grid * (S::THREADS / 64) <= 2048 || (CG && !EU && maxIter == 1))  // 1,024 SIMDs
        return launch(column_predictor_kernel<D, B, V, NP, R, CG, EU, 2>);
    }
    launch(column_predictor_kernel<D, B, V, NP, R, CG, EU>);
  }
  template <typename R, bool CG>
  static void pde(const KernelCfg& k, hipStream_t st, long n, const double* luh, const double* h, const double* dt,
                  double* lduh, double* qb, double* fb, int* pic, int maxIter, int adaptive, const LaunchOpts& o) {
    if constexpr (V == 5) {
      if (k.pde.id == kPdeEuler) {
        form<R, CG, true>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
        return;
      }
    }
    form<R, CG, false>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
  }
  static int run(const KernelCfg& k, hipStream_t st, long n, const double* luh, const double* h, const double* dt,
                 double* lduh, double* qb, double* fb, int* pic, const LaunchOpts& o) {
    // Picard rule: generic (adaptive or fixed count) or the optimised kernels'
    // (fusedSPTVI_nonlinear_cpp.template:177, tolerance exit always on)
    const int adaptive = k.dialect ? 1 : k.picard_max <= 0;
    const int maxIter = k.dialect ? (k.guess ? (B - 3 <= 1 ? 1 : B - 3) : 2 * B + 1)
                                  : (adaptive ? 2 * (k.order + 1) : k.picard_max);
    if (k.precision == 0) {
      if (k.guess)
        pde<double, true>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
      else
        pde<double, false>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
    } else {
      if (k.guess)
        pde<float, true>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
      else
        pde<float, false>(k, st, n, luh, h, dt, lduh, qb, fb, pic, maxIter, adaptive, o);
    }
    return static_cast<int>(hipGetLastError());
  }
};

}  // namespace columns
}  // namespace exa
