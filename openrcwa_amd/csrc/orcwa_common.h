// Common device/host helpers for the OpenRCWA MI355X engine.
//
// Complex numbers are interleaved double pairs (re, im), the layout of
// std::complex<double> in the reference (rcwa/defns.h:7-8).  All matrices are
// column-major unless a kernel states otherwise.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>

struct cd {
  double re, im;
};

__host__ __device__ inline cd mk(double r, double i) { cd z; z.re = r; z.im = i; return z; }
__host__ __device__ inline cd operator+(cd a, cd b) { return mk(a.re + b.re, a.im + b.im); }
__host__ __device__ inline cd operator-(cd a, cd b) { return mk(a.re - b.re, a.im - b.im); }
__host__ __device__ inline cd operator-(cd a) { return mk(-a.re, -a.im); }
__host__ __device__ inline cd operator*(cd a, cd b) {
  return mk(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
__host__ __device__ inline cd operator*(double s, cd a) { return mk(s * a.re, s * a.im); }
__host__ __device__ inline cd operator*(cd a, double s) { return mk(s * a.re, s * a.im); }
__host__ __device__ inline cd& operator+=(cd& a, cd b) { a.re += b.re; a.im += b.im; return a; }
__host__ __device__ inline cd& operator-=(cd& a, cd b) { a.re -= b.re; a.im -= b.im; return a; }
__host__ __device__ inline cd conj(cd a) { return mk(a.re, -a.im); }
__host__ __device__ inline double norm2(cd a) { return a.re * a.re + a.im * a.im; }
__host__ __device__ inline double cabs1(cd a) { return fabs(a.re) + fabs(a.im); }
__host__ __device__ inline double cabs(cd a) { return hypot(a.re, a.im); }
// a * conj(b)
__host__ __device__ inline cd mulc(cd a, cd b) {
  return mk(a.re * b.re + a.im * b.im, a.im * b.re - a.re * b.im);
}
// conj(a) * b
__host__ __device__ inline cd cmul(cd a, cd b) {
  return mk(a.re * b.re + a.im * b.im, a.re * b.im - a.im * b.re);
}
// acc + a b, acc - a b and acc + conj(a) b in four fused operations (written
// with the operators: two products of two operations and two sums)
__host__ __device__ inline cd cfma(cd acc, cd a, cd b) {
  return mk(fma(a.re, b.re, fma(-a.im, b.im, acc.re)), fma(a.re, b.im, fma(a.im, b.re, acc.im)));
}
__host__ __device__ inline cd cfnma(cd acc, cd a, cd b) {
  return mk(fma(-a.re, b.re, fma(a.im, b.im, acc.re)), fma(-a.re, b.im, fma(-a.im, b.re, acc.im)));
}
__host__ __device__ inline cd cfmac(cd acc, cd a, cd b) {
  return mk(fma(a.re, b.re, fma(a.im, b.im, acc.re)), fma(a.re, b.im, fma(-a.im, b.re, acc.im)));
}
__host__ __device__ inline cd cdiv(cd a, cd b) {
  // Smith's algorithm
  if (fabs(b.re) >= fabs(b.im)) {
    double r = b.im / b.re, d = b.re + b.im * r;
    return mk((a.re + a.im * r) / d, (a.im - a.re * r) / d);
  } else {
    double r = b.re / b.im, d = b.re * r + b.im;
    return mk((a.re * r + a.im) / d, (a.im * r - a.re) / d);
  }
}
__host__ __device__ inline cd cinv(cd b) { return cdiv(mk(1.0, 0.0), b); }

// Principal complex square root (branch cut on the negative real axis,
// Re >= 0), as std::sqrt(std::complex<double>).
__host__ __device__ inline cd csqrt_principal(cd z) {
  if (z.re == 0.0 && z.im == 0.0) return mk(0.0, z.im);
  double t = sqrt(0.5 * (fabs(z.re) + hypot(z.re, z.im)));
  if (z.re >= 0.0) return mk(t, z.im / (2.0 * t));
  return mk(fabs(z.im) / (2.0 * t), copysign(t, z.im));
}

// GammaSqrtOp (rcwa/WaveEquationSolver.cpp:8-22): principal root, negated
// if Im < 0, negated again if |Im| < |Re| and Re < 0.
__host__ __device__ inline cd gamma_sqrt(cd g) {
  cd v = csqrt_principal(g);
  if (v.im < 0) v = -v;
  if (fabs(v.im) < fabs(v.re) && v.re < 0) v = -v;
  return v;
}

__host__ __device__ inline cd cexp(cd z) {
  double e = exp(z.re);
  double s, c;
  sincos(z.im, &s, &c);
  return mk(e * c, e * s);
}

// A pointer read from a device table has no known address space, so the compiler
// moves everything behind it with flat instructions: those also count as LDS
// accesses, and waiting for an LDS read then waits for every load in flight.
// Rebuilt from its integer value in the global address space, it is known.
template <class T>
__device__ __forceinline__ T* gptr(T* p) {
  return (T*)((__attribute__((address_space(1))) T*)(unsigned long long)p);
}

typedef double v2d __attribute__((ext_vector_type(2)));

// 16-byte LDS accesses (cd alone is only 8-byte aligned to the compiler, which
// then moves it as two 8-byte halves, each with half the banks in conflict)
__device__ __forceinline__ cd lds_ld(const cd* p) {
  const v2d v = *reinterpret_cast<const v2d*>(p);
  return mk(v.x, v.y);
}
__device__ __forceinline__ void lds_st(cd* p, cd z) {
  v2d v;
  v.x = z.re;
  v.y = z.im;
  *reinterpret_cast<v2d*>(p) = v;
}

// wavefront (64-lane) helpers
// value of a uniform lane, in scalar registers
__device__ __forceinline__ double lane_value(double v, int lane) {
  union { double d; int i[2]; } u;
  u.d = v;
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], lane);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], lane);
  return u.d;
}
__device__ __forceinline__ cd lane_value(cd v, int lane) {
  return mk(lane_value(v.re, lane), lane_value(v.im, lane));
}
// sum and maximum over the wave, in every lane (all lanes active): six moves
// within the vector unit; as lane shuffles through LDS a sum took about five
// times as long, and the serial kernels are made of such sums
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double old, double v) {
  union { double d; int i[2]; } u, o;
  u.d = v;
  o.d = old;
  u.i[0] = __builtin_amdgcn_update_dpp(o.i[0], u.i[0], CTRL, ROWS, 0xf, false);
  u.i[1] = __builtin_amdgcn_update_dpp(o.i[1], u.i[1], CTRL, ROWS, 0xf, false);
  return u.d;
}
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_move<0x111, 0xf>(0.0, v);   // row_shr:1 (lanes without a source take 0)
  v += dpp_move<0x112, 0xf>(0.0, v);   // row_shr:2
  v += dpp_move<0x114, 0xf>(0.0, v);   // row_shr:4
  v += dpp_move<0x118, 0xf>(0.0, v);   // row_shr:8
  v += dpp_move<0x142, 0xa>(0.0, v);   // row_bcast:15 into rows 1 and 3
  v += dpp_move<0x143, 0xc>(0.0, v);   // row_bcast:31 into rows 2 and 3
  return lane_value(v, 63);
}
// maximum over the first 16 lanes in lane 15 (lanes without a source keep theirs)
__device__ __forceinline__ double dpp_row_reduce_max(double v) {
  v = fmax(v, dpp_move<0x111, 0xf>(v, v));
  v = fmax(v, dpp_move<0x112, 0xf>(v, v));
  v = fmax(v, dpp_move<0x114, 0xf>(v, v));
  return fmax(v, dpp_move<0x118, 0xf>(v, v));
}
__device__ __forceinline__ double wave_max(double v) {
  v = dpp_row_reduce_max(v);
  v = fmax(v, dpp_move<0x142, 0xf>(v, v));
  v = fmax(v, dpp_move<0x143, 0xf>(v, v));
  return lane_value(v, 63);
}
// q <- q with the interchanges k0 + j <-> (pivot in lane j), j < nb, applied in
// order (q in LDS, on one wave: the pivots are in its lanes, so a step costs two
// LDS latencies and no load from memory)
__device__ __forceinline__ void compose_swaps(int k0, int nb, int pivot, int* q) {
  for (int j = 0; j < nb; ++j) {
    const int k = k0 + j, p = __builtin_amdgcn_readlane(pivot, j);
    if (p != k) {
      const int a = q[k], c = q[p];
      q[k] = c;
      q[p] = a;
    }
  }
}
// orders LDS accesses between the lanes of one wavefront
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A count in LDS by which one wave hands data in LDS to others of its workgroup:
// what the publishing wave wrote before wave_publish (its other lanes: before a
// wave_fence in front of it) is there after wave_await(p, v) in any wave, once
// p has reached v.
__device__ __forceinline__ void wave_publish(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void wave_await(const int* p, int v) {
  while (__hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < v) {}
}

#define ORCWA_HIP_CHECK(expr)                                                       \
  do {                                                                              \
    hipError_t _e = (expr);                                                         \
    if (_e != hipSuccess) {                                                         \
      fprintf(stderr, "[openrcwa] HIP error %s at %s:%d: %s\n", hipGetErrorName(_e), \
              __FILE__, __LINE__, #expr);                                           \
      return ORCWA_ERR_HIP;                                                         \
    }                                                                               \
  } while (0)
