// gsg_solo.hpp -- the resident kernel of small RK4 solves: one workgroup advances one
// solve by many RK4 steps with the stage inputs in LDS (instantiated for double in
// gsg_solo64.hip and for float in gsg_solo32.hip).
//
// Why: a small solve launched stage by stage is a chain of waits.  At D = 2, k = 3, n = 5
// (1,008 coefficients) a stage launch took 15 us, all of it launch, descriptor, list and
// operand latency.  Here the lists and the 1-D blocks are read into LDS once per launch,
// the stage input stays in LDS, and a pass over the operator ends with a workgroup
// barrier.
//
// What bounds it is LDS bandwidth: with a lane per DoF every multiplication read two
// operands.  A task is therefore (direction, cell, SOLO_G fibers): a block is read once
// for SOLO_G fibers and k outputs each.  Tasks are sorted by list length (the host's
// order), so a wavefront's lists are equally long and the long ones start first.  The
// direction sums meet in LDS and one lane per DoF adds them up in direction order and
// applies the RK stage: entries in list order, modes in order, directions in order, the
// sums of the stage kernels bit for bit (float: see SEGR).
#pragma once
#include <hip/hip_runtime.h>

#include "gsg_dev.hpp"

namespace gsg {
namespace solo {

template <typename T>
struct Tab;
template <>
struct Tab<double> {
  static __device__ __forceinline__ const double* vals(const DevTables& t) { return t.val64; }
};
template <>
struct Tab<float> {
  static __device__ __forceinline__ const float* vals(const DevTables& t) { return t.val32; }
};

// acc[q][r] (and, float, accl[q][r] with the lo table) += block row r . fiber q of every
// entry of a list, for R block rows from v on; ent: packed words (block << 16) | cell; v:
// the blocks (LDS or global), vlo: elements from the hi to the lo table; off[q]: fiber q's
// element with the direction's mode digit 0, sd the digit's stride.  U entries a round.
// HI2: the hi table into accl only.
template <int K, int KD, int G, int R, int U, bool HI2, bool VL, typename T>
__device__ __forceinline__ void round_of(const uint32_t (&e)[U], const T* v, int vlo, const T* x, const int (&off)[G],
                                         int sd, T (&acc)[G][R], T (&accl)[G][R]) {
  constexpr bool HL = sizeof(T) == 4;
  T b[U][R * K], bl[U][HL ? R * K : 1], xv[U][G][K];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const T* vp = v + int(e[u] >> 16) * (K * K);
    const T* xp = x + int(e[u] & 0xffffu) * KD;
#pragma unroll
    for (int q = 0; q < R * K; ++q) {
      b[u][q] = VL ? vp[q] : gld(vp + q);
      if constexpr (HL && !HI2) bl[u][q] = VL ? vp[vlo + q] : gld(vp + vlo + q);
    }
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int j = 0; j < K; ++j) xv[u][q][j] = xp[off[q] + j * sd];
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < K; ++j) {
          if constexpr (HI2) {
            accl[q][r] += b[u][r * K + j] * xv[u][q][j];
          } else {
            acc[q][r] += b[u][r * K + j] * xv[u][q][j];
            if constexpr (HL) accl[q][r] += bl[u][r * K + j] * xv[u][q][j];
          }
        }
}
template <int K, int KD, int G, int R, int U, bool HI2, bool VL, typename T>
__device__ __forceinline__ void list(const uint32_t* ent, int p0, int p1, const T* v, int vlo, const T* x,
                                     const int (&off)[G], int sd, T (&acc)[G][R], T (&accl)[G][R]) {
  int p = p0;
  if (p + U <= p1) {
    uint32_t e[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = ent[p + u];
    do {
      uint32_t c[U];
#pragma unroll
      for (int u = 0; u < U; ++u) c[u] = e[u];
      p += U;
#pragma unroll
      for (int u = 0; u < U; ++u) e[u] = ent[min(p + u, p1 - 1)];  // the next round's words
      round_of<K, KD, G, R, U, HI2, VL>(c, v, vlo, x, off, sd, acc, accl);
    } while (p + U <= p1);
  }
  if constexpr (U > 1)
    for (; p < p1; ++p) {
      const uint32_t c[1] = {ent[p]};
      round_of<K, KD, G, R, 1, HI2, VL>(c, v, vlo, x, off, sd, acc, accl);
    }
}

// a workgroup barrier that orders LDS only: the RK state in global memory is read and
// written by its own lane alone, so its stores need not land before the barrier
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct RkRegs {
  double y, acc;
};
__device__ __forceinline__ RkRegs rk_load(int stage, const double* y, const double* acc, int64_t i) {
  RkRegs q;
  q.y = stage <= 3 ? gld(y + i) : 0.0;
  q.acc = stage >= 2 ? gld(acc + i) : 0.0;
  return q;
}
// the classical RK4 stage update of state entry i with derivative r; returns the next
// stage input
__device__ __forceinline__ double rk_stage(int stage, const SolveDesc& S, double* y, double* acc, int64_t i, const RkRegs& q,
                                           double r) {
  if (stage == 1) {
    gst(acc + i, q.y + S.dt6 * r);
    return q.y + S.dt2 * r;
  }
  if (stage == 2) {
    gst(acc + i, q.acc + S.dt3 * r);
    return q.y + S.dt2 * r;
  }
  if (stage == 3) {
    gst(acc + i, q.acc + S.dt3 * r);
    return q.y + S.dt * r;
  }
  const double yn = q.acc + S.dt6 * r;
  gst(y + i, yn);
  return yn;
}

// SEGR (float): the segmented kernel's roundings (direction sums added up in float, one
// pair of accumulators over both parts of a gradient); otherwise the plan kernel's.
// VL: the blocks are in LDS.
template <int D, int K, typename T, bool SEGR, bool VL, int G, int R, int U>
__device__ __forceinline__ void run(const SoloArgs& a, const SolveDesc& S, unsigned char* lds) {
  constexpr int KD = kpow(K, D);
  constexpr int NG = KD / (G * R);  // tasks of a cell and direction
  constexpr bool HL = sizeof(T) == 4;
  const int N = int(S.N);
  const int NT = int(blockDim.x), tid = int(threadIdx.x);
  const bool wave = S.sys == SYS_WAVE;
  const int ncell = N / KD;
  const int ne = gld(S.t.plan_ptr + int64_t(ncell) * D);
  // LDS (SoloLds): the D direction sums in double; the stage input x, or for the wave u,
  // v, the D gradient vectors and (float) u's remainder; the lists, the tasks' words, the
  // blocks
  const SoloLds L(D, K, N, int(sizeof(T)), wave, ne);
  double* P = reinterpret_cast<double*>(lds);
  T* x = reinterpret_cast<T*>(lds + L.x);
  T* vv = x + N;
  T* w = x + 2 * N;
  T* ulo = w + D * N;
  uint32_t* ent = reinterpret_cast<uint32_t*>(lds + L.ent);
  int* ptr = reinterpret_cast<int*>(lds + L.ptr);
  uint32_t* task = reinterpret_cast<uint32_t*>(lds + L.task);
  T* vl = reinterpret_cast<T*>(lds + L.vals);
  const int nv = int(S.t.val_elems);
  const T* vg = Tab<T>::vals(S.t);
  const int ntask = ncell * D;  // (direction, cell) words, NG fiber groups each
  for (int q = tid; q < ne; q += NT) ent[q] = gld(S.t.solo_ent + q);
  for (int q = tid; q <= ntask; q += NT) ptr[q] = gld(S.t.plan_ptr + q);
  for (int q = tid; q < ntask; q += NT) task[q] = gld(S.t.solo_ent + ne + q);
  if constexpr (VL)
    for (int q = tid; q < nv * (HL ? 2 : 1); q += NT) vl[q] = gld(vg + q);
  const T* v;
  if constexpr (VL)
    v = vl;
  else
    v = vg;
  double* const y = S.y;
  double* const acc = S.acc;
  const int d0 = S.dir0, d1 = S.dir0 + S.ndir;
  double coef[D];
#pragma unroll
  for (int d = 0; d < D; ++d) coef[d] = S.coef[d];

  // every task: the sums of direction d's input xin + d xs (grad: and u's remainder) into
  // P (grad: rounded, into w)
  auto pass = [&](const T* xin, int xs, bool grad, bool some) {
    for (int t = tid; t < ntask * NG; t += NT) {
      const uint32_t q0 = task[t / NG];  // (direction << 16) | cell
      const int cell = int(q0 & 0xffffu), d = int(q0 >> 16), sub = t % NG;
      if (some && (d < d0 || d >= d1)) continue;
      int sd = 1;
#pragma unroll
      for (int e = 0; e + 1 < D; ++e) sd = e < d ? sd * K : sd;
      int off[G];
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int f = (sub / (K / R)) * G + q;
        off[q] = f % sd + (f / sd) * (sd * K);
      }
      const int r0 = (sub % (K / R)) * R;
      const T* vr = v + r0 * K;
      const int p0 = ptr[cell * D + d], p1 = ptr[cell * D + d + 1];
      T ac[G][R], al[G][R];
      double s[G][R];
      auto clear = [&] {
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
          for (int r = 0; r < R; ++r) ac[q][r] = al[q][r] = T(0);
      };
      clear();
      list<K, KD, G, R, U, false, VL>(ent, p0, p1, vr, nv, xin + d * xs, off, sd, ac, al);
      if (HL && SEGR && grad) list<K, KD, G, R, U, true, VL>(ent, p0, p1, vr, nv, ulo, off, sd, ac, al);
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) s[q][r] = HL ? double(ac[q][r]) + double(al[q][r]) : double(ac[q][r]);
      if (HL && !SEGR && grad) {
        clear();
        list<K, KD, G, R, U, false, VL>(ent, p0, p1, vr, nv, ulo, off, sd, ac, al);
#pragma unroll
        for (int q = 0; q < G; ++q)
#pragma unroll
          for (int r = 0; r < R; ++r) s[q][r] += double(ac[q][r]) + double(al[q][r]);
      }
      const int o = d * N + cell * KD;
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int at = o + off[q] + (r0 + r) * sd;
          if (grad)
            w[at] = T(s[q][r]);
          else
            P[at] = s[q][r];
        }
    }
  };
  // the direction sums of DoF i added up in direction order
  auto total = [&](int i, bool scaled) -> double {
    double s = 0.0;
    T Y = T(0);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (scaled && (d < d0 || d >= d1)) continue;
      const double r = P[d * N + i];
      const double ce = scaled ? coef[d] : 1.0;
      if constexpr (SEGR)
        Y = d == 0 ? T(ce * r) : T(double(Y) + ce * r);
      else
        s += ce * r;
    }
    return SEGR ? double(Y) : s;
  };

  for (int i = tid; i < N; i += NT) {
    const double yu = gld(y + i);
    x[i] = T(yu);
    if (wave) {
      if constexpr (HL) ulo[i] = T(yu - double(T(yu)));
      vv[i] = T(gld(y + N + i));
    }
  }
  lds_barrier();
  for (int64_t st = 0; st < a.nsteps; ++st) {
    for (int stage = 1; stage <= 4; ++stage) {
      // the RK state of this lane's first DoF, in flight during the passes
      const int i0 = tid < N ? tid : 0;
      const RkRegs f0 = rk_load(stage, y, acc, i0), f1 = rk_load(stage, y, acc, wave ? int64_t(N) + i0 : i0);
      if (wave) {
        pass(x, 0, true, false);  // w_d = D_d u
        lds_barrier();
        pass(w, N, false, false);
      } else {
        pass(x, 0, false, true);
      }
      lds_barrier();
      for (int i = tid; i < N; i += NT) {
        const RkRegs qu = i == tid ? f0 : rk_load(stage, y, acc, i);
        const double s = total(i, !wave);
        if (wave) {
          const RkRegs qv = i == tid ? f1 : rk_load(stage, y, acc, int64_t(N) + i);
          const double un = rk_stage(stage, S, y, acc, i, qu, double(vv[i]));
          x[i] = T(un);
          if constexpr (HL) ulo[i] = T(un - double(T(un)));
          vv[i] = T(rk_stage(stage, S, y, acc, int64_t(N) + i, qv, s));
        } else {
          x[i] = T(rk_stage(stage, S, y, acc, i, qu, s));
        }
      }
      lds_barrier();
    }
  }
  // float: the stage launches read a step's first stage input from xs[0] (FP64: from y), so
  // it is left there as their last stage leaves it, for a solve that goes on in stage launches
  if constexpr (HL) {
    T* const x0 = static_cast<T*>(S.xs[0]);
    for (int i = tid; i < N; i += NT) {
      gst(x0 + i, x[i]);
      if (wave) {
        gst(x0 + N + i, vv[i]);
        gst(x0 + 2 * N + i, ulo[i]);
      }
    }
  }
}

template <int D, int K, typename T, bool SEGR>
__global__ __launch_bounds__(SOLO_MAXT) void k_solo(SoloArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const SolveDesc& S = a.solves[a.ids ? a.ids[blockIdx.x] : int(blockIdx.x)];
  if (!S.active) return;  // the whole workgroup
  // few tasks: one output a lane; more: the map that reads the least LDS
  constexpr SoloMap A = solo_map_small(D, K), B = solo_map_large(D, K);
  if (a.small_map) {
    if (a.vals_lds)
      run<D, K, T, SEGR, true, A.G, A.R, A.U>(a, S, lds);
    else
      run<D, K, T, SEGR, false, A.G, A.R, A.U>(a, S, lds);
  } else {
    if (a.vals_lds)
      run<D, K, T, SEGR, true, B.G, B.R, B.U>(a, S, lds);
    else
      run<D, K, T, SEGR, false, B.G, B.R, B.U>(a, S, lds);
  }
}

template <int D, int K, typename T, bool SEGR>
hipError_t launch_one(const SoloArgs& a, int nsolve, int threads, int lds_bytes, hipStream_t s) {
  if (lds_bytes > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_solo<D, K, T, SEGR>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, SOLO_LDS);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_solo<D, K, T, SEGR>), dim3(unsigned(nsolve)), dim3(unsigned(threads)), size_t(lds_bytes), s, a);
  return hipGetLastError();
}

}  // namespace solo
}  // namespace gsg
