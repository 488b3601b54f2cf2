// The GEMMs' epilogue: the outputs of a float tile in LDS (kgx_gemm.hip, kgx_split.hip).
#pragma once
#include "kgx_device.h"

namespace kgx {

// Epilogue variants, chosen at launch so that a kernel carries only its own epilogue code (a kernel holding all
// of them ran 15-25 % slower on the token GEMMs, its main loop unchanged).
enum GemmEpi {
  EPI_SCALAR,  // per-element conv_store (rows or columns not 16-byte aligned)
  EPI_GEN,     // conv_store4: any of colbias, rowmask, yt, y (+ residual), emission
  EPI_YT,      // compute-type store only
  EPI_ACC,     // float store or residual add (+ row mask) only
  EPI_GLU,     // gated output
  EPI_QKV,     // q|k|v projection
  EPI_YTMISH,  // compute-type store of mish(C)
};

// The rotation of x with its partner y (the other half of the head): x cos - y sin for the first half, y sin + x cos
// for the second, each with one explicit fused multiply-add, so that every tile configuration rounds it alike (a
// contracted expression may fuse either product, and a row must not depend on the tile it falls in).
__device__ __forceinline__ floatx4 rope4(floatx4 x, floatx4 y, floatx4 cs, floatx4 sn, bool lo) {
  floatx4 r;
#pragma unroll
  for (int k = 0; k < 4; k++)
    r[k] = lo ? __builtin_fmaf(x[k], cs[k], -(y[k] * sn[k])) : __builtin_fmaf(y[k], sn[k], x[k] * cs[k]);
  return r;
}

// PR rows from row mp and BN columns from column n0 of the result, held as floats in Et (row stride BN + 4), by NT
// threads.
template <typename T, int EPI, int PR, int BN, int NT>
__device__ __forceinline__ void gemm_tile_epilogue(const float* Et, const GemmArgs& g, const ConvOut& o, int mp, int n0,
                                                   int M, int N, int tid) {
  constexpr int ELD = BN + 4, CV = BN / 4, EV = PR * CV / NT;
  static_assert(EV * NT == PR * CV, "epilogue vectors not divisible over the threads");
  if constexpr (EPI == EPI_GLU) {
    constexpr int HV = BN / 8;  // 4-wide vectors of gated outputs per tile row
    for (int e = tid; e < PR * HV; e += NT) {
      const int r = e / HV, hc = (e % HV) * 4, lc = (hc / 16) * 32 + hc % 16;
      const int m = mp + r, f = n0 / 2 + hc;
      if (m < M && f < N / 2) {
        const floatx4 a = *(const floatx4*)(Et + r * ELD + lc), b = *(const floatx4*)(Et + r * ELD + lc + 16);
        store4<T>((T*)o.yt + (size_t)m * o.ldyt + f, act_f<ACT_SILU>(a[0]) * b[0], act_f<ACT_SILU>(a[1]) * b[1],
                  act_f<ACT_SILU>(a[2]) * b[2], act_f<ACT_SILU>(a[3]) * b[3]);
      }
    }
  } else if constexpr (EPI == EPI_QKV && NT % CV == 0) {
    // q|k|v projection: each head lies inside the tile, so the rotation partner of column n (n +- dq/2) is
    // in LDS too. A thread keeps one column quad for every row it takes (NT is a multiple of CV), so the head,
    // rotation and table indices are computed once, and the rotation tables are read for all its rows before
    // the first store (a load after a store that may alias it waits for the store).
    constexpr int RS = NT / CV;
    const QkvEpi& q = g.qkv;
    const int half = q.dq / 2;
    const int c = (tid % CV) * 4, n = n0 + c, r0 = tid / CV;
    const bool qk = n < q.nq + q.nk, isq = n < q.nq;
    const int nn = n - (isq ? 0 : q.nq), hh = nn / q.dq, rr = nn - hh * q.dq;
    const bool lo = rr < half;
    const int pp = lo ? rr : rr - half, tab = q.tables == 1 ? 0 : (isq ? hh / (q.H / q.KV) : hh);
    const bool rot = qk && q.cos;
    floatx4 cs[EV], sn[EV];
    if (rot) {
#pragma unroll
      for (int v = 0; v < EV; v++) {
        const int m = min(mp + r0 + RS * v, M - 1);
        const size_t ti = ((size_t)tab * HW + m % HW) * half + pp;
        cs[v] = *(const floatx4*)(q.cos + ti);
        sn[v] = *(const floatx4*)(q.sin + ti);
      }
    }
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int r = r0 + RS * v, m = mp + r;
      if (m < M && n < N) {
        floatx4 x = *(const floatx4*)(Et + r * ELD + c);
        if (qk) {
          if (rot) {
            const floatx4 y = *(const floatx4*)(Et + r * ELD + c + (lo ? half : -half));
            x = rope4(x, y, cs[v], sn[v], lo);
          }
          if (isq) x *= q.qscale;
        }
        store4<T>((T*)o.yt + (size_t)m * o.ldyt + n, x[0], x[1], x[2], x[3]);
      }
    }
  } else if constexpr (EPI == EPI_QKV) {
    // (The same on tiles whose thread count is not a multiple of their column quads.)
    const QkvEpi& q = g.qkv;
    const int half = q.dq / 2;
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int e = tid + NT * v, r = e / CV, c = (e % CV) * 4, m = mp + r, n = n0 + c;
      if (m < M && n < N) {
        floatx4 x = *(const floatx4*)(Et + r * ELD + c);
        if (n < q.nq + q.nk) {
          const bool isq = n < q.nq;
          const int hh = (n - (isq ? 0 : q.nq)) / q.dq, rr = (n - (isq ? 0 : q.nq)) - hh * q.dq;
          if (q.cos) {
            const bool lo = rr < half;
            const int pp = lo ? rr : rr - half, tab = q.tables == 1 ? 0 : (isq ? hh / (q.H / q.KV) : hh);
            const floatx4 y = *(const floatx4*)(Et + r * ELD + c + (lo ? half : -half));
            const size_t ti = ((size_t)tab * HW + m % HW) * half + pp;
            const floatx4 cs = *(const floatx4*)(q.cos + ti), sn = *(const floatx4*)(q.sin + ti);
            x = rope4(x, y, cs, sn, lo);
          }
          if (isq) x *= q.qscale;
        }
        store4<T>((T*)o.yt + (size_t)m * o.ldyt + n, x[0], x[1], x[2], x[3]);
      }
    }
  } else if constexpr (EPI == EPI_YT || EPI == EPI_YTMISH) {
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int e = tid + NT * v, r = e / CV, c = (e % CV) * 4, m = mp + r, n = n0 + c;
      if (m < M && n < N) {
        floatx4 x = *(const floatx4*)(Et + r * ELD + c);
        if constexpr (EPI == EPI_YTMISH) {
#pragma unroll
          for (int q = 0; q < 4; q++) x[q] = sizeof(T) == 2 ? act16<ACT_MISH>(x[q], 1.f) : act_f<ACT_MISH>(x[q]);
        }
        store4<T>((T*)o.yt + (size_t)m * o.ldyt + n, x[0], x[1], x[2], x[3]);
      }
    }
  } else if constexpr (EPI == EPI_ACC) {
    // Float output, the residual and row mask loaded ahead of the stores.
    floatx4 yres[EV];
    float rmv[EV];
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int e = tid + NT * v, m = min(mp + e / CV, M - 1), n = min(n0 + (e % CV) * 4, N - 4);
      yres[v] = o.accumulate ? *(const floatx4*)(o.y + (size_t)m * o.ldy + n) : floatx4{0.f, 0.f, 0.f, 0.f};
      rmv[v] = o.rowmask ? o.rowmask[m] : 1.f;
    }
#pragma unroll
    for (int v = 0; v < EV; v++) {
      const int e = tid + NT * v, r = e / CV, c = (e % CV) * 4, m = mp + r, n = n0 + c;
      if (m < M && n < N)
        *(floatx4*)(o.y + (size_t)m * o.ldy + n) = *(const floatx4*)(Et + r * ELD + c) * rmv[v] + yres[v];
    }
  } else {
    // Generic (EPI_GEN): one vector at a time, not unrolled, to keep the code small.
#pragma unroll 1
    for (int v = 0; v < EV; v++) {
      const int e = tid + NT * v, r = e / CV, c = (e % CV) * 4, m = mp + r, n = n0 + c;
      if (m < M && n < N) {
        const floatx4 yres = o.y && o.accumulate ? *(const floatx4*)(o.y + (size_t)m * o.ldy + n)
                                                 : floatx4{0.f, 0.f, 0.f, 0.f};
        floatx4 es = {1.f, 1.f, 1.f, 1.f}, eb = {0.f, 0.f, 0.f, 0.f};
        float mk = 1.f;
        if (o.emit.scale) {
          es = *(const floatx4*)(o.emit.scale + n);
          eb = *(const floatx4*)(o.emit.bias + n);
          mk = o.emit.mask[m];
        }
        conv_store4<T>(o, m, n, *(const floatx4*)(Et + r * ELD + c), yres, o.rowmask ? o.rowmask[m] : 1.f, es,
                       eb, mk);
      }
    }
  }
}

}  // namespace kgx
