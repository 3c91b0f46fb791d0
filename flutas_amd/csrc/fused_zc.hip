// Single-problem z-chunked slab passes (P2, P3) and their tables; the device
// bodies are in fused_chunk.hpp.
#include "fused_chunk.hpp"
#include "fused_host.hpp"

#include <type_traits>

namespace flutas {

template <typename T, int NC, int GP, int NT, bool PER>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_yz_fwd_zc(T *__restrict__ Wt, WStride ws, ZChunks zc, int nx, int nz, int msys, int kind,
                const double *__restrict__ lamx, const double *__restrict__ lamy,
                const double *__restrict__ a, const double *__restrict__ b,
                const double *__restrict__ c, int pin, const T *__restrict__ tw,
                const T *__restrict__ twh, const T *__restrict__ twq) {
  __shared__ __align__(16) T sm[2 * GP * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[Tw<T, NC>::total];
  int i, ch;
  zc_slab_of(nx, zc.nchunk, &i, &ch);
  constexpr bool OPQ = slab_opaque<T, NC, PER, false, true>();
  yz_fwd_chunk<T, NC, GP, NT, PER, OPQ>(Wt, ws, zc, nz, msys, kind, lamx, lamy, a, b, c, pin, tw,
                                        twh, twq, sm, stw, i, ch);
}

template <typename T, int NC, int GP, int NT, bool PER>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_zy_bwd_zc(T *__restrict__ Wt, WStride ws, ZChunks zc, int nx, int nz, int msys, int kind,
                const double *__restrict__ lamx, const double *__restrict__ lamy,
                const double *__restrict__ a, const double *__restrict__ b,
                const double *__restrict__ c, int pin, const T *__restrict__ tw,
                const T *__restrict__ twh, const T *__restrict__ twq) {
  __shared__ __align__(16) T sm[2 * GP * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[Tw<T, NC>::total];
  int i, ch;
  zc_slab_of(nx, zc.nchunk, &i, &ch);
  constexpr bool OPQ = slab_opaque<T, NC, PER, true, true>();
  zy_bwd_chunk<T, NC, GP, NT, PER, OPQ>(Wt, ws, zc, nz, msys, kind, lamx, lamy, a, b, c, pin, tw,
                                        twh, twq, sm, stw, i, ch);
}

// Tables of the z-chunked passes, one thread per column (i, j), with the
// operations of yz_fwd_chunk / zy_bwd_chunk (so d is bit for bit the
// passes' and the reference's): walking up, d, m (periodic: q2) before
// every plane group and the chunk sums M, SW, N; for periodic z then
// walking down group by group (factors recomputed from the stored values),
// the second solution p2 at every chunk start and the closing row's
// denominator (b(m) + lam) + c(m) p2(0) + a(m) p2(m-1).
// The pivot reciprocals are those of the chain the tables serve (zrcp<T>).
// Bound by the chain of a column's pivots, one thread's whole work: the rows
// of a group without one of the first, last and closing rows run straight
// through, up to eight at a time with their coefficients loaded ahead (a new plan
// of 32x32x2048 periodic z 1.81 -> 0.84 ms, 2x2x1000 0.78 -> 0.37).
// GP: planes of a group, 0 for gp.
constexpr int kZcMaxGroup = 16;
template <typename T, bool PER, int GP>
__global__ void __launch_bounds__(256)
    k_zchunk_tables(double *__restrict__ ckd, double *__restrict__ ckm, double *__restrict__ ckq,
                    double *__restrict__ tab, double *__restrict__ den, int nx, int ny, int nz,
                    int msys, int gp_, int cpl, int nchunk, int pin,
                    const double *__restrict__ lamx, const double *__restrict__ lamy,
                    const double *__restrict__ a, const double *__restrict__ b,
                    const double *__restrict__ c) {
#pragma clang fp contract(off)
  const long long col = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= (long long)nx * ny) return;
  const int i = (int)(col / ny), j = (int)(col - (long long)i * ny);
  const double lam = lamx[i] + lamy[j];
  const int gp = GP ? GP : gp_;
  const int ngrp = (nz + gp - 1) / gp;
  constexpr int TS = zc_tab_slots(PER), H = GP == 0 ? 1 : (GP < 8 ? GP : 8);
  double dp = 0.0, mp = 1.0, qp = 0.0, w = 1.0, sw = 0.0, ml = 0.0;
  const long long og = (long long)i * ngrp * ny + j;
  double *const t0 = tab + (long long)i * nchunk * TS * ny + j;
  int ch = 0;
  auto chunk_end = [&] {
    double *t = t0 + (long long)ch * TS * ny;
    t[0] = ml;
    t[ny] = sw;
    t[2 * ny] = w;
  };
  // a row k of the system that is neither the first nor the last
  auto row = [&](double ak, double bk, double cc) {
    const double z = zrcp<T>((bk + lam) - ak * dp);
    dp = cc * z;
    mp = (-ak * mp) * z;
    if (PER) qp = (0.0 - ak * qp) * z;
    sw = sw + w * mp;
    w = -(dp * w);
    ml = mp;
  };
  for (int g = 0; g < ngrp; ++g) {
    const int k0 = g * gp;
    if (ch + 1 < nchunk && k0 == (ch + 1) * cpl) {
      chunk_end();
      ++ch;
      mp = 1.0;
      w = 1.0;
      sw = 0.0;
      ml = 0.0;
    }
    const long long o = og + (long long)g * ny;
    ckd[o] = dp;
    if (nchunk > 1) ckm[o] = mp;
    if (PER) ckq[o] = qp;
    if (k0 > 0 && k0 + gp < msys) {
#pragma unroll 1
      for (int l = 0; l < gp; l += H) {
        double av[H], bv[H], cv[H];
        slab_rows<H>(a + k0 + l, b + k0 + l, c + k0 + l, av, bv, cv);
#pragma unroll
        for (int r = 0; r < H; ++r) row(av[r], bv[r], cv[r]);
      }
      continue;
    }
    for (int k = k0; k < min(k0 + gp, msys); ++k) {
      if (k > 0 && k < msys - 1) {
        row(a[k], b[k], c[k]);
        continue;
      }
      const double r2 = PER ? (k == msys - 1 ? -c[msys - 1] : -a[0]) : 0.0;
      double dl = 0.0;
      if (k == 0) {
        const double z = zrcp<T>(b[0] + lam);
        dp = c[0] * z;
        mp = 0.0;
        qp = r2 * z;
        dl = dp;
      } else {
        const double z = (b[k] + lam) - a[k] * dp;
        mp = (z != 0.0 && (PER || !(pin && lam == 0.0))) ? (-a[k] * mp) / z : 0.0;
        qp = (z != 0.0) ? (r2 - a[k] * qp) / z : 0.0;
      }
      sw = sw + w * mp;
      w = -(dl * w);
      ml = mp;
    }
  }
  chunk_end();
  if constexpr (PER) {
    const int m = msys;  // nz - 1
    double p2n = 0.0, p20 = 0.0, p2m1 = 0.0;
    const long long last = og + (long long)(ngrp - 1) * ny;
    double dn = ckd[last], qn = ckq[last];
    for (int g = ngrp - 1; g >= 0; --g) {
      const int k0 = g * gp;
      double d2 = dn, q2 = qn;
      // the next group's values, loaded ahead of this one's rows
      const long long o = og + (long long)max(g - 1, 0) * ny;
      dn = ckd[o];
      qn = ckq[o];
      constexpr int MG = GP ? GP : kZcMaxGroup;
      double dd[MG], qq[MG];
      if (GP && k0 > 0 && k0 + gp < m) {
#pragma unroll
        for (int h = 0; h < MG; h += H) {
          double av[H], bv[H], cv[H];
          slab_rows<H>(a + k0 + h, b + k0 + h, c + k0 + h, av, bv, cv);
#pragma unroll
          for (int l = 0; l < H; ++l) {
            const double z = zrcp<T>((bv[l] + lam) - av[l] * d2);
            d2 = cv[l] * z;
            q2 = (0.0 - av[l] * q2) * z;
            dd[h + l] = d2;
            qq[h + l] = q2;
          }
        }
#pragma unroll
        for (int l = MG - 1; l >= 0; --l) p2n = qq[l] - dd[l] * p2n;
      } else {
#pragma unroll
        for (int l = 0; l < MG; ++l) {
          const int k = k0 + l;
          if (l < gp && k < m) {
            const double ak = a[k], bk = b[k], cc = c[k];
            if (k == 0) {
              const double z = zrcp<T>(bk + lam);
              d2 = cc * z;
              q2 = -ak * z;
            } else if (k < m - 1) {
              const double z = zrcp<T>((bk + lam) - ak * d2);
              d2 = cc * z;
              q2 = (0.0 - ak * q2) * z;
            } else {
              const double z = (bk + lam) - ak * d2;
              q2 = (z != 0.0) ? (-cc - ak * q2) / z : 0.0;
            }
          }
          dd[l] = d2;
          qq[l] = q2;
        }
#pragma unroll
        for (int l = MG - 1; l >= 0; --l) {
          const int k = k0 + l;
          if (l >= gp || k >= m) continue;
          const double p2 = (k == m - 1) ? qq[l] : qq[l] - dd[l] * p2n;
          p2n = p2;
          if (k == m - 1) p2m1 = p2;
          if (k == 0) p20 = p2;
        }
      }
      // p2 of the plane after chunk ch - 1
      if (ch > 0 && k0 == ch * cpl) {
        t0[((long long)(ch - 1) * TS + 3) * ny] = p2n;
        --ch;
      }
    }
    den[(long long)i * ny + j] = ((b[m] + lam) + c[m] * p20) + a[m] * p2m1;
  }
}

// Workgroups of the chunked P2 (*r2) and P3 (*r3) slab kernels that one CU
// holds at once, from the runtime's occupancy calculator (it counts the
// kernels' registers, AGPRs included, and their LDS).
template <typename T>
static int slab_residency(int ny, int periodic, int *r2, int *r3) {
  FL_DISPATCH(ny / 2, {
    constexpr int GP = group_planes<T, NC>();
    constexpr int NTP = slab_threads<T, NC, true>();
    constexpr int NTN = slab_threads<T, NC, false>();
    if (periodic) {
      FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          r2, reinterpret_cast<const void *>(&k_yz_fwd_zc<T, NC, GP, NTP, true>), NTP, 0));
      FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          r3, reinterpret_cast<const void *>(&k_zy_bwd_zc<T, NC, GP, NTP, true>), NTP, 0));
    } else {
      FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          r2, reinterpret_cast<const void *>(&k_yz_fwd_zc<T, NC, GP, NTN, false>), NTN, 0));
      FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          r3, reinterpret_cast<const void *>(&k_zy_bwd_zc<T, NC, GP, NTN, false>), NTN, 0));
    }
  });
  return FLUTAS_OK;
}

int fused_slab_residency(int ny, int elem_bytes, int periodic, int *r2, int *r3) {
  *r2 = *r3 = 0;
  return elem_bytes == 8 ? slab_residency<double>(ny, periodic, r2, r3)
                         : slab_residency<float>(ny, periodic, r2, r3);
}

size_t zchunk_doubles(int nx, int ny, int ngrp, int nchunk, bool per) {
  // values at a plane group: d, with two chunks or more m, with periodic z q2
  const size_t col = (size_t)nx * ny, grp = 1 + (nchunk > 1) + per;
  return col * (grp * ngrp + (size_t)nchunk * zc_tab_slots(per) + per +
                (size_t)nchunk * zc_side_slots(per));
}

int build_zchunk_tables(double *mem, ZChunks *zc, int nx, int ny, int nz, int msys, int gp,
                        int cpl, int nchunk, bool per, int pin, int elem_bytes,
                        const double *lamx, const double *lamy, const double *a,
                        const double *b, const double *c, hipStream_t s) {
  if (gp < 1 || gp > kZcMaxGroup || cpl % gp != 0 || nchunk < 1 || nchunk > kMaxZChunks ||
      (nchunk - 1) * cpl > nz - 2)
    return fail(FLUTAS_EINVAL, "z chunks: bad chunk shape");
  const int ngrp = (nz + gp - 1) / gp;
  const size_t col = (size_t)nx * ny;
  // One chunk carries nothing in, its multipliers meet a zero: it reads d in
  // their place (the same lines again, no bytes of its own).
  double *ckd = mem, *ckm = nchunk > 1 ? ckd + col * ngrp : ckd;
  double *ckq = ckm + col * ngrp;
  double *tab = per ? ckq + col * ngrp : ckq;
  double *den = tab + col * nchunk * zc_tab_slots(per);
  double *side = per ? den + col : den;
  if (!per) ckq = den = nullptr;
  const int threads = 256;
  const long long blocks = ((long long)col + threads - 1) / threads;
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), 0, s, ckd, ckm, ckq, tab, den,
                       nx, ny, nz, msys, gp, cpl, nchunk, pin, lamx, lamy, a, b, c);
  };
  auto by_group = [&](auto t, auto p) {
    using T = decltype(t);
    constexpr bool P = decltype(p)::value;
    if (gp == 16) run(&k_zchunk_tables<T, P, 16>);
    else if (gp == 8) run(&k_zchunk_tables<T, P, 8>);
    else if (gp == 4) run(&k_zchunk_tables<T, P, 4>);
    else run(&k_zchunk_tables<T, P, 0>);
  };
  if (elem_bytes == 8) per ? by_group(double(), std::true_type()) : by_group(double(), std::false_type());
  else per ? by_group(float(), std::true_type()) : by_group(float(), std::false_type());
  FL_HIP(hipGetLastError());
  *zc = ZChunks{nchunk, cpl, ngrp, ckd, ckm, ckq, tab, den, side};
  return FLUTAS_OK;
}

template <typename T>
int launch_yz_fwd_zc(const LineTables &ty, int kind, T *Wt, WStride ws, const ZChunks &zc,
                     int nx, int nz, int msys, const double *lamx, const double *lamy,
                     const double *a, const double *b, const double *c, int pin, int periodic,
                     hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(ty);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  const dim3 grid(nx * zc.nchunk);
  FL_DISPATCH(ty.n / 2, {
    constexpr int GP = group_planes<T, NC>();
    constexpr int NTP = slab_threads<T, NC, true>();
    constexpr int NTN = slab_threads<T, NC, false>();
    if (zc.ngrp != (nz + GP - 1) / GP) return fail(FLUTAS_EINVAL, "z chunks: plane groups");
    if (periodic)
      hipLaunchKernelGGL((k_yz_fwd_zc<T, NC, GP, NTP, true>), grid, dim3(NTP), 0, s, Wt, ws, zc,
                         nx, nz, msys, kind, lamx, lamy, a, b, c, pin, pl.tw, th, tq);
    else
      hipLaunchKernelGGL((k_yz_fwd_zc<T, NC, GP, NTN, false>), grid, dim3(NTN), 0, s, Wt, ws, zc,
                         nx, nz, msys, kind, lamx, lamy, a, b, c, pin, pl.tw, th, tq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

template <typename T>
int launch_zy_bwd_zc(const LineTables &ty, int kind, T *Wt, WStride ws, const ZChunks &zc,
                     int nx, int nz, int msys, const double *lamx, const double *lamy,
                     const double *a, const double *b, const double *c, int pin, int periodic,
                     hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(ty);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  const dim3 grid(nx * zc.nchunk);
  FL_DISPATCH(ty.n / 2, {
    constexpr int GP = group_planes<T, NC>();
    constexpr int NTP = slab_threads<T, NC, true>();
    constexpr int NTN = slab_threads<T, NC, false>();
    if (zc.ngrp != (nz + GP - 1) / GP) return fail(FLUTAS_EINVAL, "z chunks: plane groups");
    if (periodic)
      hipLaunchKernelGGL((k_zy_bwd_zc<T, NC, GP, NTP, true>), grid, dim3(NTP), 0, s, Wt, ws, zc,
                         nx, nz, msys, kind, lamx, lamy, a, b, c, pin, pl.tw, th, tq);
    else
      hipLaunchKernelGGL((k_zy_bwd_zc<T, NC, GP, NTN, false>), grid, dim3(NTN), 0, s, Wt, ws, zc,
                         nx, nz, msys, kind, lamx, lamy, a, b, c, pin, pl.tw, th, tq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

template int launch_yz_fwd_zc<double>(const LineTables &, int, double *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_yz_fwd_zc<float>(const LineTables &, int, float *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_zy_bwd_zc<double>(const LineTables &, int, double *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_zy_bwd_zc<float>(const LineTables &, int, float *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);

}  // namespace flutas
