// Single-problem slab passes (P2, P3) over whole x-slabs; the device bodies
// are in fused_body.hpp.
#include "fused_host.hpp"

namespace flutas {

template <typename T, int NC, int GP, int NT, bool PER>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_yz_fwd(T *__restrict__ Wt, WStride ws, double *__restrict__ ck, int nx, int nz, int nzs,
             int kind, const double *__restrict__ lamx, const double *__restrict__ lamy,
             const double *__restrict__ a, const double *__restrict__ b,
             const double *__restrict__ c, int pin, const T *__restrict__ tw,
             const T *__restrict__ twh, const T *__restrict__ twq) {
  __shared__ __align__(16) T sm[2 * GP * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[Tw<T, NC>::total];
  constexpr bool OPQ = slab_opaque<T, NC, PER, false, false>();
  yz_fwd_slab<T, NC, GP, NT, PER, OPQ>(Wt, ws, ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, pin, tw,
                                       twh, twq, sm, stw, blockIdx.x);
}

template <typename T, int NC, int GP, int NT, bool PER>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_zy_bwd(T *__restrict__ Wt, WStride ws, const double *__restrict__ ck, int nx, int nz,
             int nzs, int kind,
             const double *__restrict__ lamx, const double *__restrict__ lamy,
             const double *__restrict__ a, const double *__restrict__ b,
             const double *__restrict__ c, const T *__restrict__ tw,
             const T *__restrict__ twh, const T *__restrict__ twq) {
  __shared__ __align__(16) T sm[2 * GP * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[Tw<T, NC>::total];
  constexpr bool OPQ = slab_opaque<T, NC, PER, true, false>();
  zy_bwd_slab<T, NC, GP, NT, PER, OPQ>(Wt, ws, ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, tw, twh,
                                       twq, sm, stw, blockIdx.x);
}

template <typename T>
int launch_yz_fwd(const LineTables &ty, int kind, T *Wt, WStride ws,
                  double *ck, int nx, int nz, int nzs, const double *lamx,
                  const double *lamy, const double *a, const double *b,
                  const double *c, int pin, int periodic, hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(ty);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  FL_DISPATCH(ty.n / 2, {
    constexpr int GP = group_planes<T, NC>();
    constexpr int NTP = slab_threads<T, NC, true>();
    constexpr int NTN = slab_threads<T, NC, false>();
    if (periodic)
      hipLaunchKernelGGL((k_yz_fwd<T, NC, GP, NTP, true>), dim3(nx), dim3(NTP), 0, s, Wt, ws,
                         ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, pin, pl.tw, th,
                         tq);
    else
      hipLaunchKernelGGL((k_yz_fwd<T, NC, GP, NTN, false>), dim3(nx), dim3(NTN), 0, s, Wt, ws,
                         ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, pin, pl.tw, th,
                         tq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

template <typename T>
int launch_zy_bwd(const LineTables &ty, int kind, T *Wt, WStride ws,
                  const double *ck, int nx, int nz, int nzs, const double *lamx,
                  const double *lamy, const double *a, const double *b,
                  const double *c, int periodic, hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(ty);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  FL_DISPATCH(ty.n / 2, {
    constexpr int GP = group_planes<T, NC>();
    constexpr int NTP = slab_threads<T, NC, true>();
    constexpr int NTN = slab_threads<T, NC, false>();
    if (periodic)
      hipLaunchKernelGGL((k_zy_bwd<T, NC, GP, NTP, true>), dim3(nx), dim3(NTP), 0, s, Wt, ws,
                         ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, pl.tw, th, tq);
    else
      hipLaunchKernelGGL((k_zy_bwd<T, NC, GP, NTN, false>), dim3(nx), dim3(NTN), 0, s, Wt, ws,
                         ck, nx, nz, nzs, kind, lamx, lamy, a, b, c, pl.tw, th, tq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

template int launch_yz_fwd<double>(const LineTables &, int, double *, WStride, double *, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_yz_fwd<float>(const LineTables &, int, float *, WStride, double *, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_zy_bwd<double>(const LineTables &, int, double *, WStride, const double *, int, int, int, const double *, const double *, const double *, const double *, const double *, int, hipStream_t);
template int launch_zy_bwd<float>(const LineTables &, int, float *, WStride, const double *, int, int, int, const double *, const double *, const double *, const double *, const double *, int, hipStream_t);

}  // namespace flutas
