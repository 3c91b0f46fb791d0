// Single-problem x passes (P1, P4) of the fused four-pass pressure solve and
// the tables of the compiled lengths; the device bodies and the pipeline
// description are in fused_body.hpp, the slab passes in fused_slab.hip and
// fused_zc.hip.
#include "fused_host.hpp"

namespace flutas {

using tile::cx;

// Tile of an x-pass workgroup (one-dimensional grid over ntile tiles per
// plane times the planes).  Workgroups are dealt to the 8 XCDs round robin,
// so the ids a and a + 8 run on one XCD at about the same time; they get
// the neighbouring tiles 2m and 2m + 1 of one plane.  An FP32 tile of 16
// lines covers 64 bytes of each transposed row of the work field, and its
// neighbour the other 64: on one XCD the 128-byte line is fetched (or
// written back) once instead of once per XCD.
struct XTile {
  int j0t, k;  // tile index within the plane, plane
};
__device__ __forceinline__ XTile x_tile_of(int ntile) {
  const int id = blockIdx.x, total = gridDim.x;
  int L = id;
  if ((ntile & 1) == 0 && id < (total & ~15)) {
    const int r = id & 15;
    L = (id & ~15) + 2 * (r & 7) + (r >> 3);
  }
  return {L % ntile, L / ntile};
}

template <typename T, typename Tin, int NC, int TJ, int NT>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_x_fwd(const Tin *__restrict__ in, long long is1, long long is2,
            T *__restrict__ Wt, WStride ws, int ny, int kind, const T *__restrict__ tw,
            const T *__restrict__ twh, const T *__restrict__ twq,
            double *__restrict__ absmax_part, int *nf_flag, int nf_seq) {
  __shared__ __align__(16) T sm[TJ * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[x_global_tw<T, NC>() ? 2 : Tw<T, NC>::total];
  const XTile xt = x_tile_of((ny + TJ - 1) / TJ);
  double *slot = absmax_part ? absmax_part + blockIdx.x : nullptr;
  x_fwd_tile<T, Tin, NC, TJ, NT>(in, is1, is2, Wt, ws, ny, kind, tw, twh, twq, slot, sm, stw,
                                 xt.j0t * TJ, xt.k, nf_flag, nf_seq);
}

template <typename T, typename Tout, int NC, int TJ, int NT, bool ACC, bool ALIGN>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_x_bwd(const T *__restrict__ Wt, WStride ws, Tout *__restrict__ out, long long os1,
            long long os2, int ny, int kind, T scale, const T *__restrict__ tw,
            const T *__restrict__ twh, const T *__restrict__ twq) {
  __shared__ __align__(16) T sm[TJ * line_stride<T, 2 * NC>()];
  __shared__ __align__(16) T stw[x_global_tw<T, NC>() ? 2 : Tw<T, NC>::total];
  const XTile xt = x_tile_of((ny + TJ - 1) / TJ);
  x_bwd_tile<T, Tout, NC, TJ, NT, ACC, ALIGN>(Wt, ws, out, os1, os2, ny, kind, scale, tw, twh,
                                              twq, sm, stw, xt.j0t * TJ, xt.k);
}

// ---------------------------------------------------------------- host ---

bool fused_supported(int n) {
  switch (n / 2) {
    case 16: case 24: case 32: case 40: case 48: case 50: case 64: case 80: case 96:
    case 100: case 128: case 160: case 192: case 200: case 256: case 320: case 384:
    case 400: case 512: case 1024:
      return (n % 2) == 0;
    default:
      return false;
  }
}

// Per-pass twiddles of Plan<NC>: pass s >= 1, entry (rr, j) =
// exp(-2 pi i rr j / (ns(s) r[s])), laid out [rr][j].
template <int NC>
static void pass_twiddles(std::vector<double> &out) {
  using P = tile::Plan<NC>;
  const long double pi = 3.14159265358979323846264338327950288L;
  out.assign(2 * P::tw_total(), 0.0);
  for (int s = 1; s < P::nst; ++s) {
    const int R = P::r[s], NS = P::ns(s);
    for (int rr = 0; rr < R; ++rr)
      for (int j = 0; j < NS; ++j) {
        const int m = P::tw_off(s) + rr * NS + j;
        const long double a = -2.0L * pi * (long double)(rr * j) / (long double)(NS * R);
        out[2 * m] = (double)cosl(a);
        out[2 * m + 1] = (double)sinl(a);
      }
  }
}

int build_fused_twiddles(LineTables &tab) {
  std::vector<double> h;
  FL_DISPATCH(tab.n / 2, pass_twiddles<NC>(h));
  if (tab.d_ptw) (void)hipFree(tab.d_ptw);
  if (tab.f_ptw) (void)hipFree(tab.f_ptw);
  tab.d_ptw = nullptr;
  tab.f_ptw = nullptr;
  FL_HIP(hipMalloc((void **)&tab.d_ptw, h.size() * sizeof(double)));
  FL_HIP(hipMemcpy(tab.d_ptw, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  std::vector<float> f(h.begin(), h.end());
  FL_HIP(hipMalloc((void **)&tab.f_ptw, f.size() * sizeof(float)));
  FL_HIP(hipMemcpy(tab.f_ptw, f.data(), f.size() * sizeof(float), hipMemcpyHostToDevice));
  return FLUTAS_OK;
}

template <typename T, typename Tin>
int launch_x_fwd(const LineTables &tx, int kind, const Tin *in, long long is1,
                 long long is2, T *Wt, WStride ws, int ny, int nz,
                 double *absmax_part, int *nf_flag, int nf_seq, hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(tx);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  FL_DISPATCH(tx.n / 2, {
    constexpr int NT = tile_threads<T, NC>();
    constexpr int TJ = tile_lines<T, NC>();
    dim3 grid(((ny + TJ - 1) / TJ) * nz);
    hipLaunchKernelGGL((k_x_fwd<T, Tin, NC, TJ, NT>), grid, dim3(NT), 0, s, in, is1,
                       is2, Wt, ws, ny, kind, pl.tw, th, tq, absmax_part, nf_flag,
                       nf_seq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

// FP64 outputs above this many bytes, in lines of 512 and 1024 points, are stored
// from aligned lanes (x_bwd_tile): HBM takes whole memory lines sooner, the cache
// does not mind and the further lanes cost time.  P4, lanes from the line's start /
// aligned (us): 512-point lines 512x400x320 209 / 184, 512x512x256 228 / 213,
// 512x768x320 430 / 388, 512^3 452 / 416, 512x512x1000 889 / 821 (336 MB 141 / 134, but
// the same grid 143 / 142 in another run); 1024-point lines, whose tile is 8 of them
// and not 16, gain only from 2 GB on: 1024x512x256 546 / 551, 1024x768x200 645 / 658,
// 1024x1024x256 (2.1 GB) 1095 / 1087, 1024x1024x512 2349 / 2262.  Lines of 640, 768 and
// 800 points were slower aligned (380 / 406, 518 / 554, 270 / 289; 8 lines a tile too), as
// were FP32 transforms (362 / 376).
template <int NC>
constexpr double align_bytes() {
  return NC == 256 ? 512e6 : 2e9;
}
template <typename T, typename Tout>
int launch_x_bwd(const LineTables &tx, int kind, const T *Wt, WStride ws,
                 Tout *out, long long os1, long long os2, int ny, int nz,
                 T scale, int accumulate, hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(tx);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  FL_DISPATCH(tx.n / 2, {
    constexpr int NT = tile_threads<T, NC>();
    constexpr int TJ = tile_lines<T, NC>();
    dim3 grid(((ny + TJ - 1) / TJ) * nz);
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, s, Wt, ws, out, os1, os2, ny, kind, scale,
                         pl.tw, th, tq);
    };
    if constexpr ((NC == 256 || NC == 512) && sizeof(T) == 8) {
      if (!accumulate && (double)tx.n * ny * nz * sizeof(Tout) > align_bytes<NC>()) {
        run(&k_x_bwd<T, Tout, NC, TJ, NT, false, true>);
        FL_HIP(hipGetLastError());
        return FLUTAS_OK;
      }
    }
    if (accumulate) run(&k_x_bwd<T, Tout, NC, TJ, NT, true, false>);
    else run(&k_x_bwd<T, Tout, NC, TJ, NT, false, false>);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}

int x_fwd_blocks(const LineTables &tx, int elem_bytes, int ny, int nz) {
  // tile_lines<T, NC>() evaluated at run time
  const int ls = tx.n + (elem_bytes == 8 ? 2 : 4);
  const int l = kTileBytes / (ls * elem_bytes);
  int tj = l >= 16 ? 16 : (l >= 8 ? 8 : (l >= 4 ? 4 : (l >= 2 ? 2 : 1)));
  if (elem_bytes == 8 && tx.n == 1024) tj = 8;
  if (elem_bytes == 8 && tx.n == 400) tj = 16;
  return ((ny + tj - 1) / tj) * nz;
}

int fused_group_planes(int ny, int elem_bytes) {
  int gp = 1;
  const int nc = ny / 2;
  auto f = [&](auto tag) -> int {
    using T = decltype(tag);
    switch (nc) {
      case 16: return group_planes<T, 16>();
      case 24: return group_planes<T, 24>();
      case 32: return group_planes<T, 32>();
      case 40: return group_planes<T, 40>();
      case 50: return group_planes<T, 50>();
      case 100: return group_planes<T, 100>();
      case 200: return group_planes<T, 200>();
      case 400: return group_planes<T, 400>();
      case 48: return group_planes<T, 48>();
      case 64: return group_planes<T, 64>();
      case 80: return group_planes<T, 80>();
      case 96: return group_planes<T, 96>();
      case 128: return group_planes<T, 128>();
      case 160: return group_planes<T, 160>();
      case 192: return group_planes<T, 192>();
      case 256: return group_planes<T, 256>();
      case 320: return group_planes<T, 320>();
      case 384: return group_planes<T, 384>();
      case 512: return group_planes<T, 512>();
      case 1024: return group_planes<T, 1024>();
      default: return 1;
    }
  };
  gp = (elem_bytes == 8) ? f(double()) : f(float());
  return gp;
}

template int launch_x_fwd<double, double>(const LineTables &, int, const double *, long long, long long, double *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_x_fwd<float, double>(const LineTables &, int, const double *, long long, long long, float *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_x_fwd<float, float>(const LineTables &, int, const float *, long long, long long, float *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_x_bwd<double, double>(const LineTables &, int, const double *, WStride, double *, long long, long long, int, int, double, int, hipStream_t);
template int launch_x_bwd<float, float>(const LineTables &, int, const float *, WStride, float *, long long, long long, int, int, float, int, hipStream_t);
template int launch_x_bwd<float, double>(const LineTables &, int, const float *, WStride, double *, long long, long long, int, int, float, int, hipStream_t);
}  // namespace flutas
