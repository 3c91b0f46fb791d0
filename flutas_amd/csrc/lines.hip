// Stand-alone line transforms (flutas_fft_lines, flutas_fft_guru) of the
// compiled lengths: a tile of lines per workgroup, transformed in LDS with the
// plans of the fused passes (tile_fft.hpp), in place, any strides.
#include "fused_body.hpp"
#include "fused_host.hpp"

namespace flutas {

using tile::cx;

// One workgroup: TJ lines, numbered through both levels of the batch.  Lines of
// unit stride are loaded along themselves, others across the lines (adjacent
// lines of a strided geometry lie side by side: 16 FP64 lines cover a 128-byte
// row).  Bound by its one read and write of the data: a call on 512x512x128 FP64
// takes 239 us along x and 257 across, 600 with the radices read from a table
// at run time (k_lines); 256x192x128 43 and 39 against 90 and 80.
template <typename T, int NC, int TJ, int NT, bool FWD>
__global__ void __launch_bounds__(NT, slab_waves_per_simd(NT))
    k_lines_tile(T *data, LineGeom g, int kind, const T *__restrict__ tw,
                 const T *__restrict__ twh, const T *__restrict__ twq) {
  constexpr int n = 2 * NC;
  constexpr int LS = line_stride<T, n>();
  constexpr int LD = (TJ * n + NT - 1) / NT;
  __shared__ __align__(16) T sm[TJ * LS];
  __shared__ __align__(16) T stw[x_global_tw<T, NC>() ? 2 : Tw<T, NC>::total];
  __shared__ long long base[TJ];
  const long long q0 = (long long)blockIdx.x * TJ, lines = (long long)g.L1 * g.L2;
  const int nl = (int)min((long long)TJ, lines - q0);
  if (threadIdx.x < TJ) {
    // lines past the last (partial tile) repeat it
    const long long q = q0 + min((int)threadIdx.x, nl - 1), l2 = q / g.L1;
    base[threadIdx.x] = (q - l2 * g.L1) * g.is1 + l2 * g.is2;
  }
  const bool along = g.ise == 1;
  const bool d4 = tile::is_d4(kind);
  const bool trig = tile::is_trig(kind) && !d4;
  const bool sine = tile::is_sine(kind) || kind == K_RODFT11;
  const Tw<T, NC> W = x_global_tw<T, NC>() ? Tw<T, NC>{tw, twh, twq}
                                           : stage_twiddles<T, NC, NT>(stw, tw, twh, twq);
  __syncthreads();
  T r[LD];
#pragma unroll
  for (int q = 0; q < LD; ++q) {
    const int t = min((int)threadIdx.x + q * NT, TJ * n - 1);
    const int l = along ? t / n : t % TJ, e = along ? t - (t / n) * n : t / TJ;
    r[q] = data[base[l] + e * g.ise];
  }
#pragma unroll
  for (int q = 0; q < LD; ++q) {
    const int t = threadIdx.x + q * NT;
    if (t >= TJ * n) continue;
    const int l = along ? t / n : t % TJ, e = along ? t - (t / n) * n : t / TJ;
    T x = r[q];
    int pos = e;
    if (d4) pos = tile::d4_pos(e, n);
    else if (FWD && trig) pos = tile::mk_pos(e, n);
    if ((d4 || (FWD && trig)) && sine && (e & 1)) x = -x;
    sm[l * LS + pos] = x;
  }
  __syncthreads();
  if constexpr (FWD) {
    if (d4) {
      tile::d4_pre<T, NC, TJ, NT, LS, false>(sm, W.th);
      __syncthreads();
    }
    tile::cfft<T, -1, NC, TJ, NT, LS / 2>(reinterpret_cast<cx<T> *>(sm), W.tw);
    if (d4) tile::d4_post<T, NC, TJ, NT, LS, false>(sm, W.tq, sine);
    else tile::post_fwd<T, NC, TJ, NT, LS>(sm, kind, W.th, W.tq);
  } else {
    tile::pre_inv<T, NC, TJ, NT, LS>(sm, kind, W.th, W.tq);
    tile::cfft<T, +1, NC, TJ, NT, LS / 2>(reinterpret_cast<cx<T> *>(sm), W.tw);
  }
#pragma unroll
  for (int q = 0; q < LD; ++q) {
    const int t = threadIdx.x + q * NT;
    const int l = along ? t / n : t % TJ, e = along ? t - (t / n) * n : t / TJ;
    if (t >= TJ * n || l >= nl) continue;
    int pos = e;
    T sg = T(1);
    if (!FWD && trig) {
      pos = tile::mk_pos(e, n);
      if (sine && (e & 1)) sg = T(-1);
    }
    const T v = sm[l * LS + pos];
    data[base[l] + e * g.ise] = FWD ? v : v * sg;
  }
}

// A kind and line count that launch_lines_tile runs (n a compiled length: the
// tables hold its pass twiddles).
bool lines_tile_supported(const LineTables &tab, int kind, long long lines) {
  return tab.d_ptw && kind != K_REDFT00 && kind != K_RODFT00 && lines <= 100000000LL;
}

template <typename T>
int launch_lines_tile(const LineTables &tab, int kind, T *data, const LineGeom &g,
                      hipStream_t s) {
  const LinePlan<T> pl = plan_of<T>(tab);
  const T *th, *tq;
  kind_tables(pl, kind, &th, &tq);
  const bool fwd = kind == K_R2HC || kind == K_REDFT10 || kind == K_RODFT10 ||
                   kind == K_REDFT11 || kind == K_RODFT11;
  FL_DISPATCH(tab.n / 2, {
    constexpr int NT = tile_threads<T, NC>();
    constexpr int TJ = tile_lines<T, NC>();
    const dim3 grid((unsigned)(((long long)g.L1 * g.L2 + TJ - 1) / TJ));
    if (fwd)
      hipLaunchKernelGGL((k_lines_tile<T, NC, TJ, NT, true>), grid, dim3(NT), 0, s, data, g,
                         kind, pl.tw, th, tq);
    else
      hipLaunchKernelGGL((k_lines_tile<T, NC, TJ, NT, false>), grid, dim3(NT), 0, s, data, g,
                         kind, pl.tw, th, tq);
  });
  FL_HIP(hipGetLastError());
  return FLUTAS_OK;
}
template int launch_lines_tile<double>(const LineTables &, int, double *, const LineGeom &, hipStream_t);
template int launch_lines_tile<float>(const LineTables &, int, float *, const LineGeom &, hipStream_t);

}  // namespace flutas
