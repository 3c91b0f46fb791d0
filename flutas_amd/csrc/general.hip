// Kernels and host launchers of the four passes at run-time line lengths
// (gen_body.hpp): tile shapes, radix lists and staged tables are chosen here
// from the length alone.
#include "gen_body.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace flutas {

using gen::cx;

// Tile of a workgroup: neighbouring tiles of one plane run on one XCD at
// about the same time (x_tile_of in fused.hip), so that the partial 128-byte
// rows they write meet in its L2.
__device__ __forceinline__ void gen_tile_of(int ntile, int *j0t, int *k) {
  const int id = blockIdx.x, total = gridDim.x;
  int t = id;
  if ((ntile & 1) == 0 && id < (total & ~15)) {
    const int r = id & 15;
    t = (id & ~15) + 2 * (r & 7) + (r >> 3);
  }
  *j0t = t % ntile;
  *k = t / ntile;
}

// The x and line kernels of lists without a prime above 13 hold two workgroups of
// 512 threads per CU (128 registers); the pass of a prime wants more and those
// lists keep kernels of their own (360x300x240 P1 201 us at 129 registers, 125 at
// 102; 514 points, 257 a prime, 228 us, 292 with its registers cut).
template <typename T, typename Tin, bool PRIME>
__global__ void __launch_bounds__(512, PRIME ? 3 : 4)
    k_gx_fwd(const Tin *__restrict__ in, long long is1, long long is2, T *__restrict__ Wt,
             WStride ws, int ny, int kind, gen::Plan<T> pl, int lgL,
             double *__restrict__ absmax_part, int *nf_flag, int nf_seq) {
  extern __shared__ __align__(16) unsigned char gsm[];
  int j0t, k;
  gen_tile_of((ny + (1 << lgL) - 1) >> lgL, &j0t, &k);
  gen::x_fwd<T, Tin, PRIME>(in, is1, is2, Wt, ws, ny, kind, pl, lgL,
                     absmax_part ? absmax_part + blockIdx.x : nullptr, nf_flag, nf_seq,
                     reinterpret_cast<T *>(gsm), j0t << lgL, k);
}

template <typename T, typename Tout, bool ACC, bool PRIME>
__global__ void __launch_bounds__(512, PRIME ? 3 : 4)
    k_gx_bwd(const T *__restrict__ Wt, WStride ws, Tout *__restrict__ out, long long os1,
             long long os2, int ny, int kind, T scale, gen::Plan<T> pl, int lgL) {
  extern __shared__ __align__(16) unsigned char gsm[];
  int j0t, k;
  gen_tile_of((ny + (1 << lgL) - 1) >> lgL, &j0t, &k);
  gen::x_bwd<T, Tout, ACC, PRIME>(Wt, ws, out, os1, os2, ny, kind, scale, pl, lgL,
                           reinterpret_cast<T *>(gsm), j0t << lgL, k);
}

template <typename T, int CPT, int GP, bool PER>
__global__ void __launch_bounds__(512, CPT == 1 && GP == 8 ? 4 : (CPT == 4 ? 2 : 3))
    k_gyz_fwd(T *__restrict__ Wt, WStride ws, ZChunks zc, int nx, int nz, int msys, int kind,
              const double *__restrict__ lamx, const double *__restrict__ lamy,
              const double *__restrict__ a, const double *__restrict__ b,
              const double *__restrict__ c, int pin, gen::Plan<T> pl) {
  extern __shared__ __align__(16) unsigned char gsm[];
  int i, ch;
  zc_slab_of(nx, zc.nchunk, &i, &ch);
  gen::yz_fwd<T, CPT, GP, PER>(Wt, ws, zc, nz, msys, kind, lamx, lamy, a, b, c, pin, pl,
                                   reinterpret_cast<T *>(gsm), i, ch);
}

template <typename T, int CPT, int GP, bool PER>
__global__ void __launch_bounds__(512, CPT == 1 && GP == 8 ? 4 : (CPT == 4 ? 2 : 3))
    k_gzy_bwd(T *__restrict__ Wt, WStride ws, ZChunks zc, int nx, int nz, int msys, int kind,
              const double *__restrict__ lamx, const double *__restrict__ lamy,
              const double *__restrict__ a, const double *__restrict__ b,
              const double *__restrict__ c, int pin, gen::Plan<T> pl) {
  extern __shared__ __align__(16) unsigned char gsm[];
  int i, ch;
  zc_slab_of(nx, zc.nchunk, &i, &ch);
  gen::zy_bwd<T, CPT, GP, PER>(Wt, ws, zc, nz, msys, kind, lamx, lamy, a, b, c, pin, pl,
                                   reinterpret_cast<T *>(gsm), i, ch);
}

// ---------------------------------------------------------------- host ---

static const int kRadices[] = {13, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// The radix list of N: fewest passes (each costs two barriers and a trip
// through LDS: 450-point lines in 9 x 5 x 5 run P2 at 353 us, in 5 x 5 x 3 x 3
// at 383), then the smallest largest radix; a prime factor above 13 is a
// radix of its own.  ok(R) says whether a pass of radix R fits the launch.
template <typename F>
static void radix_search(int m, int depth, int *cur, int from, RadixList &best, F ok) {
  if (m == 1) {
    if (depth < best.nst || (depth == best.nst && depth > 0 && cur[0] < best.r[0])) {
      best.nst = depth;
      std::copy(cur, cur + depth, best.r);
    }
    return;
  }
  if (depth >= gen::kMaxPass || depth + 1 > best.nst) return;
  for (int q = from; q < (int)(sizeof(kRadices) / sizeof(int)); ++q) {
    const int R = kRadices[q];
    if (m % R != 0 || !ok(R)) continue;
    cur[depth] = R;
    radix_search(m / R, depth + 1, cur, q, best, ok);
  }
}
template <typename F>
static bool radix_list(int N, RadixList &best, F ok) {
  int cur[gen::kMaxPass], depth = 0, m = N;
  for (int p = 17; p <= m; p += 2)
    while (m % p == 0) {
      bool prime = true;
      for (int q = 3; q * q <= p; q += 2) prime &= (p % q) != 0;
      if (!prime || p > 1021 || depth >= gen::kMaxPass || !ok(p)) break;
      cur[depth++] = p;
      m /= p;
    }
  best.nst = gen::kMaxPass + 1;
  radix_search(m, depth, cur, 0, best, ok);
  return best.nst <= gen::kMaxPass;
}

static int threads_for(int v) {
  // whole waves, 1, 2, 4 or 8 of them: a workgroup of five or six waves
  // leaves SIMDs that no second one of its kind fits (360-point tiles: 171 us
  // at 320 threads, 161 at 384, 137 at 512)
  int t = 64;
  while (t < v) t *= 2;
  return t;
}
static size_t gen_lds(int N, int L, int elem) {
  return ((size_t)2 * (N | 1) * L + 2 * gen::table_pairs(N)) * elem;
}
// Two x tiles of a CU share its 160 KB of LDS; lines too long for that, and
// the slab groups of the longest, take up to kGenLds.
constexpr size_t kTileLds = 76 * 1024, kGenLds = 150 * 1024;

// An x tile: as many lines as fit, 16 at most (whole 128-byte rows of the
// work field in FP64).  Eight lines instead: 360x300x240 P1 125 -> 136 us,
// 300x360x240 P1, P4 121, 135 -> 141, 155.
static GenShape x_shape(int n, int elem) {
  const int N = n / 2;
  for (int lg = 4; lg >= 0; --lg) {
    const int L = 1 << lg;
    if (gen_lds(N, L, elem) > (lg > 2 ? kTileLds : kGenLds)) continue;
    // threads a pass of radix R needs
    auto need = [&](int R) {
      const int per = (gen::kXEP + R - 1) / R, nb = N / R;
      return R > 13 ? (N * L + gen::kXEN - 1) / gen::kXEN : (nb + per - 1) / per * L;
    };
    GenShape x;
    x.rl.nst = 0;
    if (N > 1 && !radix_list(N, x.rl, [&](int R) { return need(R) <= 512; })) continue;
    int nt = (N * L + gen::kXEN - 1) / gen::kXEN;
    for (int s = 0; s < x.rl.nst; ++s) nt = std::max(nt, need(x.rl.r[s]));
    if (nt > 512) continue;
    x.lgL = lg;
    x.nt = threads_for(nt);
    return x;
  }
  return GenShape{};
}

// A slab group: 16 planes for lines of up to 256 points (their passes are a
// chain of latencies, paid once per group: 210x154x90 P2, P3 54, 50 us in
// groups of 8, 34, 36 in groups of 16), 8 planes and one column per thread up
// to 512 (300-point lines with 256 threads and two columns each, 182
// registers: P2 212 against 182 us), 8 and 4 planes beyond.
static GenShape y_shape(int n) {
  const int N = n / 2;
  GenShape y;
  y.rl.nst = 0;
  int gp = 8, cpt = 1, nt = 512;
  if (n <= 256) gp = 16, nt = threads_for(n);
  else if (n > 1024) gp = 4, cpt = 4;
  else if (n > 512) cpt = 2;
  if (nt * cpt < n || gen_lds(N, gp, 8) > kGenLds) return y;
  if (N > 1 && !radix_list(N, y.rl, [](int) { return true; })) return y;
  y.gp = gp;
  y.cpt = cpt;
  y.nt = nt;
  return y;
}

template <typename T>
static gen::Plan<T> gen_plan(const LineTables &t, const RadixList &rl, int kind) {
  gen::Plan<T> p{};
  p.n = t.n;
  p.N = t.n / 2;
  p.nst = rl.nst;
  p.lsc = p.N | 1;
  int ns = 1;
  for (int s = 0; s < rl.nst; ++s) {
    p.radix[s] = rl.r[s];
    p.ns[s] = ns;
    p.nsm[s] = gen::quot_mul(ns);
    p.tstep[s] = p.N / (ns * rl.r[s]);
    ns *= rl.r[s];
  }
  p.nm = gen::quot_mul(p.n);
  p.Nm = gen::quot_mul(p.N);
  const int o = (kind == K_REDFT11 || kind == K_RODFT11) ? 2 * gen::table_pairs(p.N) : 0;
  if constexpr (sizeof(T) == 8) p.tab = t.d_gen + o;
  else p.tab = t.f_gen + o;
  return p;
}

bool general_supported(int n) {
  return n >= 2 && (n & 1) == 0 && n <= 2048 && x_shape(n, 8).lgL >= 0 &&
         x_shape(n, 4).lgL >= 0 && y_shape(n).cpt > 0;
}
int general_group_planes(int ny) { return y_shape(ny).gp; }

// The staged tables of the usual kinds, then those of REDFT11 / RODFT11.
int build_general_tables(LineTables &tab, int n) {
  tab.release();
  tab.n = n;
  tab.N = n / 2;
  return add_general_tables(tab);
}
int add_general_tables(LineTables &tab) {
  const int n = tab.n, N = tab.N;
  tab.gen_x[0] = x_shape(n, 8);
  tab.gen_x[1] = x_shape(n, 4);
  tab.gen_y = y_shape(n);
  const long double pi = 3.14159265358979323846264338327950288L;
  std::vector<double> h;
  h.reserve(4 * gen::table_pairs(N));
  auto add = [&](long double a) {
    h.push_back((double)cosl(a));
    h.push_back((double)-sinl(a));
  };
  for (int v = 0; v < 2; ++v) {
    for (int m = 0; m < N; ++m) add(2.0L * pi * m / N);
    for (int k = 0; k <= N; ++k)
      add(v == 0 ? 2.0L * pi * k / n : pi * (4.0L * k + 1.0L) / (4.0L * n));
    for (int k = 0; k <= N; ++k) add(v == 0 ? pi * k / (2.0L * n) : pi * k / (long double)n);
  }
  FL_HIP(hipMalloc((void **)&tab.d_gen, h.size() * sizeof(double)));
  FL_HIP(hipMemcpy(tab.d_gen, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  std::vector<float> f(h.begin(), h.end());
  FL_HIP(hipMalloc((void **)&tab.f_gen, f.size() * sizeof(float)));
  FL_HIP(hipMemcpy(tab.f_gen, f.data(), f.size() * sizeof(float), hipMemcpyHostToDevice));
  return FLUTAS_OK;
}

static bool has_prime(const RadixList &rl) {
  for (int q = 0; q < rl.nst; ++q)
    if (rl.r[q] > 13) return true;
  return false;
}
bool general_has_prime(int n) { return general_supported(n) && has_prime(y_shape(n).rl); }

// Dynamic LDS beyond 64 KiB has to be asked for.  The limit belongs to the
// kernel, which all plans and threads of the process share: every launch asks
// for the same most that any shape takes, so that none lowers it between
// another's asking and its launch.
template <typename F>
static int allow_lds(F *kernel, size_t bytes) {
  if (bytes <= 64 * 1024) return FLUTAS_OK;
  FL_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGenLds));
  return FLUTAS_OK;
}

template <typename T, typename Tin>
int launch_gen_x_fwd(const LineTables &tx, int kind, const Tin *in, long long is1, long long is2,
                     T *Wt, WStride ws, int ny, int nz, double *absmax_part, int *nf_flag,
                     int nf_seq, hipStream_t s) {
  const GenShape &x = tx.gen_x[sizeof(T) == 8 ? 0 : 1];
  if (x.lgL < 0) return fail(FLUTAS_EUNSUPPORTED, "no tile for this length");
  const gen::Plan<T> pl = gen_plan<T>(tx, x.rl, kind);
  const int L = 1 << x.lgL;
  const size_t lds = gen_lds(pl.N, L, sizeof(T));
  auto run = [&](auto kernel) -> int {
    FL_TRY(allow_lds(kernel, lds));
    hipLaunchKernelGGL(kernel, dim3((ny + L - 1) / L * nz), dim3(x.nt), lds, s, in, is1, is2, Wt,
                       ws, ny, kind, pl, x.lgL, absmax_part, nf_flag, nf_seq);
    FL_HIP(hipGetLastError());
    return FLUTAS_OK;
  };
  return has_prime(x.rl) ? run(&k_gx_fwd<T, Tin, true>) : run(&k_gx_fwd<T, Tin, false>);
}

int gen_x_fwd_blocks(int n, int elem_bytes, int ny, int nz) {
  const int L = 1 << x_shape(n, elem_bytes).lgL;
  return (ny + L - 1) / L * nz;
}

template <typename T, typename Tout>
int launch_gen_x_bwd(const LineTables &tx, int kind, const T *Wt, WStride ws, Tout *out,
                     long long os1, long long os2, int ny, int nz, T scale, int accumulate,
                     hipStream_t s) {
  const GenShape &x = tx.gen_x[sizeof(T) == 8 ? 0 : 1];
  if (x.lgL < 0) return fail(FLUTAS_EUNSUPPORTED, "no tile for this length");
  const gen::Plan<T> pl = gen_plan<T>(tx, x.rl, kind);
  const int L = 1 << x.lgL;
  const size_t lds = gen_lds(pl.N, L, sizeof(T));
  const dim3 grid((ny + L - 1) / L * nz);
  auto run = [&](auto kernel) -> int {
    FL_TRY(allow_lds(kernel, lds));
    hipLaunchKernelGGL(kernel, grid, dim3(x.nt), lds, s, Wt, ws, out, os1, os2, ny, kind, scale,
                       pl, x.lgL);
    FL_HIP(hipGetLastError());
    return FLUTAS_OK;
  };
  if (has_prime(x.rl))
    return accumulate ? run(&k_gx_bwd<T, Tout, true, true>) : run(&k_gx_bwd<T, Tout, false, true>);
  return accumulate ? run(&k_gx_bwd<T, Tout, true, false>) : run(&k_gx_bwd<T, Tout, false, false>);
}

template <typename T, bool FWD, bool PRIME>
__global__ void __launch_bounds__(512, PRIME ? 3 : 4)
    k_g_lines(T *data, LineGeom g, int kind, gen::Plan<T> pl, int lgL) {
  extern __shared__ __align__(16) unsigned char raw[];
  __shared__ long long base[16];
  gen::lines<T, FWD, PRIME>(data, g, kind, pl, lgL, reinterpret_cast<T *>(raw), base,
                     (long long)blockIdx.x << lgL);
}
bool gen_lines_supported(const LineTables &tab, int kind, long long lines) {
  return tab.d_gen && kind != K_REDFT00 && kind != K_RODFT00 && lines <= 100000000LL;
}
template <typename T>
int launch_gen_lines(const LineTables &tab, int kind, T *data, const LineGeom &g, hipStream_t s) {
  const GenShape &x = tab.gen_x[sizeof(T) == 8 ? 0 : 1];
  if (x.lgL < 0) return fail(FLUTAS_EUNSUPPORTED, "no tile for this length");
  const gen::Plan<T> pl = gen_plan<T>(tab, x.rl, kind);
  const int L = 1 << x.lgL;
  const size_t lds = gen_lds(pl.N, L, sizeof(T));
  const dim3 grid((unsigned)(((long long)g.L1 * g.L2 + L - 1) / L));
  const bool fwd = kind != K_HC2R && kind != K_REDFT01 && kind != K_RODFT01;
  auto run = [&](auto kernel) -> int {
    FL_TRY(allow_lds(kernel, lds));
    hipLaunchKernelGGL(kernel, grid, dim3(x.nt), lds, s, data, g, kind, pl, x.lgL);
    FL_HIP(hipGetLastError());
    return FLUTAS_OK;
  };
  if (has_prime(x.rl)) return fwd ? run(&k_g_lines<T, true, true>) : run(&k_g_lines<T, false, true>);
  return fwd ? run(&k_g_lines<T, true, false>) : run(&k_g_lines<T, false, false>);
}
template int launch_gen_lines<double>(const LineTables &, int, double *, const LineGeom &, hipStream_t);
template int launch_gen_lines<float>(const LineTables &, int, float *, const LineGeom &, hipStream_t);

// Calls f with the compile-time shape of a slab launch.
template <int C, int G, bool P>
struct SlabTag {
  static constexpr int cpt = C, gp = G;
  static constexpr bool per = P;
};
template <typename F>
static int by_shape(const GenShape &y, bool per, F f) {
  auto go = [&](auto c, auto g) -> int {
    constexpr int C = decltype(c)::value, G = decltype(g)::value;
    return per ? f(SlabTag<C, G, true>()) : f(SlabTag<C, G, false>());
  };
  using std::integral_constant;
  if (y.cpt == 1 && y.gp == 16) return go(integral_constant<int, 1>(), integral_constant<int, 16>());
  if (y.cpt == 1 && y.gp == 8) return go(integral_constant<int, 1>(), integral_constant<int, 8>());
  if (y.cpt == 2 && y.gp == 8) return go(integral_constant<int, 2>(), integral_constant<int, 8>());
  if (y.cpt == 4 && y.gp == 4) return go(integral_constant<int, 4>(), integral_constant<int, 4>());
  return fail(FLUTAS_EUNSUPPORTED, "no slab group for this length");
}

template <typename T>
int launch_gen_yz_fwd(const LineTables &ty, int kind, T *Wt, WStride ws, const ZChunks &zc, int nx,
                      int nz, int msys, const double *lamx, const double *lamy, const double *a,
                      const double *b, const double *c, int pin, int periodic, hipStream_t s) {
  const GenShape &y = ty.gen_y;
  const gen::Plan<T> pl = gen_plan<T>(ty, y.rl, kind);
  const size_t lds = gen_lds(pl.N, y.gp, sizeof(T));
  return by_shape(y, periodic != 0, [&](auto t) -> int {
    using S = decltype(t);
    auto *k = &k_gyz_fwd<T, S::cpt, S::gp, S::per>;
    FL_TRY(allow_lds(k, lds));
    hipLaunchKernelGGL(k, dim3(nx * zc.nchunk), dim3(y.nt), lds, s, Wt, ws, zc, nx, nz, msys, kind,
                       lamx, lamy, a, b, c, pin, pl);
    FL_HIP(hipGetLastError());
    return FLUTAS_OK;
  });
}

template <typename T>
int launch_gen_zy_bwd(const LineTables &ty, int kind, T *Wt, WStride ws, const ZChunks &zc, int nx,
                      int nz, int msys, const double *lamx, const double *lamy, const double *a,
                      const double *b, const double *c, int pin, int periodic, hipStream_t s) {
  const GenShape &y = ty.gen_y;
  const gen::Plan<T> pl = gen_plan<T>(ty, y.rl, kind);
  const size_t lds = gen_lds(pl.N, y.gp, sizeof(T));
  return by_shape(y, periodic != 0, [&](auto t) -> int {
    using S = decltype(t);
    auto *k = &k_gzy_bwd<T, S::cpt, S::gp, S::per>;
    FL_TRY(allow_lds(k, lds));
    hipLaunchKernelGGL(k, dim3(nx * zc.nchunk), dim3(y.nt), lds, s, Wt, ws, zc, nx, nz, msys, kind,
                       lamx, lamy, a, b, c, pin, pl);
    FL_HIP(hipGetLastError());
    return FLUTAS_OK;
  });
}

template <typename T>
static int gen_residency(int ny, int periodic, int *r2, int *r3) {
  const GenShape y = y_shape(ny);
  const size_t lds = gen_lds(ny / 2, y.gp, sizeof(T));
  return by_shape(y, periodic != 0, [&](auto t) -> int {
    using S = decltype(t);
    auto *k2 = &k_gyz_fwd<T, S::cpt, S::gp, S::per>;
    auto *k3 = &k_gzy_bwd<T, S::cpt, S::gp, S::per>;
    FL_TRY(allow_lds(k2, lds));
    FL_TRY(allow_lds(k3, lds));
    FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(r2, reinterpret_cast<const void *>(k2),
                                                        y.nt, lds));
    FL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(r3, reinterpret_cast<const void *>(k3),
                                                        y.nt, lds));
    return FLUTAS_OK;
  });
}
int general_slab_residency(int ny, int elem_bytes, int periodic, int *r2, int *r3) {
  *r2 = *r3 = 0;
  return elem_bytes == 8 ? gen_residency<double>(ny, periodic, r2, r3)
                         : gen_residency<float>(ny, periodic, r2, r3);
}

template int launch_gen_x_fwd<double, double>(const LineTables &, int, const double *, long long, long long, double *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_gen_x_fwd<float, double>(const LineTables &, int, const double *, long long, long long, float *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_gen_x_fwd<float, float>(const LineTables &, int, const float *, long long, long long, float *, WStride, int, int, double *, int *, int, hipStream_t);
template int launch_gen_x_bwd<double, double>(const LineTables &, int, const double *, WStride, double *, long long, long long, int, int, double, int, hipStream_t);
template int launch_gen_x_bwd<float, float>(const LineTables &, int, const float *, WStride, float *, long long, long long, int, int, float, int, hipStream_t);
template int launch_gen_x_bwd<float, double>(const LineTables &, int, const float *, WStride, double *, long long, long long, int, int, float, int, hipStream_t);
template int launch_gen_yz_fwd<double>(const LineTables &, int, double *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_gen_yz_fwd<float>(const LineTables &, int, float *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_gen_zy_bwd<double>(const LineTables &, int, double *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);
template int launch_gen_zy_bwd<float>(const LineTables &, int, float *, WStride, const ZChunks &, int, int, int, const double *, const double *, const double *, const double *, const double *, int, int, hipStream_t);

}  // namespace flutas
