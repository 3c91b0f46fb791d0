// The four passes for line lengths without a compiled plan: the same
// pipeline, work field and z-chunk tables as fused_body.hpp and
// fused_chunk.hpp, with the line length, the radix list and the tile shape
// given at run time, so that every even length runs on it.
//
// What makes run-time lengths cheap is the mapping of a tile of L = 2^lgL
// lines to the lanes: lane bits select the line, the remaining bits the
// butterfly.  The 16 lines of an FP64 tile sit an odd number of complex
// values apart, so the lanes of one LDS access fall on distinct banks for
// any butterfly stride and radix (no swizzle per length), the lanes of one
// butterfly share their twiddles (LDS broadcast), and no lane divides by the
// line length.  The passes run in place (inputs to registers, barrier,
// outputs back), one LDS tile per workgroup.
//
// Against the compiled lengths (measured with compiled lengths forced onto
// these kernels) an element costs about 1.5 times the instructions: 512^3 P1
// 389 -> 695, P2 440 -> 615 us, 256^3 53 -> 71, 77 -> 86 us, so the compiled
// plans stay.  Against the five-pass line path, which ran these lengths
// before: 360x300x240 1.68 -> 0.61 ms (2.7 TB/s; P1 125, P2 181, P3 185,
// P4 137 us), 210x154x90 0.36 -> 0.10 ms, 450x450x300 4.0 -> 1.2 ms.
#pragma once

#include "fused_chunk.hpp"

namespace flutas {
namespace gen {

using tile::cx;

constexpr int kMaxPass = kGenMaxPass;
// Run-time plan of one real line length n = 2N.  Quotients by N, n and ns(s)
// go through the multipliers m = ceil(2^32 / d): umulhi(x, m) = x / d while
// x d < 2^32 (x below 2^17, d at most 4096).
template <typename T>
struct Plan {
  int n, N, nst, lsc;  // lsc: complex values between lines, odd
  int radix[kMaxPass], ns[kMaxPass], tstep[kMaxPass];
  unsigned nsm[kMaxPass];
  unsigned nm, Nm;
  const T *tab;  // table_pairs(N) pairs, see Tables
};
__host__ __device__ inline unsigned quot_mul(int d) {
  return d <= 1 ? 0u : (unsigned)((0x100000000ULL + d - 1) / d);
}
__device__ __forceinline__ int quot(int x, unsigned m) { return m ? (int)__umulhi(x, m) : x; }

// The tables a kind needs, contiguous in memory and in LDS after the tile:
// exp(-2 pi i m / N) (N), the split table (N + 1) and the phase table
// (N + 1); for REDFT11 / RODFT11 the last two are their pre and post tables.
template <typename T>
struct Tables {
  const cx<T> *tw;
  const T *th, *tq;
};
__host__ __device__ constexpr int table_pairs(int N) { return 3 * N + 2; }
template <typename T>
__device__ __forceinline__ Tables<T> tables(const T *s, const Plan<T> &pl) {
  return {reinterpret_cast<const cx<T> *>(s), s + 2 * pl.N, s + 4 * pl.N + 2};
}
// Staging in two steps: the loads are issued (before a tile's own, so that
// they need not wait for them), then written to LDS.  kStage pairs per lane
// cover the usual tiles; what is left is copied in place.
constexpr int kStage = 4;
template <typename T>
__device__ __forceinline__ void stage_load(cx<T> *r, const Plan<T> &pl) {
  const cx<T> *g = reinterpret_cast<const cx<T> *>(pl.tab);
  const int np = table_pairs(pl.N);
#pragma unroll
  for (int q = 0; q < kStage; ++q) r[q] = g[min((int)(threadIdx.x + q * blockDim.x), np - 1)];
}
template <typename T>
__device__ __forceinline__ void stage_store(const cx<T> *r, T *s, const Plan<T> &pl) {
  const cx<T> *g = reinterpret_cast<const cx<T> *>(pl.tab);
  cx<T> *d = reinterpret_cast<cx<T> *>(s);
  const int np = table_pairs(pl.N), NT = blockDim.x;
#pragma unroll
  for (int q = 0; q < kStage; ++q) {
    const int t = threadIdx.x + q * NT;
    if (t < np) d[t] = r[q];
  }
  for (int t = threadIdx.x + kStage * NT; t < np; t += NT) d[t] = g[t];
}

// ---- small DFTs beyond those of tile_fft.hpp ------------------------------
// Odd prime R: with a_q = x_q + x_{R-q}, b_q = x_q - x_{R-q},
//   X_p, X_{R-p} = x_0 + sum_q cos(2 pi pq/R) a_q +- S i sum_q sin(2 pi pq/R) b_q.
template <int R>
struct Trig;
template <>
struct Trig<7> {
  static constexpr long double c[4] = {1.0L, 0.623489801858733530525004884004239811L,
      -0.222520933956314404288902564496794759L, -0.900968867902419126236102319507445051L};
  static constexpr long double s[4] = {0.0L, 0.781831482468029808708444526674057750L,
      0.974927912181823607018131682993931217L, 0.433883739117558120475768332848358755L};
};
template <>
struct Trig<11> {
  static constexpr long double c[6] = {1.0L, 0.841253532831181168861811648919367718L,
      0.415415013001886425529274149229623204L, -0.142314838273285140443792668616369669L,
      -0.654860733945285064056925072466293553L, -0.959492973614497389890368057066327699L};
  static constexpr long double s[6] = {0.0L, 0.540640817455597582107635954318691695L,
      0.909631995354518371411715383079028460L, 0.989821441880932732376092037776718787L,
      0.755749574354258283774035843972344420L, 0.281732556841429697711417915346616899L};
};
template <>
struct Trig<13> {
  static constexpr long double c[7] = {1.0L, 0.885456025653209895900375522015098879L,
      0.568064746731155802511807559127516625L, 0.120536680255323053349067687452543582L,
      -0.354604887042535625969637892600018474L, -0.748510748171101098634630599701351384L,
      -0.970941817426052027156982276293789227L};
  static constexpr long double s[7] = {0.0L, 0.464723172043768545656015335133104778L,
      0.822983865893656394579617423439381991L, 0.992708874098053992800751649492520179L,
      0.935016242685414823439784599837830729L, 0.663122658240795202376785492666766280L,
      0.239315664287557767148753726260211895L};
};
template <typename T, int S, int R>
__device__ __forceinline__ void dprime(cx<T> *v) {
  constexpr int H = (R - 1) / 2;
  cx<T> a[H + 1], b[H + 1];
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    a[q] = tile::add(v[q], v[R - q]);
    b[q] = tile::sub(v[q], v[R - q]);
  }
  const cx<T> x0 = v[0];
#pragma unroll
  for (int q = 1; q <= H; ++q) v[0] = tile::add(v[0], a[q]);
#pragma unroll
  for (int p = 1; p <= H; ++p) {
    cx<T> A = x0, B = {T(0), T(0)};
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      const int m = (p * q) % R;
      const T c = T(Trig<R>::c[m <= H ? m : R - m]);
      const T s = m <= H ? T(Trig<R>::s[m]) : -T(Trig<R>::s[R - m]);
      A = {A.x + c * a[q].x, A.y + c * a[q].y};
      B = {B.x + s * b[q].x, B.y + s * b[q].y};
    }
    const cx<T> iB = tile::msi<T, S>(B);
    v[p] = tile::add(A, iB);
    v[R - p] = tile::sub(A, iB);
  }
}
// R = P Q with P, Q coprime (Good's mapping, no twiddles): input
// (Q p + P q) mod R, output k with k = k1 mod P, k = k2 mod Q.
template <typename T, int S, int R>
__device__ __forceinline__ void dftr(cx<T> *v);
template <typename T, int S, int P, int Q>
__device__ __forceinline__ void dgood(cx<T> *v) {
  constexpr int R = P * Q;
  cx<T> w[P][Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    cx<T> t[P];
#pragma unroll
    for (int p = 0; p < P; ++p) t[p] = v[(Q * p + P * q) % R];
    dftr<T, S, P>(t);
#pragma unroll
    for (int p = 0; p < P; ++p) w[p][q] = t[p];
  }
  // sum_q w_Q^{q k2}: both sums carry the plain roots, so the output index
  // is the one with k1 = k mod P and k2 = k mod Q
#pragma unroll
  for (int p = 0; p < P; ++p) {
    dftr<T, S, Q>(w[p]);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) {
      int k = p;
      while (k % Q != k2) k += P;
      v[k] = w[p][k2];
    }
  }
}
// 9 = 3 x 3 with the internal twiddles exp(S 2 pi i n2 k1 / 9)
template <typename T, int S>
__device__ __forceinline__ void d9(cx<T> *v) {
  constexpr long double C[5] = {1.0L, 0.766044443118978035202392650555416674L,
      0.173648177666930348851716626769314796L, 0.0L, -0.939692620785908384054109277324731470L};
  constexpr long double D[5] = {0.0L, 0.642787609686539326322643409907263433L,
      0.984807753012208059366743024589523014L, 0.0L, 0.342020143325668733044099614682259581L};
  cx<T> A[3][3];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
    cx<T> q[3] = {v[n2], v[3 + n2], v[6 + n2]};
    tile::d3<T, S>(q);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1)
      A[n2][k1] = n2 * k1 == 0 ? q[k1]
                               : tile::mul(q[k1], cx<T>{T(C[n2 * k1]), S * T(D[n2 * k1])});
  }
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    cx<T> q[3] = {A[0][k1], A[1][k1], A[2][k1]};
    tile::d3<T, S>(q);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = q[k2];
  }
}
template <typename T, int S, int R>
__device__ __forceinline__ void dftr(cx<T> *v) {
  if constexpr (R == 6) dgood<T, S, 2, 3>(v);
  else if constexpr (R == 10) dgood<T, S, 2, 5>(v);
  else if constexpr (R == 9) d9<T, S>(v);
  else if constexpr (R == 7 || R == 11 || R == 13) dprime<T, S, R>(v);
  else tile::dft<T, S, R>(v);
}

// Keeps the compiler from hoisting the LDS reads of all unrolled butterflies
// and their twiddles to the front.
__device__ __forceinline__ void read_fence() { asm volatile("" ::: "memory"); }

// Butterflies of radix R per thread when a thread's share of the tile is
// about EP complex values.
template <int EP, int R>
__host__ __device__ constexpr int per_thread() {
  return (EP + R - 1) / R;
}

// One Stockham pass in place over the L lines of the tile.
template <typename T, int S, int EP, int R>
__device__ __forceinline__ void pass(cx<T> *buf, const cx<T> *tw, const Plan<T> &pl, int s,
                                     int lgL) {
  constexpr int PER = per_thread<EP, R>();
  const int nb = pl.N / R, ns = pl.ns[s], ts = pl.tstep[s];
  const unsigned nsm = pl.nsm[s];
  const int tid = tile::lane_id<true>(), b0 = tid >> lgL, db = blockDim.x >> lgL;
  cx<T> *x = buf + (tid & ((1 << lgL) - 1)) * pl.lsc;
  cx<T> v[PER][R];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int b = b0 + u * db;
    if (b < nb) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[u][r] = x[b + r * nb];
      if (s > 0) {
        const int m = (b - ns * quot(b, nsm)) * ts;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cx<T> w = tw[r * m];
          if (S > 0) w.y = -w.y;
          v[u][r] = tile::mul(v[u][r], w);
          if (r % 3 == 0) read_fence();
        }
      }
      dftr<T, S, R>(v[u]);
      read_fence();
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int b = b0 + u * db;
    if (b < nb) {
      const int j = b - ns * quot(b, nsm);
      const int base = (b - j) * R + j;
#pragma unroll
      for (int r = 0; r < R; ++r) x[base + r * ns] = v[u][r];
    }
  }
  __syncthreads();
}

// A prime radix without a compiled butterfly: every thread forms its
// outputs (p, b) of the line as direct sums.
template <typename T, int S, int EN>
__device__ void pass_prime(cx<T> *buf, const cx<T> *tw, const Plan<T> &pl, int s, int lgL) {
  const int R = pl.radix[s], N = pl.N, nb = N / R, ns = pl.ns[s], ts = pl.tstep[s];
  const unsigned nsm = pl.nsm[s];
  const int tid = tile::lane_id<true>(), o0 = tid >> lgL, db = blockDim.x >> lgL;
  cx<T> *x = buf + (tid & ((1 << lgL) - 1)) * pl.lsc;
  cx<T> acc[EN];
#pragma unroll
  for (int u = 0; u < EN; ++u) {
    const int o = o0 + u * db;
    acc[u] = {T(0), T(0)};
    if (o < N) {
      const int p = o / nb, b = o - p * nb;
      const int j = b - ns * quot(b, nsm);
      int step = j * ts + p * nb, m = 0;  // step < 2N
      if (step >= N) step -= N;
      for (int r = 0; r < R; ++r) {
        cx<T> w = tw[m];
        if (S > 0) w.y = -w.y;
        acc[u] = tile::add(acc[u], tile::mul(x[b + r * nb], w));
        m += step;
        if (m >= N) m -= N;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EN; ++u) {
    const int o = o0 + u * db;
    if (o < N) {
      const int p = o / nb, b = o - p * nb;
      const int j = b - ns * quot(b, nsm);
      x[(b - j) * R + j + p * ns] = acc[u];
    }
  }
  __syncthreads();
}

// Complex FFT of every line of the tile.  EP bounds a thread's butterflies
// (see per_thread), EN its complex values; PRIME: the list may hold a prime
// above 13 (its pass, a call, costs the kernel registers).
template <typename T, int S, int EP, int EN, bool PRIME = true>
__device__ __forceinline__ void cfft(cx<T> *buf, const cx<T> *tw, const Plan<T> &pl, int lgL) {
  for (int s = 0; s < pl.nst; ++s) {
    switch (pl.radix[s]) {
#define FL_GEN_PASS(R) case R: pass<T, S, EP, R>(buf, tw, pl, s, lgL); break;
      FL_GEN_PASS(2) FL_GEN_PASS(3) FL_GEN_PASS(4) FL_GEN_PASS(5) FL_GEN_PASS(6)
      FL_GEN_PASS(7) FL_GEN_PASS(8) FL_GEN_PASS(9) FL_GEN_PASS(10)
#undef FL_GEN_PASS
      // (11 and 13 take too many registers where a thread's share is small)
      case 11:
        if constexpr (EP >= 8) pass<T, S, EP, 11>(buf, tw, pl, s, lgL);
        else pass_prime<T, S, EN>(buf, tw, pl, s, lgL);
        break;
      case 13:
        if constexpr (EP >= 8) pass<T, S, EP, 13>(buf, tw, pl, s, lgL);
        else pass_prime<T, S, EN>(buf, tw, pl, s, lgL);
        break;
      default:
        if constexpr (PRIME) pass_prime<T, S, EN>(buf, tw, pl, s, lgL);
        break;
    }
  }
}

// Kind of a transform, decoded once.
struct KindBits {
  bool d4, trig, sine;
};
__device__ __forceinline__ KindBits kind_bits(int kind) {
  const bool d4 = tile::is_d4(kind);
  return {d4, tile::is_trig(kind) && !d4, tile::is_sine(kind) || kind == K_RODFT11};
}

// Real split and phases after the forward FFT, in place (tile::post_fwd at
// run-time length).
template <typename T, int EN>
__device__ __forceinline__ void post_fwd(T *sm, const Plan<T> &pl, KindBits kb,
                                         const Tables<T> &tb, int lgL) {
  constexpr int PER = EN / 2 + 1;
  const int N = pl.N, n = pl.n, np = N / 2 + 1;
  const int tid = tile::lane_id<true>(), k0 = tid >> lgL, db = blockDim.x >> lgL;
  T *line = sm + (tid & ((1 << lgL) - 1)) * 2 * pl.lsc;
  const cx<T> *Z = reinterpret_cast<const cx<T> *>(line);
  T o[PER][4];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int k = k0 + u * db;
    if (k < np) {
      cx<T> Xk, Xm;
      tile::split_pair(Z[k], Z[k == 0 ? 0 : N - k], cx<T>{tb.th[2 * k], tb.th[2 * k + 1]}, Xk, Xm);
      if (!kb.trig) {
        o[u][0] = Xk.x; o[u][1] = Xk.y; o[u][2] = Xm.x; o[u][3] = Xm.y;
      } else {
        const T c = tb.tq[2 * k], s = -tb.tq[2 * k + 1];
        const T cm = tb.tq[2 * (N - k)], sm_ = -tb.tq[2 * (N - k) + 1];
        o[u][0] = T(2) * (Xk.x * c + Xk.y * s);
        o[u][1] = T(2) * (Xk.x * s - Xk.y * c);
        o[u][2] = T(2) * (Xm.x * cm + Xm.y * sm_);
        o[u][3] = T(2) * (Xm.x * sm_ - Xm.y * cm);
      }
      read_fence();
    }
  }
  __syncthreads();
  const bool rev = kb.trig && kb.sine;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int k = k0 + u * db;
    if (k < np) {
      const int km = N - k;
      line[rev ? n - 1 - k : k] = o[u][0];
      if (k > 0) line[rev ? k - 1 : n - k] = o[u][1];
      if (2 * k != N) {
        line[rev ? n - 1 - km : km] = o[u][2];
        if (k > 0) line[rev ? km - 1 : n - km] = o[u][3];
      }
    }
  }
  __syncthreads();
}

// Spectral value k of a real input line (tile::hc, tile::vprime).
template <typename T>
__device__ __forceinline__ cx<T> spec(const T *X, int k, int n, KindBits kb, const T *tq) {
  if (!kb.trig) {
    if (k == 0 || 2 * k == n) return {X[k], T(0)};
    return {X[k], X[n - k]};
  }
  const T xk = kb.sine ? X[n - 1 - k] : X[k];
  const T xnk = (k == 0) ? T(0) : (kb.sine ? X[k - 1] : X[n - k]);
  return tile::mul(cx<T>{tq[2 * k], -tq[2 * k + 1]}, cx<T>{xk, -xnk});
}
// Inverse pre-processing in place (tile::pre_inv).
template <typename T, int EN>
__device__ __forceinline__ void pre_inv(T *sm, const Plan<T> &pl, KindBits kb,
                                        const Tables<T> &tb, int lgL) {
  constexpr int PER = EN / 2 + 1;
  const int N = pl.N, n = pl.n, np = N / 2 + 1;
  const int tid = tile::lane_id<true>(), k0 = tid >> lgL, db = blockDim.x >> lgL;
  T *line = sm + (tid & ((1 << lgL) - 1)) * 2 * pl.lsc;
  cx<T> z[PER][2];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int k = k0 + u * db;
    if (k < np) {
      tile::join_pair(spec(line, k, n, kb, tb.tq), spec(line, N - k, n, kb, tb.tq),
                      cx<T>{tb.th[2 * k], -tb.th[2 * k + 1]}, z[u][0], z[u][1]);
      read_fence();
    }
  }
  __syncthreads();
  cx<T> *Z = reinterpret_cast<cx<T> *>(line);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int k = k0 + u * db;
    if (k < np) {
      Z[k] = z[u][0];
      if (k != 0 && 2 * k != N) Z[N - k] = z[u][1];
    }
  }
  __syncthreads();
}

// DCT-IV / DST-IV pre and post steps (tile::d4_pre, d4_post).
template <typename T, bool CJ>
__device__ __forceinline__ void d4_pre(T *sm, const Plan<T> &pl, const T *pre, int lgL) {
  const int tid = tile::lane_id<true>(), k0 = tid >> lgL, db = blockDim.x >> lgL;
  cx<T> *Z = reinterpret_cast<cx<T> *>(sm) + (tid & ((1 << lgL) - 1)) * pl.lsc;
  for (int m = k0; m < pl.N; m += db) {
    const cx<T> v = tile::mul(Z[m], cx<T>{pre[2 * m], pre[2 * m + 1]});
    Z[m] = CJ ? tile::cj(v) : v;
  }
  __syncthreads();
}
template <typename T, int EN, bool CJ>
__device__ __forceinline__ void d4_post(T *sm, const Plan<T> &pl, const T *post, bool sine,
                                        int lgL) {
  const int N = pl.N, n = pl.n;
  const int tid = tile::lane_id<true>(), k0 = tid >> lgL, db = blockDim.x >> lgL;
  T *line = sm + (tid & ((1 << lgL) - 1)) * 2 * pl.lsc;
  const cx<T> *Z = reinterpret_cast<const cx<T> *>(line);
  T o[EN][2];
#pragma unroll
  for (int u = 0; u < EN; ++u) {
    const int k = k0 + u * db;
    if (k < N) {
      const cx<T> W = CJ ? tile::cj(Z[k]) : Z[k];
      const cx<T> w = tile::mul(W, cx<T>{post[2 * k], post[2 * k + 1]});
      o[u][0] = T(2) * w.x;
      o[u][1] = T(-2) * w.y;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EN; ++u) {
    const int k = k0 + u * db;
    if (k < N) {
      line[sine ? n - 1 - 2 * k : 2 * k] = o[u][0];
      line[sine ? 2 * k : n - 1 - 2 * k] = o[u][1];
    }
  }
  __syncthreads();
}

// A thread's share of an x tile: butterflies of about kXEP complex values,
// kXEN complex values at most (two reals each to load and store).
constexpr int kXEP = 8, kXEN = 16;

// ---------------------------------------------------------------- P1 -----
template <typename T, typename Tin, bool PRIME>
__device__ __forceinline__ void x_fwd(const Tin *__restrict__ in, long long is1, long long is2,
                                      T *__restrict__ Wt, WStride ws, int ny, int kind,
                                      const Plan<T> &pl, int lgL, double *absmax_slot,
                                      int *nf_flag, int nf_seq, T *sm, int j0, int k) {
  const int n = pl.n, L = 1 << lgL, tot = n << lgL, NT = blockDim.x;
  const int LS = 2 * pl.lsc;
  const int nl = min(L, ny - j0);
  const KindBits kb = kind_bits(kind);
  T *const stw = sm + L * LS;
  cx<T> sr[kStage];
  stage_load(sr, pl);
  Tin r[2 * kXEN];
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    if (q * NT < tot) {
      const int t = min((int)threadIdx.x + q * NT, tot - 1);
      const int l = quot(t, pl.nm), e = t - l * n;
      r[q] = in[(long long)min(j0 + l, ny - 1) * is1 + (long long)k * is2 + e];
    } else {
      r[q] = Tin(0);
    }
  }
  stage_store(sr, stw, pl);
  const Tables<T> tb = tables(stw, pl);
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    const int t = threadIdx.x + q * NT;
    if (t < tot) {
      const int l = quot(t, pl.nm), e = t - l * n;
      T x = (T)r[q];
      int pos = e;
      if (kb.trig || kb.d4) {
        pos = kb.trig ? tile::mk_pos(e, n) : tile::d4_pos(e, n);
        if (kb.sine && (e & 1)) x = -x;
      }
      sm[l * LS + pos] = x;
    }
  }
  if (absmax_slot) {
    // clamped loads repeat entries of the tile, the rest are zero
    double am = 0.0;
#pragma unroll
    for (int q = 0; q < 2 * kXEN; ++q) am = nan_max(am, (double)r[q]);
    __shared__ double wmax[8];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) am = nan_max(am, __shfl_xor(am, off));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = am;
    __syncthreads();
    if (threadIdx.x == 0) {
      double m = wmax[0];
      for (int w = 1; w < (NT >> 6); ++w) m = nan_max(m, wmax[w]);
      *absmax_slot = m;
    }
  }
  if (nf_flag) {
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 2 * kXEN; ++q) bad |= !(fabs((double)r[q]) <= 1.7976931348623157e308);
    if (bad) *nf_flag = nf_seq;
  }
  __syncthreads();
  cx<T> *const buf = reinterpret_cast<cx<T> *>(sm);
  if (kb.d4) d4_pre<T, false>(sm, pl, tb.th, lgL);
  cfft<T, -1, kXEP, kXEN, PRIME>(buf, tb.tw, pl, lgL);
  if (kb.d4) d4_post<T, kXEN, false>(sm, pl, tb.tq, kb.sine, lgL);
  else post_fwd<T, kXEN>(sm, pl, kb, tb, lgL);
  // transposed store: lanes along the lines
  const int l = threadIdx.x & (L - 1);
  if (l < nl) {
    T *plane = Wt + (long long)k * ws.wk + j0 + l;
    const T *src = sm + l * LS;
    const int db = NT >> lgL;
#pragma unroll 4
    for (int i = threadIdx.x >> lgL; i < n; i += db) {
      if constexpr (sizeof(T) == 8) st_nt(src[i], plane + ws.ioff(i));
      else plane[ws.ioff(i)] = src[i];
    }
  }
}

// ---------------------------------------------------------------- P4 -----
template <typename T, typename Tout, bool ACC, bool PRIME>
__device__ __forceinline__ void x_bwd(const T *__restrict__ Wt, WStride ws,
                                      Tout *__restrict__ out, long long os1, long long os2,
                                      int ny, int kind, T scale, const Plan<T> &pl, int lgL,
                                      T *sm, int j0, int k) {
  const int n = pl.n, L = 1 << lgL, tot = n << lgL, NT = blockDim.x;
  const int LS = 2 * pl.lsc;
  const int nl = min(L, ny - j0);
  const KindBits kb = kind_bits(kind);
  T *const stw = sm + L * LS;
  const int ll = threadIdx.x & (L - 1), i0 = threadIdx.x >> lgL, db = NT >> lgL;
  const T *plane = Wt + (long long)k * ws.wk + min(j0 + ll, ny - 1);
  cx<T> sr[kStage];
  stage_load(sr, pl);
  T r[2 * kXEN];
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    if (q * db < n) r[q] = plane[ws.ioff(min(i0 + q * db, n - 1))];
    if (q % 4 == 3) read_fence();
  }
  stage_store(sr, stw, pl);
  const Tables<T> tb = tables(stw, pl);
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    const int i = i0 + q * db;
    if (i < n) {
      T x = r[q];
      int pos = i;
      if (kb.d4) {
        pos = tile::d4_pos(i, n);
        if (kb.sine && (i & 1)) x = -x;
      }
      sm[ll * LS + pos] = x;
    }
  }
  __syncthreads();
  cx<T> *const buf = reinterpret_cast<cx<T> *>(sm);
  if (kb.d4) d4_pre<T, true>(sm, pl, tb.th, lgL);
  else pre_inv<T, kXEN>(sm, pl, kb, tb, lgL);
  cfft<T, +1, kXEP, kXEN, PRIME>(buf, tb.tw, pl, lgL);
  if (kb.d4) d4_post<T, kXEN, true>(sm, pl, tb.tq, kb.sine, lgL);
#pragma unroll 4
  for (int t = threadIdx.x; t < tot; t += NT) {
    const int l = quot(t, pl.nm), e = t - l * n;
    if (l >= nl) break;
    int pos = e;
    T sg = scale;
    if (kb.trig) {
      pos = tile::mk_pos(e, n);
      if (kb.sine && (e & 1)) sg = -scale;
    }
    const T v = sm[l * LS + pos] * sg;
    Tout *o = out + (long long)(j0 + l) * os1 + (long long)k * os2 + e;
    if constexpr (ACC) *o = (Tout)((double)*o + (double)v);
    else if constexpr (sizeof(T) == 8) st_nt((Tout)v, o);
    else *o = (Tout)v;
  }
}

// ---- stand-alone lines -----------------------------------------------------
// In-place transform of L lines, numbered through both levels of the batch from
// q0 on; lines of unit stride are loaded along themselves, others across the
// lines.  base: L line offsets.
template <typename T, bool FWD, bool PRIME>
__device__ __forceinline__ void lines(T *data, const LineGeom &g, int kind, const Plan<T> &pl,
                                      int lgL, T *sm, long long *base, long long q0) {
  const int n = pl.n, L = 1 << lgL, tot = n << lgL, NT = blockDim.x;
  const int LS = 2 * pl.lsc;
  const int nl = (int)min((long long)L, (long long)g.L1 * g.L2 - q0);
  const KindBits kb = kind_bits(kind);
  const bool along = g.ise == 1;
  T *const stw = sm + L * LS;
  if (threadIdx.x < L) {
    // lines past the last repeat it
    const long long q = q0 + min((int)threadIdx.x, nl - 1), l2 = q / g.L1;
    base[threadIdx.x] = (q - l2 * g.L1) * g.is1 + l2 * g.is2;
  }
  cx<T> sr[kStage];
  stage_load(sr, pl);
  stage_store(sr, stw, pl);
  const Tables<T> tb = tables(stw, pl);
  __syncthreads();
  auto line_of = [&](int t) { return along ? quot(t, pl.nm) : t & (L - 1); };
  auto elem_of = [&](int t, int l) { return along ? t - l * n : t >> lgL; };
  T r[2 * kXEN];
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    if (q * NT < tot) {
      const int t = min((int)threadIdx.x + q * NT, tot - 1), l = line_of(t);
      r[q] = data[base[l] + elem_of(t, l) * g.ise];
    }
  }
#pragma unroll
  for (int q = 0; q < 2 * kXEN; ++q) {
    const int t = threadIdx.x + q * NT;
    if (t < tot) {
      const int l = line_of(t), e = elem_of(t, l);
      T x = r[q];
      int pos = e;
      if (kb.d4) pos = tile::d4_pos(e, n);
      else if (FWD && kb.trig) pos = tile::mk_pos(e, n);
      if ((kb.d4 || (FWD && kb.trig)) && kb.sine && (e & 1)) x = -x;
      sm[l * LS + pos] = x;
    }
  }
  __syncthreads();
  cx<T> *const buf = reinterpret_cast<cx<T> *>(sm);
  if constexpr (FWD) {
    if (kb.d4) d4_pre<T, false>(sm, pl, tb.th, lgL);
    cfft<T, -1, kXEP, kXEN, PRIME>(buf, tb.tw, pl, lgL);
    if (kb.d4) d4_post<T, kXEN, false>(sm, pl, tb.tq, kb.sine, lgL);
    else post_fwd<T, kXEN>(sm, pl, kb, tb, lgL);
  } else {
    pre_inv<T, kXEN>(sm, pl, kb, tb, lgL);
    cfft<T, +1, kXEP, kXEN, PRIME>(buf, tb.tw, pl, lgL);
  }
#pragma unroll 4
  for (int t = threadIdx.x; t < tot; t += NT) {
    const int l = line_of(t), e = elem_of(t, l);
    if (l >= nl) continue;
    int pos = e;
    bool neg = false;
    if (!FWD && kb.trig) {
      pos = tile::mk_pos(e, n);
      neg = kb.sine && (e & 1);
    }
    const T v = sm[l * LS + pos];
    data[base[l] + e * g.ise] = neg ? -v : v;
  }
}

// Columns of a thread: j = tid + u NT, u < CPT (whole waves of idle columns
// skip the elimination).
template <typename T, int CPT>
__device__ __forceinline__ void get_cols(const T *__restrict__ line, T *v, int n) {
#pragma unroll
  for (int u = 0; u < CPT; ++u) v[u] = line[min((int)threadIdx.x + u * (int)blockDim.x, n - 1)];
}
template <typename T, int CPT>
__device__ __forceinline__ void put_cols(T *__restrict__ line, const T *v, int n) {
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int j = threadIdx.x + u * blockDim.x;
    if (j < n) line[j] = v[u];
  }
}

// ---------------------------------------------------------------- P2 -----
// The chunk body of fused_chunk.hpp (yz_fwd_chunk) for y-lines of run-time
// length: GP planes per group, one LDS tile.  zc.nchunk may be 1.
template <typename T, int CPT, int GP, bool PER>
__device__ __forceinline__ void yz_fwd(T *__restrict__ Wt, WStride ws, const ZChunks &zc, int nz,
                                       int msys, int kind, const double *__restrict__ lamx,
                                       const double *__restrict__ lamy,
                                       const double *__restrict__ a,
                                       const double *__restrict__ b,
                                       const double *__restrict__ c, int pin, const Plan<T> &pl,
                                       T *sm, int i, int ch) {
#pragma clang fp contract(off)
  constexpr int lgL = GP == 16 ? 4 : (GP == 8 ? 3 : 2), EN = GP / 2 * CPT, LD = EN;
  static_assert(GP == 1 << lgL, "a group's planes are the lines of the tile");
  using V2 = typename Pair<T>::type;
  const int n = pl.n, N = pl.N, LS = 2 * pl.lsc, NT = blockDim.x;
  const KindBits kb = kind_bits(kind);
  {
    cx<T> sr[kStage];
    stage_load(sr, pl);
    stage_store(sr, sm + GP * LS, pl);
  }
  const Tables<T> tb = tables(sm + GP * LS, pl);
  cx<T> *const buf = reinterpret_cast<cx<T> *>(sm);
  const int ks = ch * zc.cpl, ke = ch == zc.nchunk - 1 ? nz : (ch + 1) * zc.cpl;
  const int gb = ks / GP, ge = (ke + GP - 1) / GP;
  T *line0 = Wt + ws.ioff(i);
  const double lx = lamx[i];
  double lam[CPT], dprev[CPT], pprev[CPT], w[CPT], S[CPT], E[CPT], ym[CPT];
  get_cols<double, CPT>(zc.ckd + ((long long)i * zc.ngrp + gb) * n, dprev, n);
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int j = threadIdx.x + u * NT;
    lam[u] = (j < n) ? lx + lamy[j] : 0.0;
    pprev[u] = S[u] = E[u] = ym[u] = 0.0;
    w[u] = 1.0;
  }
  // element pairs of a group: pair t of the tile is (plane t / N, t % N);
  // branch free, entries past the group or the chunk repeat valid ones
  V2 r[LD];
  auto load = [&](int g) {
    const int tid = tile::lane_id<true>();
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int t = min(tid + q * NT, GP * N - 1);
      const int l = quot(t, pl.Nm), e = 2 * (t - l * N);
      r[q] = *reinterpret_cast<const V2 *>(line0 + (long long)min(g * GP + l, ke - 1) * ws.wk + e);
    }
  };
  // a group's results leave after the next group's loads have arrived (see
  // yz_fwd_slab); hold[l] past the chunk repeats its last plane
  T hold[GP][CPT];
  auto flush = [&](int g) {
    const int tid = tile::lane_id<true>();
#pragma unroll
    for (int l = 0; l < GP; ++l) {
      T *line = line0 + (long long)min(g * GP + l, ke - 1) * ws.wk;
#pragma unroll
      for (int u = 0; u < CPT; ++u)
        if (tid + u * NT < n) st_nt(hold[l][u], line + tid + u * NT);
    }
  };
  load(gb);
  for (int g = gb; g < ge; ++g) {
    const int k0 = g * GP, np = min(GP, ke - k0), tid = tile::lane_id<true>();
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int t = tid + q * NT;
      if (t < GP * N) {
        const int l = quot(t, pl.Nm), e = 2 * (t - l * N);
        const int p0 = kb.trig ? (e >> 1) : e;
        const int p1 = kb.trig ? n - 1 - (e >> 1) : (kb.d4 ? n - 1 - e : e + 1);
        sm[l * LS + p0] = r[q].x;
        sm[l * LS + p1] = ((kb.trig || kb.d4) && kb.sine) ? -r[q].y : r[q].y;
      }
    }
    __syncthreads();
    if (g > gb) flush(g - 1);
    load(min(g + 1, ge - 1));
    if (kb.d4) d4_pre<T, false>(sm, pl, tb.th, lgL);
    cfft<T, -1, EN, EN>(buf, tb.tw, pl, lgL);
    if (kb.d4) d4_post<T, EN, false>(sm, pl, tb.tq, kb.sine, lgL);
    else post_fwd<T, EN>(sm, pl, kb, tb, lgL);
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int j = threadIdx.x + u * NT;
      if (j >= n) continue;
      T y[GP];
#pragma unroll
      for (int l = 0; l < GP; ++l) y[l] = sm[l * LS + j];
      zc_eliminate<T, GP, PER>(a, b, c, k0, np, msys, pin, lam[u], y, dprev[u], pprev[u], w[u],
                               S[u], E[u], ym[u]);
#pragma unroll
      for (int l = 0; l < GP; ++l) hold[l][u] = y[l];
    }
    __syncthreads();
  }
  flush(ge - 1);
  double *sd = zc.side + ((long long)i * zc.nchunk + ch) * zc_side_slots(PER) * n;
  put_cols<double, CPT>(sd, E, n);
  put_cols<double, CPT>(sd + n, S, n);
  if (PER && ch == zc.nchunk - 1) put_cols<double, CPT>(sd + 2 * n, ym, n);
}

// ---------------------------------------------------------------- P3 -----
template <typename T, int CPT, int GP, bool PER>
__device__ __forceinline__ void zy_bwd(T *__restrict__ Wt, WStride ws, const ZChunks &zc, int nz,
                                       int msys, int kind, const double *__restrict__ lamx,
                                       const double *__restrict__ lamy,
                                       const double *__restrict__ a,
                                       const double *__restrict__ b,
                                       const double *__restrict__ c, int pin, const Plan<T> &pl,
                                       T *sm, int i, int ch) {
#pragma clang fp contract(off)
  constexpr int lgL = GP == 16 ? 4 : (GP == 8 ? 3 : 2), EN = GP / 2 * CPT, LD = EN;
  using V2 = typename Pair<T>::type;
  const int n = pl.n, N = pl.N, LS = 2 * pl.lsc, NT = blockDim.x;
  const KindBits kb = kind_bits(kind);
  {
    cx<T> sr[kStage];
    stage_load(sr, pl);
    stage_store(sr, sm + GP * LS, pl);
  }
  const Tables<T> tb = tables(sm + GP * LS, pl);
  cx<T> *const buf = reinterpret_cast<cx<T> *>(sm);
  const int ks = ch * zc.cpl, ke = ch == zc.nchunk - 1 ? nz : (ch + 1) * zc.cpl;
  const int gb = ks / GP, ge = (ke + GP - 1) / GP;
  T *line0 = Wt + ws.ioff(i);
  const double lx = lamx[i];
  double lam[CPT], Pc[CPT], pn[CPT], pn2[CPT], xm[CPT];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int j = threadIdx.x + u * NT;
    lam[u] = (j < n) ? lx + lamy[j] : 0.0;
    Pc[u] = pn[u] = pn2[u] = xm[u] = 0.0;
  }
  zc_carries<CPT, PER>(zc, n, zc.nchunk, i, ch, nz, a, b, c, pin, lam, Pc, pn, pn2, xm,
                       [n](const double *line, double *v) { get_cols<double, CPT>(line, v, n); });
  T pv[GP][CPT];
  double dck[CPT], mck[CPT], qck[CPT];
  auto load = [&](int g) {
    const int tid = tile::lane_id<true>();
    const long long o = ((long long)i * zc.ngrp + g) * n;
    get_cols<double, CPT>(zc.ckd + o, dck, n);
    get_cols<double, CPT>(zc.ckm + o, mck, n);
    if constexpr (PER) get_cols<double, CPT>(zc.ckq + o, qck, n);
#pragma unroll
    for (int l = 0; l < GP; ++l) {
      const long long k = min(g * GP + l, ke - 1);
#pragma unroll
      for (int u = 0; u < CPT; ++u) {
        const int j = min(tid + u * NT, n - 1);
        pv[l][u] = line0[k * ws.wk + j];
      }
    }
  };
  auto flush = [&](int g) {
    const int k0 = g * GP, np = min(GP, ke - k0), tid = tile::lane_id<true>();
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int t = tid + q * NT;
      const int l = quot(t, pl.Nm), e = 2 * (t - l * N);
      if (t >= GP * N || l >= np) continue;
      V2 v;
      if (kb.trig) {
        v.x = sm[l * LS + (e >> 1)];
        v.y = kb.sine ? -sm[l * LS + n - 1 - (e >> 1)] : sm[l * LS + n - 1 - (e >> 1)];
      } else {
        v = *reinterpret_cast<const V2 *>(sm + l * LS + e);
      }
      st_nt2(v.x, v.y, line0 + (long long)(k0 + l) * ws.wk + e);
    }
  };
  load(ge - 1);
  for (int g = ge - 1; g >= gb; --g) {
    const int k0 = g * GP, np = min(GP, ke - k0);
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      if ((int)threadIdx.x + u * NT >= n) continue;
      zc_substitute<T, GP, PER>(
          a, b, c, k0, np, msys, pin, lam[u], dck[u], mck[u], PER ? qck[u] : 0.0, Pc[u], xm[u],
          pn[u], pn2[u], [&](int l) -> T & { return pv[l][u]; });
    }
    if (g + 1 < ge) {
      flush(g + 1);
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int j = threadIdx.x + u * NT;
      if (j >= n) continue;
      const int jp = kb.d4 ? tile::d4_pos(j, n) : j;
      const bool neg = kb.d4 && kb.sine && (j & 1);
#pragma unroll
      for (int l = 0; l < GP; ++l) sm[l * LS + jp] = neg ? -pv[l][u] : pv[l][u];
    }
    __syncthreads();
    if (g > gb) load(g - 1);
    if (kb.d4) d4_pre<T, true>(sm, pl, tb.th, lgL);
    else pre_inv<T, EN>(sm, pl, kb, tb, lgL);
    cfft<T, +1, EN, EN>(buf, tb.tw, pl, lgL);
    if (kb.d4) d4_post<T, EN, true>(sm, pl, tb.tq, kb.sine, lgL);
  }
  flush(gb);
}

}  // namespace gen
}  // namespace flutas
