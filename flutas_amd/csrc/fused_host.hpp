// Host side shared by the launchers of the compiled four passes: dispatch on
// the complex line length, and the tables a launch hands to its kernels.
#pragma once

#include "fused_body.hpp"

namespace flutas {

#define FL_DISPATCH(NCV, ...)                                \
  switch (NCV) {                                             \
    case 16: { constexpr int NC = 16; __VA_ARGS__; } break;   \
    case 24: { constexpr int NC = 24; __VA_ARGS__; } break;   \
    case 32: { constexpr int NC = 32; __VA_ARGS__; } break;   \
    case 40: { constexpr int NC = 40; __VA_ARGS__; } break;   \
    case 50: { constexpr int NC = 50; __VA_ARGS__; } break;   \
    case 100: { constexpr int NC = 100; __VA_ARGS__; } break; \
    case 200: { constexpr int NC = 200; __VA_ARGS__; } break; \
    case 400: { constexpr int NC = 400; __VA_ARGS__; } break; \
    case 48: { constexpr int NC = 48; __VA_ARGS__; } break;   \
    case 64: { constexpr int NC = 64; __VA_ARGS__; } break;   \
    case 80: { constexpr int NC = 80; __VA_ARGS__; } break;   \
    case 96: { constexpr int NC = 96; __VA_ARGS__; } break;   \
    case 128: { constexpr int NC = 128; __VA_ARGS__; } break; \
    case 160: { constexpr int NC = 160; __VA_ARGS__; } break; \
    case 192: { constexpr int NC = 192; __VA_ARGS__; } break; \
    case 256: { constexpr int NC = 256; __VA_ARGS__; } break; \
    case 320: { constexpr int NC = 320; __VA_ARGS__; } break; \
    case 384: { constexpr int NC = 384; __VA_ARGS__; } break; \
    case 512: { constexpr int NC = 512; __VA_ARGS__; } break; \
    case 1024: { constexpr int NC = 1024; __VA_ARGS__; } break; \
    default: return fail(FLUTAS_EUNSUPPORTED, "no fused kernel for this length"); \
  }

// The fused kernels use the per-pass twiddle tables in place of the plain
// exp(-2 pi i m/N) table.
template <typename T>
inline LinePlan<T> plan_of(const LineTables &t) {
  LinePlan<T> p;
  if constexpr (sizeof(T) == 8) { p = t.dplan(); p.tw = t.d_ptw; }
  else { p = t.fplan(); p.tw = t.f_ptw; }
  return p;
}

// The tables a kind's tile kernels stage as their split and phase tables:
// the DCT-IV/DST-IV pre/post twiddles for REDFT11/RODFT11.
template <typename T>
inline void kind_tables(const LinePlan<T> &pl, int kind, const T **th, const T **tq) {
  if (kind == K_REDFT11 || kind == K_RODFT11) {
    *th = pl.t4;
    *tq = pl.t4 + 2 * (pl.N + 1);
  } else {
    *th = pl.twh;
    *tq = pl.twq;
  }
}

}  // namespace flutas
