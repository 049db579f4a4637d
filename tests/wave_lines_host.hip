// Host-side checks of the wave lines over every listed box length: where the staged x
// pass's LDS tiles start, that an exchange layout gives each element of a wave a slot of
// its own, and both transforms through that layout, lane by lane, against a direct DFT in
// double precision. Prints one line per failure and exits non-zero on any.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "../gradwave_amd/csrc/gw_wave_x.h"

using namespace gw;

static int g_fail = 0, g_lengths = 0;

// FP32 tiles move as 16-byte pairs: their start, row stride and second tile are whole pairs.
template <int M, int S> static void check_stage_tiles() {
  using W = WaveLine<float, M * S, M, S>;
  ++g_lengths;
  for (int nwx : {2, 4, 8}) {
    const size_t ex = (size_t)nwx * W::E_PER_WAVE * sizeof(typename W::EX);
    const size_t start = ex + stage_tw(M * S) * sizeof(float2), row = (size_t)(nwx * W::LW + kXTilePad) * sizeof(float2);
    const int na = M * S - 2;
    const bool ok = start % sizeof(cpx2f) == 0 && row % sizeof(cpx2f) == 0 && stage_tw(M * S) >= M * S &&
                    stage_lds_bytes(M * S, na, nwx * W::LW, ex, sizeof(float2)) == start + 2 * (na + 2) * row;
    if (ok) continue;
    ++g_fail;
    printf("stage tiles n=%d waves=%d start %zu row %zu FAIL\n", M * S, nwx, start, row);
  }
}

// Slots l L + s SS + k K, each once and inside the area; even sizes keep what follows aligned.
template <int M, int S> static void check_exchange() {
  constexpr int LW = 64 / S;
  using X = ExLayout<M, S, LW>;
  std::vector<int> seen(X::SIZE, 0);
  bool ok = X::SIZE % 2 == 0;
  for (int l = 0; l < LW; ++l)
    for (int s = 0; s < S; ++s)
      for (int k = 0; k < M; ++k) {
        const int at = l * X::L + s * X::SS + k * X::K;
        if (at < 0 || at >= X::SIZE || seen[at]++) ok = false;
      }
  int lw = 0, es = 0, sm = 0;
  ok = ok && wave_any_info(M * S, &lw, &es, &sm) && lw == LW && es == X::SIZE && sm == S;
  if (ok) return;
  ++g_fail;
  printf("exchange %d x %d FAIL\n", M, S);
}

// The LW lines of a wave: pass 1 of every part, the exchange, pass 2 of every part.
template <int M, int S> static void check_lines() {
  constexpr int N = M * S, LW = 64 / S;
  using W = WaveLine<double, N, M, S>;
  using X = ExLayout<M, S, LW>;
  std::vector<double2> tw(N), a(LW * N), got(LW * N), E(X::SIZE);
  for (int m = 0; m < N; ++m) tw[m] = double2{std::cos(2 * M_PI * m / N), std::sin(2 * M_PI * m / N)};
  unsigned r = 12345u + N;
  auto rnd = [&] { r = r * 1664525u + 1013904223u; return (double)r / 4294967296.0 - 0.5; };
  for (auto& v : a) v = double2{rnd(), rnd()};
  for (int sign : {+1, -1}) {
    for (int l = 0; l < LW; ++l) {
      if (sign > 0) {
        for (int t = 0; t < S; ++t) {
          double2 x[M];
          for (int q = 0; q < M; ++q) x[q] = a[l * N + W::gpos(t, q)];
          dft<M, +1, double>(x);
          for (int k = 0; k < M; ++k)
            E[l * X::L + t * X::SS + k * X::K] = W::PFA || k == 0 ? x[k] : twmul<+1, double>(x[k], tw[t * k]);
        }
      } else {
        for (int t = 0; t < M; ++t) {
          double2 y[S];
          for (int s = 0; s < S; ++s) y[s] = a[l * N + W::rpos(t, s)];
          dft<S, -1, double>(y);
          for (int s = 0; s < S; ++s)
            E[l * X::L + s * X::SS + t * X::K] = W::PFA || s == 0 ? y[s] : twmul<-1, double>(y[s], tw[t * s]);
        }
      }
    }
    for (int l = 0; l < LW; ++l) {
      if (sign > 0) {
        for (int t = 0; t < M; ++t) {
          double2 y[S];
          for (int s = 0; s < S; ++s) y[s] = E[l * X::L + s * X::SS + t * X::K];
          dft<S, +1, double>(y);
          for (int s = 0; s < S; ++s) got[l * N + W::rpos(t, s)] = y[s];
        }
      } else {
        for (int t = 0; t < S; ++t) {
          double2 x[M];
          for (int k = 0; k < M; ++k) x[k] = E[l * X::L + t * X::SS + k * X::K];
          dft<M, -1, double>(x);
          for (int q = 0; q < M; ++q) got[l * N + W::gpos(t, q)] = x[q];
        }
      }
    }
    double err = 0;
    for (int l = 0; l < LW; ++l)
      for (int k = 0; k < N; ++k) {
        double re = 0, im = 0;
        for (int j = 0; j < N; ++j) {
          const double2 w = tw[(long)j * k % N], v = a[l * N + j];
          re += v.x * w.x - sign * v.y * w.y;
          im += sign * v.x * w.y + v.y * w.x;
        }
        err = std::max(err, std::hypot(got[l * N + k].x - re, got[l * N + k].y - im));
      }
    if (err < 1e-14 * N) continue;
    ++g_fail;
    printf("lines %d = %d x %d sign %d error %.2e FAIL\n", N, M, S, sign, err);
  }
}

int main() {
#define GW_CASE(M, S)        \
  check_stage_tiles<M, S>(); \
  check_exchange<M, S>();    \
  check_lines<M, S>();
  GW_WAVE_SMALL(GW_CASE)
  GW_WAVE_LARGE(GW_CASE)
#undef GW_CASE
  printf("lengths %d failures %d\n", g_lengths, g_fail);
  return g_fail ? 1 : 0;
}
