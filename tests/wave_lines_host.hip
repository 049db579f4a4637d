// Host-side checks of the wave-line x pass over every listed box length: where the
// staged kernel's LDS tiles start. Prints one line per failure and exits non-zero on any.
#include <cstdio>

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

int main() {
#define GW_CASE(M, S) check_stage_tiles<M, S>();
  GW_WAVE_SMALL(GW_CASE)
  GW_WAVE_LARGE(GW_CASE)
#undef GW_CASE
  printf("lengths %d failures %d\n", g_lengths, g_fail);
  return g_fail ? 1 : 0;
}
