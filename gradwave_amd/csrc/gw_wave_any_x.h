// Launchers of the x passes over every listed box length.
#pragma once

#include "gw_wave_x.h"

namespace gw {

constexpr int kXWaves = 4;  // waves per workgroup

// f(chunks of lines, work items of `groups` band groups, grid) for the split (M, S) of n1
#define GW_X_SWITCH(CASE)                                                                 \
  switch (g.n1) {                                                                         \
    GW_WAVE_SMALL(CASE)                                                                   \
    GW_WAVE_LARGE(CASE)                                                                   \
    default: set_error("no wave-line split for n1 = %d", g.n1); return GW_ERR_UNSUPPORTED; \
  }                                                                                       \
  GW_CHECK_HIP(hipGetLastError());                                                        \
  return GW_OK;

template <typename T>
int wave_x_apply(const Geom& g, int nbt, cpx<T>* box, const T* vx, const cpx<T>* twx, hipStream_t st) {
  int lw = 1, es = 0, sm = 0;
  (void)wave_any_info(g.n1, &lw, &es, &sm);
  const int lines = kXWaves * lw, nchunk = (g.n2 * g.n3 + lines - 1) / lines;
  // bands per workgroup: V(r) and the set-up are paid once per group, but the chip
  // wants a few thousand workgroups
  const int bgroup = (int)std::max<long>(1, std::min<long>(sizeof(T) == 8 ? 8 : 16, (long)nchunk * nbt / 2048));
  const long total = (long)nchunk * ((nbt + bgroup - 1) / bgroup);
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
  if constexpr (sizeof(T) == 4) {
    // staged tiles where they move in pairs (n2 n3 even) and several bands share a
    // workgroup: 72^3, 133 bands 130 -> 111 us (90^3, 160 bands 310 -> 235)
    const size_t lds = stage_lds_bytes(g.n1, g.na, lines, kXWaves * (size_t)es * 8, sizeof(cpx<T>));
    if (bgroup >= 4 && g.n2 * g.n3 % 2 == 0 && lds <= kLdsPerCu / 2) {
#define GW_CASE(M, S)                                                                                           \
  case (M) * (S):                                                                                               \
    hipLaunchKernelGGL((k_xpass_stage<T, (M) * (S), M, S, kXWaves, true>), grid, dim3(64 * kXWaves), lds, st, g, \
                       nbt, bgroup, box, vx, twx, nchunk, total);                                               \
    break;
      GW_X_SWITCH(GW_CASE)
#undef GW_CASE
    }
  }
#define GW_CASE(M, S)                                                                                               \
  case (M) * (S):                                                                                                   \
    hipLaunchKernelGGL((k_xpass_wave<T, (M) * (S), M, S, kXWaves>), grid, dim3(64 * kXWaves), 0, st, g, nbt, bgroup, \
                       box, vx, twx, nchunk, total);                                                                \
    break;
  GW_X_SWITCH(GW_CASE)
#undef GW_CASE
}

template <typename T>
int wave_x_adjv(const Geom& g, int nbt, const cpx<T>* boxc, const cpx<T>* boxg, const cpx<T>* twx, double* part,
                hipStream_t st) {
  int lw = 1, es = 0, sm = 0;
  (void)wave_any_info(g.n1, &lw, &es, &sm);
  const int lines = 4 * lw, nchunk = (g.n2 * g.n3 + lines - 1) / lines;
  const long total = (long)nchunk * ((nbt + kAdjBandGroup - 1) / kAdjBandGroup);
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
#define GW_CASE(M, S)                                                                                          \
  case (M) * (S):                                                                                              \
    hipLaunchKernelGGL((k_xpass_adjv_wave<T, (M) * (S), M, S>), grid, dim3(256), 0, st, g, nbt, kAdjBandGroup, \
                       boxc, boxg, twx, nchunk, total, part);                                                  \
    break;
  GW_X_SWITCH(GW_CASE)
#undef GW_CASE
}

template <typename T>
int wave_x_density(const Geom& g, int nbt, const cpx<T>* box, const double* wts, const cpx<T>* twx, double* part,
                   hipStream_t st) {
  int lw = 1, es = 0, sm = 0;
  (void)wave_any_info(g.n1, &lw, &es, &sm);
  const int lines = 4 * lw, nchunk = (g.n2 * g.n3 + lines - 1) / lines;
  const long total = (long)nchunk * ((nbt + kAdjBandGroup - 1) / kAdjBandGroup);
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
#define GW_CASE(M, S)                                                                                             \
  case (M) * (S):                                                                                                 \
    hipLaunchKernelGGL((k_xpass_density_wave<T, (M) * (S), M, S>), grid, dim3(256), 0, st, g, nbt, kAdjBandGroup, \
                       box, wts, twx, nchunk, total, part);                                                       \
    break;
  GW_X_SWITCH(GW_CASE)
#undef GW_CASE
}

// ---- ragged batches: the x pass of every cell in one launch ----
template <typename T, int SM>
__global__ void __launch_bounds__(64 * kRagWaves)
k_xpass_rag_any(const RagInst<T>* __restrict__ R, int n, long total) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long w = xcd_work_id(total);
  if (w < 0) return;
  const RagInst<T>& d = R[rag_find(R, n, w, true)];
  const long local = w - d.w2;
  const int chunk = (int)(local % d.nchunk), bgi = (int)(local / d.nchunk);
#define GW_CASE(M, S)                                                                                           \
  case (M) * (S):                                                                                               \
    if constexpr ((S) <= SM) {                                                                                  \
      using W = WaveLine<T, (M) * (S), (M), (S)>;                                                               \
      typename W::EX* E = reinterpret_cast<typename W::EX*>(smem_raw);                                          \
      xpass_wave_body<T, (M) * (S), (M), (S), kRagWaves>(d.g, d.nbt, kRagBandGroup, chunk, bgi, d.box, d.vp, d.twx, E, \
                                                         reinterpret_cast<cpx<T>*>(E + kRagWaves * W::E_PER_WAVE)); \
    }                                                                                                           \
    break;
  switch (d.g.n1) {
    GW_WAVE_SMALL(GW_CASE)
    GW_WAVE_LARGE(GW_CASE)
    default: break;
  }
#undef GW_CASE
}

template <typename T> size_t wave_rag_x_lds(const Geom& g, int* nchunk) {
  int lw = 1, es = 0, sm = 0;
  if (!wave_any_info(g.n1, &lw, &es, &sm)) return 0;
  const int lines = kRagWaves * lw;
  *nchunk = (g.n2 * g.n3 + lines - 1) / lines;
  return (size_t)kRagWaves * es * 8 + (size_t)g.n1 * sizeof(cpx<T>);
}

template <typename T>
int wave_rag_x(int smax, const RagInst<T>* R, int n, long total, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
  if (smax <= 10)
    hipLaunchKernelGGL((k_xpass_rag_any<T, 10>), grid, dim3(64 * kRagWaves), lds, st, R, n, total);
  else
    hipLaunchKernelGGL((k_xpass_rag_any<T, 16>), grid, dim3(64 * kRagWaves), lds, st, R, n, total);
  GW_CHECK_HIP(hipGetLastError());
  return GW_OK;
}

template <typename T> void wave_x_attrs(int want) {
  constexpr auto A = hipFuncAttributeMaxDynamicSharedMemorySize;
  (void)hipFuncSetAttribute((const void*)k_xpass_rag_any<T, 10>, A, want);
  (void)hipFuncSetAttribute((const void*)k_xpass_rag_any<T, 16>, A, want);
  if constexpr (sizeof(T) == 4) {
#define GW_CASE(M, S) (void)hipFuncSetAttribute((const void*)k_xpass_stage<T, (M) * (S), M, S, kXWaves, true>, A, want);
    GW_WAVE_SMALL(GW_CASE)
    GW_WAVE_LARGE(GW_CASE)
#undef GW_CASE
  }
}

#define GW_X_INST(T)                                                                                           \
  template int wave_x_apply<T>(const Geom&, int, cpx<T>*, const T*, const cpx<T>*, hipStream_t);               \
  template int wave_x_adjv<T>(const Geom&, int, const cpx<T>*, const cpx<T>*, const cpx<T>*, double*, hipStream_t); \
  template int wave_x_density<T>(const Geom&, int, const cpx<T>*, const double*, const cpx<T>*, double*, hipStream_t); \
  template size_t wave_rag_x_lds<T>(const Geom&, int*);                                                        \
  template int wave_rag_x<T>(int, const RagInst<T>*, int, long, size_t, hipStream_t);                          \
  template void wave_x_attrs<T>(int);

}  // namespace gw
