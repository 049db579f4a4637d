// Device helpers shared by the local-term kernels (hpsi_local.hip, wave_planes*.hip, wave_x*.hip).
#pragma once

#include "gw_internal.h"
#include "gw_regfft.h"

namespace gw {

template <typename T> __device__ __forceinline__ cpx<T> czero() { cpx<T> z; z.x = 0; z.y = 0; return z; }

// Range-checked buffer access (raw buffer resource, stride 0): a lane whose byte
// offset lies past `bytes` reads zero and its store is discarded by the memory
// unit, so masked loads and stores need no branch and every lane issues the
// same instruction stream (the wait counts before dependent uses stay exact).
// The base must be wave-uniform; bytes < 2^31.
constexpr int kBufOff = 0x7fffff00;  // offset of a masked lane
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
using u32x2 = unsigned int __attribute__((ext_vector_type(2)));
using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ cpx<T> buf_load(__amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (sizeof(cpx<T>) == 8)
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  else
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
// two adjacent FP32 complex values, moved as one 16-byte access
struct alignas(16) cpx2f { float2 a, b; };
__device__ __forceinline__ cpx2f buf_load2(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(cpx2f, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ void buf_store2(cpx2f v, __amdgpu_buffer_rsrc_t r, int off) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0);
}
template <typename T> __device__ __forceinline__ void buf_store(cpx<T> v, __amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (sizeof(cpx<T>) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0);
}

// the same with a wave-uniform part of the offset
template <typename T> __device__ __forceinline__ cpx<T> buf_load_s(__amdgpu_buffer_rsrc_t r, int off, int soff) {
  if constexpr (sizeof(cpx<T>) == 8)
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
  else
    return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
}
template <typename T>
__device__ __forceinline__ void buf_store_s(cpx<T> v, __amdgpu_buffer_rsrc_t r, int off, int soff) {
  if constexpr (sizeof(cpx<T>) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, soff, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, soff, 0);
}

// Linear workgroup id -> work id so that consecutive work ids share an XCD
// (dispatch places workgroup L on XCD L % 8). Returns -1 for the padding ids.
__device__ __forceinline__ long xcd_work_id(long total) {
  const long L = blockIdx.x;
  const long per = (total + 7) / 8;
  const long w = (L % 8) * per + L / 8;
  return w < total ? w : -1;
}

// Coefficients c[si[i]] of one batch of a plane's points, as separate re / im
// registers (an array of FP64 complex was placed in scratch by the compiler).
template <typename T, int KB>
__device__ __forceinline__ void gather_points(const cpx<T>* __restrict__ cb, const int (&si)[KB], T (&re)[KB],
                                              T (&im)[KB]) {
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const cpx<T> v = cb[si[i]];
    re[i] = v.x;
    im[i] = v.y;
  }
}

struct PlaneItem {
  int a, k, b0, b1;
};
__device__ __forceinline__ PlaneItem plane_item(long wid, int na, int nb, int bpw) {
  const int ngrp = (nb + bpw - 1) / bpw;
  const long rest = wid / na;
  PlaneItem it;
  it.a = (int)(wid % na);
  it.k = (int)(rest / ngrp);
  it.b0 = (int)(rest % ngrp) * bpw;
  it.b1 = min(nb, it.b0 + bpw);
  return it;
}

constexpr int kMaxLds = 160 * 1024;
constexpr size_t kLdsPerCu = 160 * 1024;
constexpr int kAdjBandGroup = 16;  // bands reduced per x-pass workgroup in the V adjoint and the density

// Geometry of one apply, passed to the kernels by value.
struct Geom {
  int n1, n2, n3, na, nst_max, npw_max, nb;
  int xlo, xhi;  // active x-planes = [0, xlo) U [xhi, n1), or xlo = -1
  int st_max_plane;
  int fx0, fx1, fy0, fy1, fz0, fz1;
  int fx2, fy2, fz2;  // third factor of each axis split (1: two factors)
  const int* planes;
  const int* st_plane_ptr;
  const int* st_i1;
  const int* st_pt_ptr;
  const int* pt_src;
  const int* pt_yz;
  const int* npw;
  // any-length wave lines: rows of each (k, plane) in LDS, row(y) = (y + off) mod n2
  int rows_max;
  const int* st_off;   // (nk, na)
  const int* st_nrow;  // (nk, na)
  const int* pt_row;   // (nk, npw_max) LDS position row * (n3 | 1) + z of each point
};
Geom geom_of(const Plan* p, int nb);

// ---- wave lines of any listed length (wave_planes*.hip, wave_x*.hip) ----
// The (M, S) splits built, N = M S: every 2-3-5-7-smooth length from 15 to 160 that
// splits with M <= 10 and S <= 16, the most balanced split. SMALL(M, S): S <= 10.
#define GW_WAVE_SMALL(X)                                                                                     \
  X(3, 5) X(4, 4) X(3, 6) X(4, 5) X(3, 7) X(4, 6) X(5, 5) X(3, 9) X(4, 7) X(5, 6) X(4, 8) X(5, 7) X(6, 6)    \
  X(5, 8) X(6, 7) X(5, 9) X(6, 8) X(7, 7) X(5, 10) X(6, 9) X(7, 8) X(6, 10) X(7, 9) X(8, 8) X(7, 10) X(8, 9) \
  X(8, 10) X(9, 9) X(9, 10) X(10, 10)
#define GW_WAVE_LARGE(X)                                                                                      \
  X(5, 15) X(7, 12) X(8, 12) X(7, 14) X(7, 15) X(9, 12) X(8, 14) X(10, 12) X(9, 14) X(8, 16) X(9, 15) X(10, 14) \
  X(9, 16) X(10, 15) X(10, 16)

// lines per wave, exchange elements per wave and S of a listed length; false if not listed
inline bool wave_any_info(int n, int* lw, int* esize, int* smax) {
#define GW_CASE(M, S)                                   \
  case (M) * (S):                                       \
    *lw = 64 / (S);                                     \
    *esize = ExLayout<(M), (S), 64 / (S)>::SIZE;        \
    *smax = (S);                                        \
    return true;
  switch (n) { GW_WAVE_SMALL(GW_CASE) GW_WAVE_LARGE(GW_CASE) default: return false; }
#undef GW_CASE
}

int plane_bands_knob(bool fp32, bool inv);  // GW_TUNE_PLANE_BANDS, 0 unset
template <typename T> bool wave_planes_fit(const Plan& P);
template <typename T> int wave_planes_per_cu(const Plan& P);  // plane workgroups that a CU's LDS holds
// the any-length wave lines take this plan's local term
inline bool wave_any_ok(const Plan& P, int precision) {
  if ((P.flags & GW_PLAN_LEGACY) || !P.any_ok) return false;
  const size_t e = precision == GW_FP64 ? 16 : 8;
  if ((double)P.na * P.n[1] * P.n[2] * e > (double)kBufOff) return false;  // one band's planes, a buffer resource
  return precision == GW_FP64 ? wave_planes_fit<double>(P) : wave_planes_fit<float>(P);
}
// P1 (inv) or P3 of the whole block, nk k-points of g.nb bands
template <typename T>
int wave_any_planes(bool inv, const Plan& P, const Geom& g, int nk, const cpx<T>* c, long ldc, long sc, cpx<T>* box,
                    const T* t, cpx<T>* out, long ldo, long so, T scale, bool kin, hipStream_t st);
// x passes: x V(r); the V(r) adjoint and the band density into part[group][r]
template <typename T>
int wave_x_apply(const Geom& g, int nbt, cpx<T>* box, const T* vx, const cpx<T>* twx, hipStream_t st);
template <typename T>
int wave_x_adjv(const Geom& g, int nbt, const cpx<T>* boxc, const cpx<T>* boxg, const cpx<T>* twx, double* part,
                hipStream_t st);
template <typename T>
int wave_x_density(const Geom& g, int nbt, const cpx<T>* box, const double* wts, const cpx<T>* twx, double* part,
                   hipStream_t st);
template <typename T> void wave_any_attrs(int want);
template <typename T> void wave_x_attrs(int want);

// One cell of a ragged batch: its blocks, tables and first work items.
template <typename T>
struct RagInst {
  Geom g;
  const cpx<T>* c;
  long ldc, sc;
  cpx<T>* out;
  long ldo, so;
  const T* t;
  const T* vp;  // V(r): natural order (any-length wave lines) or permuted (generic passes)
  const cpx<T>* twx;
  const cpx<T>* twy;
  const cpx<T>* twz;
  cpx<T>* box;
  T scale;
  int XL, nbt, nchunk, kin;
  int emax;      // exchange elements per wave of the plane passes (any-length)
  long w13, w2;  // first work item of this instance in the plane passes / in the x pass
};
// Instance of work item w: the last whose first item is <= w (instances that sit a
// call out share their first item with the next one).
template <typename T>
__device__ __forceinline__ int rag_find(const RagInst<T>* R, int n, long w, bool xpass) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((xpass ? R[mid].w2 : R[mid].w13) <= w) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}
constexpr int kRagWaves = 4;     // waves per workgroup of the ragged passes
constexpr int kRagBandGroup = 8; // bands per ragged x-pass workgroup
// LDS of one ragged plane / x workgroup for this cell, and its exchange elements
template <typename T> size_t wave_rag_plane_lds(const Geom& g, int* emax);
template <typename T> size_t wave_rag_x_lds(const Geom& g, int* nchunk);
// the ragged passes over every cell: P1 (pass 0), x (1), P3 (2); smax = largest S of the batch
template <typename T>
int wave_rag_planes(bool inv, int smax, const RagInst<T>* R, int n, long total, size_t lds, hipStream_t st);
template <typename T>
int wave_rag_x(int smax, const RagInst<T>* R, int n, long total, size_t lds, hipStream_t st);
// sums the band groups' partials: gv[e] += scale * sum_i part[i][e]
int launch_group_sum(long n, int ngroups, double scale, const double* part, double* gv, hipStream_t st);

}  // namespace gw
