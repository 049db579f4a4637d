// Plane passes of the local term on wave lines of any listed length, cubic or not.
//
//   P1  per (x-plane, bands of one k): scatter the plane's points into stick rows in
//       LDS, inverse z on the rows in place, inverse y on every column, natural-order
//       rows out to the box
//   P3  per (x-plane, bands of one k): forward y on the box's columns into stick rows,
//       forward z in place, gather + t c
//
// Each pass is a run over lines (z rows, then y columns) of a box length picked by
// a switch on the uniform length, so one kernel takes every pair of lengths while
// each length's transform is compiled for its split (a kernel whose codelets, and
// not its lengths, were picked at run time kept both register arrays alive across
// the switches: 250 VGPRs FP64, spills, 3x slower). A plane's sticks are a cyclic
// interval of y (gw_internal.h), so the LDS row of a y-position is a running sum
// modulo n2 and no map is read.
//
// What it replaced: LDS tiles of whole planes (one or two workgroups per CU, a
// barrier between every pass, digit-permuted order), and, where an FP64 plane
// above 95 x 95 did not fit, two extra passes over the sticks in HBM.
#pragma once

#include "gw_local.h"

namespace gw {

// v, opaque to the compiler: values that depend on the lane and a length alone would
// otherwise be computed for every length before the loops and kept in registers
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// f(u, voffset, uniform offset) for the S r-space positions of a lane (part t < M) in
// a box plane of rows of rowb bytes, at column byte col: a Cooley-Tukey split's are
// M rows apart for every lane, a prime-factor split's wrap around n per lane.
template <typename W, int M, int S, typename F>
__device__ __forceinline__ void each_rpos(int t, int col, int rowb, F&& f) {
  constexpr int N = M * S;
  if constexpr (W::PFA) {
    const int wrap = N * rowb, step = (W::CS % N) * rowb;
    int v = opaque((W::CM * t) % N) * rowb;
#pragma unroll
    for (int u = 0; u < S; ++u) {
      f(u, col + v, 0);
      v += step;
      v = v >= wrap ? v - wrap : v;
    }
  } else {
    const int v = col + t * rowb;
#pragma unroll
    for (int u = 0; u < S; ++u) f(u, v, u * M * rowb);
  }
}

// One run over lines.
template <typename T> struct LineRun {
  cpx<T>* rows;   // stick rows in LDS
  int rs;         // row stride
  int nline;      // lines of this run
  int nrow, off;  // y lines: rows present and row of y = 0
  void* E;        // the wave's exchange area
  const cpx<T>* tw;
  int n3;         // box row length (y lines)
  bool zline;
};

// Inverse transforms: z lines LDS -> LDS in place, y lines LDS -> box plane rb.
template <typename T, int M, int S>
__device__ __forceinline__ void lines_inv(const LineRun<T>& R, __amdgpu_buffer_rsrc_t rb, int wave, int nw, int lane_) {
  constexpr int N = M * S;
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  const int lane = opaque(lane_);
  const int t = lane / LW, l = lane - t * LW;
  const bool part = t < S;
  typename W::EX* E = reinterpret_cast<typename W::EX*>(R.E);
  // positions scaled by the element stride of a line: 1 along a z row, rs along a column
  const int es = R.zline ? 1 : R.rs, ls = R.zline ? R.rs : 1;
  const int wrap = N * es, step = S * es, lim = R.zline ? N : R.nrow * es;
  int g0 = part ? W::gpos(t, 0) + (R.zline ? 0 : R.off) : 0;
  g0 = (g0 >= N ? g0 - N : g0) * es;
  const int rowb = R.n3 * (int)sizeof(cpx<T>);
  for (int c0 = wave * LW; c0 < R.nline; c0 += nw * LW) {
    const int line = c0 + l;
    const bool ok = t < M && line < R.nline;
    cpx<T>* base = R.rows + min(line, R.nline - 1) * ls;
    cpx<T> x[M], y[S];
    int v = g0;
#pragma unroll
    for (int q = 0; q < M; ++q) {
      x[q] = v < lim ? base[v] : czero<T>();
      v += step;
      v = v >= wrap ? v - wrap : v;
    }
    W::inverse(x, y, t, l, part, E, R.tw);
    if (R.zline) {
      if (ok) {
#pragma unroll
        for (int u = 0; u < S; ++u) base[W::rpos(t, u)] = y[u];
      }
    } else {
      each_rpos<W, M, S>(t, line * (int)sizeof(cpx<T>), rowb, [&](int u, int v, int sv) {
        buf_store_s<T>(y[u], rb, ok ? v : kBufOff, sv);
      });
    }
  }
}

// Forward transforms: y lines box plane rb -> LDS rows, z lines LDS -> LDS in place.
// PF: the next columns' box values load during a transform (their registers cost
// a wave per SIMD in FP64 and in the classes above 10, where they are not).
template <typename T, int M, int S, bool PF>
__device__ __forceinline__ void lines_fwd(const LineRun<T>& R, __amdgpu_buffer_rsrc_t rb, int wave, int nw, int lane_) {
  constexpr int N = M * S;
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  const int lane = opaque(lane_);
  const int t = lane / LW, l = lane - t * LW;
  const bool part = t < S;
  typename W::EX* E = reinterpret_cast<typename W::EX*>(R.E);
  const int es = R.zline ? 1 : R.rs, ls = R.zline ? R.rs : 1;
  const int wrap = N * es, step = S * es, lim = R.zline ? N : R.nrow * es;
  int g0 = part ? W::gpos(t, 0) + (R.zline ? 0 : R.off) : 0;
  g0 = (g0 >= N ? g0 - N : g0) * es;
  const int rowb = R.n3 * (int)sizeof(cpx<T>);
  cpx<T> yn[PF ? S : 1];
  auto load = [&](int c0, cpx<T>* yn) {  // a column group's box values (masked lanes read zero)
    const int line = c0 + l;
    const bool ok = t < M && line < R.nline;
    each_rpos<W, M, S>(t, line * (int)sizeof(cpx<T>), rowb, [&](int u, int v, int sv) {
      yn[u] = buf_load_s<T>(rb, ok ? v : kBufOff, sv);
    });
  };
  const int c00 = wave * LW;
  if constexpr (PF) {
    if (!R.zline && c00 < R.nline) load(c00, yn);
  }
  for (int c0 = c00; c0 < R.nline; c0 += nw * LW) {
    const int line = c0 + l;
    cpx<T>* base = R.rows + min(line, R.nline - 1) * ls;
    cpx<T> x[M], y[S];
    if (R.zline) {
      const int tm = min(t, M - 1);
#pragma unroll
      for (int u = 0; u < S; ++u) y[u] = base[W::rpos(tm, u)];
    } else if constexpr (PF) {
#pragma unroll
      for (int u = 0; u < S; ++u) y[u] = yn[u];
      if (c0 + nw * LW < R.nline) load(c0 + nw * LW, yn);
    } else {
      load(c0, y);
    }
    W::forward(y, x, t, l, part, E, R.tw);
    if (part && line < R.nline) {
      int v = g0;
#pragma unroll
      for (int q = 0; q < M; ++q) {
        if (v < lim) base[v] = x[q];
        v += step;
        v = v >= wrap ? v - wrap : v;
      }
    }
  }
}

template <typename T, int SM, bool INV>
__device__ __forceinline__ void lines_any(int n, const LineRun<T>& R, __amdgpu_buffer_rsrc_t rb, int wave, int nw,
                                          int lane) {
#define GW_CASE(M, S)                                                        \
  case (M) * (S):                                                            \
    if constexpr ((S) <= SM) {                                               \
      if constexpr (INV) lines_inv<T, M, S>(R, rb, wave, nw, lane);          \
      else lines_fwd<T, M, S, sizeof(T) == 4 && SM <= 10>(R, rb, wave, nw, lane);                        \
    }                                                                        \
    break;
  switch (n) {
    GW_WAVE_SMALL(GW_CASE)
    GW_WAVE_LARGE(GW_CASE)
    default: break;
  }
#undef GW_CASE
}

// LDS: exchange areas (nw x emax elements of 8 bytes), y and z twiddles, stick rows
template <typename T, int SM, bool LOOP>
__device__ __forceinline__ void plane_inv_any_body(const Geom& g, const PlaneItem& it, int emax,
                                                   const cpx<T>* __restrict__ c, long ldc, long sc,
                                                   cpx<T>* __restrict__ box, const cpx<T>* __restrict__ twyg,
                                                   const cpx<T>* __restrict__ twzg, unsigned char* smem) {
  constexpr int KB = 4;
  const int NT = blockDim.x, nw = NT >> 6;
  cpx<T>* twy = reinterpret_cast<cpx<T>*>(smem + (size_t)nw * emax * 8);
  cpx<T>* twz = twy + g.n2;
  cpx<T>* rows = twz + g.n3;
  const int a = it.a, k = it.k;
  const int* sp = g.st_plane_ptr + (long)k * (g.na + 1);
  const int s0 = sp[a], s1 = sp[a + 1];
  const int* pp = g.st_pt_ptr + (long)k * (g.nst_max + 1);
  const int* src = g.pt_src + (long)k * g.npw_max;
  const int* prow = g.pt_row + (long)k * g.npw_max;
  const int nrow = g.st_nrow[(long)k * g.na + a];
  const cpx<T>* ck = c + (long)k * sc;
  const int p0 = pp[s0], p1 = pp[s1];
  const int q0 = p0 + threadIdx.x;
  // the plane's points in batches of KB per thread, their loads in flight together
  // (from clamped in-range slots; an empty plane reads slot 0 and places nothing)
  int pv[KB], si[KB];
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int q = p1 > p0 ? min(q0 + i * NT, p1 - 1) : 0;
    pv[i] = prow[q];
    si[i] = src[q];
  }
  T pr[KB], pim[KB];
  gather_points<T, KB>(ck + (long)it.b0 * ldc, si, pr, pim);
  for (int i = threadIdx.x; i < g.n2; i += NT) twy[i] = twyg[i];
  for (int i = threadIdx.x; i < g.n3; i += NT) twz[i] = twzg[i];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  LineRun<T> R;
  R.rows = rows; R.rs = g.n3 | 1; R.nrow = nrow; R.off = g.st_off[(long)k * g.na + a];
  R.E = smem + (size_t)wave * emax * 8;
  R.n3 = g.n3;
  const int n23 = g.n2 * g.n3;
  const int b_end = LOOP ? it.b1 : it.b0 + 1;  // one band per item unless LOOP
  for (int b = it.b0; b < b_end; ++b) {
    const cpx<T>* cb = ck + (long)b * ldc;
    for (int e = threadIdx.x; e < nrow * R.rs; e += NT) rows[e] = czero<T>();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KB; ++i)
      if (q0 + i * NT < p1) rows[pv[i]] = cpx<T>{pr[i], pim[i]};
    for (int qq = q0 + KB * NT; qq < p1; qq += KB * NT) {  // planes of more than KB * NT points
      int v2[KB], s2[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int q = min(qq + i * NT, p1 - 1);
        v2[i] = prow[q];
        s2[i] = src[q];
      }
      T r2[KB], i2[KB];
      gather_points<T, KB>(cb, s2, r2, i2);
#pragma unroll
      for (int i = 0; i < KB; ++i)
        if (qq + i * NT < p1) rows[v2[i]] = cpx<T>{r2[i], i2[i]};
    }
    __syncthreads();
    if (LOOP && b + 1 < b_end) gather_points<T, KB>(cb + ldc, si, pr, pim);  // the next band's first batch
    const auto rb = buf_rsrc(box + (((long)k * g.nb + b) * g.na + a) * n23, (unsigned)(n23 * (int)sizeof(cpx<T>)));
#pragma nounroll
    for (int ph = 0; ph < 2; ++ph) {  // z rows, then y columns: one copy of the transforms
      R.zline = ph == 0;
      R.nline = ph == 0 ? nrow : g.n3;
      R.tw = ph == 0 ? twz : twy;
      lines_any<T, SM, true>(ph == 0 ? g.n3 : g.n2, R, rb, wave, nw, lane);
      __syncthreads();
    }
  }
}

template <typename T, int SM, bool LOOP>
__device__ __forceinline__ void plane_fwd_any_body(const Geom& g, const PlaneItem& it, int emax,
                                                   const cpx<T>* __restrict__ box, const cpx<T>* __restrict__ c,
                                                   long ldc, long sc, const T* __restrict__ tk_all,
                                                   cpx<T>* __restrict__ out, long ldo, long so, T scale, bool kin,
                                                   const cpx<T>* __restrict__ twyg, const cpx<T>* __restrict__ twzg,
                                                   unsigned char* smem) {
  constexpr int KB = 2;
  const int NT = blockDim.x, nw = NT >> 6;
  cpx<T>* twy = reinterpret_cast<cpx<T>*>(smem + (size_t)nw * emax * 8);
  cpx<T>* twz = twy + g.n2;
  cpx<T>* rows = twz + g.n3;
  const int a = it.a, k = it.k;
  if (a == 0) {  // padded slots of these bands are zero (reference: out * mask)
    for (int b = it.b0; b < it.b1; ++b) {
      cpx<T>* ob = out + (long)k * so + (long)b * ldo;
      for (int q = g.npw[k] + threadIdx.x; q < g.npw_max; q += NT) ob[q] = czero<T>();
    }
  }
  const int* sp = g.st_plane_ptr + (long)k * (g.na + 1);
  const int s0 = sp[a], s1 = sp[a + 1];
  if (s1 == s0) return;
  const int* pp = g.st_pt_ptr + (long)k * (g.nst_max + 1);
  const int* src = g.pt_src + (long)k * g.npw_max;
  const int* prow = g.pt_row + (long)k * g.npw_max;
  const cpx<T>* ck = c + (long)k * sc;
  const T* tk = tk_all + (long)k * g.npw_max;
  const int p0 = pp[s0], p1 = pp[s1];  // p1 > p0: the plane has sticks, each with points
  const int q0 = p0 + threadIdx.x;
  int gs[KB], gv[KB];
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int q = min(q0 + i * NT, p1 - 1);
    gs[i] = src[q];
    gv[i] = prow[q];
  }
  // the first band's t c, loaded now so its latency overlaps the transforms
  T gr[KB], gi[KB], tt[KB];
#pragma unroll
  for (int i = 0; i < KB; ++i) tt[i] = gr[i] = gi[i] = T(0);
  if (kin) {
#pragma unroll
    for (int i = 0; i < KB; ++i) tt[i] = tk[gs[i]];
    gather_points<T, KB>(ck + (long)it.b0 * ldc, gs, gr, gi);
  }
  for (int i = threadIdx.x; i < g.n2; i += NT) twy[i] = twyg[i];
  for (int i = threadIdx.x; i < g.n3; i += NT) twz[i] = twzg[i];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  LineRun<T> R;
  R.rows = rows; R.rs = g.n3 | 1; R.nrow = g.st_nrow[(long)k * g.na + a]; R.off = g.st_off[(long)k * g.na + a];
  R.E = smem + (size_t)wave * emax * 8;
  R.n3 = g.n3;
  const int n23 = g.n2 * g.n3;
  __syncthreads();  // twiddles
  const int b_end = LOOP ? it.b1 : it.b0 + 1;
  for (int b = it.b0; b < b_end; ++b) {
    const cpx<T>* cb = ck + (long)b * ldc;
    cpx<T>* ob = out + (long)k * so + (long)b * ldo;
    const auto rb = buf_rsrc(box + (((long)k * g.nb + b) * g.na + a) * n23, (unsigned)(n23 * (int)sizeof(cpx<T>)));
#pragma nounroll
    for (int ph = 0; ph < 2; ++ph) {  // y columns, then z rows
      R.zline = ph == 1;
      R.nline = ph == 1 ? R.nrow : g.n3;
      R.tw = ph == 1 ? twz : twy;
      lines_any<T, SM, false>(ph == 1 ? g.n3 : g.n2, R, rb, wave, nw, lane);
      __syncthreads();
    }
    auto put = [&](int s, int v, cpx<T> kc) {
      cpx<T> r = rows[v];
      r.x = r.x * scale + kc.x;
      r.y = r.y * scale + kc.y;
      ob[s] = r;
    };
#pragma unroll
    for (int i = 0; i < KB; ++i)
      if (q0 + i * NT < p1) put(gs[i], gv[i], cpx<T>{tt[i] * gr[i], tt[i] * gi[i]});
    if (LOOP && kin && b + 1 < b_end) gather_points<T, KB>(cb + ldc, gs, gr, gi);  // the next band's first batch
    for (int q = q0 + KB * NT; q < p1; q += NT) {  // planes of more than KB * NT points
      const int s = src[q];
      cpx<T> kc = czero<T>();
      if (kin) { const cpx<T> cv = cb[s]; const T tv = tk[s]; kc.x = tv * cv.x; kc.y = tv * cv.y; }
      put(s, prow[q], kc);
    }
    __syncthreads();  // the rows are rewritten for the next band
  }
}

// Waves per SIMD the kernels are compiled for: 4 (128 registers) unless the class's
// largest codelets would spill more than a few.
template <typename T, int SM, bool LOOP, bool INV> constexpr int any_waves() {
  if (sizeof(T) == 4) return 4;
  return INV ? (LOOP && SM > 8 ? 3 : 4) : (SM > 8 ? 3 : 4);
}

template <typename T, int SM, bool LOOP>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(any_waves<T, SM, LOOP, true>())))
k_plane_inv_any(Geom g, int emax, long total, int bpw, const cpx<T>* __restrict__ c, long ldc, long sc,
                cpx<T>* __restrict__ box, const cpx<T>* __restrict__ twy, const cpx<T>* __restrict__ twz) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  plane_inv_any_body<T, SM, LOOP>(g, plane_item(wid, g.na, g.nb, bpw), emax, c, ldc, sc, box, twy, twz, smem_raw);
}

template <typename T, int SM, bool LOOP>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(any_waves<T, SM, LOOP, false>())))
k_plane_fwd_any(Geom g, int emax, long total, int bpw, const cpx<T>* __restrict__ box, const cpx<T>* __restrict__ c,
                long ldc, long sc, const T* __restrict__ t, cpx<T>* __restrict__ out, long ldo, long so, T scale,
                int kin, const cpx<T>* __restrict__ twy, const cpx<T>* __restrict__ twz) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  plane_fwd_any_body<T, SM, LOOP>(g, plane_item(wid, g.na, g.nb, bpw), emax, box, c, ldc, sc, t, out, ldo, so, scale, kin,
                            twy, twz, smem_raw);
}

// ---- ragged batches: one launch over every cell's (plane, band) items ----
template <typename T> __device__ __forceinline__ PlaneItem rag_item(const RagInst<T>& d, long local) {
  PlaneItem it;
  it.a = (int)(local % d.g.na);
  const int bi = (int)(local / d.g.na);
  it.k = bi / d.g.nb;
  it.b0 = bi - it.k * d.g.nb;
  it.b1 = it.b0 + 1;
  return it;
}

template <typename T, int SM>
__global__ void __launch_bounds__(64 * kRagWaves) __attribute__((amdgpu_waves_per_eu(any_waves<T, SM, false, true>())))
k_plane_inv_rag_any(const RagInst<T>* __restrict__ R, int n, long total) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long w = xcd_work_id(total);
  if (w < 0) return;
  const RagInst<T>& d = R[rag_find(R, n, w, false)];
  plane_inv_any_body<T, SM, false>(d.g, rag_item(d, w - d.w13), d.emax, d.c, d.ldc, d.sc, d.box, d.twy, d.twz,
                                   smem_raw);
}

template <typename T, int SM>
__global__ void __launch_bounds__(64 * kRagWaves) __attribute__((amdgpu_waves_per_eu(any_waves<T, SM, false, false>())))
k_plane_fwd_rag_any(const RagInst<T>* __restrict__ R, int n, long total) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const long w = xcd_work_id(total);
  if (w < 0) return;
  const RagInst<T>& d = R[rag_find(R, n, w, false)];
  plane_fwd_any_body<T, SM, false>(d.g, rag_item(d, w - d.w13), d.emax, d.box, d.c, d.ldc, d.sc, d.t, d.out, d.ldo,
                                   d.so, d.scale, d.kin != 0, d.twy, d.twz, smem_raw);
}

// ------------------------------------------------------------------ host

template <typename T> static size_t any_plane_lds(const Geom& g, int emax, int nw) {
  return (size_t)nw * emax * 8 + ((size_t)g.n2 + g.n3 + (size_t)g.rows_max * (g.n3 | 1)) * sizeof(cpx<T>);
}

// Waves per plane workgroup (8, 4 or 2) and the exchange elements per wave: the
// count whose LDS keeps the most waves resident per CU, no more than the y and z
// lines keep busy, the larger on a tie; 0 if none fits.
template <typename T> static int any_plane_waves(const Geom& g, size_t cap, int* emax) {
  int lwy = 1, ey = 0, lwz = 1, ez = 0, sm;
  if (!wave_any_info(g.n2, &lwy, &ey, &sm) || !wave_any_info(g.n3, &lwz, &ez, &sm)) return 0;
  *emax = std::max(ey, ez);
  const int busy = std::max(1, std::max((g.n3 + lwy - 1) / lwy, (g.rows_max + lwz - 1) / lwz));
  int best = 0, best_res = 0;
  for (int nw : {8, 4, 2}) {
    if (nw > 2 && nw / 2 >= busy) continue;
    const size_t lds = any_plane_lds<T>(g, *emax, nw);
    if (lds > cap) continue;
    const int res = std::min(16, nw * (int)(kLdsPerCu / lds));
    if (res > best_res) { best = nw; best_res = res; }
  }
  return best;
}

template <typename T>
int wave_any_planes(bool inv, const Plan& P, const Geom& g, int nk, const cpx<T>* c, long ldc, long sc, cpx<T>* box,
                    const T* t, cpx<T>* out, long ldo, long so, T scale, bool kin, hipStream_t st) {
  int emax = 0;
  const int nw = any_plane_waves<T>(g, (size_t)std::min(P.lds_max, kMaxLds), &emax);
  GW_REQUIRE(nw > 0, GW_ERR_UNSUPPORTED, "x-plane sticks exceed LDS");
  const size_t lds = any_plane_lds<T>(g, emax, nw);
  // one workgroup per CU: four bands in turn (one band's stores drain and the next
  // band's points load while a band transforms), else one
  const int knob = plane_bands_knob(sizeof(T) == 4, inv);
  const int bpw = std::min(g.nb, knob > 0 ? knob : kLdsPerCu / lds <= 1 ? 4 : 1);
  const long items = (long)g.na * nk * ((g.nb + bpw - 1) / bpw);
  const dim3 grid((unsigned)(8 * ((items + 7) / 8)));
  const cpx<T>*twy = tw_of<T>(&P, 1), *twz = tw_of<T>(&P, 2);
  int lw, es, sy = 0, sz = 0;
  (void)wave_any_info(g.n2, &lw, &es, &sy);
  (void)wave_any_info(g.n3, &lw, &es, &sz);
  auto go = [&](auto smc, auto loop) {
    constexpr int SM = decltype(smc)::value;
    constexpr bool L = decltype(loop)::value;
    if (inv)
      hipLaunchKernelGGL((k_plane_inv_any<T, SM, L>), grid, dim3(64 * nw), lds, st, g, emax, items, bpw, c, ldc, sc, box,
                         twy, twz);
    else
      hipLaunchKernelGGL((k_plane_fwd_any<T, SM, L>), grid, dim3(64 * nw), lds, st, g, emax, items, bpw, box, c, ldc, sc,
                         t, out, ldo, so, scale, kin ? 1 : 0, twy, twz);
  };
  auto pick = [&](auto loop) {
    const int s = std::max(sy, sz);
    if (s <= 8) go(std::integral_constant<int, 8>{}, loop);
    else if (s <= 10) go(std::integral_constant<int, 10>{}, loop);
    else go(std::integral_constant<int, 16>{}, loop);
  };
  if (bpw > 1) pick(std::true_type{});
  else pick(std::false_type{});
  GW_CHECK_HIP(hipGetLastError());
  return GW_OK;
}

template <typename T> bool wave_planes_fit(const Plan& P) {
  int emax;
  return any_plane_waves<T>(geom_of(&P, 1), (size_t)std::min(P.lds_max, kMaxLds), &emax) > 0;
}

template <typename T> int wave_planes_per_cu(const Plan& P) {
  int emax;
  const Geom g = geom_of(&P, 1);
  const int nw = any_plane_waves<T>(g, (size_t)std::min(P.lds_max, kMaxLds), &emax);
  return nw > 0 ? (int)(kLdsPerCu / any_plane_lds<T>(g, emax, nw)) : 0;
}

template <typename T> size_t wave_rag_plane_lds(const Geom& g, int* emax) {
  int lw, ey = 0, ez = 0, sm;
  if (!wave_any_info(g.n2, &lw, &ey, &sm) || !wave_any_info(g.n3, &lw, &ez, &sm)) return 0;
  *emax = std::max(ey, ez);
  return any_plane_lds<T>(g, *emax, kRagWaves);
}

template <typename T>
int wave_rag_planes(bool inv, int smax, const RagInst<T>* R, int n, long total, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
  auto go = [&](auto smc) {
    constexpr int SM = decltype(smc)::value;
    if (inv)
      hipLaunchKernelGGL((k_plane_inv_rag_any<T, SM>), grid, dim3(64 * kRagWaves), lds, st, R, n, total);
    else
      hipLaunchKernelGGL((k_plane_fwd_rag_any<T, SM>), grid, dim3(64 * kRagWaves), lds, st, R, n, total);
  };
  if (smax <= 10) go(std::integral_constant<int, 10>{});
  else go(std::integral_constant<int, 16>{});
  GW_CHECK_HIP(hipGetLastError());
  return GW_OK;
}

template <typename T, int SM> static void rag_attr(int want) {
  constexpr auto A = hipFuncAttributeMaxDynamicSharedMemorySize;
  (void)hipFuncSetAttribute((const void*)k_plane_inv_rag_any<T, SM>, A, want);
  (void)hipFuncSetAttribute((const void*)k_plane_fwd_rag_any<T, SM>, A, want);
}

template <typename T, int SM, bool L> static void any_attr(int want) {
  constexpr auto A = hipFuncAttributeMaxDynamicSharedMemorySize;
  (void)hipFuncSetAttribute((const void*)k_plane_inv_any<T, SM, L>, A, want);
  (void)hipFuncSetAttribute((const void*)k_plane_fwd_any<T, SM, L>, A, want);
}
template <typename T> void wave_any_attrs(int want) {
  any_attr<T, 8, false>(want); any_attr<T, 8, true>(want);
  any_attr<T, 10, false>(want); any_attr<T, 10, true>(want);
  any_attr<T, 16, false>(want); any_attr<T, 16, true>(want);
  rag_attr<T, 10>(want); rag_attr<T, 16>(want);
}

#define GW_PLANES_INST(T)                                                                                          \
  template int wave_any_planes<T>(bool, const Plan&, const Geom&, int, const cpx<T>*, long, long, cpx<T>*, const T*, \
                                  cpx<T>*, long, long, T, bool, hipStream_t);                                     \
  template void wave_any_attrs<T>(int);                                                                            \
  template bool wave_planes_fit<T>(const Plan&);                                                                   \
  template int wave_planes_per_cu<T>(const Plan&);                                                                 \
  template size_t wave_rag_plane_lds<T>(const Geom&, int*);                                                        \
  template int wave_rag_planes<T>(bool, int, const RagInst<T>*, int, long, size_t, hipStream_t);

}  // namespace gw
