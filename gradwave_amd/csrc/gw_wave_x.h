// x passes on wave lines (gw_regfft.h), shared by the cubic and the any-length
// wave-line paths.
#pragma once

#include "gw_local.h"

namespace gw {

// y V(r), never fused into the transform that follows: the direct and the staged
// pass then round alike whatever the compiler picks around them.
template <typename T> __device__ __forceinline__ cpx<T> times_v(cpx<T> y, T v) {
#pragma clang fp contract(off)
  y.x *= v;
  y.y *= v;
  return y;
}

// P2 with wave-cooperative lines (gw_regfft.h): each x-line is spread over S
// lanes, the transpose between the two DFT passes stays inside the wave's own
// LDS area, V(r) (natural x order) is held in registers across the band group,
// and only the sphere's x-planes are loaded and stored.
template <typename T, int N, int M, int S, int NWX>
__device__ __forceinline__ void xpass_wave_body(const Geom& g, int nbt, int bgroup, int chunk, int bgi,
                                                cpx<T>* __restrict__ box, const T* __restrict__ vx,
                                                const cpx<T>* __restrict__ twx,
                                                typename WaveLine<T, N, M, S>::EX* E, cpx<T>* tw) {
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twx[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = lane / LW, l = lane - t * LW;
  const bool part = t < S;
  const int n23 = g.n2 * g.n3;
  const int j = (chunk * NWX + wave) * LW + l;
  const bool jok = j < n23;
  typename W::EX* Ew = E + wave * W::E_PER_WAVE;
  // the sphere's x-planes are [0, xlo) U [xhi, N)
  auto slot = [&](int i0) { return i0 < g.xlo ? i0 : (i0 >= g.xhi ? g.xlo + i0 - g.xhi : -1); };
  T vr[S];
#pragma unroll
  for (int s = 0; s < S; ++s) vr[s] = (t < M && jok) ? vx[(long)W::rpos(t, s) * n23 + j] : T(0);
  // byte offsets of this lane's elements inside one band's planes (kBufOff: none)
  int off[M];
#pragma unroll
  for (int q = 0; q < M; ++q) {
    const int sl = part ? slot(W::gpos(t, q)) : -1;
    off[q] = (jok && sl >= 0) ? (sl * n23 + j) * (int)sizeof(cpx<T>) : kBufOff;
  }
  const unsigned band_bytes = (unsigned)((long)g.na * n23 * sizeof(cpx<T>));
  auto load = [&](int bi, cpx<T> (&v)[M]) {
    const auto r = buf_rsrc(box + (long)bi * g.na * n23, band_bytes);
#pragma unroll
    for (int q = 0; q < M; ++q) v[q] = buf_load<T>(r, off[q]);
  };
  const int b0 = bgi * bgroup;
  const int nbg = min(bgroup, nbt - b0);
  if (nbg <= 0) return;
  cpx<T> x[M], xn[M], y[S];
  // The first band's loads complete before the loop, so no load is pending at
  // the loop head; inside, the next band's loads (an empty range after the last
  // band: zeros, no traffic) overlap this band's transforms, and the copy at the
  // end waits for them only, not for this band's stores.
  load(b0, x);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  for (int bg = 0; bg < nbg; ++bg) {
    const int bi = b0 + bg;
    {
      const bool more = bg + 1 < nbg;
      const auto rn = buf_rsrc(box + (long)(more ? bi + 1 : bi) * g.na * n23, more ? band_bytes : 0u);
#pragma unroll
      for (int q = 0; q < M; ++q) xn[q] = buf_load<T>(rn, off[q]);
    }
    W::inverse(x, y, t, l, part, Ew, tw);
#pragma unroll
    for (int s = 0; s < S; ++s) y[s] = times_v<T>(y[s], vr[s]);
    W::forward(y, x, t, l, part, Ew, tw);
    const auto r = buf_rsrc(box + (long)bi * g.na * n23, band_bytes);
#pragma unroll
    for (int q = 0; q < M; ++q) buf_store<T>(x[q], r, off[q]);
#pragma unroll
    for (int q = 0; q < M; ++q) x[q] = xn[q];
  }
}

template <typename T, int N, int M, int S, int NWX = 4>
__global__ void __launch_bounds__(64 * NWX)
k_xpass_wave(Geom g, int nbt, int bgroup, cpx<T>* __restrict__ box, const T* __restrict__ vx,
             const cpx<T>* __restrict__ twx, int nchunk, long total) {
  using W = WaveLine<T, N, M, S>;
  __shared__ __align__(16) typename W::EX E[NWX * W::E_PER_WAVE];
  __shared__ cpx<T> tw[N];
  // neighbouring line chunks share cache lines of every plane row: keep them on one XCD
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  xpass_wave_body<T, N, M, S, NWX>(g, nbt, bgroup, (int)(wid % nchunk), (int)(wid / nchunk), box, vx, twx, E, tw);
}

constexpr int kXTilePad = 0;  // extra elements per row of the staged x-pass tiles (1, 2, 4 measured slower)

// LDS of k_xpass_stage: exchange areas (ex_bytes, a multiple of 16), the n x
// twiddles, two tiles of na + 2 rows. The twiddles take a whole number of pairs, so
// that the tiles start on 16 bytes for odd n too: FP32 tiles move as pairs.
constexpr int stage_tw(int n) { return (n + 1) & ~1; }
inline size_t stage_lds_bytes(int n, int na, int lines, size_t ex_bytes, size_t elem) {
  return ex_bytes + (stage_tw(n) + 2 * (size_t)(na + 2) * (lines + kXTilePad)) * elem;
}

// P2 with the band's sphere planes staged through LDS. A workgroup of NWX waves
// owns a chunk of LC = NWX*LW yz-lines; one band's na planes of that chunk form
// a tile of na rows x LC contiguous elements, which arrives with row-contiguous
// range-checked loads (each wave instruction covers LC-element row segments
// instead of S planes x LW elements) and leaves the same way. Each wave reads its
// LW lines out of the tile (a zero row stands in for the planes outside the
// sphere), transforms them in registers as in k_xpass_wave and writes them back
// in place (a discard row takes the outside planes). Two tiles alternate, so the
// next band's loads are in flight during this band's transforms.
template <typename T, int N, int M, int S, int NWX, bool PAIR = (N % 2 == 0)>
__global__ void __launch_bounds__(64 * NWX)
k_xpass_stage(Geom g, int nbt, int bgroup, cpx<T>* __restrict__ box, const T* __restrict__ vx,
              const cpx<T>* __restrict__ twx, int nchunk, long total) {
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  constexpr int LC = NWX * LW;                  // lines per workgroup
  constexpr int NT = 64 * NWX;
  // FP32 tiles move in pairs of adjacent lines (16-byte accesses): every tile row
  // starts at an even line (PAIR: n2*n3 is even, as LC and j0 are), so a pair never
  // straddles a row or the last line; in LDS the tiles start on 16 bytes and their
  // rows are whole pairs
  constexpr int PK = (sizeof(T) == 4 && LC % 2 == 0 && PAIR) ? 2 : 1;
  using SV = typename std::conditional<PK == 2, cpx2f, cpx<T>>::type;
  constexpr int LCU = LC / PK;                  // staging units per tile row
  constexpr int KS = (N * LCU + NT - 1) / NT;   // staged units per thread (na <= N rows)
  constexpr int LDT = LC + kXTilePad;           // tile row stride
  static_assert(PK == 1 || (LDT % 2 == 0 && (NWX * W::E_PER_WAVE * sizeof(typename W::EX) +
                                             stage_tw(N) * sizeof(cpx<T>)) % sizeof(SV) == 0), "pairs on 16 bytes");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typename W::EX* E = reinterpret_cast<typename W::EX*>(smem_raw);
  cpx<T>* tw = reinterpret_cast<cpx<T>*>(E + NWX * W::E_PER_WAVE);  // E_PER_WAVE is even
  cpx<T>* tiles = tw + stage_tw(N);              // 2 x (na + 2) rows of LC
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  const int chunk = (int)(wid % nchunk), bgi = (int)(wid / nchunk);
  const int b0 = bgi * bgroup;
  const int nbg = min(bgroup, nbt - b0);
  if (nbg <= 0) return;
  const int na = g.na, n23 = g.n2 * g.n3;
  const int tstride = (na + 2) * LDT;            // one tile: rows 0..na-1, zero row na, discard row na+1
  if constexpr (!W::PFA) {
    for (int i = threadIdx.x; i < N; i += NT) tw[i] = twx[i];
  }
  for (int i = threadIdx.x; i < LC; i += NT) {
    tiles[na * LDT + i] = czero<T>();
    tiles[tstride + na * LDT + i] = czero<T>();
  }
  const int j0 = chunk * LC;
  // staging map: thread unit k is tile unit e = threadIdx.x + k*NT = a*LCU + jj/PK
  // <-> box[band][a][j0 + jj .. + PK-1]; units past the tile or the last line are masked
  const int ne = na * LCU;
  const int ks = (ne + NT - 1) / NT;  // staged units per thread actually needed (uniform)
  int soff[KS], tix[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const int e = threadIdx.x + k * NT;
    const int a = e / LCU, jj = (e - a * LCU) * PK;
    soff[k] = (e < ne && j0 + jj < n23) ? (a * n23 + j0 + jj) * (int)sizeof(cpx<T>) : kBufOff;
    tix[k] = e < ne ? a * LDT + jj : 0;
  }
  auto sload = [](__amdgpu_buffer_rsrc_t r, int off) -> SV {
    if constexpr (PK == 2) return buf_load2(r, off);
    else return buf_load<T>(r, off);
  };
  auto sstore = [](SV v, __amdgpu_buffer_rsrc_t r, int off) {
    if constexpr (PK == 2) buf_store2(v, r, off);
    else buf_store<T>(v, r, off);
  };
  const unsigned band_bytes = (unsigned)((long)na * n23 * sizeof(cpx<T>));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = lane / LW, l = lane - t * LW;
  const bool part = t < S;
  const int col = wave * LW + l;
  const bool jok = j0 + col < n23;
  typename W::EX* Ew = E + wave * W::E_PER_WAVE;
  auto slot = [&](int i0) { return i0 < g.xlo ? i0 : (i0 >= g.xhi ? g.xlo + i0 - g.xhi : -1); };
  // tile entries of this lane's elements: read from the zero row, write to the
  // discard row for planes outside the sphere (and idle lanes)
  int rd[M], wr[M];
#pragma unroll
  for (int q = 0; q < M; ++q) {
    const int sl = part ? slot(W::gpos(t, q)) : -1;
    rd[q] = (sl >= 0 ? sl : na) * LDT + min(col, LC - 1);
    wr[q] = (sl >= 0 ? sl : na + 1) * LDT + min(col, LC - 1);
  }
  T vr[S];
#pragma unroll
  for (int s = 0; s < S; ++s) vr[s] = (t < M && jok) ? vx[(long)W::rpos(t, s) * n23 + j0 + col] : T(0);
  SV st[KS];
  {
    const auto r = buf_rsrc(box + (long)b0 * na * n23, band_bytes);
#pragma unroll
    for (int k = 0; k < KS; ++k)
      if (k < ks) st[k] = sload(r, soff[k]);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int e = threadIdx.x + k * NT;
      if (k < ks && e < ne) *reinterpret_cast<SV*>(tiles + tix[k]) = st[k];
    }
  }
  // V(r) and the first tile have landed on every path: no load is pending at the
  // loop head, so the waits inside the loop concern the next band's tile only
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  cpx<T> x[M], y[S];
  for (int bg = 0; bg < nbg; ++bg) {
    const int bi = b0 + bg;
    cpx<T>* cur = tiles + (bg & 1) * tstride;
    cpx<T>* nxt = tiles + ((bg + 1) & 1) * tstride;
    {  // next band's tile entries (an empty range after the last band: zeros, no traffic)
      const bool more = bg + 1 < nbg;
      const auto r = buf_rsrc(box + (long)(more ? bi + 1 : bi) * na * n23, more ? band_bytes : 0u);
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < ks) st[k] = sload(r, soff[k]);
    }
#pragma unroll
    for (int q = 0; q < M; ++q) x[q] = cur[rd[q]];
    W::inverse(x, y, t, l, part, Ew, tw);
#pragma unroll
    for (int s = 0; s < S; ++s) y[s] = times_v<T>(y[s], vr[s]);
    W::forward(y, x, t, l, part, Ew, tw);
#pragma unroll
    for (int q = 0; q < M; ++q) cur[wr[q]] = x[q];
    __syncthreads();
    {
      const auto r = buf_rsrc(box + (long)bi * na * n23, band_bytes);
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < ks) sstore(*reinterpret_cast<const SV*>(cur + tix[k]), r, soff[k]);
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int e = threadIdx.x + k * NT;
      if (k < ks && e < ne) *reinterpret_cast<SV*>(nxt + tix[k]) = st[k];
    }
    __syncthreads();
  }
}

// ---- adjoint of the local term with respect to V(r) ----
// grad_V(r) += (1/N) sum_{k,b} Re[conj(phi(r)) psi(r)], psi = N ifftn(scatter c),
// phi = N ifftn(scatter g): both boxes come from P1, this x-pass finishes the
// two inverse transforms and reduces over a group of bands into partial sums
// [group][x][y*n3 + z] (natural order), summed by k_adjv_reduce.
template <typename T, int N, int M, int S>
__global__ void __launch_bounds__(256)
k_xpass_adjv_wave(Geom g, int nbt, int bgroup, const cpx<T>* __restrict__ boxc, const cpx<T>* __restrict__ boxg,
                  const cpx<T>* __restrict__ twx, int nchunk, long total, double* __restrict__ part) {
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  __shared__ __align__(16) typename W::EX E[4 * W::E_PER_WAVE];
  __shared__ cpx<T> tw[N];
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  const int chunk = (int)(wid % nchunk), bgi = (int)(wid / nchunk);
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twx[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = lane / LW, l = lane - t * LW;
  const bool part_ = t < S;
  const int n23 = g.n2 * g.n3;
  const int j = (chunk * 4 + wave) * LW + l;
  const bool jok = j < n23;
  typename W::EX* Ew = E + wave * W::E_PER_WAVE;
  auto slot = [&](int i0) { return i0 < g.xlo ? i0 : (i0 >= g.xhi ? g.xlo + i0 - g.xhi : -1); };
  double acc[S];
#pragma unroll
  for (int s = 0; s < S; ++s) acc[s] = 0.0;
  const int b0 = bgi * bgroup;
  const int nbg = min(bgroup, nbt - b0);
  for (int bg = 0; bg < nbg; ++bg) {
    const long off = (long)(b0 + bg) * g.na * n23 + j;
    cpx<T> x[M], yc[S], yg[S];
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int sl = part_ ? slot(W::gpos(t, q)) : -1;
      x[q] = (jok && sl >= 0) ? boxc[off + (long)sl * n23] : czero<T>();
    }
    W::inverse(x, yc, t, l, part_, Ew, tw);
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int sl = part_ ? slot(W::gpos(t, q)) : -1;
      x[q] = (jok && sl >= 0) ? boxg[off + (long)sl * n23] : czero<T>();
    }
    W::inverse(x, yg, t, l, part_, Ew, tw);
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] += (double)yg[s].x * yc[s].x + (double)yg[s].y * yc[s].y;
  }
  if (t < M && jok) {
    double* pp = part + (long)bgi * N * n23;
#pragma unroll
    for (int s = 0; s < S; ++s) pp[(long)W::rpos(t, s) * n23 + j] = acc[s];
  }
}

// ---- band density: rho(r) += sum_{k,b} w_kb |psi_kb(r)|^2, psi = N ifftn(scatter c) ----
// (core/batch.py:562-587 without the final 1/volume.) P1 fills the box, this
// x-pass finishes the inverse transform of a group of bands and reduces
// w |psi|^2 in FP64 into partials [group][x][y*n3 + z], summed by k_adjv_reduce.
template <typename T, int N, int M, int S>
__global__ void __launch_bounds__(256)
k_xpass_density_wave(Geom g, int nbt, int bgroup, const cpx<T>* __restrict__ box, const double* __restrict__ wts,
                     const cpx<T>* __restrict__ twx, int nchunk, long total, double* __restrict__ part) {
  using W = WaveLine<T, N, M, S>;
  constexpr int LW = W::LW;
  __shared__ __align__(16) typename W::EX E[4 * W::E_PER_WAVE];
  __shared__ cpx<T> tw[N];
  const long wid = xcd_work_id(total);
  if (wid < 0) return;
  const int chunk = (int)(wid % nchunk), bgi = (int)(wid / nchunk);
  for (int i = threadIdx.x; i < N; i += blockDim.x) tw[i] = twx[i];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = lane / LW, l = lane - t * LW;
  const bool part_ = t < S;
  const int n23 = g.n2 * g.n3;
  const int j = (chunk * 4 + wave) * LW + l;
  const bool jok = j < n23;
  typename W::EX* Ew = E + wave * W::E_PER_WAVE;
  auto slot = [&](int i0) { return i0 < g.xlo ? i0 : (i0 >= g.xhi ? g.xlo + i0 - g.xhi : -1); };
  double acc[S];
#pragma unroll
  for (int s = 0; s < S; ++s) acc[s] = 0.0;
  const int b0 = bgi * bgroup;
  const int nbg = min(bgroup, nbt - b0);
  for (int bg = 0; bg < nbg; ++bg) {
    const long off = (long)(b0 + bg) * g.na * n23 + j;
    const double wb = wts[b0 + bg];
    cpx<T> x[M], y[S];
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int sl = part_ ? slot(W::gpos(t, q)) : -1;
      x[q] = (jok && sl >= 0) ? box[off + (long)sl * n23] : czero<T>();
    }
    W::inverse(x, y, t, l, part_, Ew, tw);
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] += wb * ((double)y[s].x * y[s].x + (double)y[s].y * y[s].y);
  }
  if (t < M && jok) {
    double* pp = part + (long)bgi * N * n23;
#pragma unroll
    for (int s = 0; s < S; ++s) pp[(long)W::rpos(t, s) * n23 + j] = acc[s];
  }
}

}  // namespace gw
