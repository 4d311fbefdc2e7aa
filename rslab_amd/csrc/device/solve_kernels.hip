// Multi-RHS triangular solves on the supernodal panels (gfx950).
//
// Computes x = D_s P L^-T D_bk^-1 L^-1 P^T (D_s b) with b, x row-major n x nrhs,
// as LdltSolver::solve_many (src/numeric/sparse_solver.rs:302-327) around
// solve_ldlt_block (src/dense/ldlt_generic.rs:618-714). The sweeps run level by
// level over the supernode tree directly on the factored panels:
//   forward  : a supernode first gathers its children's terms (which hold
//              their subtrees', children ascending), solves its own unit-lower
//              block (the 2x2 coupling row is D, not L), and leaves its
//              off-diagonal products plus the children's terms on those rows
//              to its parent;
//   D block  : 1x1 / 2x2 inverse per pivot block;
//   backward : a supernode gathers its off-diagonal rows from already solved
//              ancestors, then back-substitutes its own block.
// Every output entry is written by one thread in a fixed order: no atomic
// sums, run-to-run identical.
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <type_traits>

#include "devtypes.hpp"
#include "prof.hpp"
#include "scalar.hpp"

namespace rsl {

constexpr int SNT = 256;
constexpr int RCH = 8;  // right-hand sides per accumulator chunk

template <class T>
__global__ void k_gather_rhs(int32_t n, int32_t nrhs, const int32_t* __restrict__ perm_e,
                             const double* __restrict__ scale, const T* __restrict__ b,
                             T* __restrict__ y) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * nrhs) return;
  int64_t e = idx / nrhs, c = idx % nrhs;
  int32_t u = perm_e[e];
  y[idx] = F<T>::scale(b[(int64_t)u * nrhs + c], scale[u]);
}

template <class T>
__global__ void k_scatter_sol(int32_t n, int32_t nrhs, const int32_t* __restrict__ perm_e,
                              const double* __restrict__ scale, const T* __restrict__ y,
                              T* __restrict__ x) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * nrhs) return;
  int64_t e = idx / nrhs, c = idx % nrhs;
  int32_t u = perm_e[e];
  x[(int64_t)u * nrhs + c] = F<T>::scale(y[idx], scale[u]);
}

// ---------------------------------------------------------------------------
// Own-block and update building blocks. Every loop that reads global memory
// issues its loads as one batch into registers before using them, so a
// workgroup keeps many loads in flight instead of waiting on one at a time.
// ---------------------------------------------------------------------------
constexpr int TB = 64;   // triangular block
constexpr int NWV = SNT / 64;  // waves per workgroup

// lane p's value, made wave-uniform (p wave-uniform)
__device__ inline double lane_bcast(double v, int p) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), p);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), p);
  return __hiloint2double(hi, lo);
}
__device__ inline cplx lane_bcast(cplx v, int p) { return {lane_bcast(v.re, p), lane_bcast(v.im, p)}; }

// sum over the 64 lanes (DPP partial sums inside rows of 16, then across the
// rows); the total lands in lane 63. Fixed order: run-to-run identical.
template <int CTRL, int RM>
__device__ inline double dpp_take(double v) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, RM, 0xF, false);
  hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, RM, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ inline double wave_sum_to63(double v) {
  v = v + dpp_take<0x111, 0xF>(v);
  v = v + dpp_take<0x112, 0xF>(v);
  v = v + dpp_take<0x114, 0xF>(v);
  v = v + dpp_take<0x118, 0xF>(v);
  v = v + dpp_take<0x142, 0xA>(v);
  v = v + dpp_take<0x143, 0xC>(v);
  return v;
}
__device__ inline cplx wave_sum_to63(cplx v) { return {wave_sum_to63(v.re), wave_sum_to63(v.im)}; }

// Stage the strictly lower part of the own block's 64-block at j0 in LDS:
// Ld[p * TB + i] = L[j0+i][j0+p] for i > p, zero elsewhere and on the 2x2
// coupling entries (held in D, not in L).
template <class T>
__device__ void stage_block_lower(const T* P, int64_t h, const uint8_t* two, int j0, int nbk, T* Ld) {
  constexpr int PER = TB * TB / SNT;
  T v[PER];
  uint8_t tw[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x + u * SNT, i = t % TB, p = t / TB;
    const bool in = p < nbk && i < nbk && i > p;
    v[u] = in ? P[(int64_t)(j0 + i) + (int64_t)(j0 + p) * h] : F<T>::zero();
    tw[u] = (in && i == p + 1) ? two[j0 + p] : 0;
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) Ld[threadIdx.x + u * SNT] = tw[u] ? F<T>::zero() : v[u];
  __syncthreads();
}

// Transposed: Lt[p * (TB+1) + i] = L[j0+p][j0+i] for p > i (read along the
// panel's columns, padded against LDS bank conflicts).
template <class T>
__device__ void stage_block_upper(const T* P, int64_t h, const uint8_t* two, int j0, int nbk, T* Lt) {
  constexpr int PER = TB * TB / SNT;
  T v[PER];
  uint8_t tw[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x + u * SNT, p = t % TB, i = t / TB;
    const bool in = p < nbk && i < nbk && p > i;
    v[u] = in ? P[(int64_t)(j0 + p) + (int64_t)(j0 + i) * h] : F<T>::zero();
    tw[u] = (in && p == i + 1) ? two[j0 + i] : 0;
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x + u * SNT, p = t % TB, i = t / TB;
    Lt[p * (TB + 1) + i] = tw[u] ? F<T>::zero() : v[u];
  }
  __syncthreads();
}

// Forward substitution with the staged block: one wave per right-hand side,
// two right-hand sides interleaved per wave; lane i holds y_i and takes
// y_p from lane p once it is final.
template <class T>
__device__ void fwd_block_solve(const T* Ld, int eo, int j0, int nbk, int32_t nrhs, T* y) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t row = eo + j0 + lane;
  for (int c = wv; c < nrhs; c += 2 * NWV) {
    const int c2 = c + NWV;
    const bool two_rhs = c2 < nrhs;
    T y0 = lane < nbk ? y[row * nrhs + c] : F<T>::zero();
    T y1 = (two_rhs && lane < nbk) ? y[row * nrhs + c2] : F<T>::zero();
#pragma unroll 8
    for (int p = 0; p + 1 < nbk; ++p) {
      const T l = Ld[p * TB + lane];
      const T a0 = lane_bcast(y0, p), a1 = lane_bcast(y1, p);
      y0 = y0 - l * a0;
      y1 = y1 - l * a1;
    }
    if (lane < nbk) {
      y[row * nrhs + c] = y0;
      if (two_rhs) y[row * nrhs + c2] = y1;
    }
  }
}

// Back substitution with L^T of the staged block (Lt from stage_block_upper).
template <class T>
__device__ void bwd_block_solve(const T* Lt, int eo, int j0, int nbk, int32_t nrhs, T* y) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t row = eo + j0 + lane;
  for (int c = wv; c < nrhs; c += 2 * NWV) {
    const int c2 = c + NWV;
    const bool two_rhs = c2 < nrhs;
    T y0 = lane < nbk ? y[row * nrhs + c] : F<T>::zero();
    T y1 = (two_rhs && lane < nbk) ? y[row * nrhs + c2] : F<T>::zero();
#pragma unroll 8
    for (int p = nbk - 1; p > 0; --p) {
      const T l = Lt[p * (TB + 1) + lane];
      const T a0 = lane_bcast(y0, p), a1 = lane_bcast(y1, p);
      y0 = y0 - l * a0;
      y1 = y1 - l * a1;
    }
    if (lane < nbk) {
      y[row * nrhs + c] = y0;
      if (two_rhs) y[row * nrhs + c2] = y1;
    }
  }
}

// red[r][k] = sum_{p in [c_lo, c_hi)} L[row0 + r][p] * y[(eo + p) * nrhs + c0 + k]
// for r < nr (<= 64), k < nc (<= RCH). Thread (r, q): columns c_lo + q + 4m,
// 8 of them per batch of 32; the batch's y rows are staged in LDS. zr/zc name one
// entry (relative row, absolute column) read as zero: a 2x2 coupling entry
// that falls outside the diagonal block, or -1.
template <class T>
__device__ void rows_times_y(const T* P, int64_t h, int64_t row0, int nr, int c_lo, int c_hi, int eo,
                             int32_t nrhs, int c0, int nc, const T* __restrict__ y, int zr, int zc, T* ys,
                             T* red) {
  const int r = threadIdx.x & 63, q = threadIdx.x >> 6;
  constexpr int CB = 32;  // columns per batch
  T acc[RCH];
#pragma unroll
  for (int k = 0; k < RCH; ++k) acc[k] = F<T>::zero();
  for (int pb = c_lo; pb < c_hi; pb += CB) {
    const int ncb = min(CB, c_hi - pb);
    // y rows of the batch: CB x RCH values, one per thread
    {
      const int t = threadIdx.x, p = t / RCH, k = t % RCH;
      ys[t] = (p < ncb && k < nc) ? y[(int64_t)(eo + pb + p) * nrhs + c0 + k] : F<T>::zero();
    }
    T l[CB / NWV];
#pragma unroll
    for (int m = 0; m < CB / NWV; ++m) {
      const int p = q + NWV * m;
      l[m] = (r < nr && p < ncb) ? P[(row0 + r) + (int64_t)(pb + p) * h] : F<T>::zero();
      if (r == zr && pb + p == zc) l[m] = F<T>::zero();
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < CB / NWV; ++m) {
      const T* yp = ys + (q + NWV * m) * RCH;
#pragma unroll
      for (int k = 0; k < RCH; ++k) acc[k] = acc[k] + l[m] * yp[k];
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < RCH; ++k) red[(q * 64 + r) * RCH + k] = acc[k];
  __syncthreads();
  // fixed-order sum over the four column groups into group 0's slots
  for (int t = threadIdx.x; t < 64 * RCH; t += SNT) {
    T v = red[t];
    v = v + red[64 * RCH + t];
    v = v + red[2 * 64 * RCH + t];
    v = v + red[3 * 64 * RCH + t];
    red[t] = v;
  }
  __syncthreads();
}

// part[p][k] = sum_{i < nr} L[r0 + i][j0 + p] * x[(eo + r0 + i) * nrhs + c0 + k]
// (transposed product of a 64-row chunk of the own block), p < nbk, k < nc:
// L chunk and x rows staged in LDS, thread (p, k-pair) sums 64 terms.
template <class T>
__device__ void chunk_t_times_x(const T* P, int64_t h, const uint8_t* two, int eo, int j0, int nbk, int r0, int nr,
                                int32_t nrhs, int c0, int nc, const T* __restrict__ y, T* Ls, T* xs, T* out) {
  constexpr int PER = TB * TB / SNT;
  T v[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x + u * SNT, i = t % TB, p = t / TB;
    v[u] = (p < nbk && i < nr) ? P[(int64_t)(r0 + i) + (int64_t)(j0 + p) * h] : F<T>::zero();
  }
  T xv[TB * RCH / SNT];
#pragma unroll
  for (int u = 0; u < TB * RCH / SNT; ++u) {
    const int t = threadIdx.x + u * SNT, i = t / RCH, k = t % RCH;
    xv[u] = (i < nr && k < nc) ? y[(int64_t)(eo + r0 + i) * nrhs + c0 + k] : F<T>::zero();
  }
  // a 2x2 coupling entry (j0+p+1, j0+p) can only sit in this chunk at its
  // first row, when the chunk starts right below the block
  const bool zc = r0 == j0 + nbk && nbk > 0 && two[j0 + nbk - 1];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x + u * SNT, i = t % TB, p = t / TB;
    Ls[i * (TB + 1) + p] = (zc && i == 0 && p == nbk - 1) ? F<T>::zero() : v[u];
  }
#pragma unroll
  for (int u = 0; u < TB * RCH / SNT; ++u) xs[threadIdx.x + u * SNT] = xv[u];
  __syncthreads();
  const int p = threadIdx.x & 63, kq = threadIdx.x >> 6;
  T a0 = F<T>::zero(), a1 = F<T>::zero();
#pragma unroll 8
  for (int i = 0; i < TB; ++i) {
    const T l = Ls[i * (TB + 1) + p];
    a0 = a0 + l * xs[i * RCH + kq];
    a1 = a1 + l * xs[i * RCH + kq + NWV];
  }
  out[p * RCH + kq] = a0;
  out[p * RCH + kq + NWV] = a1;
  __syncthreads();
}

// Forward, gather: own rows of a level's supernodes take the contributions of
// their children (which hold their subtrees'), ascending; 64-row chunks.
template <class T>
__global__ __launch_bounds__(SNT) void k_fgather(DevSym S, DevFac<T> Fc, const int2* __restrict__ items,
                                                 int32_t nrhs, T* __restrict__ y, const T* __restrict__ u) {
  const int2 it = items[blockIdx.x];
  const int s = it.x, r0 = it.y;
  const int w = S.sn_ncol[s], first = S.sn_first[s];
  const int nr = min(64, w - r0);
  for (int t = threadIdx.x; t < nr * nrhs; t += SNT) {
    const int gl = r0 + t % nr, c = t / nr;
    const int g = first + gl;
    const int64_t e = Fc.e_of_g[g];
    T acc = y[e * nrhs + c];
    int64_t q = S.gat_ptr[S.rs_off[s] + gl];
    const int64_t qe = S.gat_ptr[S.rs_off[s] + gl + 1];
    for (; q + 4 <= qe; q += 4) {
      int64_t ix[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) ix[m] = S.gat_idx[q + m];
      T v[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) v[m] = u[ix[m] * nrhs + c];
#pragma unroll
      for (int m = 0; m < 4; ++m) acc = acc - v[m];
    }
    for (; q < qe; ++q) acc = acc - u[S.gat_idx[q] * nrhs + c];
    y[e * nrhs + c] = acc;
  }
}

// Forward own-block solve of a narrow supernode (w <= 32): one workgroup.
template <class T>
__global__ __launch_bounds__(SNT) void k_fwd_tri(DevSym S, DevFac<T> Fc,
                                                 const int32_t* __restrict__ list, int32_t nrhs,
                                                 T* __restrict__ y) {
  __shared__ T Ld[TB * TB];
  __shared__ T ys[64 * RCH];
  __shared__ T red[4 * 64 * RCH];
  const int s = list[blockIdx.x];
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s];
  const T* P = Fc.pool + S.panel_off[s];
  const uint8_t* two = Fc.two + eo;
  for (int j0 = 0; j0 < w; j0 += TB) {
    const int nbk = min(TB, w - j0);
    stage_block_lower(P, h, two, j0, nbk, Ld);
    fwd_block_solve(Ld, eo, j0, nbk, nrhs, y);
    __syncthreads();
    const int rb = j0 + nbk;
    for (int r0 = rb; r0 < w; r0 += 64) {
      const int nr = min(64, w - r0);
      const int zr = (r0 == rb && two[rb - 1]) ? 0 : -1;
      for (int c0 = 0; c0 < nrhs; c0 += RCH) {
        const int nc = min(RCH, nrhs - c0);
        rows_times_y(P, h, r0, nr, j0, rb, eo, nrhs, c0, nc, y, zr, rb - 1, ys, red);
        for (int t = threadIdx.x; t < nr * RCH; t += SNT) {
          const int rr = t / RCH, k = t % RCH;
          if (k < nc) {
            const int64_t o = (int64_t)(eo + r0 + rr) * nrhs + c0 + k;
            y[o] = y[o] - red[rr * RCH + k];
          }
        }
        __syncthreads();
      }
    }
  }
}

// Forward, part 2: u_s = L21 y_own plus the children's terms on the same rows,
// for 64-row chunks of the off-diagonal rows (items are (supernode, row
// offset) pairs of one level). A product thus moves up the tree one parent at
// a time, and a gather has the few children's rows to read instead of every
// descendant's.
template <class T>
__global__ __launch_bounds__(SNT) void k_fwd_update(DevSym S, DevFac<T> Fc,
                                                    const int2* __restrict__ items, int32_t nrhs,
                                                    const T* __restrict__ y, T* u) {
  __shared__ T ys[64 * RCH];
  __shared__ T red[4 * 64 * RCH];
  const int2 it = items[blockIdx.x];
  const int s = it.x, r0 = it.y;
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s];
  const int nr = (int)min<int64_t>(64, h - w - r0);
  const int64_t uo = S.u_off[s] + r0;
  for (int c0 = 0; c0 < nrhs; c0 += RCH) {
    const int nc = min(RCH, nrhs - c0);
    rows_times_y(Fc.pool + S.panel_off[s], h, (int64_t)w + r0, nr, 0, w, eo, nrhs, c0, nc, y, -1, -1, ys, red);
    for (int t = threadIdx.x; t < nr * RCH; t += SNT) {
      const int rr = t / RCH, k = t % RCH;
      if (k < nc) {
        T v = red[rr * RCH + k];
        const int64_t g = S.rs_off[s] + w + r0 + rr;
        for (int64_t q = S.gat_ptr[g]; q < S.gat_ptr[g + 1]; ++q) v = v + u[S.gat_idx[q] * nrhs + c0 + k];
        u[(uo + rr) * nrhs + c0 + k] = v;
      }
    }
    __syncthreads();
  }
}

// y_own[p] -= sum_{i >= w} L[i][p] x[rs[i]] for the 16 columns p0.. of
// supernode s. xs holds RB * RCH values of LDS, is RB row indices. A pass's x
// rows are gathered eight lanes to a row (its RCH values, one 64-byte line),
// their indices shared through is.
constexpr int BW_RB = 512, BW_CW = 4;  // rows per pass, columns per wave
static_assert(RCH == 8, "a gathered x row is one lane octet");
template <class T>
__device__ void bwd_update_cols(const DevSym& S, const DevFac<T>& Fc, int s, int p0, int32_t nrhs,
                                T* __restrict__ y, T* xs, int32_t* is) {
  constexpr int RB = BW_RB, CW = BW_CW;
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s], ib0 = w, ie = h;
  const T* P = Fc.pool + S.panel_off[s];
  const int32_t* re = Fc.rs_e + S.rs_off[s];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int pw = p0 + wv * CW;  // this wave's first column
  for (int c0 = 0; c0 < nrhs; c0 += RCH) {
    const int nc = min(RCH, nrhs - c0);
    T acc[CW][RCH];
#pragma unroll
    for (int a = 0; a < CW; ++a)
#pragma unroll
      for (int k = 0; k < RCH; ++k) acc[a][k] = F<T>::zero();
    // row indices of the next pass, loaded one pass ahead (real field; the
    // complex field's registers hold no second set): a pass then waits on
    // one round of loads (its x rows and L entries together)
    constexpr bool AHEAD = sizeof(T) == sizeof(double);
    int32_t en[RB / SNT];
    auto load_idx = [&](int64_t ib) {
#pragma unroll
      for (int q = 0; q < RB / SNT; ++q) {
        const int64_t r = ib + threadIdx.x + q * SNT;
        en[q] = r < ie ? re[r] : -1;
      }
    };
    if (AHEAD) load_idx(ib0);
    for (int64_t ib = ib0; ib < ie; ib += RB) {
      const int nr = (int)min<int64_t>(RB, ie - ib);
      if (!AHEAD) load_idx(ib);
#pragma unroll
      for (int q = 0; q < RB / SNT; ++q) is[threadIdx.x + q * SNT] = en[q];
      __syncthreads();
      // x rows of the pass: thread t takes row t / 8 + 32 q, value t % 8
      constexpr int XR = RB * RCH / SNT;
      const int xk = threadIdx.x & 7, xr0 = threadIdx.x >> 3;
      T xv[XR];
#pragma unroll
      for (int q = 0; q < XR; ++q) {
        const int32_t ee = is[xr0 + 32 * q];
        xv[q] = (ee >= 0 && xk < nc) ? y[(int64_t)ee * nrhs + c0 + xk] : F<T>::zero();
      }
      auto stage_x = [&]() {
#pragma unroll
        for (int q = 0; q < XR; ++q) xs[xk * RB + xr0 + 32 * q] = xv[q];  // [k][row]
      };
      // complex field: x staged before the L loads (registers)
      if (!AHEAD) stage_x();
      T l[RB / 64][CW];
#pragma unroll
      for (int sb = 0; sb < RB / 64; ++sb)
#pragma unroll
        for (int a = 0; a < CW; ++a) {
          const int ir = sb * 64 + lane, p = pw + a;
          l[sb][a] = (ir < nr && p < w) ? P[(ib + ir) + (int64_t)p * h] : F<T>::zero();
        }
      if (AHEAD && ib + RB < ie) load_idx(ib + RB);
      if (AHEAD) stage_x();
      __syncthreads();
#pragma unroll
      for (int sb = 0; sb < RB / 64; ++sb) {
        T xr[RCH];
#pragma unroll
        for (int k = 0; k < RCH; ++k) xr[k] = xs[k * RB + sb * 64 + lane];
#pragma unroll
        for (int a = 0; a < CW; ++a)
#pragma unroll
          for (int k = 0; k < RCH; ++k) acc[a][k] = acc[a][k] + l[sb][a] * xr[k];
      }
      __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < CW; ++a)
#pragma unroll
      for (int k = 0; k < RCH; ++k) {
        const T v = wave_sum_to63(acc[a][k]);
        if (lane == 63 && k < nc && pw + a < w && pw + a < p0 + 16) {
          const int64_t o2 = (int64_t)(eo + pw + a) * nrhs + c0 + k;
          y[o2] = y[o2] - v;
        }
      }
  }
}

// Backward, part 1: y_own[p] -= sum_{i>=w} L[i][p] x[rs[i]] for 16-column
// chunks (items (supernode, column offset)). Lanes run over rows, 512 rows
// per pass (their x rows gathered into LDS; each pass costs a dependent
// gather, so few large passes), each wave owns four columns; the lane
// partial sums (lane l: rows = l mod 64, ascending) are reduced once at the
// end.
template <class T>
__global__ __launch_bounds__(SNT) void k_bwd_update(DevSym S, DevFac<T> Fc,
                                                    const int2* __restrict__ items, int32_t nrhs,
                                                    T* __restrict__ y) {
  __shared__ T xs[BW_RB * RCH];
  __shared__ int32_t is[BW_RB];
  const int2 it = items[blockIdx.x];
  bwd_update_cols(S, Fc, it.x, it.y, nrhs, y, xs, is);
}

// Backward own-block solve of a narrow supernode (w <= 32): one workgroup
// back-substitutes L11^T x = y from the last 64-block up.
template <class T>
__global__ __launch_bounds__(SNT) void k_bwd_tri(DevSym S, DevFac<T> Fc,
                                                 const int32_t* __restrict__ list, int32_t nrhs,
                                                 T* __restrict__ y) {
  __shared__ T Lt[TB * (TB + 1)];
  __shared__ T xs[TB * RCH];
  __shared__ T out[TB * RCH];
  const int s = list[blockIdx.x];
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s];
  const T* P = Fc.pool + S.panel_off[s];
  const uint8_t* two = Fc.two + eo;
  const int nblk = (w + TB - 1) / TB;
  for (int b = nblk - 1; b >= 0; --b) {
    const int j0 = b * TB, nbk = min(TB, w - j0), jend = j0 + nbk;
    // contributions of the already solved own rows below this block
    for (int r0 = jend; r0 < w; r0 += 64) {
      const int nr = min(64, w - r0);
      for (int c0 = 0; c0 < nrhs; c0 += RCH) {
        const int nc = min(RCH, nrhs - c0);
        chunk_t_times_x(P, h, two, eo, j0, nbk, r0, nr, nrhs, c0, nc, y, Lt, xs, out);
        for (int t = threadIdx.x; t < nbk * RCH; t += SNT) {
          const int p = t / RCH, k = t % RCH;
          if (k < nc) {
            const int64_t o = (int64_t)(eo + j0 + p) * nrhs + c0 + k;
            y[o] = y[o] - out[t];
          }
        }
        __syncthreads();
      }
    }
    stage_block_upper(P, h, two, j0, nbk, Lt);
    bwd_block_solve(Lt, eo, j0, nbk, nrhs, y);
    __syncthreads();
  }
}

// ---- wide supernodes: one launch per 64-column block step ----
// Every unit of a step solves the step's diagonal block itself (its y rows
// are read only within the launch) into LDS; the diagonal unit stores it in z,
// and the other units apply it: forward to 64 own rows below the block,
// backward (push form) to an earlier own block. z is copied back to y once
// the level's steps are done.

// A step issues every global load of a right-hand-side chunk (the diagonal
// block, its y entries, the unit's 64 x 64 L operand and the y entries it
// updates) before using any of them, so one memory latency covers the step
// instead of one per phase. Arithmetic per unit: the block solve is
// fwd/bwd_block_solve's (lane i holds y_i, one pair of right-hand sides per
// wave); a forward row unit sums L[r][j0 + p] * y_p over 32-column batches
// (thread (r, q) on columns q + 4m, then a fixed-order sum over q), as
// rows_times_y; a backward push unit sums L[j0 + i][i0 + p] * x_i over the
// block's 64 rows in order, as chunk_t_times_x.
static_assert(RCH == 2 * NWV, "one pair of right-hand sides per wave and chunk");
constexpr int TPER = TB * TB / SNT;  // 64 x 64 block entries per thread

// forward step: units [0, nu) are row units (s, j0, r0), the rest diagonal units
template <class T>
__global__ __launch_bounds__(SNT) void k_ftri_step(DevSym S, DevFac<T> Fc, const SItem* __restrict__ items, int nu,
                                                   int32_t nrhs, T* __restrict__ y, T* __restrict__ z) {
  __shared__ T Ld[TB * TB];
  __shared__ T sb[TB * RCH];
  __shared__ T red[4 * 64 * RCH];
  const SItem it = items[blockIdx.x];
  const bool diag = (int)blockIdx.x >= nu;
  const int s = it.s, j0 = it.j0;
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s];
  const T* P = Fc.pool + S.panel_off[s];
  const uint8_t* two = Fc.two + eo;
  const int nbk = min(TB, w - j0), rb = j0 + nbk;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // the block's strict lower part (stage_block_lower's entries)
  T vst[TPER];
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int t = tid + u * SNT, i = t % TB, p = t / TB;
    const bool in = p < nbk && i < nbk && i > p && !(i == p + 1 && two[j0 + p]);
    vst[u] = in ? P[(int64_t)(j0 + i) + (int64_t)(j0 + p) * h] : F<T>::zero();
  }
  // row unit: L[r0 + r][j0 + p] for r = lane, p = pb + wv + NWV m (rows_times_blk's operand)
  const int r0 = diag ? 0 : it.r0, nr = diag ? 0 : min(64, w - r0);
  const int zr = (!diag && r0 == rb && two[rb - 1]) ? 0 : -1;
  T lr[TPER];
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int p = (u / 8) * 32 + wv + NWV * (u % 8);
    lr[u] = (lane < nr && p < nbk) ? P[(int64_t)(r0 + lane) + (int64_t)(j0 + p) * h] : F<T>::zero();
    if (lane == zr && j0 + p == rb - 1) lr[u] = F<T>::zero();
  }
  for (int c0 = 0; c0 < nrhs; c0 += RCH) {
    const int nc = min(RCH, nrhs - c0);
    const int k = wv, k2 = wv + NWV;
    const int64_t brow = eo + j0 + lane;
    T y0 = (k < nc && lane < nbk) ? y[brow * nrhs + c0 + k] : F<T>::zero();
    T y1 = (k2 < nc && lane < nbk) ? y[brow * nrhs + c0 + k2] : F<T>::zero();
    T yr[RCH * 64 / SNT];
#pragma unroll
    for (int u = 0; u < RCH * 64 / SNT; ++u) {
      const int t = tid + u * SNT, rr = t / RCH, kk = t % RCH;
      yr[u] = (rr < nr && kk < nc) ? y[(int64_t)(eo + r0 + rr) * nrhs + c0 + kk] : F<T>::zero();
    }
    if (c0 == 0) {
#pragma unroll
      for (int u = 0; u < TPER; ++u) Ld[tid + u * SNT] = vst[u];
    }
    for (int t = tid; t < TB * RCH; t += SNT) sb[t] = F<T>::zero();
    __syncthreads();
    if (k < nc) {
#pragma unroll 8
      for (int p = 0; p + 1 < nbk; ++p) {
        const T l = Ld[p * TB + lane];
        const T a0 = lane_bcast(y0, p), a1 = lane_bcast(y1, p);
        y0 = y0 - l * a0;
        y1 = y1 - l * a1;
      }
      sb[lane * RCH + k] = y0;
      if (k2 < nc) sb[lane * RCH + k2] = y1;
    }
    __syncthreads();
    if (diag) {
      for (int t = tid; t < nbk * RCH; t += SNT) {
        const int p = t / RCH, kk = t % RCH;
        if (kk < nc) z[(int64_t)(eo + j0 + p) * nrhs + c0 + kk] = sb[t];
      }
    } else {
      T acc[RCH];
#pragma unroll
      for (int kk = 0; kk < RCH; ++kk) acc[kk] = F<T>::zero();
#pragma unroll
      for (int u = 0; u < TPER; ++u) {
        const int pb = (u / 8) * 32, p = pb + wv + NWV * (u % 8);
        if (pb < nbk && p < nbk) {
          const T* yp = sb + p * RCH;
#pragma unroll
          for (int kk = 0; kk < RCH; ++kk) acc[kk] = acc[kk] + lr[u] * yp[kk];
        }
      }
#pragma unroll
      for (int kk = 0; kk < RCH; ++kk) red[(wv * 64 + lane) * RCH + kk] = acc[kk];
      __syncthreads();
      for (int t = tid; t < 64 * RCH; t += SNT) {
        T v = red[t];
        v = v + red[64 * RCH + t];
        v = v + red[2 * 64 * RCH + t];
        v = v + red[3 * 64 * RCH + t];
        red[t] = v;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < RCH * 64 / SNT; ++u) {
        const int t = tid + u * SNT, rr = t / RCH, kk = t % RCH;
        if (rr < nr && kk < nc) y[(int64_t)(eo + r0 + rr) * nrhs + c0 + kk] = yr[u] - red[rr * RCH + kk];
      }
    }
    __syncthreads();
  }
}

// backward step (last block first): units [0, nd) are diagonal units, the
// rest push units (s, j0, i0)
template <class T>
__global__ __launch_bounds__(SNT) void k_btri_step(DevSym S, DevFac<T> Fc, const SItem* __restrict__ items, int nd,
                                                   int32_t nrhs, T* __restrict__ y, T* __restrict__ z) {
  __shared__ T Lt[TB * (TB + 1)];
  __shared__ T sb[TB * RCH];
  __shared__ T out[TB * RCH];
  const SItem it = items[blockIdx.x];
  const bool diag = (int)blockIdx.x < nd;
  const int s = it.s, j0 = it.j0;
  const int w = S.sn_ncol[s], eo = S.e_off[s];
  const int64_t h = S.sn_nrow[s];
  const T* P = Fc.pool + S.panel_off[s];
  const uint8_t* two = Fc.two + eo;
  const int nbk = min(TB, w - j0);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // the block's transposed strict lower part (stage_block_upper's entries)
  T vst[TPER];
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int t = tid + u * SNT, p = t % TB, i = t / TB;
    const bool in = p < nbk && i < nbk && p > i && !(p == i + 1 && two[j0 + i]);
    vst[u] = in ? P[(int64_t)(j0 + p) + (int64_t)(j0 + i) * h] : F<T>::zero();
  }
  // push unit: L[j0 + i][i0 + p] (blk_t_times_sb's operand, rows j0.. of block i0's columns)
  const int i0 = diag ? 0 : it.r0;
  const bool zc = !diag && j0 == i0 + TB && two[i0 + TB - 1];
  T vp[TPER];
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int t = tid + u * SNT, i = t % TB, p = t / TB;
    vp[u] = (!diag && i < nbk) ? P[(int64_t)(j0 + i) + (int64_t)(i0 + p) * h] : F<T>::zero();
    if (zc && i == 0 && p == TB - 1) vp[u] = F<T>::zero();
  }
  for (int c0 = 0; c0 < nrhs; c0 += RCH) {
    const int nc = min(RCH, nrhs - c0);
    const int k = wv, k2 = wv + NWV;
    const int64_t brow = eo + j0 + lane;
    T y0 = (k < nc && lane < nbk) ? y[brow * nrhs + c0 + k] : F<T>::zero();
    T y1 = (k2 < nc && lane < nbk) ? y[brow * nrhs + c0 + k2] : F<T>::zero();
    T yt[RCH * TB / SNT];
#pragma unroll
    for (int u = 0; u < RCH * TB / SNT; ++u) {
      const int t = tid + u * SNT, p = t / RCH, kk = t % RCH;
      yt[u] = (!diag && kk < nc) ? y[(int64_t)(eo + i0 + p) * nrhs + c0 + kk] : F<T>::zero();
    }
#pragma unroll
    for (int u = 0; u < TPER; ++u) {
      const int t = tid + u * SNT, p = t % TB, i = t / TB;
      Lt[p * (TB + 1) + i] = vst[u];
    }
    for (int t = tid; t < TB * RCH; t += SNT) sb[t] = F<T>::zero();
    __syncthreads();
    if (k < nc) {
#pragma unroll 8
      for (int p = nbk - 1; p > 0; --p) {
        const T l = Lt[p * (TB + 1) + lane];
        const T a0 = lane_bcast(y0, p), a1 = lane_bcast(y1, p);
        y0 = y0 - l * a0;
        y1 = y1 - l * a1;
      }
      sb[lane * RCH + k] = y0;
      if (k2 < nc) sb[lane * RCH + k2] = y1;
    }
    __syncthreads();
    if (diag) {
      for (int t = tid; t < nbk * RCH; t += SNT) {
        const int p = t / RCH, kk = t % RCH;
        if (kk < nc) z[(int64_t)(eo + j0 + p) * nrhs + c0 + kk] = sb[t];
      }
      __syncthreads();
    } else {
#pragma unroll
      for (int u = 0; u < TPER; ++u) {
        const int t = tid + u * SNT, i = t % TB, p = t / TB;
        Lt[i * (TB + 1) + p] = vp[u];
      }
      __syncthreads();
      const int p = lane, kq = wv;
      T a0 = F<T>::zero(), a1 = F<T>::zero();
#pragma unroll 8
      for (int i = 0; i < TB; ++i) {
        const T l = Lt[i * (TB + 1) + p];
        a0 = a0 + l * sb[i * RCH + kq];
        a1 = a1 + l * sb[i * RCH + kq + NWV];
      }
      out[p * RCH + kq] = a0;
      out[p * RCH + kq + NWV] = a1;
      __syncthreads();
#pragma unroll
      for (int u = 0; u < RCH * TB / SNT; ++u) {
        const int t = tid + u * SNT, pp = t / RCH, kk = t % RCH;
        if (kk < nc) y[(int64_t)(eo + i0 + pp) * nrhs + c0 + kk] = yt[u] - out[t];
      }
      __syncthreads();
    }
  }
}

// y := z on the own blocks of a level's wide supernodes
template <class T>
__global__ __launch_bounds__(SNT) void k_zcopy(DevSym S, const SItem* __restrict__ items, int32_t nrhs,
                                               const T* __restrict__ z, T* __restrict__ y) {
  const SItem it = items[blockIdx.x];
  const int w = S.sn_ncol[it.s], eo = S.e_off[it.s];
  const int nbk = min(TB, w - it.j0);
  const int64_t base = (int64_t)(eo + it.j0) * nrhs, n = (int64_t)nbk * nrhs;
  for (int64_t t = threadIdx.x; t < n; t += SNT) y[base + t] = z[base + t];
}

template <class T>
__global__ void k_dsolve(int32_t n, int32_t nrhs, const T* __restrict__ d,
                         const T* __restrict__ ds, const uint8_t* __restrict__ two,
                         T* __restrict__ y) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)n * nrhs) return;
  int32_t e = (int32_t)(idx / nrhs), c = (int32_t)(idx % nrhs);
  if (two[e] && e + 1 < n) {
    T d11 = d[e], d21 = ds[e], d22 = d[e + 1];
    T detinv = F<T>::recip(d11 * d22 - d21 * d21);
    T z0 = y[(int64_t)e * nrhs + c], z1 = y[(int64_t)(e + 1) * nrhs + c];
    y[(int64_t)e * nrhs + c] = (d22 * z0 - d21 * z1) * detinv;
    y[(int64_t)(e + 1) * nrhs + c] = (d11 * z1 - d21 * z0) * detinv;
  } else if (!(e > 0 && two[e - 1])) {
    y[idx] = y[idx] * F<T>::recip(d[e]);
  }
}

// ---------------------------------------------------------------------------
// Dependency-driven sweeps: one launch per sweep, one workgroup per unit.
// A unit's workgroup takes a ticket (an atomic counter, so units start in
// plan order whatever order the hardware dispatches workgroups in) and waits
// only on units with earlier tickets, which belong to workgroups that are
// already running or finished; only a chain also waits on the helpers right
// after it. So the launch makes progress wherever one workgroup more than it
// has chunks of right-hand sides is resident: 5 of a card's 256, one a CU. A
// producer publishes a counter with an agent-scope release after its stores; a
// consumer polls it and acquires before reading.
//   forward unit (s, -1): the chain of s, every own 64-row block in order;
//     publishes its block counter = blocks solved;
//   forward unit (s, c), 1 <= c < nblk: helper of own block c -- gather the
//     children's terms (waits for the off-diagonal chunks of every child that
//     has units; they hold their subtrees' terms), subtract the terms of the
//     blocks before c - 2 (waiting for each), leave the result in z, publish by
//     the helper counter = c, in order;
//   forward unit (s, c), c >= nblk: 64 off-diagonal rows of s, u = L21 y_own
//     over every own block, plus the children's terms on those rows (terms are
//     subtracted where they are gathered), publish by its chunk counter += 1;
//   backward off unit (s, -1 - q): once the parent (and so every ancestor)
//     is solved, subtract L21^T x from the own entries of
//     the 16 columns 16q.. (one writer per entry), publish by its counter += 1;
//   backward units (s, c), c = nblk - 1 .. 0: the chain (the first) and the
//     helpers of the transposed own block, blocks counted from the last.
// A chain's tickets come right before its helpers', so only the newest chains
// (one per chunk of right-hand sides) can wait on a helper that has not
// started, and every earlier unit finishes without it.
// Sums run in a fixed order per output entry: run-to-run identical.
// Right-hand sides go DN = 16 at a time, and every chunk of them is a set of units
// and counters of its own in the same launch (up to DEP_CHUNKS): the chunks'
// chains run beside each other, so 64 right-hand sides take little longer
// than 16. (One chain walked once per chunk, or one launch per level and block
// step, which wider solves took before, makes the chain's latency a factor of
// the width: 7.8 ms for 32 right-hand sides on a 36^3 grid.) A ticket
// is unit * chunks + chunk: a unit still waits only on earlier tickets.
// ---------------------------------------------------------------------------
constexpr uint64_t kSpinTicks = 200000000ull;  // 2 s of the 100 MHz constant clock
// counters of supernode s: cnt[s * CSTRIDE + CKINDS * chunk + kind], one 128-byte line per supernode
constexpr int CSTRIDE = 32, CKINDS = 8;
constexpr int CF_BLK = 0, CF_U = 1, CB_BLK = 2, CB_OFF = 3, CF_H = 4, CB_H = 5;
static_assert(DEP_CHUNKS * CKINDS <= CSTRIDE, "a supernode's counters are one line");

__device__ inline int32_t* counter(const SolveSync& sy, int s, int kind) {
  return sy.cnt + (int64_t)s * CSTRIDE + kind;
}

// Poll *p until it reaches target and return the value read. Returns target
// at once when the solve is aborted: this wait or an earlier one of the same
// solve ran past kSpinTicks. A poll is one load; a counter more than one
// step short of its target is polled about every 0.8 us (hundreds of
// waiting workgroups polling at full rate slow every poll down), one step
// short about every 30 ns. The abort word and the clock are read every 32nd
// poll.
__device__ inline int32_t wait_ge(int32_t* p, int32_t target, uint32_t* ctl) {
  int32_t v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (v >= target) return v;
  const uint64_t t0 = (uint64_t)wall_clock64();
  for (uint32_t it = 1;; ++it) {
    if (target - v > 1) __builtin_amdgcn_s_sleep(31);
    else __builtin_amdgcn_s_sleep(1);
    v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v >= target) return v;
    if ((it & 31u) == 0) {
      if (__hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return target;
      if ((uint64_t)wall_clock64() - t0 > kSpinTicks) {
        __hip_atomic_store(ctl + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(ctl + 3, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return target;
      }
    }
  }
}

// The workgroup's stores, then the counter. Every wave waits for its own
// stores to complete before the barrier (the barrier does not wait for
// them); then thread 0 writes the L2 back at agent scope and waits for that
// write-back (an explicit wait: the fence alone is not followed by one when
// an atomic comes next) before it stores / adds the counter. s_waitcnt
// immediate: vmcnt 0, expcnt and lgkmcnt not waited on.
__device__ inline void wg_publish(int32_t* p, int32_t v, bool add) {
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __builtin_amdgcn_s_waitcnt(0x0F70);
    if (add) __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__device__ inline int take_ticket(uint32_t* ctr, int* slot) {
  if (threadIdx.x == 0) *slot = (int)__hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return *slot;
}

// Counters and control words at the start of a solve: zero (the sticky timeout
// count, ctl[3], is kept).
__global__ void k_sync_init(int32_t* __restrict__ cnt, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cnt[i] = 0;
}

// ---- the sweeps' matrix-core operands ----
// A unit's products are 16x16x4 FP64 matrix-core steps: 16 rows by up to 16
// right-hand sides, four terms a step. Lane l holds, for a 16-column group of
// a tile, A(row l % 16, column 4 r + l / 16) in register r = 0..3, the matching
// four right-hand-side rows in B, and rows 4 r + l / 16 of column l % 16 of
// the result: a result's registers are the B operand of the next product, so
// a 64-row block solve chains products without moving data between lanes.
typedef double dv4 __attribute__((ext_vector_type(4)));

template <class T>
struct Acc;
template <>
struct Acc<double> {
  dv4 v = {0.0, 0.0, 0.0, 0.0};
  __device__ double get(int r) const { return v[r]; }
  __device__ void set(int r, double x) { v[r] = x; }
  __device__ void add(const Acc& o) { v += o.v; }
};
template <>
struct Acc<cplx> {
  dv4 re = {0.0, 0.0, 0.0, 0.0}, im = {0.0, 0.0, 0.0, 0.0};
  __device__ cplx get(int r) const { return {re[r], im[r]}; }
  __device__ void set(int r, cplx x) {
    re[r] = x.re;
    im[r] = x.im;
  }
  __device__ void add(const Acc& o) {
    re += o.re;
    im += o.im;
  }
};

// acc += a b
__device__ __forceinline__ void mac(Acc<double>& acc, double a, double b) {
  acc.v = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc.v, 0, 0, 0);
}
__device__ __forceinline__ void mac(Acc<cplx>& acc, cplx a, cplx b) {
  acc.re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, acc.re, 0, 0, 0);
  acc.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, acc.im, 0, 0, 0);
  acc.re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, acc.re, 0, 0, 0);
  acc.im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, acc.im, 0, 0, 0);
}
// acc -= a b
__device__ __forceinline__ void msub(Acc<double>& acc, double a, double b) { mac(acc, -a, b); }
__device__ __forceinline__ void msub(Acc<cplx>& acc, cplx a, cplx b) { mac(acc, cplx{-a.re, -a.im}, b); }

// ---- the own blocks' diagonal 64x64 blocks, as the block solve reads them ----
// Per 64 own columns of a supernode, 14 tiles of 16x16 in operand order
// (register r of lane l at r * 64 + l): the inverses of the four unit-lower
// diagonal tiles, the tiles themselves, and the six below them; entries past
// the last column and 2x2 couplings (held in D) are zero. A last block of nt
// < 4 diagonal tiles has only those: nt inverses, nt tiles, nt (nt - 1) / 2
// below (whole blocks for every narrow supernode of a band made the pack
// several times the panels). The block solve
// multiplies by an inverse instead of substituting row by row. Its operands
// are fetched whole and in order, one instruction a register: read from the
// panel with their addresses and coupling flags, they took the solving wave
// longer than the solve (5 to 14 us a block).
constexpr int PK_INV = 0, PK_UNIT = 1, PK_LOW = 2;
static_assert(PACK_TILE == 256, "16x16 tiles");
// Block c of supernode s starts at tile dep_tile[s] + PACK_TILES * c.
// Place of tile (r, c) of a kind (r == c but for PK_LOW) in a block of nt
// diagonal tiles.
__host__ __device__ constexpr int pack_place(int nt, int kind, int r, int c) {
  return kind == PK_LOW ? 2 * nt + r * (r - 1) / 2 + c : kind * nt + r;
}
static_assert(pack_place(4, PK_LOW, 3, 2) == PACK_TILES - 1, "the last one");
// diagonal tiles of block c of w columns
__host__ __device__ inline int block_tiles(int w, int c) { return w - 64 * c >= 64 ? 4 : (w - 64 * c + 15) / 16; }
// What a tile's inverse needs, two bits a tile in the block's flags. Entries up
// to INV_PLAIN: nothing. Above: one correction with the tile's own residual,
// after which the inverse's rounding is out of the result (on ill-conditioned
// interior-point systems the plain product's backward error was up to 3 times
// that of substitution, the corrected one's is not above it). Above INV_MAX
// (Bunch-Kaufman panels stay below about 10): substitution, since the
// correction only converges while the entries are far below 1 / eps.
constexpr double INV_PLAIN = 1.25, INV_MAX = 64.0;

template <class T>
__global__ __launch_bounds__(SNT) void k_diag_pack(DevSym S, DevFac<T> Fc, const int2* __restrict__ items) {
  __shared__ T Lb[64 * 65];  // row i, column j at i * 65 + j
  __shared__ T Iv[4][16][17];
  __shared__ unsigned flags;
  const int2 it = items[blockIdx.x];
  const int s = it.x, w = S.sn_ncol[s], eo = S.e_off[s], c0 = 64 * it.y;
  const int64_t h = S.sn_nrow[s];
  const T* P = Fc.pool + S.panel_off[s];
  const int tid = threadIdx.x;
#pragma unroll 4
  for (int e = tid; e < 64 * 64; e += SNT) {
    const int i = e & 63, j = e >> 6;
    T v = F<T>::zero();
    if (i > j && c0 + i < w && !(i == j + 1 && Fc.two[eo + c0 + j])) v = P[(c0 + i) + (int64_t)(c0 + j) * h];
    if (i == j && c0 + i < w) v = F<T>::one();
    Lb[i * 65 + j] = v;
  }
  if (tid == 0) flags = 0;
  __syncthreads();
  if (tid < 64) {
    // lane (q, j): column j of tile q's inverse by forward substitution
    const int q = tid >> 4, j = tid & 15;
    T x[16];
    double mx = 0.0;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      T t = i == j ? F<T>::one() : F<T>::zero();
#pragma unroll
      for (int k = 0; k < i; ++k) t = t - Lb[(16 * q + i) * 65 + 16 * q + k] * x[k];
      x[i] = t;
      const double m = F<T>::magsq(t);
      mx = fmax(mx, m);
      bad = bad || !(m <= INV_MAX * INV_MAX);  // (NaN too)
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      Iv[q][i][j] = (c0 + 16 * q + i < w && c0 + 16 * q + j < w) ? x[i] : F<T>::zero();
    if (bad) atomicOr(&flags, 2u << (2 * q));
    else if (mx > INV_PLAIN * INV_PLAIN) atomicOr(&flags, 1u << (2 * q));
  }
  __syncthreads();
  const int64_t first = S.dep_tile[s] + (int64_t)PACK_TILES * it.y;
  const int nt = block_tiles(w, it.y);
  T* out = Fc.dpack + first * PACK_TILE + tid;
  const int m = tid & 15, k = 4 * (tid >> 6) + ((tid & 63) >> 4);  // tid = 64 r + l
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b >= nt) break;
    out[pack_place(nt, PK_INV, b, b) * PACK_TILE] = Iv[b][m][k];
    out[pack_place(nt, PK_UNIT, b, b) * PACK_TILE] = Lb[(16 * b + m) * 65 + 16 * b + k];
#pragma unroll
    for (int c = 0; c < b; ++c) out[pack_place(nt, PK_LOW, b, c) * PACK_TILE] = Lb[(16 * b + m) * 65 + 16 * c + k];
  }
  if (tid == 0) Fc.dflags[first] = flags;
}

// ---- own index order ----
// Both sweeps solve a unit-lower system over the own index a = 0, 1, ... in
// blocks of 64: forward a is the own row, backward a counts the own rows of
// the transposed block from the end (W = w rounded up to blocks; the places
// past w come first and are zero), so one code serves both.
template <class T, bool BWD>
struct Own {
  const T* P;
  const uint8_t* two;
  int64_t h;
  int w, W, eo, tile;  // tile: the diagonal pack's first of own block 0
  __device__ int row(int a) const { return BWD ? W - 1 - a : a; }  // own row of index a (valid if < w)
  __device__ bool valid(int a) const { return row(a) < w; }
  // entry (a, b), a > b
  __device__ T at(int a, int b) const {
    if constexpr (BWD) return row(b) < w ? P[row(b) + (int64_t)row(a) * h] : F<T>::zero();
    else return row(a) < w ? P[row(a) + (int64_t)row(b) * h] : F<T>::zero();
  }
  // own block i counted from the first column, and its first tile in the pack
  __device__ int block(int i) const { return BWD ? W / 64 - 1 - i : i; }
  __device__ int64_t pack(int i) const { return tile + (int64_t)PACK_TILES * block(i); }
  // is entry (b + 1, b) a 2x2 coupling (held in D)?
  __device__ bool coupled(int b) const {
    const int p = BWD ? row(b + 1) : row(b);
    return p >= 0 && p < w && two[p] != 0;
  }
};

constexpr int DNW = 4;             // waves that own rows (16 each)
// and two that solve diagonal blocks in turn. At 197 / 204 registers (256 in the
// complex field) a SIMD holds two waves, so a CU one workgroup of six: units
// that use four waves leave half of it idle, which shows where a level has
// thousands of small supernodes (see solve_split).
constexpr int DNT = 64 * (DNW + 2);
constexpr int DN = DEP_RHS;        // right-hand sides per unit
static_assert(DN == 16, "one column of a matrix-core result each");
constexpr int FKC = 2;             // blocks before its own that the chain subtracts itself
static_assert(FKC == 2, "the chain keeps one middle and one last tile");

// 64 x 16 values in LDS: row i of right-hand side n at i * 16 + n
template <class T>
__device__ __forceinline__ void lds_b(const T* v, int bb, int l, T (&B)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) B[r] = v[(16 * bb + 4 * r + (l >> 4)) * DN + (l & 15)];
}

// Rows 16 q + l % 16 of tile (i, j), j < i, of the own triangle, all 64
// columns, as A operands. No load depends on a lane's place: rows past the end
// read the last one (their results are not kept), and only the backward
// sweep's first block, whose leading places are empty, takes zeros. cp gets 1
// on the lanes whose last entry is a 2x2 coupling (the tile right below the
// diagonal); the caller zeroes it when the tile has arrived.
template <class T, bool BWD>
__device__ __forceinline__ void load_tile(const Own<T, BWD>& O, int i, int j, int q, int l, T (&A)[16], int& cp) {
  const int a = 64 * i + 16 * q + (l & 15), g = l >> 4;
  if constexpr (BWD) {
    const T* p = O.P + (O.W - 1 - 64 * j - g) + (int64_t)(O.W - 1 - a) * O.h;
    if (j > 0 || O.W == O.w) {
#pragma unroll
      for (int k = 0; k < 16; ++k) A[k] = p[-4 * k];
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        A[k] = F<T>::zero();
        if (O.W - 1 - g - 4 * k < O.w) A[k] = p[-4 * k];
      }
    }
  } else {
    const T* p = O.P + min(a, O.w - 1) + (int64_t)(64 * j + g) * O.h;
#pragma unroll
    for (int k = 0; k < 16; ++k) A[k] = p[(int64_t)(4 * k) * O.h];
  }
  const int two = j + 1 == i ? (int)O.coupled(64 * i - 1) : 0;
  cp = two && q == 0 && l == 48;  // row 64 i, column 64 i - 1
}

// The chain's diagonal-block operands of one wave (the diagonal tiles
// themselves only in the real field: the complex field's registers do not hold
// them, and a correction there fetches its tile).
template <class T>
struct DiagOps {
  static constexpr bool UNIT = sizeof(T) == sizeof(double);
  T inv[4][4], unit[UNIT ? 4 : 1][4], low[6][4];
  unsigned flags;
};

// Register r of a lane in tile t of a pack, for tile (row group b2, column
// group b) of the own order's block: the backward order's tile is the
// transposed mirror image of the forward tile (3 - b, 3 - b2).
template <bool BWD>
__device__ __forceinline__ int pack_lane(int l) {
  const int m = 15 - (l & 15);
  return BWD ? (m >> 2) * 64 + (m & 3) * 16 + 15 - (l >> 4) : l;
}
template <class T, bool BWD>
__device__ __forceinline__ const T* pack_block(const Own<T, BWD>& O, const DevFac<T>& Fc, int i, int l) {
  return Fc.dpack + O.pack(i) * PACK_TILE + pack_lane<BWD>(l);
}
// (the forward tile's row and column group: it is there where the row group is)
template <bool BWD>
__device__ __forceinline__ constexpr int pack_row(int b2, int b) {
  return BWD ? 3 - b : b2;
}
template <bool BWD>
__device__ __forceinline__ constexpr int pack_tile(int nt, int kind, int b2, int b) {
  return PACK_TILE * pack_place(nt, kind, pack_row<BWD>(b2, b), BWD ? 3 - b2 : b);
}

template <class T, bool BWD>
__device__ __forceinline__ void load_diag(const Own<T, BWD>& O, const DevFac<T>& Fc, int i, int l,
                                          DiagOps<T>& D) {
  constexpr int st = BWD ? -4 : 64;  // one register on
  const T* v = pack_block(O, Fc, i, l);
  auto tile = [&](int nt, int kind, int b2, int b, T (&x)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = v[pack_tile<BWD>(nt, kind, b2, b) + st * r];
  };
  auto load = [&](int nt, auto&& fetch) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      fetch(nt, PK_INV, b, b, D.inv[b]);
      if constexpr (DiagOps<T>::UNIT) fetch(nt, PK_UNIT, b, b, D.unit[b]);
#pragma unroll
      for (int b2 = b + 1; b2 < 4; ++b2) fetch(nt, PK_LOW, b2, b, D.low[b2 * (b2 - 1) / 2 + b]);
    }
  };
  const int nt = block_tiles(O.w, O.block(i));
  if (nt == 4) {
    load(4, tile);
  } else {
    load(nt, [&](int n, int kind, int b2, int b, T (&x)[4]) {
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = F<T>::zero();
      if (pack_row<BWD>(b2, b) < n) tile(n, kind, b2, b, x);
    });
  }
  D.flags = Fc.dflags[O.pack(i)];
}

// x of L x = b on one 16-row group whose inverse is not used, by substitution
// in place on 16 x 16 values of LDS (one wave).
template <class T, bool BWD>
__device__ __attribute__((noinline)) void substitute16(Own<T, BWD> O, int a0, T* v) {
  const int l = threadIdx.x & 63, n = l & 15;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (l < 16) {
    for (int i = 1; i < 16; ++i) {
      T t = v[i * DN + n];
      for (int k = 0; k < i; ++k) {
        if (k + 1 == i && O.coupled(a0 + k)) continue;
        t = t - O.at(a0 + i, a0 + k) * v[k * DN + n];
      }
      v[i * DN + n] = t;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Chain unit: one workgroup solves every own block of supernode s in order, so
// consecutive blocks pass no counter between workgroups. Block i takes
// t_i = b_i - sum_{j < i-2} L[i, j] y_j from its helper unit (z rows of the
// block, published in block order through `kh`); the four row waves subtract
// the two nearest blocks' terms, y_j from an LDS ring of the last two solved
// blocks, and hand the 64 x 16 values to a solver wave, which chains 16x16
// inverses and products in registers (40 matrix-core steps, and eight more for
// each tile that is corrected). The solver
// waves take turns, so each has a block's time to fetch its next operands; the
// row waves do the farther near term of the next block and fetch its tiles
// meanwhile. One block costs one 64-term product, the block solve and two
// barriers. Block 0's b comes from the caller's `first` values.
// Bound by latency: a block takes 5.1 us in the real field (11 on the vector
// units with the right-hand sides broadcast from LDS and a 64-step
// substitution; 13 with two workgroups handing blocks to each other). The
// forward sweep of one right-hand side on a 48^3 grid, 120 blocks in a row,
// went from 1034 to 758 us, the backward one from 1076 to 905; 32 of them on a
// 36^3 grid from 921 to 531 and from 1071 to 715; a complex 40^3 grid's 16
// from 1909 to 1013 and from 3010 to 1092. A complex block takes 17 us: four
// times the matrix-core work, one set of tiles ahead, and 71 (forward) and 29
// (backward) registers in scratch memory.
template <class T, bool BWD, class Init>
__device__ __forceinline__ void dep_chain(const Own<T, BWD>& O, const DevFac<T>& Fc, const SolveSync& sy, int32_t nrhs, int nc,
                          T* __restrict__ y, const T* __restrict__ z, int s, T* xs, T* ring, Init&& first) {
  constexpr int kb = BWD ? CB_BLK : CF_BLK, kh = BWD ? CB_H : CF_H;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = l & 15, g = l >> 4;
  const int nblk = O.W / 64;
  if (wv < DNW) {
    // tiles (i, i - 1) and (i + 1, i - 1) of iteration i in la[i % NB] and
    // mid[i % NB], loaded NB iterations ahead (the complex field's registers
    // hold one set)
    constexpr int NB = sizeof(T) == sizeof(double) ? 2 : 1;
    T t[4], la[NB][16], mid[NB][16];
    int lc[NB], mc;
    first(t);
    if (nblk > 1) load_tile(O, 1, 0, wv, l, la[1 % NB], lc[1 % NB]);
    if (nblk > 2) load_tile(O, 2, 0, wv, l, mid[1 % NB], mc);
    if (NB > 1 && nblk > 2) load_tile(O, 2, 1, wv, l, la[0], lc[0]);
    if (NB > 1 && nblk > 3) load_tile(O, 3, 1, wv, l, mid[0], mc);
    Acc<T> acc;
    int seen = 0;  // helpers 1 .. seen published and acquired
    auto block = [&](int i, T (&A)[16], int& ac, T (&M)[16]) {
      const T* yr = ring + ((i - 1) & 1) * 64 * DN;
      if (i > 0) {
        if (ac) A[15] = F<T>::zero();
        Acc<T> a0, a1;
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
          T B[4], C[4];
          lds_b(yr, bb, l, B);
          lds_b(yr, bb + 2, l, C);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            msub(a0, A[4 * bb + r], B[r]);
            msub(a1, A[4 * (bb + 2) + r], C[r]);
          }
        }
        a0.add(a1);
        acc.add(a0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) xs[(16 * wv + 4 * r + g) * DN + n] = t[r] + acc.get(r);
      __syncthreads();  // xs is whole
      if (i + 1 < nblk) {
        if (seen < i + 1) {
          int v = 0;
          if (l == 0) v = wait_ge(counter(sy, s, kh), i + 1, sy.ctl);
          seen = __builtin_amdgcn_readfirstlane(v);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        // (loads are used in the order they go out)
        const T* zp = z + (int64_t)O.eo * nrhs + min(n, nc - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          t[r] = zp[(int64_t)min(O.row(64 * (i + 1) + 16 * wv + 4 * r + g), O.w - 1) * nrhs];
        acc = Acc<T>();
        if (i > 0) {
          if (i + NB < nblk) load_tile(O, i + NB, i + NB - 1, wv, l, A, ac);
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) {
            T B[4];
            lds_b(yr, bb, l, B);
#pragma unroll
            for (int r = 0; r < 4; ++r) msub(acc, M[4 * bb + r], B[r]);
          }
          if (i + NB + 1 < nblk) load_tile(O, i + NB + 1, i + NB - 1, wv, l, M, mc);
        }
      }
      __syncthreads();  // y_i is in the ring
    };
    for (int i = 0; i < nblk; i += 2) {
      block(i, la[0], lc[0], mid[0]);
      if (i + 1 < nblk) block(i + 1, la[1 % NB], lc[1 % NB], mid[1 % NB]);
    }
  } else {
    const int mine = wv - DNW;  // blocks of this parity
    DiagOps<T> D;
    if (mine < nblk) load_diag(O, Fc, mine, l, D);
    for (int i = 0; i < nblk; ++i) {
      __syncthreads();
      const bool own = (i & 1) == mine;
      // Row groups in order, each minus the products with the ones before it.
      // The real field keeps all four (a solved group's products with the
      // later ones are independent of each other); the complex field's
      // registers hold one beside the operands, so it reads the values it has
      // solved back from the ring, a lane its own.
      constexpr bool KEEP = DiagOps<T>::UNIT;
      T* yr = ring + (i & 1) * 64 * DN;
      Acc<T> X[KEEP ? 4 : 1];
      auto get = [&](Acc<T>& x, const T* v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x.set(r, v[(4 * r + g) * DN + n]);
      };
      auto put = [&](T* v, const Acc<T>& x) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[(4 * r + g) * DN + n] = x.get(r);
      };
      if (own) {
        if constexpr (KEEP) {
#pragma unroll
          for (int b = 0; b < 4; ++b) get(X[b], xs + 16 * b * DN);
        }
        const int nt = block_tiles(O.w, O.block(i));
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          Acc<T>& x = X[KEEP ? b : 0];
          T* const v = yr + 16 * b * DN;
          // (places without columns: not kept forward, zero backward)
          if (pack_row<BWD>(b, b) >= nt) {
            if constexpr (BWD) put(v, Acc<T>());
            continue;
          }
          // (row group b2's product with group b is entry b2 (b2 - 1) / 2 + b of `low`)
          if constexpr (!KEEP) {
            get(x, xs + 16 * b * DN);
#pragma unroll
            for (int b1 = 0; b1 < b; ++b1)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                msub(x, D.low[b * (b - 1) / 2 + b1][r], yr[(16 * b1 + 4 * r + g) * DN + n]);
          }
          const unsigned need = (D.flags >> (2 * (BWD ? 3 - b : b))) & 3u;
          if (need & 2u) {
            put(v, x);
            substitute16(O, 64 * i + 16 * b, v);
            get(x, v);
          } else {
            Acc<T> p;
#pragma unroll
            for (int r = 0; r < 4; ++r) mac(p, D.inv[b][r], x.get(r));
            if (need) {
              const T* u = pack_block(O, Fc, i, l) + pack_tile<BWD>(nt, PK_UNIT, b, b);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                if constexpr (DiagOps<T>::UNIT) msub(x, D.unit[b][r], p.get(r));
                else msub(x, u[(BWD ? -4 : 64) * r], p.get(r));
              }
#pragma unroll
              for (int r = 0; r < 4; ++r) mac(p, D.inv[b][r], x.get(r));
            }
            x = p;
          }
          if constexpr (KEEP) {
#pragma unroll
            for (int b2 = b + 1; b2 < 4; ++b2)
#pragma unroll
              for (int r = 0; r < 4; ++r) msub(X[b2], D.low[b2 * (b2 - 1) / 2 + b][r], x.get(r));
          }
          put(v, x);
        }
      }
      __syncthreads();
      if (own) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int a = 64 * i + 16 * b + 4 * r + g;
            T v;
            if constexpr (KEEP) v = X[b].get(r);
            else v = yr[(16 * b + 4 * r + g) * DN + n];
            if (O.valid(a) && n < nc) y[(int64_t)(O.eo + O.row(a)) * nrhs + n] = v;
          }
        // this wave wrote the whole block: its stores, the L2, the counter
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __builtin_amdgcn_s_waitcnt(0x0F70);
        if (l == 0) __hip_atomic_store(counter(sy, s, kb), i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (i + 2 < nblk) load_diag(O, Fc, i + 2, l, D);
      }
    }
  }
}

// acc -= sum over blocks j < jn of tile(j) y_j, the blocks taken as they are
// published (four waves; `tile` loads this wave's A operands of block j, the
// right-hand sides come from the solution; none of these tiles touches the
// diagonal). The next block's operands load while the current one multiplies.
template <class T, bool BWD, class Tile>
__device__ __forceinline__ void dep_products(const Own<T, BWD>& O, const SolveSync& sy, int32_t nrhs, int nc,
                                             const T* __restrict__ y, int s, int jn, int* s_ready, Tile&& tile,
                                             Acc<T>& acc) {
  constexpr int kb = BWD ? CB_BLK : CF_BLK;
  const int l = threadIdx.x & 63, n = min(l & 15, nc - 1), g = l >> 4;
  int ready = 0;  // blocks seen solved (and acquired)
  T A[2][16], B[16];
  // (places past the block read its last row: their A entries are zero)
  auto load_y = [&](int j) {
    const T* p = y + (int64_t)O.eo * nrhs + n;
#pragma unroll
    for (int k = 0; k < 16; ++k) B[k] = p[(int64_t)min(O.row(64 * j + 4 * k + g), O.w - 1) * nrhs];
  };
  auto step = [&](int j, T (&Ac)[16], T (&An)[16]) {
    if (j >= ready) {
      if (threadIdx.x == 0) {
        *s_ready = wait_ge(counter(sy, s, kb), j + 1, sy.ctl);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      }
      __syncthreads();
      ready = __builtin_amdgcn_readfirstlane(*s_ready);
      __syncthreads();  // read by all before it is written again
    }
    load_y(j);
    if (j + 1 < jn) tile(j + 1, An);
    // a block's terms are summed apart from the running sum: less rounding
    // than one chain over all of them, and two chains for the matrix core
    Acc<T> a0, a1;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      msub(a0, Ac[k], B[k]);
      msub(a1, Ac[8 + k], B[8 + k]);
    }
    a0.add(a1);
    acc.add(a0);
  };
  if (jn > 0) tile(0, A[0]);
  for (int j = 0; j < jn; j += 2) {
    step(j, A[0], A[1]);
    if (j + 1 < jn) step(j + 1, A[1], A[0]);
  }
}

template <class T>
__global__ __launch_bounds__(DNT) void k_fwd_dep(DevSym S, DevFac<T> Fc, const int2* __restrict__ items, SolveSync sy,
                                                 int32_t nrhs, int first, int chunks, T* __restrict__ y,
                                                 T* __restrict__ u, T* __restrict__ z) {
  __shared__ T xs[64 * DN], ring[2 * 64 * DN];
  __shared__ int s_t, s_ready;
  const int tk = take_ticket(sy.ctl, &s_t), ch = tk % chunks;
  const int2 it = items[tk / chunks];
  const int s = it.x, c = it.y;
  // this unit's right-hand sides: columns 0 .. nc - 1 from here on
  const int rhs0 = first + ch * DN, nc = min(DN, nrhs - rhs0);
  y += rhs0;
  u += rhs0;
  z += rhs0;
  sy.cnt += ch * CKINDS;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = l & 15, g = l >> 4;
  const int w = S.sn_ncol[s], eo = S.e_off[s], nblk = (w + 63) / 64;
  const int64_t h = S.sn_nrow[s];
  const Own<T, false> O{Fc.pool + S.panel_off[s], Fc.two + eo, h, w, 64 * nblk, eo, S.dep_tile[s]};
  // the children's terms on four panel rows of this lane (row r: `rows` + 4 r
  // + g, if `in`), summed in order: GN entries of each row at a time, the
  // first ones' indices loaded before the wait for the children
  constexpr int GN = 2;
  auto gather = [&](int64_t rows, const bool (&in)[4], T (&t)[4]) {
    int64_t q[4], qe[4], ix[4][GN];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      q[r] = qe[r] = 0;
      t[r] = F<T>::zero();
      if (in[r]) {
        const int64_t p = S.rs_off[s] + (rows < 0 ? Fc.lperm[eo + (-1 - rows) + 4 * r + g] : rows + 4 * r + g);
        q[r] = S.gat_ptr[p];
        qe[r] = S.gat_ptr[p + 1];
      }
    }
    auto indices = [&]() {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < GN; ++m) ix[r][m] = q[r] + m < qe[r] ? S.gat_idx[q[r] + m] : -1;
    };
    indices();
    for (int e = S.kid_ptr[s] + l; e < S.kid_ptr[s + 1]; e += 64) {
      const int k = S.kid_idx[e];
      (void)wait_ge(counter(sy, k, CF_U), (S.sn_nrow[k] - S.sn_ncol[k] + 63) / 64, sy.ctl);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    for (;;) {
      bool more = false;
      T v[4][GN];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int m = 0; m < GN; ++m) {
          v[r][m] = F<T>::zero();
          if (ix[r][m] >= 0 && n < nc) v[r][m] = u[ix[r][m] * nrhs + n];
        }
        q[r] += GN;
        more = more || q[r] < qe[r];
      }
      const bool any = __any(more);
      if (any) indices();
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < GN; ++m) t[r] = t[r] + v[r][m];
      if (!any) break;
    }
  };
  // b of own block i: the right-hand side minus the children's terms
  auto block_b = [&](int i, T (&t)[4]) {
    bool in[4];
    T b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int a = 64 * i + 16 * wv + 4 * r + g;
      in[r] = a < w;
      b[r] = F<T>::zero();
      if (in[r] && n < nc) b[r] = y[(int64_t)(eo + a) * nrhs + n];
    }
    gather(-1 - (64 * i + 16 * wv), in, t);
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = b[r] - t[r];
  };
  if (c < 0) {
    dep_chain<T, false>(O, Fc, sy, nrhs, nc, y, z, s, xs, ring, [&](T (&t)[4]) { block_b(0, t); });
    return;
  }
  if (wv >= DNW) return;
  Acc<T> acc;
  if (c < nblk) {
    // helper of block c: b minus the terms of blocks before c - 2, into z
    T t[4];
    block_b(c, t);
    dep_products(O, sy, nrhs, nc, y, s, max(0, c - FKC), &s_ready,
                 [&](int j, T (&A)[16]) { int cp; load_tile(O, c, j, wv, l, A, cp); }, acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int a = 64 * c + 16 * wv + 4 * r + g;
      if (a < w && n < nc) z[(int64_t)(eo + a) * nrhs + n] = t[r] + acc.get(r);
    }
    // helpers publish in block order (the chain waits for CF_H >= c)
    if (threadIdx.x == 0 && c > 1) (void)wait_ge(counter(sy, s, CF_H), c - 1, sy.ctl);
    wg_publish(counter(sy, s, CF_H), c, false);
  } else {
    // 64 off-diagonal rows: u = L21 y over every own block, plus the
    // children's terms on those rows (gathered while the chain runs)
    const int64_t row0 = w + (int64_t)(c - nblk) * 64 + 16 * wv, row = min(row0 + n, h - 1);
    const T* P = O.P;
    bool in[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) in[r] = row0 + 4 * r + g < h;
    T t[4];
    gather(row0, in, t);
    dep_products(O, sy, nrhs, nc, y, s, nblk, &s_ready,
                 [&](int j, T (&A)[16]) {
                   const T* p = P + row + (int64_t)(64 * j + g) * h;
                   if (64 * j + 64 <= w) {
#pragma unroll
                     for (int k = 0; k < 16; ++k) A[k] = p[(int64_t)(4 * k) * h];
                   } else {
#pragma unroll
                     for (int k = 0; k < 16; ++k) {
                       A[k] = F<T>::zero();
                       if (64 * j + 4 * k + g < w) A[k] = p[(int64_t)(4 * k) * h];
                     }
                   }
                 },
                 acc);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (in[r] && n < nc) u[(S.u_off[s] + (row0 - w) + 4 * r + g) * nrhs + n] = t[r] - acc.get(r);
    wg_publish(counter(sy, s, CF_U), 1, true);
  }
}

template <class T>
__global__ __launch_bounds__(DNT) void k_bwd_dep(DevSym S, DevFac<T> Fc, const int2* __restrict__ items, SolveSync sy,
                                                 int32_t nrhs, int first, int chunks, T* __restrict__ y,
                                                 T* __restrict__ u, T* __restrict__ z) {
  __shared__ T xs[64 * DN], ring[2 * 64 * DN];
  __shared__ int s_t, s_ready;
  const int tk = take_ticket(sy.ctl + 1, &s_t), ch = tk % chunks;
  const int2 it = items[tk / chunks];
  const int s = it.x, c = it.y;
  // this unit's right-hand sides: columns 0 .. nc - 1 from here on
  const int rhs0 = first + ch * DN, nc = min(DN, nrhs - rhs0);
  y += rhs0;
  u += rhs0;
  z += rhs0;
  sy.cnt += ch * CKINDS;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = l & 15, g = l >> 4;
  const int w = S.sn_ncol[s], eo = S.e_off[s], nblk = (w + 63) / 64;
  const int64_t h = S.sn_nrow[s];
  const Own<T, true> O{Fc.pool + S.panel_off[s], Fc.two + eo, h, w, 64 * nblk, eo, S.dep_tile[s]};
  const int ng = (w + 15) / 16, nch = bwd_row_chunks(w, h - w);
  if (c < 0) {
    // off unit: the terms of 16 own columns from one chunk of the off-
    // diagonal rows, once the parent (and so every ancestor) is solved; 64 rows
    // a wave and pass, the next pass's row indices loaded with them, and the
    // waves' sums added in order at the end
    if (wv >= DNW) return;
    const int p0 = 16 * ((-1 - c) % ng), rc = (-1 - c) / ng;
    const int64_t ib0 = w + (int64_t)rc * BWD_CHUNK, ie = nch > 1 ? min<int64_t>(h, ib0 + BWD_CHUNK) : h;
    const int32_t* re = Fc.rs_e + S.rs_off[s];
    const T* P = O.P + (int64_t)min(p0 + n, w - 1) * h;  // this lane's column
    const bool col = p0 + n < w;
    int32_t ix[16];
    T A[16];
    auto load_idx = [&](int64_t ib) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int64_t i = ib + 4 * k + g;
        ix[k] = i < ie ? re[i] : -1;
      }
    };
    auto load_a = [&](int64_t ib) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int64_t i = ib + 4 * k + g;
        A[k] = F<T>::zero();
        if (i < ie && col) A[k] = P[i];
      }
    };
    int64_t ib = ib0 + 64 * wv;
    load_idx(ib);
    load_a(ib);
    {
      // (the parent waited for its own ancestors, which hold all these rows)
      const int a = S.parent[s];
      if (l == 0) (void)wait_ge(counter(sy, a, CB_BLK), (S.sn_ncol[a] + 63) / 64, sy.ctl);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    Acc<T> acc;
    for (; ib < ie; ib += 64 * DNW) {
      T B[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        B[k] = F<T>::zero();
        if (ix[k] >= 0 && n < nc) B[k] = y[(int64_t)ix[k] * nrhs + n];
      }
      load_idx(ib + 64 * DNW);
      Acc<T> a0, a1;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        mac(a0, A[k], B[k]);
        mac(a1, A[8 + k], B[8 + k]);
      }
      a0.add(a1);
      acc.add(a0);
      load_a(ib + 64 * DNW);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) xs[256 * wv + (4 * r + g) * DN + n] = acc.get(r);
    __syncthreads();
    {
      const int t = threadIdx.x, p = p0 + t / DN, k = t % DN;
      T v = xs[t];
#pragma unroll
      for (int q = 1; q < DNW; ++q) v = v + xs[256 * q + t];
      if (p < w && k < nc) {
        if (nch > 1) {
          u[(S.u_off[s] + (int64_t)rc * w + p) * nrhs + k] = v;
        } else {
          const int64_t o = (int64_t)(eo + p) * nrhs + k;
          y[o] = y[o] - v;
        }
      }
    }
    wg_publish(counter(sy, s, CB_OFF), 1, true);
    return;
  }
  // rows of own block i once the off units are done: minus the row chunks'
  // sums (ascending chunks, summed first) when they were stored apart
  auto rows = [&](int i, T (&t)[4]) {
    if (h > w) {
      if (l == 0) (void)wait_ge(counter(sy, s, CB_OFF), ng * nch, sy.ctl);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int a = 64 * i + 16 * wv + 4 * r + g;
      t[r] = F<T>::zero();
      if (!O.valid(a) || n >= nc) continue;
      t[r] = y[(int64_t)(eo + O.row(a)) * nrhs + n];
      if (nch > 1) {
        T q = F<T>::zero();
        for (int e = 0; e < nch; ++e) q = q + u[(S.u_off[s] + (int64_t)e * w + O.row(a)) * nrhs + n];
        t[r] = t[r] - q;
      }
    }
  };
  const int i = nblk - 1 - c;  // the units of a supernode come last block first
  if (i == 0) {
    dep_chain<T, true>(O, Fc, sy, nrhs, nc, y, z, s, xs, ring, [&](T (&t)[4]) { rows(0, t); });
    return;
  }
  if (wv >= DNW) return;
  T t[4];
  rows(i, t);
  Acc<T> acc;
  dep_products(O, sy, nrhs, nc, y, s, max(0, i - FKC), &s_ready,
               [&](int j, T (&A)[16]) { int cp; load_tile(O, i, j, wv, l, A, cp); }, acc);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int a = 64 * i + 16 * wv + 4 * r + g;
    if (O.valid(a) && n < nc) z[(int64_t)(eo + O.row(a)) * nrhs + n] = t[r] + acc.get(r);
  }
  if (threadIdx.x == 0 && i > 1) (void)wait_ge(counter(sy, s, CB_H), i - 1, sy.ctl);
  wg_publish(counter(sy, s, CB_H), i, false);
}

// ---- launchers ----
template <class T>
void launch_gather_rhs(int32_t n, int32_t nrhs, const int32_t* perm_e, const double* scale,
                       const T* b, T* y, hipStream_t st, LaunchProfiler* pf) {
  int64_t tot = (int64_t)n * nrhs;
  if (tot <= 0) return;
  ProfScope ps(pf, LK_SOLVE_GATHER, 0.0, 2.0 * sizeof(T) * tot, st);
  hipLaunchKernelGGL(k_gather_rhs<T>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, n,
                     nrhs, perm_e, scale, b, y);
}
template <class T>
void launch_scatter_sol(int32_t n, int32_t nrhs, const int32_t* perm_e, const double* scale,
                        const T* y, T* x, hipStream_t st, LaunchProfiler* pf) {
  int64_t tot = (int64_t)n * nrhs;
  if (tot <= 0) return;
  ProfScope ps(pf, LK_SOLVE_SCATTER, 0.0, 2.0 * sizeof(T) * tot, st);
  hipLaunchKernelGGL(k_scatter_sol<T>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, n,
                     nrhs, perm_e, scale, y, x);
}
template <class T>
void launch_fgather(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count, int32_t nrhs, T* y,
                    const T* u, hipStream_t st, LaunchProfiler* pf) {
  if (count <= 0) return;
  ProfScope ps(pf, LK_SOLVE_GATHER, 0.0, 0.0, st);
  hipLaunchKernelGGL(k_fgather<T>, dim3(count), dim3(SNT), 0, st, S, Fc, items, nrhs, y, u);
}
template <class T>
void launch_fwd_tri(const DevSym& S, const DevFac<T>& Fc, const int32_t* list, int count,
                    int32_t nrhs, T* y, double bytes, hipStream_t st, LaunchProfiler* pf) {
  if (count <= 0) return;
  ProfScope ps(pf, LK_FWD_TRI, 0.0, bytes, st);
  hipLaunchKernelGGL(k_fwd_tri<T>, dim3(count), dim3(SNT), 0, st, S, Fc, list, nrhs, y);
}
// one 64-column block step of the wide supernodes (one launch)
template <class T>
void launch_ftri_step(const DevSym& S, const DevFac<T>& Fc, const SItem* items, const SolveStep& stp,
                      int32_t nrhs, T* y, T* z, hipStream_t st, LaunchProfiler* pf) {
  if (stp.d_end <= stp.u_beg) return;
  ProfScope ps(pf, LK_FWD_TRI, 0.0, 0.0, st);
  hipLaunchKernelGGL(k_ftri_step<T>, dim3((unsigned)(stp.d_end - stp.u_beg)), dim3(SNT), 0, st, S, Fc,
                     items + stp.u_beg, (int)(stp.u_end - stp.u_beg), nrhs, y, z);
}
template <class T>
void launch_btri_step(const DevSym& S, const DevFac<T>& Fc, const SItem* items, const SolveStep& stp,
                      int32_t nrhs, T* y, T* z, hipStream_t st, LaunchProfiler* pf) {
  if (stp.u_end <= stp.d_beg) return;
  ProfScope ps(pf, LK_BWD_TRI, 0.0, 0.0, st);
  hipLaunchKernelGGL(k_btri_step<T>, dim3((unsigned)(stp.u_end - stp.d_beg)), dim3(SNT), 0, st, S, Fc,
                     items + stp.d_beg, (int)(stp.d_end - stp.d_beg), nrhs, y, z);
}
template <class T>
void launch_zcopy(const DevSym& S, const SItem* items, int count, int32_t nrhs, const T* z, T* y, hipStream_t st) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_zcopy<T>, dim3((unsigned)count), dim3(SNT), 0, st, S, items, nrhs, z, y);
}
template <class T>
void launch_fwd_update(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count,
                       int32_t nrhs, const T* y, T* u, double bytes, hipStream_t st, LaunchProfiler* pf) {
  if (count <= 0) return;
  ProfScope ps(pf, LK_FWD_UPDATE, 0.0, bytes, st);
  hipLaunchKernelGGL(k_fwd_update<T>, dim3(count), dim3(SNT), 0, st, S, Fc, items, nrhs, y, u);
}
template <class T>
void launch_dsolve(int32_t n, int32_t nrhs, const T* d, const T* ds, const uint8_t* two, T* y,
                   hipStream_t st, LaunchProfiler* pf) {
  int64_t tot = (int64_t)n * nrhs;
  if (tot <= 0) return;
  ProfScope ps(pf, LK_DSOLVE, 0.0, 2.0 * sizeof(T) * tot, st);
  hipLaunchKernelGGL(k_dsolve<T>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, n, nrhs,
                     d, ds, two, y);
}
template <class T>
void launch_bwd_update(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count,
                       int32_t nrhs, T* y, double bytes, hipStream_t st, LaunchProfiler* pf) {
  if (count <= 0) return;
  ProfScope ps(pf, LK_BWD_UPDATE, 0.0, bytes, st);
  hipLaunchKernelGGL(k_bwd_update<T>, dim3(count), dim3(SNT), 0, st, S, Fc, items, nrhs, y);
}
template <class T>
void launch_bwd_tri(const DevSym& S, const DevFac<T>& Fc, const int32_t* list, int count,
                    int32_t nrhs, T* y, double bytes, hipStream_t st, LaunchProfiler* pf) {
  if (count <= 0) return;
  ProfScope ps(pf, LK_BWD_TRI, 0.0, bytes, st);
  hipLaunchKernelGGL(k_bwd_tri<T>, dim3(count), dim3(SNT), 0, st, S, Fc, list, nrhs, y);
}

void launch_sync_init(int32_t* cnt, int32_t ns, hipStream_t st) {
  const int64_t n = (int64_t)ns * CSTRIDE + 3;
  hipLaunchKernelGGL(k_sync_init, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, cnt, n);
}
template <class T>
void launch_diag_pack(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count, hipStream_t st) {
  if (count > 0) hipLaunchKernelGGL(k_diag_pack<T>, dim3((unsigned)count), dim3(SNT), 0, st, S, Fc, items);
}
// right-hand sides first .. first + DEP_RHS * chunks - 1 (as far as there are)
template <class T>
void launch_fwd_dep(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count, const SolveSync& sy,
                    int32_t nrhs, int first, int chunks, T* y, T* u, T* z, double bytes, hipStream_t st,
                    LaunchProfiler* pf) {
  if (count <= 0 || chunks <= 0) return;
  if (chunks > DEP_CHUNKS) throw std::runtime_error("solve: more chunks than a launch has counters for");
  ProfScope ps(pf, LK_FWD_TRI, 0.0, bytes, st);
  hipLaunchKernelGGL(k_fwd_dep<T>, dim3((unsigned)(count * chunks)), dim3(DNT), 0, st, S, Fc, items, sy, nrhs, first,
                     chunks, y, u, z);
}
template <class T>
void launch_bwd_dep(const DevSym& S, const DevFac<T>& Fc, const int2* items, int count, const SolveSync& sy,
                    int32_t nrhs, int first, int chunks, T* y, T* u, T* z, double bytes, hipStream_t st,
                    LaunchProfiler* pf) {
  if (count <= 0 || chunks <= 0) return;
  if (chunks > DEP_CHUNKS) throw std::runtime_error("solve: more chunks than a launch has counters for");
  ProfScope ps(pf, LK_BWD_TRI, 0.0, bytes, st);
  hipLaunchKernelGGL(k_bwd_dep<T>, dim3((unsigned)(count * chunks)), dim3(DNT), 0, st, S, Fc, items, sy, nrhs, first,
                     chunks, y, u, z);
}

#define RSL_SINST(T)                                                                           \
  template void launch_gather_rhs<T>(int32_t, int32_t, const int32_t*, const double*, const T*, \
                                     T*, hipStream_t, LaunchProfiler*);                        \
  template void launch_scatter_sol<T>(int32_t, int32_t, const int32_t*, const double*,          \
                                      const T*, T*, hipStream_t, LaunchProfiler*);             \
  template void launch_fgather<T>(const DevSym&, const DevFac<T>&, const int2*, int, int32_t, T*, \
                                  const T*, hipStream_t, LaunchProfiler*);                     \
  template void launch_fwd_tri<T>(const DevSym&, const DevFac<T>&, const int32_t*, int, int32_t, \
                                  T*, double, hipStream_t, LaunchProfiler*);                   \
  template void launch_ftri_step<T>(const DevSym&, const DevFac<T>&, const SItem*, const SolveStep&, \
                                    int32_t, T*, T*, hipStream_t, LaunchProfiler*);            \
  template void launch_btri_step<T>(const DevSym&, const DevFac<T>&, const SItem*, const SolveStep&, \
                                    int32_t, T*, T*, hipStream_t, LaunchProfiler*);            \
  template void launch_zcopy<T>(const DevSym&, const SItem*, int, int32_t, const T*, T*, hipStream_t); \
  template void launch_fwd_update<T>(const DevSym&, const DevFac<T>&, const int2*, int, int32_t, \
                                     const T*, T*, double, hipStream_t, LaunchProfiler*);      \
  template void launch_dsolve<T>(int32_t, int32_t, const T*, const T*, const uint8_t*, T*,      \
                                 hipStream_t, LaunchProfiler*);                                \
  template void launch_bwd_update<T>(const DevSym&, const DevFac<T>&, const int2*, int, int32_t, \
                                     T*, double, hipStream_t, LaunchProfiler*);                \
  template void launch_bwd_tri<T>(const DevSym&, const DevFac<T>&, const int32_t*, int, int32_t, \
                                  T*, double, hipStream_t, LaunchProfiler*);                   \
  template void launch_fwd_dep<T>(const DevSym&, const DevFac<T>&, const int2*, int, const SolveSync&, \
                                  int32_t, int, int, T*, T*, T*, double, hipStream_t, LaunchProfiler*); \
  template void launch_diag_pack<T>(const DevSym&, const DevFac<T>&, const int2*, int, hipStream_t); \
  template void launch_bwd_dep<T>(const DevSym&, const DevFac<T>&, const int2*, int, const SolveSync&, \
                                  int32_t, int, int, T*, T*, T*, double, hipStream_t, LaunchProfiler*);

RSL_SINST(double)
RSL_SINST(cplx)

}  // namespace rsl
