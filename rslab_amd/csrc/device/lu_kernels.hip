// Device kernels of the LU twin: supernodal left-looking LU with threshold
// partial pivoting restricted to each supernode's own rows
// (lu_ll_factor_node, src/numeric/multifrontal_lu.rs:1629-2347), and its
// supernodal forward / backward solve (the arithmetic of solve_lu_block,
// :3209-3283, grouped by supernode).
//
// Storage per supernode s (h rows, w own columns, rows in rs[s] order with the
// own rows first): L panel h x w column-major (unit-lower L below the
// diagonal, U11 on and above it) and U12 w x (h - w) column-major. The own
// rows of the panel are interchanged by the pivoting (rperm records which
// row-structure row sits at each position); the deep rows never are.
//
// Launch sequence of a tree level: cmod (every target tile of the level's
// supernodes sums its updaters' products L_k[rows] U_k[:, cols]), then per
// panel index: getf2 (one workgroup per supernode panel), apply (the panel's
// interchanges on the other columns and the triangular solve of the later
// own columns and of U12, the deep rows' transform), and the trailing GEMM.
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "lu_types.hpp"
#include "scalar.hpp"
#include "tile_mfma.hpp"
#include "wave.hpp"

namespace rsl {

namespace {

template <class T>
__device__ inline T lu_fma(T a, T b, T c) {
  return c + a * b;
}
template <>
__device__ inline double lu_fma<double>(double a, double b, double c) {
  return fma(a, b, c);
}

// value of lane q (wave-uniform) across the wave, read through the scalar unit
__device__ inline double lu_bcast(double v, int q) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), q);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), q);
  return __hiloint2double(hi, lo);
}
__device__ inline cplx lu_bcast(cplx v, int q) { return {lu_bcast(v.re, q), lu_bcast(v.im, q)}; }

// perturb_pivot (multifrontal_ldlt.rs:786-795)
template <class T>
__device__ inline T lu_perturb(T d, double floor) {
  const double mag = F<T>::mag(d);
  if (mag >= floor) return d;
  if (mag == 0.0) return F<T>::from_real(floor);
  return F<T>::scale(d, floor / mag);
}

// A 16x16 tile on the matrix cores: mac adds four terms (lane l: entry (l %
// 16, l / 16) of a, (l / 16, l % 16) of b); register r is entry (4 r + l / 16,
// l % 16). The terms add one after another, each as a fused multiply-add.
template <class T>
struct LuTile;
template <>
struct LuTile<double> {
  mf_d4 v = {0.0, 0.0, 0.0, 0.0};
  __device__ double get(int r) const { return v[r]; }
  __device__ void mac(double a, double b) { v = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, v, 0, 0, 0); }
};
template <>
struct LuTile<cplx> {
  mf_d4 re = {0.0, 0.0, 0.0, 0.0}, im = {0.0, 0.0, 0.0, 0.0};
  __device__ cplx get(int r) const { return {re[r], im[r]}; }
  __device__ void mac(cplx a, cplx b) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, im, 0, 0, 0);
  }
};

// f(0), f(1), .. f(N - 1) with compile-time arguments: the register columns of
// a step need constant places, and the step's body is past what the loop
// unroller takes
template <int N, int Q = 0, class Fn>
__device__ __forceinline__ void static_steps(Fn&& f) {
  if constexpr (Q < N) {
    f(std::integral_constant<int, Q>{});
    static_steps<N, Q + 1>(f);
  }
}

}  // namespace

// Scatter of the equilibrated, permuted values into the zeroed L and U12
// storage (the assembly of lu_ll_factor_node, multifrontal_lu.rs:1670-1686).
template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_assemble(LuSymDev S, LuFacDev<T> Fc, const T* __restrict__ vals) {
  const int64_t k = (int64_t)blockIdx.x * LU_NT + threadIdx.x;
  if (k >= S.nnz) return;
  const int64_t d = S.amap[k];
  if (d >= 0) Fc.l[d] = vals[k];
  else Fc.u[-1 - d] = vals[k];
}

// cmod of the real field on the matrix cores (v_mfma_f64_16x16x4f64): one
// workgroup per 64x64 target tile, its updaters ascending, the sum subtracted
// once; operands gathered into LDS
// 32 columns of K at a time (the next chunk's loads issued before the current
// chunk's products), every updater's product accumulated in FP64.
__global__ __launch_bounds__(LU_NT) void k_lu_cmod_mfma(LuSymDev S, LuFacDev<double> Fc,
                                                        const LuItem* __restrict__ items,
                                                        const CTask* __restrict__ tasks) {
  typedef TileCfgW<TP_F64> C;
  constexpr int KCW = C::KC, PER = KCW * 64 / LU_NT;
  __shared__ __align__(16) double As[C::ELEMS];
  __shared__ __align__(16) double Bs[C::ELEMS];
  const int tid = threadIdx.x;
  const LuItem it = items[blockIdx.x];
  double va[PER], vb[PER];
  auto fetch = [&](int tt, int cc) {
    const CTask tk = tasks[tt];
    const int k = tk.k, nck = S.sn_ncol[k];
    const int64_t hk = S.sn_nrow[k];
    const double* Lk = Fc.l + S.l_off[k];
    const double* Uk = Fc.u + S.u_off[k];
    const int kc = min(KCW, nck - cc);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + LU_NT * u, r = e & 63, c = e >> 6;
      const uint64_t below = (1ull << r) - 1ull;
      va[u] = 0.0;
      vb[u] = 0.0;
      if (c < kc) {
        if ((tk.rmask >> r) & 1ull) va[u] = Lk[(nck + tk.a0 + __popcll(tk.rmask & below)) + (int64_t)(cc + c) * hk];
        if ((tk.cmask >> r) & 1ull) vb[u] = Uk[(cc + c) + (int64_t)(tk.b0 + __popcll(tk.cmask & below)) * nck];
      }
    }
  };
  int t = it.t_beg, c0 = 0;
  int nck_t = S.sn_ncol[tasks[t].k];
  fetch(t, 0);
  TileAcc<TP_F64> acc;
  tile_zero(acc);
  for (;;) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + LU_NT * u, r = e & 63, c = e >> 6;
      stage_store_w<TP_F64>(As, r, c, va[u]);
      stage_store_w<TP_F64>(Bs, r, c, vb[u]);
    }
    __syncthreads();
    int tn = t, cn = c0 + KCW, nck_n = nck_t;
    if (cn >= nck_t) {
      tn = t + 1;
      cn = 0;
      if (tn < it.t_end) nck_n = S.sn_ncol[tasks[tn].k];
    }
    if (tn < it.t_end) fetch(tn, cn);
    tile_mma_w<TP_F64>(As, Bs, acc);
    __syncthreads();
    if (tn >= it.t_end) break;
    t = tn;
    c0 = cn;
    nck_t = nck_n;
  }
  const int s = it.s;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s];
  double* P;
  int64_t ld, mr, mc;
  if (it.region == 0) {
    P = Fc.l + S.l_off[s];
    ld = h;
    mr = h - it.r0;
    mc = w - it.c0;
  } else {
    P = Fc.u + S.u_off[s];
    ld = w;
    mr = w - it.r0;
    mc = h - w - it.c0;
  }
  // the targets read as one batch, then updated
  double old[16];
  int n = 0;
  tile_for_each<TP_F64>(acc, [&](int i, int j, double) {
    old[n++] = (i < mr && j < mc) ? P[(it.r0 + i) + (int64_t)(it.c0 + j) * ld] : 0.0;
  });
  n = 0;
  tile_for_each<TP_F64>(acc, [&](int i, int j, double v) {
    if (i < mr && j < mc) P[(it.r0 + i) + (int64_t)(it.c0 + j) * ld] = old[n] - v;
    ++n;
  });
}

// cmod of the complex field: the real product of A = [re im] with B = [re -im]
// for the real part and [im re] for the imaginary one, 16 columns of K at a
// time, all staged at once (the four products apart, staged pairwise, took
// eight barriers a chunk: 5.10 ms in 8 launches on a 26^3 grid, 4.78 now).
// Chunks are fetched two ahead, and what their addresses come from (the task,
// then its updater's sizes and offsets) one and two tasks before that; the
// real field, whose chunk is 32 columns and two barriers, gained nothing from
// that (7.08 and 7.42 ms in 16 launches, 40^3).
struct LuCmodTask {
  CTask tk;
  int nck;
  int64_t hk, l, u;
};

__global__ __launch_bounds__(LU_NT) void k_lu_cmod_mfma_c64(LuSymDev S, LuFacDev<cplx> Fc,
                                                            const LuItem* __restrict__ items,
                                                            const CTask* __restrict__ tasks) {
  typedef cplx T;
  typedef TileCfgW<TP_F64> C;
  constexpr int KX = C::KC / 2, PER = KX * 64 / LU_NT;
  __shared__ __align__(16) double As[C::ELEMS];
  __shared__ __align__(16) double Bs[2][C::ELEMS];
  const int tid = threadIdx.x;
  const LuItem it = items[blockIdx.x];
  auto resolve = [&](const CTask& tk) {
    return LuCmodTask{tk, S.sn_ncol[tk.k], S.sn_nrow[tk.k], S.l_off[tk.k], S.u_off[tk.k]};
  };
  auto task = [&](int t) { return tasks[min(t, it.t_end - 1)]; };
  int t = it.t_beg, c0 = 0;  // the next chunk to fetch
  LuCmodTask cur = resolve(task(t)), nxt = resolve(task(t + 1));
  CTask raw = task(t + 2);
  T va[2][PER], vb[2][PER];
  int ka[2], kb[2];  // columns of a fetched chunk that this thread's row / column takes
  // Thread r of each wave stages A's row r and B's column r, wave v columns v,
  // v + 4, .. of the chunk. A place's entry is the count of the mask's bits
  // below it; places without one and columns past the chunk's read a valid
  // entry (no load depends on a lane's place) and are zeroed when staged.
  const int r = tid & 63, v0 = tid >> 6;
  const uint64_t below = (1ull << r) - 1ull;
  auto fetch = [&](T (&a)[PER], T (&b)[PER], int& na, int& nb) {
    if (t >= it.t_end) return false;
    const int kc = min(KX, cur.nck - c0);
    const bool ina = (cur.tk.rmask >> r) & 1ull, inb = (cur.tk.cmask >> r) & 1ull;
    na = ina ? kc : 0;
    nb = inb ? kc : 0;
    const T* pa = Fc.l + cur.l + (cur.nck + cur.tk.a0 + (ina ? __popcll(cur.tk.rmask & below) : 0)) + (int64_t)c0 * cur.hk;
    const T* pb = Fc.u + cur.u + c0 + (int64_t)(cur.tk.b0 + (inb ? __popcll(cur.tk.cmask & below) : 0)) * cur.nck;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int c = min(v0 + (LU_NT / 64) * u, kc - 1);
      a[u] = pa[(int64_t)c * cur.hk];
      b[u] = pb[c];
    }
    c0 += KX;
    if (c0 >= cur.nck) {
      c0 = 0;
      ++t;
      cur = nxt;
      nxt = resolve(raw);
      raw = task(t + 2);
    }
    return true;
  };
  TileAcc<TP_F64> acc[2];
  tile_zero(acc[0]);
  tile_zero(acc[1]);
  auto chunk = [&](T (&a)[PER], T (&b)[PER], int& na, int& nb) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int c = v0 + (LU_NT / 64) * u;
      const T av = choose(c < na, a[u], F<T>::zero()), bv = choose(c < nb, b[u], F<T>::zero());
      stage_store_w<TP_F64>(As, r, c, av.re);
      stage_store_w<TP_F64>(As, r, c + KX, av.im);
      stage_store_w<TP_F64>(Bs[0], r, c, bv.re);
      stage_store_w<TP_F64>(Bs[0], r, c + KX, -bv.im);
      stage_store_w<TP_F64>(Bs[1], r, c, bv.im);
      stage_store_w<TP_F64>(Bs[1], r, c + KX, bv.re);
    }
    __syncthreads();
    const bool more = fetch(a, b, na, nb);
    tile_mma_w<TP_F64>(As, Bs[0], acc[0]);
    tile_mma_w<TP_F64>(As, Bs[1], acc[1]);
    __syncthreads();
    return more;
  };
  bool h0 = fetch(va[0], vb[0], ka[0], kb[0]), h1 = fetch(va[1], vb[1], ka[1], kb[1]);
  while (h0) {
    h0 = chunk(va[0], vb[0], ka[0], kb[0]);
    if (!h1) break;
    h1 = chunk(va[1], vb[1], ka[1], kb[1]);
  }
  const int s = it.s;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s];
  T* P;
  int64_t ld, mr, mc;
  if (it.region == 0) {
    P = Fc.l + S.l_off[s];
    ld = h;
    mr = h - it.r0;
    mc = w - it.c0;
  } else {
    P = Fc.u + S.u_off[s];
    ld = w;
    mr = w - it.r0;
    mc = h - w - it.c0;
  }
  // the targets read as one batch, then updated
  T old[16];
  int n = 0;
  tile_for_each<TP_F64>(acc[0], [&](int i, int j, double) {
    old[n] = F<T>::zero();
    if (i < mr && j < mc) old[n] = P[(it.r0 + i) + (int64_t)(it.c0 + j) * ld];
    ++n;
  });
  n = 0;
  tile_for_each<TP_F64>(acc[1], [&](int, int, double v) { old[n++].im -= v; });
  n = 0;
  tile_for_each<TP_F64>(acc[0], [&](int, int, double v) { old[n++].re -= v; });
  n = 0;
  tile_for_each<TP_F64>(acc[0], [&](int i, int j, double) {
    if (i < mr && j < mc) P[(it.r0 + i) + (int64_t)(it.c0 + j) * ld] = old[n];
    ++n;
  });
}

// getf2 on the own rows of one panel (multifrontal_lu.rs:2064-2111): per
// column, the pivot is the first row of largest magnitude in [k, w); the rows
// are interchanged only when the diagonal is below u times it; the
// interchange is applied to the panel's columns here and recorded (ipiv,
// rperm) for the other columns; then the column is scaled and the panel's
// later columns get the rank-1 update.
//
// The 16 columns of a panel are a serial chain of pivot searches over up to
// thousands of rows, one workgroup per supernode, so the time is the latency
// of a step. The panel's rows sit in registers (thread t holds rows t, t +
// 1024, ...), C columns at a time: a step is a local maximum, one exchange of
// the waves' maxima, one of the pivot row (and of the diagonal row it changes
// places with), and the rank-1 update, two barriers and no memory access.
// Waves without rows leave at once. C is 16 as long as the rows' columns take
// 64 of the 128 registers a thread of 1024 has (2 rows a thread in the real
// field, 1 in the complex), 8 or 4 beyond (the step's own values and addresses
// take the rest and, at the widest forms, 4 registers of scratch memory in the
// real field and 24 in the complex one); the panel's
// other columns then take a finished group of C from memory, the rows gathered
// by the group's composite interchange (src). The operations on an entry and
// their order are those of one rank-1 update per step. With the panel in
// memory and a serial scan of the 16 waves' maxima a panel took 73 us on a
// 40^3 grid (own rows up to 1600), 340 of them in a row: 25 of 57 ms.
template <class T>
struct LuPanelLds {
  double red_m[LU_GT / 64];
  int red_i[LU_GT / 64];
  double dsq;
  T prow[2][LU_PANEL], drow[2][LU_PANEL];  // by step parity: a step without a search has one barrier
  int pint[2][2], dint[2][2];
  T lb[8][8], ub[8][4];
};

template <class T, int R, int C>
__device__ __forceinline__ void lu_getf2_reg(const LuSymDev& S, const LuFacDev<T>& Fc, int s, int kb, int ke,
                                             LuPanelLds<T>& sh) {
  const int64_t h = S.sn_nrow[s];
  const int first = S.sn_first[s], m = S.sn_ncol[s] - kb, pw = ke - kb;
  T* const L = Fc.l + S.l_off[s] + (int64_t)kb * h + kb;  // panel entry (i, j) = L[i + j h], i < m
  int32_t* const rperm = Fc.rperm + first + kb;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (wv * 64 >= m) return;
  const int nw = min(LU_GT / 64, (m + 63) / 64);  // waves with rows
  const bool search = Fc.thresh_sq > 0.0;
  int rp[R];
#pragma unroll
  for (int r = 0; r < R; ++r) rp[r] = rperm[min(tid + LU_GT * r, m - 1)];
  int par = 0;
  for (int c0 = 0; c0 < pw; c0 += C) {
    const int nc = min(C, pw - c0);
    T x[R][C];
    int src[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = tid + LU_GT * r;
      src[r] = row;
#pragma unroll
      for (int j = 0; j < C; ++j) x[r][j] = L[min(row, m - 1) + (int64_t)(c0 + min(j, nc - 1)) * h];
    }
    static_steps<C>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      if (q >= nc) return;
      const int kk = c0 + q;
      int p = kk;
      bool swap = false;
      if (search) {
        // the wave's largest magnitude and its first row; the largest high
        // word usually singles the row out (NaN never competes)
        double v[R];
        uint32_t hm = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int row = tid + LU_GT * r;
          const double a = F<T>::magsq(x[r][q]);
          v[r] = (row >= kk && row < m && a >= 0.0) ? a : -1.0;
          hm = max(hm, v[r] >= 0.0 ? (uint32_t)__double2hiint(v[r]) : 0u);
        }
        hm = wave_umax_dpp(hm);
        unsigned long long b[R];
        int hits = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          b[r] = __ballot(v[r] >= 0.0 && (uint32_t)__double2hiint(v[r]) == hm);
          hits += __popcll(b[r]);
        }
        double wm = -1.0;
        if (hits != 1) {
#pragma unroll
          for (int r = 0; r < R; ++r) wm = fmax(wm, v[r]);
          wm = wave_max_dpp(wm);
#pragma unroll
          for (int r = 0; r < R; ++r) b[r] = __ballot(v[r] == wm);
        }
        int wl = 0, wr = 0;
#pragma unroll
        for (int r = R - 1; r >= 0; --r)
          if (b[r]) {
            wl = __ffsll((long long)b[r]) - 1;
            wr = r;
          }
        if (hits == 1) {
          double vv = v[0];
#pragma unroll
          for (int r = 1; r < R; ++r) vv = wr == r ? v[r] : vv;
          wm = lu_bcast(vv, wl);
        }
        if (lane == 0) {
          sh.red_m[wv] = wm;
          sh.red_i[wv] = 64 * wv + wl + LU_GT * wr;
        }
        if (tid == kk) sh.dsq = F<T>::magsq(x[0][q]);
        __syncthreads();
        const int o = lane & 15;
        const double om = o < nw ? sh.red_m[min(o, nw - 1)] : -2.0;
        const int oi = sh.red_i[min(o, nw - 1)];
        double gm = om;
        gm = fmax(gm, dpp_move<0x111, 0xF, 0xF>(gm));
        gm = fmax(gm, dpp_move<0x112, 0xF, 0xF>(gm));
        gm = fmax(gm, dpp_move<0x114, 0xF, 0xF>(gm));
        gm = fmax(gm, dpp_move<0x118, 0xF, 0xF>(gm));
        gm = lu_bcast(gm, 15);
        // the first row among the waves that reach it (complemented: a maximum)
        const uint32_t inv = om == gm ? ~(uint32_t)oi : 0u;
        const int bi = (int)~wave_umax_dpp(inv);
        swap = bi != kk && sh.dsq < Fc.thresh_sq * gm;
        if (swap) p = bi;
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int row = tid + LU_GT * r;
        if (row == p) {
#pragma unroll
          for (int j = 0; j < C; ++j) sh.prow[par][j] = x[r][j];
          sh.pint[par][0] = rp[r];
          sh.pint[par][1] = src[r];
        }
        if (r == 0 && swap && row == kk) {
#pragma unroll
          for (int j = 0; j < C; ++j) sh.drow[par][j] = x[0][j];
          sh.dint[par][0] = rp[0];
          sh.dint[par][1] = src[0];
        }
      }
      __syncthreads();
      T piv = sh.prow[par][q];
      if (Fc.pol.have_floor) {
        if (F<T>::mag(piv) < Fc.pol.floor) {
          piv = lu_perturb(piv, Fc.pol.floor);
          if (tid == 0) atomicAdd(&Fc.counters[0], 1ull);
        }
      } else if (F<T>::is_zero(piv) && tid == 0) {
        Fc.status[0] = 1;
        atomicMin(&Fc.counters[1], (unsigned long long)(first + kb + kk));
      }
      if (tid == 0) Fc.ipiv[first + kb + kk] = kb + p;
      const T pinv = F<T>::recip(piv);
      if (swap) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int row = tid + LU_GT * r;
          if (row == p) {
#pragma unroll
            for (int j = 0; j < C; ++j) x[r][j] = sh.drow[par][j];
            rp[r] = sh.dint[par][0];
            src[r] = sh.dint[par][1];
          }
          if (r == 0 && row == kk) {
#pragma unroll
            for (int j = 0; j < C; ++j) x[0][j] = sh.prow[par][j];
            rp[0] = sh.pint[par][0];
            src[0] = sh.pint[par][1];
          }
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool below = r > 0 || tid > kk;
        const T l = x[r][q] * pinv;
        if (below) {
          x[r][q] = l;
#pragma unroll
          for (int j = q + 1; j < C; ++j) x[r][j] = x[r][j] - l * sh.prow[par][j];
        } else if (tid == kk) {
          x[r][q] = piv;
        }
      }
      par ^= 1;
    });
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = tid + LU_GT * r;
#pragma unroll
      for (int j = 0; j < C; ++j)
        if (j < nc && row >= c0 && row < m) L[row + (int64_t)(c0 + j) * h] = x[r][j];
    }
    if constexpr (C < LU_PANEL) {
      // the panel's other columns: interchanges (left of the group), and the
      // group's steps (right of it), JC columns at a time (as many
      // registers as the step's own values)
      constexpr int JC = 8 / (R * (int)(sizeof(T) / 8));
      if (tid >= c0 && tid < c0 + nc) {
#pragma unroll
        for (int j = 0; j < C; ++j) sh.lb[tid - c0][j] = x[0][j];
      }
      for (int j0 = 0; j0 < pw; j0 += JC) {
        if (j0 >= c0 && j0 < c0 + nc) continue;  // (JC divides C)
        const bool right = j0 >= c0 + nc;
        const int je = min(JC, (right ? pw : c0) - j0);
        T v[R][JC];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int u = 0; u < JC; ++u) v[r][u] = L[min(src[r], m - 1) + (int64_t)(j0 + min(u, je - 1)) * h];
        if (right && tid >= c0 && tid < c0 + nc) {
#pragma unroll
          for (int u = 0; u < JC; ++u) sh.ub[tid - c0][u] = v[0][u];
        }
        __syncthreads();  // every gather is done before a store
        if (right) {
          if (tid < JC) {
            for (int a = 1; a < nc; ++a) {
              T t = sh.ub[a][tid];
              for (int e = 0; e < a; ++e) t = t - sh.lb[a][e] * sh.ub[e][tid];
              sh.ub[a][tid] = t;
            }
          }
          __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int row = tid + LU_GT * r;
          if (right) {
            if (r == 0 && row < c0 + nc) {
#pragma unroll
              for (int u = 0; u < JC; ++u)
                if (row >= c0) v[0][u] = sh.ub[row - c0][u];
            } else {
#pragma unroll
              for (int e = 0; e < C; ++e)
                if (e < nc) {
#pragma unroll
                  for (int u = 0; u < JC; ++u) v[r][u] = v[r][u] - x[r][e] * sh.ub[e][u];
                }
            }
          }
          if (row >= c0 && row < m) {
#pragma unroll
            for (int u = 0; u < JC; ++u)
              if (u < je) L[row + (int64_t)(j0 + u) * h] = v[r][u];
          }
        }
        __syncthreads();  // before ub is written again, and before the next group reads the columns
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = tid + LU_GT * r;
    if (row < m) rperm[row] = rp[r];
  }
}

// One workgroup per panel. Panels of more than 4096 own rows do not fit the
// registers: one supernode of that width is past 64^3 unknowns on a regular
// grid, and its panel stays in memory.
template <class T>
__global__ __launch_bounds__(LU_GT) void k_lu_getf2(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units) {
  __shared__ LuPanelLds<T> lds;
  constexpr bool CPLX = sizeof(T) == 16;
  const LuUnit un = units[blockIdx.x];
  const int s = un.s, kb = un.kb;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s], first = S.sn_first[s], ke = min(kb + S.nb[s], w);
  if (w - kb <= LU_GT) return lu_getf2_reg<T, 1, 16>(S, Fc, s, kb, ke, lds);
  if (w - kb <= 2 * LU_GT) return lu_getf2_reg<T, 2, CPLX ? 8 : 16>(S, Fc, s, kb, ke, lds);
  if (w - kb <= 4 * LU_GT) return lu_getf2_reg<T, 4, CPLX ? 4 : 8>(S, Fc, s, kb, ke, lds);
  __shared__ double red_m[LU_GT / 64];
  __shared__ int red_i[LU_GT / 64];
  __shared__ T ukj[128];
  __shared__ int sh_p;
  __shared__ T sh_pinv;
  T* L = Fc.l + S.l_off[s];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int k = kb; k < ke; ++k) {
    T* ck = L + (int64_t)k * h;
    int p = k;
    if (Fc.thresh_sq > 0.0) {
      double m = -1.0;
      int mi = INT_MAX;
      for (int i = k + tid; i < w; i += LU_GT) {
        const double v = F<T>::magsq(ck[i]);
        if (v > m) {
          m = v;
          mi = i;
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const double om = __shfl_xor(m, off);
        const int oi = __shfl_xor(mi, off);
        if (om > m || (om == m && oi < mi)) {
          m = om;
          mi = oi;
        }
      }
      if (lane == 0) {
        red_m[wv] = m;
        red_i[wv] = mi;
      }
      __syncthreads();
      if (tid == 0) {
        double bm = red_m[0];
        int bi = red_i[0];
        for (int q = 1; q < LU_GT / 64; ++q)
          if (red_m[q] > bm || (red_m[q] == bm && red_i[q] < bi)) {
            bm = red_m[q];
            bi = red_i[q];
          }
        const double dsq = F<T>::magsq(ck[k]);
        sh_p = (bi != k && dsq < Fc.thresh_sq * bm) ? bi : k;
      }
      __syncthreads();
      p = sh_p;
    }
    if (p != k) {
      for (int j = kb + tid; j < ke; j += LU_GT) {
        T* cj = L + (int64_t)j * h;
        const T t = cj[k];
        cj[k] = cj[p];
        cj[p] = t;
      }
      if (tid == 0) {
        int32_t* rp = Fc.rperm + first;
        const int32_t t = rp[k];
        rp[k] = rp[p];
        rp[p] = t;
      }
    }
    __syncthreads();
    if (tid == 0) {
      Fc.ipiv[first + k] = p;
      T piv = ck[k];
      if (Fc.pol.have_floor) {
        if (F<T>::mag(piv) < Fc.pol.floor) {
          piv = lu_perturb(piv, Fc.pol.floor);
          atomicAdd(&Fc.counters[0], 1ull);
        }
      } else if (F<T>::is_zero(piv)) {
        Fc.status[0] = 1;
        atomicMin(&Fc.counters[1], (unsigned long long)(first + k));
      }
      ck[k] = piv;
      sh_pinv = F<T>::recip(piv);
    }
    for (int j = k + 1 + tid; j < ke; j += LU_GT) ukj[j - kb] = L[(int64_t)j * h + k];
    __syncthreads();
    const T pinv = sh_pinv;
    for (int i = k + 1 + tid; i < w; i += LU_GT) {
      const T lik = ck[i] * pinv;
      ck[i] = lik;
      for (int j = k + 1; j < ke; ++j) {
        const T m = ukj[j - kb];
        if (!F<T>::is_zero(m)) {
          T* cj = L + (int64_t)j * h;
          cj[i] = cj[i] - lik * m;
        }
      }
    }
    __syncthreads();
  }
}

// After a panel's getf2: column units apply the panel's interchanges to the
// columns outside the panel (the finished ones left of it, the later own
// columns and U12) and, on the later ones, the unit-lower triangular solve
// with L11 (the TRSM of :2157-2199); deep-row units apply the panel transform
// to the rows below the own rows (apply_panel_trailing, :1357-1387). The
// panel's diagonal block and pivot reciprocals sit in LDS, each thread's
// column or row segment in registers (the same operations in the same order
// as on the stored values), all places known at compile time. Bound by latency:
// one round of loads, the block's staging and a 16-step chain. Units are one
// wave of 64 columns or rows: a lane reads along its own column, so a wave's
// load touches 64 lines, and four waves a workgroup left most of the chip idle
// (10.8 us a launch with 256 columns a unit, 8.4 with 64, 15.9 with the chain
// selecting its registers at run time; 340 launches of a 40^3 grid).
template <class T>
__global__ __launch_bounds__(LU_COLS) void k_lu_apply(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units) {
  __shared__ T Ls[LU_PANEL][LU_PANEL + 1];  // the panel's diagonal block: Ls[r][c] = entry (kb + r, kb + c)
  __shared__ T pinv[LU_PANEL];
  __shared__ int pv[LU_PANEL];
  const LuUnit un = units[blockIdx.x];
  const int s = un.s, kb = un.kb;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s], first = S.sn_first[s], ke = min(kb + S.nb[s], w), pw = ke - kb;
  T* L = Fc.l + S.l_off[s];
  // this thread's column or row segment, its loads out before the panel's
  // block is staged (a thread past the unit's last one reads that one)
  const int64_t nlater = w - ke, ncols = kb + nlater + (h - w);
  const bool row = un.b != 0;
  const int64_t place = (int64_t)un.a + threadIdx.x, count = row ? h - w : ncols;
  const bool live = place < count;
  const int64_t c = min(place, count - 1);
  const bool later = c >= kb;
  T* seg;
  if (row) seg = L + (int64_t)kb * h + w + c;
  else if (c < kb) seg = L + c * h + kb;
  else if (c < kb + nlater) seg = L + (ke + c - kb) * h + kb;
  else seg = Fc.u + S.u_off[s] + (c - kb - nlater) * w + kb;
  const int64_t ld = row ? h : 1;
  T v[LU_PANEL];
#pragma unroll
  for (int r = 0; r < LU_PANEL; ++r) v[r] = seg[min(r, pw - 1) * ld];
  #pragma unroll
  for (int e = threadIdx.x; e < LU_PANEL * LU_PANEL; e += LU_COLS) {
    const int r = e % LU_PANEL, c = e / LU_PANEL;
    Ls[r][c] = (r < pw && c < pw) ? L[(int64_t)(kb + c) * h + kb + r] : F<T>::zero();
  }
  if (threadIdx.x < LU_PANEL) pv[threadIdx.x] = threadIdx.x < pw ? Fc.ipiv[first + kb + threadIdx.x] : 0;
  __syncthreads();
  if (threadIdx.x < LU_PANEL) pinv[threadIdx.x] = threadIdx.x < pw ? F<T>::recip(Ls[threadIdx.x][threadIdx.x]) : F<T>::zero();
  __syncthreads();
  if (!live) return;
  if (!row) {
    // interchanges inside the panel are register moves, the others one
    // exchange with the column
    T* const col = seg - kb;
    bool moved = false;
    static_steps<LU_PANEL>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const int p = __builtin_amdgcn_readfirstlane(pv[q]);
      if (q < pw && p != kb + q) {
        moved = true;
        const T t = v[q];
        if (p >= ke) {
          v[q] = col[p];
          col[p] = t;
        } else {
#pragma unroll
          for (int i = q + 1; i < LU_PANEL; ++i) {
            const bool at = kb + i == p;
            v[q] = choose(at, v[i], v[q]);
            v[i] = choose(at, t, v[i]);
          }
        }
      }
    });
    if (later) {
      // column by column of L11: every entry's terms in ascending order
      static_steps<LU_PANEL - 1>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
#pragma unroll
        for (int r = q + 1; r < LU_PANEL; ++r) v[r] = v[r] - Ls[r][q] * v[q];
      });
    }
    if (later || moved) {
#pragma unroll
      for (int r = 0; r < LU_PANEL; ++r)
        if (r < pw) col[kb + r] = v[r];
    }
  } else {
    static_steps<LU_PANEL>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      if (q < pw) {
        v[q] = v[q] * pinv[q];
#pragma unroll
        for (int jj = q + 1; jj < LU_PANEL; ++jj) {
          const T m = Ls[q][jj];
          v[jj] = choose(F<T>::is_zero(m), v[jj], v[jj] - v[q] * m);
        }
      }
    });
#pragma unroll
    for (int q = 0; q < LU_PANEL; ++q)
      if (q < pw) seg[q * ld] = v[q];
  }
}

// Trailing GEMMs of a panel (:2206-2280): L[ke.., ke..w) -= L[ke.., kb..ke)
// U[kb..ke, ke..w) and U12[ke..w, :] -= L[ke..w, kb..ke) U12[kb..ke, :], one
// 64x64 tile per workgroup. With 16 terms an entry a tile is one round of
// loads: every wave fetches its operands and targets (16 rows, all columns)
// straight into matrix-core registers, no LDS and no barrier. The transposed
// product, so that a register's lanes hold 16 rows of a column. Bound by that
// round's latency. The terms add in ascending order, as on the vector units.
template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_gemm(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units) {
  const LuUnit un = units[blockIdx.x];
  const int s = un.s, kb = un.kb;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s], ke = min(kb + S.nb[s], w), pw = ke - kb;
  const T* L = Fc.l + S.l_off[s];
  const bool upart = un.a < 0;
  const int64_t r0 = (int64_t)ke + (int64_t)(upart ? -1 - un.a : un.a) * 64;
  const int64_t c0 = (int64_t)un.b * 64;
  T* P;
  int64_t ld, mr, mc;
  const T* B;
  if (!upart) {
    P = Fc.l + S.l_off[s] + (int64_t)ke * h;  // column ke + c0 + j at P + (c0 + j) h
    ld = h;
    mr = h - r0;
    mc = w - ke - c0;
    B = L + (int64_t)ke * h + kb;
  } else {
    P = Fc.u + S.u_off[s];
    ld = w;
    mr = w - r0;
    mc = h - w - c0;
    B = Fc.u + S.u_off[s] + kb;
  }
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, n = l & 15, g = l >> 4;
  const int i = 16 * wv + n;  // this lane's row; places past the end read the last one
  if (16 * wv >= mr) return;
  const T* Lp = L + (int64_t)kb * h + r0 + min<int64_t>(i, mr - 1);
  static_assert(LU_PANEL == 16, "four steps of four terms");
  T lv[4], uv[4][4], old[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r) lv[r] = Lp[(int64_t)min(4 * r + g, pw - 1) * h];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const T* Bp = B + (c0 + min<int64_t>(16 * ct + n, mc - 1)) * ld;
#pragma unroll
    for (int r = 0; r < 4; ++r) uv[ct][r] = Bp[min(4 * r + g, pw - 1)];
  }
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      old[ct][r] = P[(r0 + min<int64_t>(i, mr - 1)) + (c0 + min<int64_t>(16 * ct + 4 * r + g, mc - 1)) * ld];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * r + g >= pw) lv[r] = F<T>::zero();
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * r + g >= pw) uv[ct][r] = F<T>::zero();
    LuTile<T> acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc.mac(uv[ct][r], lv[r]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * ct + 4 * r + g;
      if (i < mr && j < mc) P[(r0 + i) + (c0 + j) * ld] = old[ct][r] - acc.get(r);
    }
  }
}

// ---- solve (row-major n x nrhs vectors)

// bh[g] = d_row[o] b[o] for the original row o = perm[g]
template <class T>
__global__ void k_lu_sprep(int32_t n, int32_t nrhs, const int32_t* __restrict__ perm, const double* __restrict__ d_row,
                           const T* __restrict__ b, T* __restrict__ bh) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)n * nrhs) return;
  const int64_t g = e / nrhs, c = e - g * nrhs, o = perm[g];
  bh[e] = F<T>::scale(b[o * nrhs + c], d_row[o]);
}

// x[o] = d_col[o] y[e] for the original column o = perm[e]
template <class T>
__global__ void k_lu_sfinish(int32_t n, int32_t nrhs, const int32_t* __restrict__ perm,
                             const double* __restrict__ d_col, const T* __restrict__ y, T* __restrict__ x) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)n * nrhs) return;
  const int64_t g = e / nrhs, c = e - g * nrhs, o = perm[g];
  x[o * nrhs + c] = F<T>::scale(y[e], d_col[o]);
}

// Forward gather, 64 own rows of one supernode per unit (s, -, first row):
// y_s[p] = b[pivot row of p] minus the descendants' off-diagonal products
// that land on that row.
template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_fgather(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units,
                                                      int32_t nrhs, const T* __restrict__ bh, const T* __restrict__ scr,
                                                      T* __restrict__ y) {
  const LuUnit un = units[blockIdx.x];
  const int s = un.s, w = S.sn_ncol[s], first = S.sn_first[s];
  const int64_t m = min(64, w - un.a);
  for (int64_t e = threadIdx.x; e < m * nrhs; e += LU_NT) {
    const int64_t p = un.a + e / nrhs, c = e % nrhs;
    const int64_t g = first + Fc.rperm[first + p];
    T v = bh[g * nrhs + c];
#pragma unroll 4
    for (int64_t q = S.gat_ptr[g]; q < S.gat_ptr[g + 1]; ++q) v = v - scr[S.gat_idx[q] * nrhs + c];
    y[(first + p) * nrhs + c] = v;
  }
}

// Backward U12 terms, 16 own rows per unit (s, -, first row), the trailing
// columns split over 16 slices summed in LDS, 8 right-hand sides at a time:
// y_s[p] -= U12[p, :] x[rs[w..]] (the ancestors' x, final, in x).
template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_boff(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units,
                                                   int32_t nrhs, T* __restrict__ y, const T* __restrict__ x) {
  constexpr int CW = 8;
  __shared__ T part[16][16][CW + 1];
  const LuUnit un = units[blockIdx.x];
  const int s = un.s;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s], first = S.sn_first[s];
  const T* U = Fc.u + S.u_off[s];
  const int32_t* rs = S.rs_idx + S.rs_off[s] + w;
  const int64_t nt = h - w;
  const int i = threadIdx.x & 15, sl = threadIdx.x >> 4;
  const int64_t p = un.a + i;
  for (int c0 = 0; c0 < nrhs; c0 += CW) {
    const int cw = min(CW, nrhs - c0);
    T acc[CW];
#pragma unroll
    for (int c = 0; c < CW; ++c) acc[c] = F<T>::zero();
    if (p < w) {
      // QB columns of the slice per pass, their loads issued together; the
      // next pass's row indices are loaded with them, so a pass waits on one
      // round of loads (ascending columns: the sums keep their order)
      constexpr int QB = 8;
      int64_t t = sl;
      int32_t rn[QB];
#pragma unroll
      for (int q = 0; q < QB; ++q) rn[q] = t + 16 * q < nt ? rs[t + 16 * q] : 0;
      for (; t + 16 * (QB - 1) < nt; t += 16 * QB) {
        T u[QB];
        const T* xr[QB];
#pragma unroll
        for (int q = 0; q < QB; ++q) {
          u[q] = U[p + (t + 16 * q) * w];
          xr[q] = x + (int64_t)rn[q] * nrhs + c0;
        }
        T xv[QB][CW];
#pragma unroll
        for (int q = 0; q < QB; ++q)
#pragma unroll
          for (int c = 0; c < CW; ++c) xv[q][c] = c < cw ? xr[q][c] : F<T>::zero();
#pragma unroll
        for (int q = 0; q < QB; ++q) {
          const int64_t tn = t + 16 * QB + 16 * q;
          rn[q] = tn < nt ? rs[tn] : 0;
        }
#pragma unroll
        for (int q = 0; q < QB; ++q)
#pragma unroll
          for (int c = 0; c < CW; ++c)
            if (c < cw) acc[c] = lu_fma(u[q], xv[q][c], acc[c]);
      }
      for (; t < nt; t += 16) {
        const T u1 = U[p + t * w];
        const T* x1 = x + (int64_t)rs[t] * nrhs + c0;
#pragma unroll
        for (int c = 0; c < CW; ++c)
          if (c < cw) acc[c] = lu_fma(u1, x1[c], acc[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < CW; ++c) part[sl][i][c] = acc[c];
    __syncthreads();
    if (threadIdx.x < 16 * CW) {
      const int ii = threadIdx.x & 15, c = threadIdx.x >> 4;
      const int64_t pp = un.a + ii;
      if (pp < w && c < cw) {
        T sum = part[0][ii][c];
        for (int q = 1; q < 16; ++q) sum = sum + part[q][ii][c];
        T* d = y + (first + pp) * nrhs + c0 + c;
        *d = *d - sum;
      }
    }
    __syncthreads();
  }
}

// The block solves of the steps below: LU_BS rows, a lane each, NK right-hand
// sides of a wave as interleaved chains.
template <int NK, bool BWD, class T>
__device__ __forceinline__ void lu_block_solve(const T (*D)[LU_BS + 1], const T* dinv, int m, int lane, T* v) {
  const int row = min(lane, LU_BS - 1);
#pragma unroll 8
  for (int t = 0; t < m; ++t) {
    const int q = BWD ? m - 1 - t : t;
    const T dq = D[row][q];
    T di = F<T>::zero();
    if constexpr (BWD) di = dinv[q];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if constexpr (BWD) v[k] = choose(lane == q, v[k] * di, v[k]);
      const T vq = lu_bcast(v[k], q);
      const T nv = lu_fma(F<T>::zero() - dq, vq, v[k]);
      v[k] = choose(BWD ? lane < q : lane > q && lane < m, nv, v[k]);
    }
  }
}

// One forward block step of a supernode's own block, units (s, j0, first
// row, writer): every unit solves the diagonal block [j0, j0 + m) of L11 from
// the updated, not yet solved values in y (unit-lower substitution, one wave
// per right-hand side, lane per row, the block's L in LDS), then updates its
// 64 rows below the block with it: own rows in y, off-diagonal rows into the
// supernode's scratch rows (written by the first block, added to after). The
// writer unit stores the solved block into yo; no unit of the launch writes
// rows another one reads.
// Bound by latency: a step is a launch, one round of loads, the substitution
// and a product; LU_BS rows in both fields, since the complex field's 32, which
// kept its LDS small, took twice the launches (4.7 and 3.8 ms of steps on a
// 26^3 grid). The rows' entries and their targets are fetched with the
// block, before the substitution, and the product runs on the matrix cores
// (16 rows by 16 right-hand sides a wave, its terms in ascending order), where
// it fetched the entries column by column after it.
// The backward step is the same on U11 from below (back substitution with the
// pivots, whose reciprocals are taken once): own rows above the block.
template <class T, bool BWD>
__device__ __forceinline__ void lu_step(const LuSymDev& S, const LuFacDev<T>& Fc, const LuUnit& un, int32_t nrhs,
                                        T* y, T* yo, T* scr) {
  constexpr int CW = 16;
  __shared__ T D[LU_BS][LU_BS + 1];
  __shared__ T yb[LU_BS][CW + 1];
  __shared__ T dinv[LU_BS];
  const int s = un.s, j0 = un.kb;
  const int64_t h = S.sn_nrow[s];
  const int w = S.sn_ncol[s], first = S.sn_first[s], m = min(LU_BS, w - j0);
  const T* L = Fc.l + S.l_off[s];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n = lane & 15, g = lane >> 4;
  const int64_t r0 = un.a + 16 * wv, rend = BWD ? j0 : h;  // this wave's 16 rows
  // the block's loads and the rows' issued together, then the LDS stores
  constexpr int PER = LU_BS * LU_BS / LU_NT;
  T b[PER], A[LU_BS / 4];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + u * LU_NT, r = e % LU_BS, q = e / LU_BS;
    b[u] = F<T>::zero();
    if (BWD ? q < m && r <= q : r < m && q < r) b[u] = L[(int64_t)(j0 + q) * h + j0 + r];
  }
  const T* row = L + (int64_t)j0 * h + max<int64_t>(0, min<int64_t>(r0 + n, rend - 1));
#pragma unroll
  for (int k = 0; k < LU_BS / 4; ++k) A[k] = row[(int64_t)min(4 * k + g, m - 1) * h];
  T* d[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t i = r0 + 4 * r + g;
    d[r] = nullptr;
    if (i < rend) d[r] = (i < w ? y + (first + i) * nrhs : scr + (S.s_off[s] + i - w) * nrhs) + n;
  }
  const bool add = BWD || j0 > 0;  // (off-diagonal rows: the first block's terms are stored)
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + u * LU_NT;
    D[e % LU_BS][e / LU_BS] = b[u];
  }
  __syncthreads();
  if constexpr (BWD) {
    if (threadIdx.x < m) dinv[threadIdx.x] = F<T>::recip(D[threadIdx.x][threadIdx.x]);
    __syncthreads();
  }
  for (int c0 = 0; c0 < nrhs; c0 += CW) {
    const int cw = min(CW, nrhs - c0);
    // a wave's right-hand sides: columns wv, wv + 4, ...
    constexpr int NW = LU_NT / 64, CPW = CW / NW;
    T v[CPW], t[4];
    const T* yc = y + (int64_t)(first + j0 + min(lane, m - 1)) * nrhs + c0;
#pragma unroll
    for (int k = 0; k < CPW; ++k) v[k] = yc[min(wv + k * NW, cw - 1)];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      t[r] = F<T>::zero();
      if (d[r] && n < cw && (add || r0 + 4 * r + g < w)) t[r] = d[r][c0];
    }
    if (cw > 2 * NW) lu_block_solve<4, BWD>(D, dinv, m, lane, v);
    else if (cw > NW) lu_block_solve<2, BWD>(D, dinv, m, lane, v);
    else lu_block_solve<1, BWD>(D, dinv, m, lane, v);
    if (lane < LU_BS) {
#pragma unroll
      for (int k = 0; k < CPW; ++k) {
        const int c = wv + k * NW;
        const bool in = lane < m && c < cw;
        yb[lane][c] = choose(in, v[k], F<T>::zero());
        if (in && un.b) yo[(int64_t)(first + j0 + lane) * nrhs + c0 + c] = v[k];
      }
    }
    __syncthreads();
    if (r0 < rend) {
      LuTile<T> acc;
#pragma unroll
      for (int k = 0; k < LU_BS / 4; ++k) acc.mac(choose(4 * k + g < m, A[k], F<T>::zero()), yb[4 * k + g][n]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (!d[r] || n >= cw) continue;
        if (r0 + 4 * r + g < w) d[r][c0] = t[r] - acc.get(r);
        else d[r][c0] = add ? t[r] + acc.get(r) : acc.get(r);
      }
    }
    __syncthreads();
  }
}

template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_fstep(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units,
                                                    int32_t nrhs, T* __restrict__ y, T* __restrict__ yo,
                                                    T* __restrict__ scr) {
  lu_step<T, false>(S, Fc, units[blockIdx.x], nrhs, y, yo, scr);
}

// (the writer stores the solved block into xo)
template <class T>
__global__ __launch_bounds__(LU_NT) void k_lu_bstep(LuSymDev S, LuFacDev<T> Fc, const LuUnit* __restrict__ units,
                                                    int32_t nrhs, T* __restrict__ y, T* __restrict__ xo) {
  lu_step<T, true>(S, Fc, units[blockIdx.x], nrhs, y, xo, nullptr);
}

// ---- launchers
template <class T>
void launch_lu_assemble(const LuSymDev& S, const LuFacDev<T>& Fc, const T* vals, hipStream_t st) {
  if (S.nnz <= 0) return;
  hipLaunchKernelGGL(k_lu_assemble<T>, dim3((unsigned)((S.nnz + LU_NT - 1) / LU_NT)), dim3(LU_NT), 0, st, S, Fc, vals);
}
template <class T>
void launch_lu_cmod(const LuSymDev& S, const LuFacDev<T>& Fc, const LuItem* items, int nitems, const CTask* tasks,
                    hipStream_t st) {
  if (nitems <= 0) return;
  if constexpr (sizeof(T) == 8)
    hipLaunchKernelGGL(k_lu_cmod_mfma, dim3((unsigned)nitems), dim3(LU_NT), 0, st, S, Fc, items, tasks);
  else
    hipLaunchKernelGGL(k_lu_cmod_mfma_c64, dim3((unsigned)nitems), dim3(LU_NT), 0, st, S, Fc, items, tasks);
}
template <class T>
void launch_lu_getf2(const LuSymDev& S, const LuFacDev<T>& Fc, const LuUnit* units, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lu_getf2<T>, dim3((unsigned)n), dim3(LU_GT), 0, st, S, Fc, units);
}
template <class T>
void launch_lu_apply(const LuSymDev& S, const LuFacDev<T>& Fc, const LuUnit* units, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lu_apply<T>, dim3((unsigned)n), dim3(LU_COLS), 0, st, S, Fc, units);
}
template <class T>
void launch_lu_gemm(const LuSymDev& S, const LuFacDev<T>& Fc, const LuUnit* units, int n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_lu_gemm<T>, dim3((unsigned)n), dim3(LU_NT), 0, st, S, Fc, units);
}
template <class T>
void launch_lu_sprep(int32_t n, int32_t nrhs, const int32_t* perm, const double* d_row, const T* b, T* bh,
                     hipStream_t st) {
  const int64_t m = (int64_t)n * nrhs;
  if (m <= 0) return;
  hipLaunchKernelGGL(k_lu_sprep<T>, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, n, nrhs, perm, d_row, b, bh);
}
template <class T>
void launch_lu_sfinish(int32_t n, int32_t nrhs, const int32_t* perm, const double* d_col, const T* y, T* x,
                       hipStream_t st) {
  const int64_t m = (int64_t)n * nrhs;
  if (m <= 0) return;
  hipLaunchKernelGGL(k_lu_sfinish<T>, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, n, nrhs, perm, d_col, y, x);
}
// kind: 0 gather (into y), 1 forward block step (y -> yo), 3 backward U12
// terms (on y, x of the ancestors in yo), 4 backward block step (y -> yo)
template <class T>
void launch_lu_sstep(int kind, const LuSymDev& S, const LuFacDev<T>& Fc, const LuUnit* units, int n, int32_t nrhs,
                     const T* bh, T* scr, T* y, T* yo, hipStream_t st) {
  if (n <= 0) return;
  const dim3 g((unsigned)n), b(LU_NT);
  switch (kind) {
    case 0: hipLaunchKernelGGL(k_lu_fgather<T>, g, b, 0, st, S, Fc, units, nrhs, bh, scr, y); break;
    case 1: hipLaunchKernelGGL((k_lu_fstep<T>), g, b, 0, st, S, Fc, units, nrhs, y, yo, scr); break;
    case 3: hipLaunchKernelGGL(k_lu_boff<T>, g, b, 0, st, S, Fc, units, nrhs, y, yo); break;
    default: hipLaunchKernelGGL((k_lu_bstep<T>), g, b, 0, st, S, Fc, units, nrhs, y, yo); break;
  }
}

#define RSL_LU_INST(T)                                                                                          \
  template void launch_lu_assemble<T>(const LuSymDev&, const LuFacDev<T>&, const T*, hipStream_t);              \
  template void launch_lu_cmod<T>(const LuSymDev&, const LuFacDev<T>&, const LuItem*, int, const CTask*,         \
                                  hipStream_t);                                                                 \
  template void launch_lu_getf2<T>(const LuSymDev&, const LuFacDev<T>&, const LuUnit*, int, hipStream_t);       \
  template void launch_lu_apply<T>(const LuSymDev&, const LuFacDev<T>&, const LuUnit*, int, hipStream_t);       \
  template void launch_lu_gemm<T>(const LuSymDev&, const LuFacDev<T>&, const LuUnit*, int, hipStream_t);        \
  template void launch_lu_sprep<T>(int32_t, int32_t, const int32_t*, const double*, const T*, T*, hipStream_t);  \
  template void launch_lu_sfinish<T>(int32_t, int32_t, const int32_t*, const double*, const T*, T*, hipStream_t); \
  template void launch_lu_sstep<T>(int, const LuSymDev&, const LuFacDev<T>&, const LuUnit*, int, int32_t, const T*, \
                                   T*, T*, T*, hipStream_t);
RSL_LU_INST(double)
RSL_LU_INST(cplx)

}  // namespace rsl
