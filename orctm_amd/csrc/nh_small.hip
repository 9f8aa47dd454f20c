// nh_small.hip -- the inner PCG iteration of launches of few columns.
//
// A system of a few thousand columns leaves the streaming kernels (nh_kernels.hip: one column per lane,
// marching over the levels) with a handful of wavefronts, each a chain of dependent memory round trips: on
// 512x4x100 a mixed iteration took 75 us for 10 MB of data. Here a block of 12 wavefronts takes WC columns of
// one row with all their levels: its threads load and store the levels side by side, and only the
// recurrences that must run level by level -- the line solve's two sweeps and the sums along a column --
// run in one wavefront each, out of LDS, at an instruction's latency per level instead of a memory round trip.
//
//   k_col   r -= alpha q, both sweeps of the line solve (z), r.z and r.r
//   k_mv    p = z + beta p_old, x += alpha p_old, q = C p, p.q
//
// z goes to memory whole, so the matvec's neighbours need no recurrence of their own: p of the rows to the
// north and south is z + beta p_old of two loads.
//
// The scalars are folded into the kernels: every block forms the system totals from the sums that the
// kernel before it left (their loads go out before its own data's), and one block of the system writes the
// new state to the other of two copies, as other blocks may still read the old one. So an iteration is two
// launches, not four. The values are the streaming kernels' bit for bit: the same operations per cell and
// along a column, and the same tree over a row of 64, over groups of 4 rows and over the groups' slots.
//
// WC = 64 leaves the sums of its row (one value a block). WC = 32 and 16, for systems that would not fill the
// device with 64, leave the columns' sums, and the totals begin with the rows' trees: 2 or 4 times as many
// blocks share the loads (one CU draws about 55 GB/s from beyond its L2), for a few more reads each.
#include "nh_dev.h"
#include "nh_small.h"

namespace onh {
namespace {

constexpr int NW = 12;  // wavefronts of a block: k_reduce's, whose order the totals keep
constexpr int NS = 64 * NW;
static_assert(NS == NT, "the totals' order is that of k_reduce");
constexpr int kBatch = kSmallBatch;
__host__ __device__ constexpr int padded(int nz) { return (nz + kBatch - 1) / kBatch * kBatch; }

enum { SUMS_MATVEC = 0, SUMS_UPDATE = 1 };

// A kernel's sums: 2 values for each row of 64 columns (WC = 64) or each column (WC < 64).
template <typename T, int WC>
__device__ __forceinline__ gptr<T> sums_of(const Sys& s, int which) {
  return G<T>(s.rowsum) + (size_t)which * 2 * s.tiles_x * s.ny * (WC == 64 ? 1 : 64);
}

// Block -> place. One system: from the block's number, each XCD (which gets every 8th block) a contiguous run
// of places; several: from the list.
struct Place {
  int sys, bx, j;
};
template <int WC>
__device__ __forceinline__ Place place_of(int tiles_x) {
  const int nb = gridDim.x, b = blockIdx.x, per = nb >> 3, rem = nb & 7, x = b & 7;
  const int n = x * per + (x < rem ? x : rem) + (b >> 3), w = tiles_x * (64 / WC);
  const int j = n / w;
  return Place{0, n - j * w, j};
}

// The system totals in every thread: thread t sums the slots t, t + NS, ... of 4 rows each, then block_sum2
// (the order of k_reduce). The first sums are loaded by the constructor.
template <typename T, int WC>
struct Totals {
  static constexpr int RU = 3;  // rows per wavefront loaded ahead (WC < 64)
  gptr<const T> part;
  const Sys& s;
  T va[4], vb[4];
  __device__ void slot(int t) {
    const int g = t / s.tiles_x, bx = t - g * s.tiles_x;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * g + q, rr = row < s.ny ? row : s.ny - 1;
      const size_t n = 2 * ((size_t)rr * s.tiles_x + bx);
      const T x = part[n], y = part[n + 1];
      va[q] = row < s.ny ? x : T(0);
      vb[q] = row < s.ny ? y : T(0);
    }
  }
  __device__ Totals(const Sys& sys, int which) : part(sums_of<T, WC>(sys, which)), s(sys) {
    if constexpr (WC == 64) {
      const int t = s.nslots <= 64 ? threadIdx.x & 63 : threadIdx.x;
      slot(t < s.nslots ? t : 0);
    } else {
      const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, rows = s.tiles_x * s.ny;
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const int r = wv + NW * u < rows ? wv + NW * u : 0;
        va[u] = part[2 * ((size_t)r * 64 + lane)];
        vb[u] = part[2 * ((size_t)r * 64 + lane) + 1];
      }
    }
  }
  __device__ void get(T& a, T& b) {
    __shared__ T all[2];
    a = T(0);
    b = T(0);
    // up to 64 slots all lie with the first wavefront (the others' sums are 0): every wavefront forms them itself
    const bool few = s.nslots <= 64;
    if constexpr (WC == 64) {
      if (few) {
        const bool in = (threadIdx.x & 63) < s.nslots;
        a = T(0) + wave_sum(in ? T(0) + ((va[0] + va[1]) + (va[2] + va[3])) : T(0));
        b = T(0) + wave_sum(in ? T(0) + ((vb[0] + vb[1]) + (vb[2] + vb[3])) : T(0));
        return;
      }
      for (int t = threadIdx.x; t < s.nslots; t += NS) {
        if (t >= NS) slot(t);
        a += (va[0] + va[1]) + (va[2] + va[3]);
        b += (vb[0] + vb[1]) + (vb[2] + vb[3]);
      }
    } else {
      __shared__ T rs[2][kSmallColumns / 64];
      const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, rows = s.tiles_x * s.ny;
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const T x = wave_sum(va[u]), y = wave_sum(vb[u]);
        if (lane == 0 && wv + NW * u < rows) {
          rs[0][wv + NW * u] = x;
          rs[1][wv + NW * u] = y;
        }
      }
      for (int r = wv + NW * RU; r < rows; r += NW) {
        const T x = wave_sum(part[2 * ((size_t)r * 64 + lane)]), y = wave_sum(part[2 * ((size_t)r * 64 + lane) + 1]);
        if (lane == 0) {
          rs[0][r] = x;
          rs[1][r] = y;
        }
      }
      __syncthreads();
      for (int t = few ? lane : threadIdx.x; t < s.nslots; t += NS) {
        const int g = t / s.tiles_x, bx = t - g * s.tiles_x;
        T wa[4], wb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = 4 * g + q;
          wa[q] = row < s.ny ? rs[0][row * s.tiles_x + bx] : T(0);
          wb[q] = row < s.ny ? rs[1][row * s.tiles_x + bx] : T(0);
        }
        a += (wa[0] + wa[1]) + (wa[2] + wa[3]);
        b += (wb[0] + wb[1]) + (wb[2] + wb[3]);
      }
      if (few) {
        a = T(0) + wave_sum(a);
        b = T(0) + wave_sum(b);
        return;
      }
    }
    block_sum2<T, NW>(a, b);
    if (threadIdx.x == 0) {
      all[0] = a;
      all[1] = b;
    }
    __syncthreads();
    a = all[0];
    b = all[1];
  }
};

// The sums of this block's columns, by one wavefront whose lane c < WC holds column c's.
template <typename T, int WC>
__device__ __forceinline__ void put_sums(const Sys& s, int which, const Place& at, bool ok, T a, T b) {
  const int c = threadIdx.x & 63;
  a = ok ? a : T(0);
  b = ok ? b : T(0);
  gptr<T> p = sums_of<T, WC>(s, which);
  if constexpr (WC == 64) {
    a = wave_sum(a);
    b = wave_sum(b);
    if (c == 0) {
      const size_t n = 2 * ((size_t)at.j * s.tiles_x + at.bx);
      p[n] = a;
      p[n + 1] = b;
    }
  } else if (c < WC) {
    const size_t n = 2 * ((size_t)at.j * s.tiles_x * 64 + at.bx * WC + c);
    p[n] = a;
    p[n + 1] = b;
  }
}

// A recurrence down or up a column in LDS, in batches of kBatch levels: a batch is read while the one before is
// worked on. ld(k, u) reads level k into slot u of the batch in hand's other half, op(k, u) works on it.
template <bool DOWN, typename Ld, typename Op>
__device__ __forceinline__ void sweep(int nzp, Ld&& ld, Op&& op) {
  constexpr int B = kBatch;
  auto load = [&](int k0, auto half) {
    const int kk = k0 < 0 ? 0 : k0 < nzp ? k0 : nzp - B;
#pragma unroll
    for (int u = 0; u < B; ++u) ld(kk + u, decltype(half)::value * B + u);
  };
  auto run = [&](int k0, auto half) {
#pragma unroll
    for (int v = 0; v < B; ++v) {
      const int u = DOWN ? v : B - 1 - v;
      op(k0 + u, decltype(half)::value * B + u);
    }
  };
  constexpr std::integral_constant<int, 0> H0{};
  constexpr std::integral_constant<int, 1> H1{};
  const int n = nzp / B;
  auto at = [&](int q) { return DOWN ? q * B : nzp - B - q * B; };
  load(at(0), H0);
  for (int q = 0; q < n; q += 2) {
    load(at(q + 1), H1);
    run(at(q), H0);
    if (q + 1 >= n) break;
    load(at(q + 2), H0);
    run(at(q + 1), H1);
  }
}

// U: levels (and the padding's) per thread at most. ONE: the launch's only system is passed by value and its places follow from
// the blocks' numbers, which spares every kernel two dependent reads (about 1 us).
template <typename T, int WC, int U, bool ONE, bool INIT>
__global__ __launch_bounds__(NS) void k_col(const Sys one, const Sys* __restrict__ systems,
                                            const Tile* __restrict__ tiles, int nzmax) {
  extern __shared__ __align__(16) char raw[];
  constexpr int LV = NS / WC;  // levels side by side
  T* R = reinterpret_cast<T*>(raw);  // r, then z
  T* L = R + (size_t)nzmax * WC;
  T* Y = L + (size_t)nzmax * WC;
  T* W = Y + (size_t)nzmax * WC;
  using FS = typename Fac<T>::S;
  Place at;
  if constexpr (ONE) at = place_of<WC>(one.tiles_x);
  else at = Place{tiles[blockIdx.x].sys, tiles[blockIdx.x].bx, tiles[blockIdx.x].by};
  const Sys& s = ONE ? one : systems[at.sys];
  const int c = threadIdx.x & (WC - 1), lev = threadIdx.x / WC;
  const int i = at.bx * WC + c, nz = s.nz, nzp = padded(nz);
  const bool ok = i < s.nx;
  const size_t P = s.plane, col = (size_t)at.j * s.pitch + (ok ? i : s.nx - 1);
  const bool writer = at.bx == 0 && at.j == 0 && threadIdx.x == 0;
  Outer* o = s.outer;
  Inner<T> in;
  if (!INIT) in = *reinterpret_cast<const Inner<T>*>(s.inner);
  Totals<T, WC> tot(s, SUMS_MATVEC);
  gptr<T> r = G<T>(s.r);
  gptr<const T> q = G<const T>(s.q);
  gptr<const FS> Lg = G<const FS>(s.L), Dg = G<const FS>(s.invD);
  T rk[U], qk[U];
  FS lk[U], dk[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    const size_t idx = col + (size_t)(k < nz ? k : nz - 1) * P;
    rk[u] = r[idx];
    if (!INIT) qk[u] = q[idx];
    lk[u] = Lg[idx];
    dk[u] = Dg[idx];
  }
  T cs = T(1);
  if constexpr (std::is_same<T, float>::value) cs = G<const float>(s.dscale)[col];
  T alpha = T(0);
  if (INIT) {
    if (o->odone != RUN) return;
  } else {
    Inner<T>* next = reinterpret_cast<Inner<T>*>(s.inner2);
    if (in.done != RUN) {
      if (writer) *next = in;
      return;
    }
    T pq, unused;
    tot.get(pq, unused);
    inner_after_matvec(in, pq);
    if (writer) {
      *next = in;
      if (in.done == BREAKDOWN && in.iter == 0) o->odone = BREAKDOWN;
    }
    if (in.done != RUN) return;
    alpha = in.alpha;
  }
  // levels nz .. nzp - 1 pad the sweeps to whole batches: r = l = 1/D = 0 there adds nothing to the sums
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    if (k < nz) {
      if (INIT) {
        if (ok) G<T>(s.x)[col + (size_t)k * P] = T(0);
      } else {
        rk[u] = fmad(-alpha, qk[u], rk[u]);
        if (ok) r[col + (size_t)k * P] = rk[u];
      }
      R[k * WC + c] = rk[u];
      L[k * WC + c] = Fac<T>::dec(lk[u]);
    } else if (k < nzp) {
      R[k * WC + c] = T(0);
      L[k * WC + c] = T(0);
      Y[k * WC + c] = T(0);
      W[k * WC + c] = T(0);
    }
  }
  __syncthreads();
  // forward elimination (wavefront 0) beside r.r (wavefront 1)
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  T rr = T(0);
  if (wv == 0 && lane < WC) {
    T vr[2 * kBatch], vl[2 * kBatch], y = T(0);
    sweep<true>(nzp, [&](int k, int u) { vr[u] = R[k * WC + lane], vl[u] = L[k * WC + lane]; },
                [&](int k, int u) {
                  y = fmad(-vl[u], y, vr[u]);
                  Y[k * WC + lane] = y;
                });
  } else if (wv == 1 && lane < WC) {
    T vr[2 * kBatch];
    sweep<true>(nzp, [&](int k, int u) { vr[u] = R[k * WC + lane]; }, [&](int, int u) { rr = fmad(vr[u], vr[u], rr); });
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    if (k < nz) W[k * WC + c] = Y[k * WC + c] * (Fac<T>::dec(dk[u]) * cs);
  }
  __syncthreads();
  // back substitution (wavefront 0) beside r.z (wavefront 1)
  if (wv == 0 && lane < WC) {
    T vw[2 * kBatch], vl[2 * kBatch], z = T(0), l = T(0);
    sweep<false>(nzp, [&](int k, int u) { vw[u] = W[k * WC + lane], vl[u] = L[k * WC + lane]; },
                 [&](int k, int u) {
                   z = fmad(-l, z, vw[u]);
                   l = vl[u];
                   R[k * WC + lane] = z;
                 });
  } else if (wv == 1) {
    T vy[2 * kBatch], vw[2 * kBatch], rho = T(0);
    if (lane < WC)
      sweep<true>(nzp, [&](int k, int u) { vy[u] = Y[k * WC + lane], vw[u] = W[k * WC + lane]; },
                  [&](int, int u) { rho = fmad(vy[u], vw[u], rho); });
    put_sums<T, WC>(s, SUMS_UPDATE, at, lane < WC && at.bx * WC + lane < s.nx, rho, rr);
  }
  __syncthreads();
  gptr<T> zg = G<T>(s.z);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    if (k < nz && ok) zg[col + (size_t)k * P] = R[k * WC + c];
  }
}

// FOLD: the column update before it was an iteration's, and its scalars are formed here.
template <typename T, int WC, int U, bool ONE, bool FOLD>
__global__ __launch_bounds__(NS) void k_mv(const Sys one, const Sys* __restrict__ systems,
                                           const Tile* __restrict__ tiles, int nzmax) {
  extern __shared__ __align__(16) char raw[];
  constexpr int LV = NS / WC, LP = WC + 2;
  T* Pl = reinterpret_cast<T*>(raw);  // p of the block's columns and one on either side
  T* A = Pl + (size_t)nzmax * LP;     // C p
  Place at;
  if constexpr (ONE) at = place_of<WC>(one.tiles_x);
  else at = Place{tiles[blockIdx.x].sys, tiles[blockIdx.x].bx, tiles[blockIdx.x].by};
  const Sys& s = ONE ? one : systems[at.sys];
  const int c = threadIdx.x & (WC - 1), lev = threadIdx.x / WC;
  const int nx = s.nx, ny = s.ny, nz = s.nz, nzp = padded(nz), i0 = at.bx * WC, i = i0 + c, j = at.j;
  const size_t P = s.plane, IP = s.pitch;
  const bool active = i < nx;
  const bool writer = at.bx == 0 && at.j == 0 && threadIdx.x == 0;
  Outer* o = s.outer;
  Inner<T> in = *reinterpret_cast<const Inner<T>*>(FOLD ? s.inner2 : s.inner);
  Totals<T, WC> tot(s, SUMS_UPDATE);
  // own column (past the domain's end: the periodic image, or p = 0), the rows to the north and south, and
  // one column west and east of the block for 2 threads of each level
  int mi = i, mj = j;
  const bool val = map_ij(mi, mj, nx, ny, s.cyc_x, s.cyc_y);
  const int ci = val ? mi : 0;
  const size_t col = (size_t)j * IP + ci;
  int ni = 0, nj = j - 1, si = 0, sj = j + 1;
  const bool hn = map_ij(ni, nj, nx, ny, s.cyc_x, s.cyc_y), hs = map_ij(si, sj, nx, ny, s.cyc_x, s.cyc_y);
  const size_t cn = (size_t)(hn ? nj : j) * IP + ci, cs = (size_t)(hs ? sj : j) * IP + ci;
  const int ek = threadIdx.x >> 1, eside = threadIdx.x & 1;
  int ei = eside ? i0 + WC : i0 - 1, ej = j;
  const bool ev = ek < nz && map_ij(ei, ej, nx, ny, s.cyc_x, s.cyc_y);
  const size_t ce = ev ? (size_t)ek * P + (size_t)j * IP + ei : 0;
  gptr<const T> z = G<const T>(s.z);
  gptr<T> x = G<T>(s.x);
  T zk[U], pk[U], xk[U];
  const T ze = z[ce];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    const size_t idx = col + (size_t)(k < nz ? k : nz - 1) * P;
    zk[u] = z[idx];
    xk[u] = x[idx];
  }
  const int pb = in.pbuf ^ (FOLD ? 1 : 0);
  gptr<const T> pold = G<const T>(pb ? s.pb : s.pa);
  gptr<T> pnew = G<T>(pb ? s.pa : s.pb);
  const T pe = pold[ce];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    pk[u] = pold[col + (size_t)(k < nz ? k : nz - 1) * P];
  }
  // row data and neighbours' z and p_old, a batch of levels ahead of their use
  constexpr int UB = sizeof(T) == 4 ? (U < 5 ? U : 5) : (U < 3 ? U : 3);
  struct Row {
    T zn, pn, zs, ps, zw, zw1, zp;
    unsigned f;
  };
  Row ra[UB], rb[UB];
  const bool tab = s.tab != 0;
  ZCol<T> zcol;
  T cc[7];
  {
    gptr<const T> cpi = G<const T>(s.col_in);
#pragma unroll
    for (int m = 0; m < 7; ++m) cc[m] = cpi[m * P + col];
    if (tab)
      zcol.load(G<const T>(s.tw_in), G<const T>(s.tp_in), s.xk, G<const T>(s.xw_in), G<const T>(s.xp_in), s.xf, P, col);
  }
  gptr<const T> zwi = G<const T>(s.zw_in), zpi = G<const T>(s.zp_in);
  gptr<const uint16_t> flg = G<const uint16_t>(s.flg);
  auto load_rows = [&](int u0, Row* rd) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int kr = lev + LV * (u0 + u), k = kr < nz ? kr : nz - 1;
      const size_t o3 = (size_t)k * P;
      rd[u].zn = z[cn + o3];
      rd[u].pn = pold[cn + o3];
      rd[u].zs = z[cs + o3];
      rd[u].ps = pold[cs + o3];
      if (tab) {
        rd[u].zw = zcol.tw[k];
        rd[u].zw1 = zcol.tw[k + 1];
        rd[u].zp = zcol.tp[k];
      } else {
        rd[u].zw = zwi[col + o3];
        rd[u].zw1 = zwi[col + o3 + P];
        rd[u].zp = zpi[col + o3];
      }
      rd[u].f = flg[col + o3];
    }
  };
  load_rows(0, ra);
  if (FOLD) {
    Inner<T>* next = reinterpret_cast<Inner<T>*>(s.inner);
    if (in.done != RUN) {
      if (writer) *next = in;
      return;
    }
    T rho, rr;
    tot.get(rho, rr);
    inner_after_update(in, rho, rr);
    if (writer) {
      *next = in;
      o->inner_total += 1;
    }
  }
  if (in.done != RUN) return;
  const bool first = in.first != 0;
  const T beta = in.beta, alpha = in.alpha;
  auto dir = [&](T zv, T pv) { return first ? zv : fmad(beta, pv, zv); };
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = lev + LV * u;
    if (k < nz) {
      const size_t idx = col + (size_t)k * P;
      const T pm = dir(zk[u], pk[u]);
      Pl[k * LP + c + 1] = val ? pm : T(0);
      if (active) {
        pnew[idx] = pm;
        if (!first) x[idx] = fmad(alpha, pk[u], xk[u]);
      }
    } else if (k < nzp) {  // pads the sum below to whole batches
      Pl[k * LP + c + 1] = T(0);
      A[k * WC + c] = T(0);
    }
  }
  if (ek < nz) Pl[ek * LP + (eside ? LP - 1 : 0)] = ev ? dir(ze, pe) : T(0);
  if (U > UB) load_rows(UB, rb);
  __syncthreads();
  gptr<T> q = G<T>(s.q);
  auto rows = [&](int u0, const Row* rd) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int k = lev + LV * (u0 + u);
      if (u0 + u < U && k < nz) {
        const T* pc = Pl + k * LP + c + 1;
        const T zwk = tab ? zcol.template zw_or<true>(k, rd[u].zw) : rd[u].zw, zwk1 = tab ? zcol.template zw_or<true>(k + 1, rd[u].zw1) : rd[u].zw1;
        const T zpk = tab ? zcol.template zp_or<true>(k, rd[u].zp) : rd[u].zp;
        T c7[7];
        inner_row<T, true>(cc, zwk, zwk1, zpk, rd[u].f, c7);
        T acc = c7[0] * pc[0];
        acc = fmad(c7[1], pc[-1], acc);
        acc = fmad(c7[2], pc[1], acc);
        acc = fmad(c7[3], hn ? dir(rd[u].zn, rd[u].pn) : T(0), acc);
        acc = fmad(c7[4], hs ? dir(rd[u].zs, rd[u].ps) : T(0), acc);
        acc = fmad(c7[5], k > 0 ? pc[-LP] : T(0), acc);
        acc = fmad(c7[6], k < nz - 1 ? pc[LP] : T(0), acc);
        if (active) q[col + (size_t)k * P] = acc;
        A[k * WC + c] = acc;
      }
    }
  };
#pragma unroll
  for (int u0 = 0; u0 < U; u0 += 2 * UB) {
    rows(u0, ra);
    if (u0 + UB >= U) break;
    if (u0 + 2 * UB < U) load_rows(u0 + 2 * UB, ra);
    rows(u0 + UB, rb);
    if (u0 + 3 * UB < U) load_rows(u0 + 3 * UB, rb);
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (wv == 0) {  // p.q along the columns, bottom-up
    T vp[2 * kBatch], vq[2 * kBatch], dot = T(0);
    if (lane < WC)
      sweep<false>(nzp, [&](int k, int u) { vp[u] = Pl[k * LP + lane + 1], vq[u] = A[k * WC + lane]; },
                   [&](int, int u) { dot = fmad(vp[u], vq[u], dot); });
    put_sums<T, WC>(s, SUMS_MATVEC, at, lane < WC && i0 + lane < nx, dot, T(0));
  }
}

// The scalars of the last column update of a run (or of the first one of an inner solve), one block per system.
template <typename T, int WC, bool INIT>
__global__ __launch_bounds__(NS) void k_end(const Sys* __restrict__ systems) {
  const Sys& s = systems[blockIdx.x];
  Outer* o = s.outer;
  Inner<T>* dst = reinterpret_cast<Inner<T>*>(s.inner);
  Inner<T> in = *reinterpret_cast<const Inner<T>*>(INIT ? s.inner : s.inner2);
  Totals<T, WC> tot(s, SUMS_UPDATE);
  if (INIT && o->odone != RUN) return;
  if (!INIT && in.done != RUN) {
    if (threadIdx.x == 0) *dst = in;
    return;
  }
  T rho, rr;
  tot.get(rho, rr);
  if (threadIdx.x != 0) return;
  if (INIT) {
    inner_begin(in, rho, rr);
    if (in.done == BREAKDOWN) o->odone = BREAKDOWN;
  } else {
    inner_after_update(in, rho, rr);
    o->inner_total += 1;
  }
  *dst = in;
}

size_t col_lds(const SmallLaunch& l) { return (size_t)padded(l.nz) * 4 * l.wc * (l.fp32 ? 4 : 8); }
size_t mv_lds(const SmallLaunch& l) { return (size_t)padded(l.nz) * (2 * l.wc + 2) * (l.fp32 ? 4 : 8); }

template <int V>
using Int = std::integral_constant<int, V>;

// f(WC, U, ONE): the form of a launch, U at least the levels per thread.
template <typename F>
hipError_t by_form(const SmallLaunch& l, F&& f) {
  const int u = (padded(l.nz) * l.wc + NS - 1) / NS;
  if (l.wc == 16 && l.one) {
    if (u <= 1) return f(Int<16>{}, Int<1>{}, std::true_type{});
    if (u <= 3) return f(Int<16>{}, Int<3>{}, std::true_type{});
    if (u <= 5) return f(Int<16>{}, Int<5>{}, std::true_type{});
  } else if (l.wc == 32 && l.one) {
    if (u <= 3) return f(Int<32>{}, Int<3>{}, std::true_type{});
    if (u <= 5) return f(Int<32>{}, Int<5>{}, std::true_type{});
    if (u <= 9) return f(Int<32>{}, Int<9>{}, std::true_type{});
  } else if (l.wc == 64 && l.one) {
    if (u <= 3) return f(Int<64>{}, Int<3>{}, std::true_type{});
    if (u <= 5) return f(Int<64>{}, Int<5>{}, std::true_type{});
    if (u <= 9) return f(Int<64>{}, Int<9>{}, std::true_type{});
    if (u <= 13) return f(Int<64>{}, Int<13>{}, std::true_type{});
  } else if (l.wc == 64) {
    if (u <= 3) return f(Int<64>{}, Int<3>{}, std::false_type{});
    if (u <= 5) return f(Int<64>{}, Int<5>{}, std::false_type{});
    if (u <= 9) return f(Int<64>{}, Int<9>{}, std::false_type{});
    if (u <= 13) return f(Int<64>{}, Int<13>{}, std::false_type{});
  }
  return hipErrorInvalidValue;
}

template <typename T, bool INIT>
hipError_t col(hipStream_t st, const SmallLaunch& l) {
  return by_form(l, [&](auto wc, auto u, auto one) {
    hipLaunchKernelGGL((k_col<T, decltype(wc)::value, decltype(u)::value, decltype(one)::value, INIT>),
                       dim3(l.nblocks), dim3(NS), col_lds(l), st, l.sys, l.d_sys, l.d_rows, padded(l.nz));
    return hipGetLastError();
  });
}

template <typename T, bool FOLD>
hipError_t mv(hipStream_t st, const SmallLaunch& l) {
  return by_form(l, [&](auto wc, auto u, auto one) {
    hipLaunchKernelGGL((k_mv<T, decltype(wc)::value, decltype(u)::value, decltype(one)::value, FOLD>),
                       dim3(l.nblocks), dim3(NS), mv_lds(l), st, l.sys, l.d_sys, l.d_rows, padded(l.nz));
    return hipGetLastError();
  });
}

template <typename T, bool INIT>
hipError_t end(hipStream_t st, const SmallLaunch& l) {
  if (l.wc < 64) hipLaunchKernelGGL((k_end<T, 16, INIT>), dim3(l.nsys), dim3(NS), 0, st, l.d_sys);
  else hipLaunchKernelGGL((k_end<T, 64, INIT>), dim3(l.nsys), dim3(NS), 0, st, l.d_sys);
  return hipGetLastError();
}

template <typename T>
hipError_t setup(const SmallLaunch& l) {
  return by_form(l, [&](auto wc, auto u, auto one) {
    constexpr int WC = decltype(wc)::value, U = decltype(u)::value;
    constexpr bool ONE = decltype(one)::value;
    const void* fs[] = {(const void*)&k_col<T, WC, U, ONE, true>, (const void*)&k_col<T, WC, U, ONE, false>,
                        (const void*)&k_mv<T, WC, U, ONE, true>, (const void*)&k_mv<T, WC, U, ONE, false>};
    for (const void* f : fs) {
      const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  });
}

template <typename T>
hipError_t begin(hipStream_t st, const SmallLaunch& l) {
  const hipError_t e = col<T, true>(st, l);
  return e != hipSuccess ? e : end<T, true>(st, l);
}

template <typename T>
hipError_t iterations(hipStream_t st, const SmallLaunch& l, int n) {
  hipError_t e = hipSuccess;
  for (int it = 0; it < n && e == hipSuccess; ++it) {
    e = it ? mv<T, true>(st, l) : mv<T, false>(st, l);
    if (e == hipSuccess) e = col<T, false>(st, l);
  }
  return e != hipSuccess ? e : end<T, false>(st, l);
}

}  // namespace

hipError_t small_setup(const SmallLaunch& l) { return l.fp32 ? setup<float>(l) : setup<double>(l); }

hipError_t small_begin(hipStream_t st, const SmallLaunch& l) {
  return l.fp32 ? begin<float>(st, l) : begin<double>(st, l);
}

hipError_t small_iterations(hipStream_t st, const SmallLaunch& l, int n) {
  return l.fp32 ? iterations<float>(st, l, n) : iterations<double>(st, l, n);
}

hipError_t small_matvec(hipStream_t st, const SmallLaunch& l) {
  return l.fp32 ? mv<float, false>(st, l) : mv<double, false>(st, l);
}

hipError_t small_update(hipStream_t st, const SmallLaunch& l) {
  return l.fp32 ? col<float, false>(st, l) : col<double, false>(st, l);
}

hipError_t small_finish(hipStream_t st, const SmallLaunch& l) {
  return l.fp32 ? end<float, false>(st, l) : end<double, false>(st, l);
}

}  // namespace onh
