// nh_stream.hip -- the two kernels of an inner PCG iteration on launches of many columns.
//
// k_update takes a column down and up again: r -= alpha q and the forward elimination, w kept in registers, then the
// back substitution, which leaves z in memory. k_matvec takes p = z + beta p_old from z of the column and of its
// neighbours, so that it needs no line solve of halo columns, no LDS and no barrier. Both move 12 words and 2 factors
// a cell and iteration, as the tiled pair does (z written and read in place of w).
//
// What bounds them is memory: 1024x768x60 in FP32 runs at 4.9 TB/s of a copy's 6.1 with every level read. So each
// column stops at the levels in use (Sys::use): its depth, or what r holds below it, made equal over 64 bytes of a
// row so that stores fill whole pieces. Dry cells have no couplings: where r is 0 the rest of their vectors is 0 and
// adds nothing to a sum, hence the same values (a zero's sign apart). The other loss was the pipeline of loads, which
// a chain of ?: or an exit in the middle of the loop empties (the compiler waits for every load where paths meet):
// selects one after the other, whole turns of the ring of levels, and the loads of a level fixed in place before its
// arithmetic.
//
// us per iteration (matvec + update), tiled -> these, on basins of 0.5 to 0.6 wet cells: 1024x768x60 mixed 270 + 168
// -> 220 + 156, FP64 535 + 429 -> 429 + 336; 512x443x49 74 + 65 -> 62 + 41, FP64 144 + 90 -> 116 + 87; 203x194x35
// 26 + 14 -> 20 + 15, FP64 45 + 22 -> 24 + 18. Blocks of 8 or 12 rows, in step by a barrier a level, re-read fewer
// rows but end with their deepest: 234 instead of 220.
#include "nh_dev.h"
#include "nh_stream.h"

namespace onh {
namespace {

constexpr int H = kOuterRows;  // rows of a block: a wavefront each
constexpr int NZ = kStreamLevels;

// FP32: pairs of tiles from which a lane takes two columns, which halves the memory instructions, instead of one, which
// doubles the wavefronts. us per iteration with one and with two: 384x384x40 (288 pairs) 77 and 84, 448x448x45 (392)
// 107 and 107, 512x443x49 (444) 131 and 122.
constexpr int kPairs = 400;

// V adjacent columns of a lane.
template <typename T, int V>
struct Vec {
  typedef T type __attribute__((ext_vector_type(V)));
};
template <typename T>
struct Vec<T, 1> {
  typedef T type;
};
template <typename T, int V>
using vec = typename Vec<T, V>::type;

template <typename T, int V>
__device__ __forceinline__ T get(const vec<T, V>& v, int c) {
  if constexpr (V == 1) return v;
  else return v[c];
}
template <typename T, int V>
__device__ __forceinline__ void put(vec<T, V>& v, int c, T x) {
  if constexpr (V == 1) v = x;
  else v[c] = x;
}

// Loads and stores through a descriptor: vo the lane's byte offset, so the level's.
template <typename E, int AUX>
__device__ __forceinline__ E ldb(Rsrc r, uint32_t vo, uint32_t so) {
  if constexpr (sizeof(E) == 2) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b16(r, vo, so, AUX));
  else if constexpr (sizeof(E) == 4) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, AUX));
  else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, AUX));
}
template <typename E, int AUX>
__device__ __forceinline__ void stb(Rsrc r, uint32_t vo, uint32_t so, E v) {
  typedef unsigned int U2 __attribute__((ext_vector_type(2)));
  if constexpr (sizeof(E) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, vo, so, AUX);
  else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, vo, so, AUX);
}

template <typename T>
__device__ __forceinline__ T half_sum(T v) {
  return fold_add<1>(fold_add<2>(fold_add<4>(fold_add<8>(fold_add<16>(v)))));
}

// Row sums of a block (wavefront w: row w of its tile, or of both tiles of its pair) to the 4-row slots.
template <typename T, int V>
__device__ __forceinline__ void publish(const Sys& s, const Tile& t, bool vert, const T* a, const T* b) {
  __shared__ T sh[2][2 * H];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  T x, y;
  if constexpr (V == 1) {
    x = wave_sum(a[0]);
    y = wave_sum(b[0]);
    if (l == 0) sh[0][w] = x, sh[0][H + w] = y;
  } else {
    x = half_sum(a[0]) + half_sum(a[1]);
    y = half_sum(b[0]) + half_sum(b[1]);
    if ((l & 31) == 0) sh[l >> 5][w] = x, sh[l >> 5][H + w] = y;
  }
  __syncthreads();
  if (threadIdx.x < V * (H / RG)) {
    const int half = threadIdx.x / (H / RG), g = threadIdx.x % (H / RG);
    const int grow = (t.by + (vert ? half : 0)) * (H / RG) + g, tx = t.bx + (vert ? 0 : half);
    if (grow * RG < s.ny && tx < s.tiles_x) {
      const T* v = sh[half];
      gptr<T> part = G<T>(s.partials);
      const size_t slot = (size_t)grow * s.tiles_x + tx;
      part[2 * slot] = (v[4 * g] + v[4 * g + 1]) + (v[4 * g + 2] + v[4 * g + 3]);
      part[2 * slot + 1] = (v[H + 4 * g] + v[H + 4 * g + 1]) + (v[H + 4 * g + 2] + v[H + 4 * g + 3]);
    }
  }
}

// The largest of the lanes' m (0 .. 127).
__device__ __forceinline__ int wave_max(int m) {
  int t = 0;
#pragma unroll
  for (int b = 64; b; b >>= 1)
    if (__ballot(m >= t + b)) t += b;
  return t;
}

// Factors of V columns as stored, and column c's value.
template <typename T, int V>
struct FacV {
  using S = vec<T, V>;
  __device__ static T dec(const S& v, int c) { return get<T, V>(v, c); }
};
template <>
struct FacV<float, 1> {
  using S = uint16_t;
  __device__ static float dec(S v, int) { return half_val(v); }
};
template <>
struct FacV<float, 2> {
  using S = uint32_t;
  __device__ static float dec(S v, int c) { return half_val((uint16_t)(c ? v >> 16 : v & 0xffffu)); }
};

// Column update with both sweeps of the line solve: r -= alpha q, y and w = y / D top-down, w kept in registers,
// z bottom-up to memory; r.z = sum y w, r.r. INIT: r as it is, x = 0.
// U: levels of a batch of loads, one batch ahead. LKEEP: l kept too (two columns of FP32: 233 VGPRs, 2 wavefronts a
// SIMD; FP64: 256 and 46 AGPRs, 1), else read a second time (one column of FP32: 128, 4). 1024x768x60, us: FP32
// two columns kept 156, one column read again 167; FP64 kept 336, read again 351.
template <typename T, int V, int U, bool INIT, bool LKEEP>
__global__ __launch_bounds__(64 * H) void k_update(const Sys* __restrict__ systems, const Tile* __restrict__ tiles) {
  using VT = vec<T, V>;
  using FS = typename FacV<T, V>::S;
  const Tile t = tiles[blockIdx.x];
  if (t.sys < 0) return;  // an empty tile of a work-balanced list
  const Sys& s = systems[t.sys];
  const bool vert = V == 2 && t.local != 0;
  const int l = threadIdx.x & 63;
  const int i = t.bx * TX + V * (vert ? (l & 31) : l), j = (t.by + (vert ? (l >> 5) : 0)) * H + (threadIdx.x >> 6);
  const int nx = s.nx, ny = s.ny, nz = s.nz;
  const size_t P = s.plane;
  bool ok[V];
#pragma unroll
  for (int c = 0; c < V; ++c) ok[c] = i + c < nx && j < ny;
  const uint32_t col = (uint32_t)((size_t)j * s.pitch + i);
  const uint32_t oe = ok[0] ? col * (uint32_t)sizeof(T) : kOob, of = ok[0] ? col * (uint32_t)(sizeof(FS) / V) : kOob;
  const uint32_t PB = (uint32_t)(P * sizeof(T)), PF = (uint32_t)(P * (sizeof(FS) / V));
  const uint32_t AB = PB * (uint32_t)nz, AF = PF * (uint32_t)nz;
  // the levels in use are asked for before the state is looked at: one wait for both
  const int used = ok[0] && s.tab ? s.use[col] : nz;
  Inner<T>* in = reinterpret_cast<Inner<T>*>(s.inner);
  if ((INIT ? s.outer->odone : in->done) != RUN) return;
  const T alpha = INIT ? T(0) : in->alpha;
  const int use = ok[0] ? min(used, nz) : 0, top = wave_max(use);
  T cs[V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    cs[c] = T(1);
    if constexpr (std::is_same<T, float>::value)
      cs[c] = ok[0] ? G<const float>(s.dscale)[(size_t)col + c] : 0.f;
  }
  VT w[NZ];
  FS lf[LKEEP ? NZ : 1];
  T y[V], rho[V], rr[V];
#pragma unroll
  for (int c = 0; c < V; ++c) y[c] = rho[c] = rr[c] = T(0);
  struct Batch {
    VT r[U], q[U];
    FS d[U], l[U];
  };
  Batch ba, bb;
  const Rsrc r_r = buf_of(s.r, AB), r_q = buf_of(s.q, AB), r_d = buf_of(s.invD, AF), r_l = buf_of(s.L, AF);
  const Rsrc r_z = buf_of(s.z, AB);
  auto at = [&](int k) { return k < use ? oe : kOob; };
  auto fat = [&](int k) { return k < use ? of : kOob; };
  auto lev = [&](int k) { return (uint32_t)(k < nz ? k : 0); };  // levels from nz on are masked everywhere
  if (INIT) {
    const Rsrc r_x = buf_of(s.x, AB);
    VT zero;
#pragma unroll
    for (int c = 0; c < V; ++c) put<T, V>(zero, c, T(0));
    for (int k = 0; k < nz; ++k) stb<VT, kAuxNt>(r_x, oe, (uint32_t)k * PB, zero);
  }
  auto load = [&](int k0, Batch& b) {
    if (k0 >= top) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u;
      const uint32_t e = at(k), f = fat(k);
      b.r[u] = ldb<VT, kAuxNt>(r_r, e, lev(k) * PB);
      b.l[u] = ldb<FS, LKEEP ? kAuxNt : kAuxNone>(r_l, f, lev(k) * PF);
      if (LKEEP) lf[k] = b.l[u];
      b.d[u] = ldb<FS, kAuxNt>(r_d, f, lev(k) * PF);
      if (!INIT) b.q[u] = ldb<VT, kAuxNt>(r_q, e, lev(k) * PB);
    }
  };
  auto down = [&](int k0, const Batch& b) {
    __builtin_amdgcn_sched_barrier(0);
    if (k0 >= top) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u;
      VT rv;
#pragma unroll
      for (int c = 0; c < V; ++c) {
        T rk = get<T, V>(b.r[u], c);
        if (!INIT) rk = fmad(-alpha, get<T, V>(b.q[u], c), rk);
        put<T, V>(rv, c, rk);
        rr[c] = fmad(rk, rk, rr[c]);
        y[c] = fmad(-FacV<T, V>::dec(b.l[u], c), y[c], rk);
        const T wv = y[c] * (FacV<T, V>::dec(b.d[u], c) * cs[c]);
        rho[c] = fmad(y[c], wv, rho[c]);
        put<T, V>(w[k], c, wv);
      }
      if (!INIT) stb<VT, kAuxNt>(r_r, at(k), lev(k) * PB, rv);
    }
  };
  load(0, ba);
#pragma unroll
  for (int k0 = 0; k0 < NZ; k0 += 2 * U) {
    if (k0 + U < NZ) load(k0 + U, bb);
    down(k0, ba);
    if (k0 + U >= NZ) break;
    if (k0 + 2 * U < NZ) load(k0 + 2 * U, ba);
    down(k0 + U, bb);
  }
  T z[V], lc[V];
#pragma unroll
  for (int c = 0; c < V; ++c) z[c] = lc[c] = T(0);
  FS la[U], lb[U];
  auto load_l = [&](int k0, FS* v) {  // levels k0 .. k0 - U + 1
    if (k0 - U + 1 >= top) return;
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ldb<FS, kAuxNt>(r_l, fat(k0 - u), lev(k0 - u) * PF);
  };
  auto up = [&](int k0, const FS* v) {
    if (k0 - U + 1 >= top) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 - u;
      VT zv;
#pragma unroll
      for (int c = 0; c < V; ++c) {
        z[c] = fmad(-lc[c], z[c], get<T, V>(w[k], c));
        lc[c] = FacV<T, V>::dec(LKEEP ? lf[LKEEP ? k : 0] : v[u], c);
        put<T, V>(zv, c, z[c]);
      }
      stb<VT, kAuxNt>(r_z, at(k), lev(k) * PB, zv);
    }
  };
  if (!LKEEP) load_l(NZ - 1, la);
#pragma unroll
  for (int k0 = NZ - 1; k0 >= 0; k0 -= 2 * U) {
    if (!LKEEP && k0 - U >= 0) load_l(k0 - U, lb);
    up(k0, la);
    if (k0 - U < 0) break;
    if (!LKEEP && k0 - 2 * U >= 0) load_l(k0 - 2 * U, la);
    up(k0 - U, lb);
  }
#pragma unroll
  for (int c = 0; c < V; ++c)
    if (!ok[c]) rho[c] = rr[c] = T(0);
  publish<T, V>(s, t, vert, rho, rr);
}

// Lane l - 1's value (lane 0: `edge`), lane l + 1's (lane 63: `edge`).
__device__ __forceinline__ unsigned from_west(unsigned v, unsigned edge) {
  return __builtin_amdgcn_update_dpp(edge, v, 0x138, 0xf, 0xf, false);  // wave_shr:1
}
__device__ __forceinline__ unsigned from_east(unsigned v, unsigned edge) {
  return __builtin_amdgcn_update_dpp(edge, v, 0x130, 0xf, 0xf, false);  // wave_shl:1
}
__device__ __forceinline__ float west_of(float v, float e) {
  return __uint_as_float(from_west(__float_as_uint(v), __float_as_uint(e)));
}
__device__ __forceinline__ float east_of(float v, float e) {
  return __uint_as_float(from_east(__float_as_uint(v), __float_as_uint(e)));
}
__device__ __forceinline__ double west_of(double v, double e) {
  const unsigned long long a = (unsigned long long)__double_as_longlong(v), b = (unsigned long long)__double_as_longlong(e);
  const unsigned lo = from_west((unsigned)a, (unsigned)b), hi = from_west((unsigned)(a >> 32), (unsigned)(b >> 32));
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
__device__ __forceinline__ double east_of(double v, double e) {
  const unsigned long long a = (unsigned long long)__double_as_longlong(v), b = (unsigned long long)__double_as_longlong(e);
  const unsigned lo = from_east((unsigned)a, (unsigned)b), hi = from_east((unsigned)(a >> 32), (unsigned)(b >> 32));
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// Matvec: p = z + beta p_old (the neighbours' too, from their z and p_old), x += alpha p_old, q = C p, p.q, bottom-up;
// a wavefront takes a row of 64 V columns on its own. Neighbours along x come from the lanes beside, those past the
// wavefront's row from memory. TAB: ZW, ZP and the couplings from the table and the wet depths; neighbours are read
// down to what couples. WRAP: some column's east neighbour is the domain's first.
// D: levels in flight (FP32 two columns 140 VGPRs, one column 91, FP64 148). us with D = 1 and with the one taken:
// 203x194x35 FP32 21.3 and 20.2, FP64 25.3 and 24.2; 1024x768x60 alike.
template <typename T, int V, bool TAB, bool WRAP, int D>
__global__ __launch_bounds__(64 * H) void k_matvec(const Sys* __restrict__ systems, const Tile* __restrict__ tiles) {
  using VT = vec<T, V>;
  const Tile t = tiles[blockIdx.x];
  if (t.sys < 0) return;
  const Sys& s = systems[t.sys];
  Inner<T>* in = reinterpret_cast<Inner<T>*>(s.inner);
  if (in->done != RUN) return;
  const bool vert = V == 2 && t.local != 0;
  const int l = threadIdx.x & 63, hl = vert ? (l & 31) : l;
  const int i = t.bx * TX + V * hl, j = (t.by + (vert ? (l >> 5) : 0)) * H + (threadIdx.x >> 6);
  const int nx = s.nx, ny = s.ny, nz = s.nz;
  const size_t P = s.plane;
  const bool first = __builtin_amdgcn_readfirstlane(in->first) != 0;
  const int pb = __builtin_amdgcn_readfirstlane(in->pbuf);
  // The first iteration has no p_old and no x: both read as 0, and z + -0.0 is z to the sign of a zero.
  const T beta = first ? T(-0.0) : in->beta, alpha = first ? T(0) : in->alpha;
  bool ok[V];
#pragma unroll
  for (int c = 0; c < V; ++c) ok[c] = i + c < nx && j < ny;
  const uint32_t row = (uint32_t)s.pitch, W = (uint32_t)sizeof(T);
  const uint32_t col = ok[0] ? (uint32_t)j * row + (uint32_t)i : 0u;
  const int jn = j > 0 ? j - 1 : s.cyc_y ? ny - 1 : -1, js = j < ny - 1 ? j + 1 : s.cyc_y ? 0 : -1;
  const uint32_t oc = ok[0] ? col * W : kOob;
  const uint32_t on = ok[0] && jn >= 0 ? ((uint32_t)jn * row + (uint32_t)i) * W : kOob;
  const uint32_t os = ok[0] && js >= 0 ? ((uint32_t)js * row + (uint32_t)i) * W : kOob;
  const uint32_t oh = ok[0] ? col * 2u : kOob;
  // the columns west and east of the wavefront's row (or half row); WRAP: and of the domain's sides
  const bool at_w = hl == 0, at_e = hl == (vert ? 31 : 63);
  uint32_t ow = kOob, oo = kOob;  // west edge; east edge
  bool wrap_e0 = false, wrap_e1 = false;
  if (ok[0]) {
    if (at_w) {
      const int iw = i > 0 ? i - 1 : s.cyc_x ? nx - 1 : -1;
      if (iw >= 0) ow = ((uint32_t)j * row + (uint32_t)iw) * W;
    }
    const int ie = i + V;  // east of the lane's columns
    if (at_e && ie < nx) oo = ((uint32_t)j * row + (uint32_t)ie) * W;
    if (WRAP && s.cyc_x) {
      wrap_e0 = i == nx - 1;
      wrap_e1 = V == 2 && i + 1 == nx - 1;
      if (wrap_e0 || wrap_e1) oo = (uint32_t)j * row * W;
    }
  }
  const uint32_t oedge = at_w ? ow : oo;  // without WRAP no lane has both
  const uint32_t PB = (uint32_t)(P * W), P2 = (uint32_t)(P * 2), AB = PB * (uint32_t)nz, A2 = P2 * (uint32_t)nz;
  const Rsrc r_z = buf_of(s.z, AB), r_po = buf_of(pb ? s.pb : s.pa, first ? 0u : AB), r_pn = buf_of(pb ? s.pa : s.pb, AB);
  const Rsrc r_x = buf_of(s.x, first ? 0u : AB), r_q = buf_of(s.q, AB);
  const Rsrc r_f = buf_of(s.flg, TAB ? 0u : A2);
  const bool tab = TAB || s.tab != 0;
  const Rsrc r_zw = buf_of(s.zw_in, tab ? 0u : AB), r_zp = buf_of(s.zp_in, tab ? 0u : AB);
  typedef __attribute__((address_space(4))) const T* cptr;
  const cptr ctw = (cptr)s.tw_in, ctp = (cptr)s.tp_in;

  T cc[V][7], zwb[V], pc[V], pd[V], dot[V];  // pc, pd: p of this level and the one below
  ZCol<T> zc[V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    gptr<const T> cpi = G<const T>(s.col_in);
    const size_t cl = (size_t)col + (ok[c] ? c : 0);
#pragma unroll
    for (int m = 0; m < 7; ++m) cc[c][m] = cpi[m * P + cl];
    if (tab) {
      zc[c].load(G<const T>(s.tw_in), G<const T>(s.tp_in), s.xk, G<const T>(s.xw_in), G<const T>(s.xp_in), s.xf, P, cl);
      zc[c].clamp();
    }
    pd[c] = dot[c] = T(0);
  }
  // levels in use: the lane's columns, what their couplings reach north and south and past the wavefront's row
  int use = !ok[0] ? 0 : tab ? min(s.use[col], nz) : nz, un = nz, us = nz, uw = nz, ue = nz;
  if (tab) {
    un = max(zc[0].kn, zc[V - 1].kn);
    us = max(zc[0].ks, zc[V - 1].ks);
    uw = zc[0].kw;
    ue = WRAP && wrap_e0 ? zc[0].ke : zc[V - 1].ke;
  }
  const int uedge = at_w ? uw : ue;
  const int top = max(1, wave_max(use));
#pragma unroll
  for (int c = 0; c < V; ++c) {
    const size_t cl = (size_t)col + (ok[c] ? c : 0);
    zwb[c] = tab ? zc[c].zw(top) : G<const T>(s.zw_in)[(size_t)top * P + cl];
  }
  auto dir = [&](T zv, T pv) { return fmad(beta, pv, zv); };
  struct Own {
    VT z, p, x;
  };
  struct Row {
    VT zn, pn, zs, ps, zw, zp;
    T ze, pe, zo, po;
    T tw, tp;
    unsigned f;
  };
  auto load_own = [&](int m, Own& o) {
    const uint32_t so = (uint32_t)(m > 0 ? m : 0) * PB, vo = m < use ? oc : kOob;
    o.z = ldb<VT, kAuxNone>(r_z, vo, so);
    o.p = ldb<VT, kAuxNone>(r_po, vo, so);
    o.x = ldb<VT, kAuxNt>(r_x, vo, so);
  };
  auto load_row = [&](int m, Row& r) {
    const uint32_t mm = (uint32_t)(m > 0 ? m : 0), so = mm * PB;
    const uint32_t vn = m < un ? on : kOob, vs = m < us ? os : kOob;
    r.zn = ldb<VT, kAuxNone>(r_z, vn, so);
    r.pn = ldb<VT, kAuxNone>(r_po, vn, so);
    r.zs = ldb<VT, kAuxNone>(r_z, vs, so);
    r.ps = ldb<VT, kAuxNone>(r_po, vs, so);
    const uint32_t ve = WRAP ? (m < uw ? ow : kOob) : m < uedge ? oedge : kOob;
    r.ze = ldb<T, kAuxNone>(r_z, ve, so);
    r.pe = ldb<T, kAuxNone>(r_po, ve, so);
    if (WRAP) {
      const uint32_t vv = m < ue ? oo : kOob;
      r.zo = ldb<T, kAuxNone>(r_z, vv, so);
      r.po = ldb<T, kAuxNone>(r_po, vv, so);
    }
    if (!TAB) {
      r.zw = ldb<VT, kAuxNt>(r_zw, oc, so);
      r.zp = ldb<VT, kAuxNt>(r_zp, oc, so);
    }
    r.tw = tab ? ctw[mm] : T(0);
    r.tp = tab ? ctp[mm] : T(0);
    if constexpr (!TAB) {
      if constexpr (V == 1) r.f = ldb<uint16_t, kAuxNt>(r_f, oh, mm * P2);
      else r.f = ldb<uint32_t, kAuxNt>(r_f, oh, mm * P2);
    }
  };
  // p and x of level m
  auto advance = [&](int m, const Own& o, T* p) {
    VT pv, xv;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      p[c] = dir(get<T, V>(o.z, c), get<T, V>(o.p, c));
      put<T, V>(pv, c, p[c]);
      put<T, V>(xv, c, fmad(alpha, get<T, V>(o.p, c), get<T, V>(o.x, c)));
    }
    const uint32_t so = (uint32_t)m * PB, vo = m < use ? oc : kOob;
    stb<VT, kAuxNt>(r_pn, vo, so, pv);
    stb<VT, kAuxNt>(r_x, vo, so, xv);
  };
  auto step = [&](int k, const Row& r, const T* pu) {  // pu: p of level k - 1
    T e[2], w[V], ea[V];
    const T pe = dir(r.ze, r.pe), po = WRAP ? dir(r.zo, r.po) : pe;
    T west = west_of(pc[V - 1], pe), east = east_of(pc[0], po);
    if (V == 2) {
      if (at_w) west = pe;
      if (at_e) east = po;
    }
    VT qv;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      T pw = c == 0 ? west : pc[0], px = c == V - 1 ? east : pc[V - 1];
      if (WRAP) px = (c == 0 ? wrap_e0 : wrap_e1) ? po : px;
      const T zwk = TAB ? zc[c].template zw_or<true>(k, r.tw) : tab ? zc[c].template zw_or<true>(k, r.tw) : get<T, V>(r.zw, c);
      const T zpk = TAB ? zc[c].template zp_or<true>(k, r.tp) : tab ? zc[c].template zp_or<true>(k, r.tp) : get<T, V>(r.zp, c);
      T c7[7];
      if constexpr (TAB) inner_row<T>(cc[c], zwk, zwb[c], zpk, k, zc[c], c7);
      else inner_row<T, true>(cc[c], zwk, zwb[c], zpk, V == 1 ? r.f : c ? r.f >> 16 : r.f & 0xffffu, c7);
      zwb[c] = zwk;
      T acc = c7[0] * pc[c];
      acc = fmad(c7[1], pw, acc);
      acc = fmad(c7[2], px, acc);
      acc = fmad(c7[3], dir(get<T, V>(r.zn, c), get<T, V>(r.pn, c)), acc);
      acc = fmad(c7[4], dir(get<T, V>(r.zs, c), get<T, V>(r.ps, c)), acc);
      acc = fmad(c7[5], pu[c], acc);
      acc = fmad(c7[6], pd[c], acc);
      acc = ok[c] ? acc : T(0);
      put<T, V>(qv, c, acc);
      dot[c] = fmad(pc[c], acc, dot[c]);
    }
    stb<VT, kAuxNt>(r_q, k < use ? oc : kOob, (uint32_t)k * PB, qv);
#pragma unroll
    for (int c = 0; c < V; ++c) {
      pd[c] = pc[c];
      pc[c] = pu[c];
    }
  };
  Own o[D + 1];  // level k - 1's at step k, with D levels after it in flight
  Row r[D + 1];  // level k's, likewise
  T none[V];
#pragma unroll
  for (int c = 0; c < V; ++c) none[c] = T(0);
  {
    Own last;
    load_own(top - 1, last);
#pragma unroll
    for (int u = 0; u < D; ++u) {
      load_own(top - 2 - u, o[u]);
      load_row(top - 1 - u, r[u]);
    }
    advance(top - 1, last, pc);
  }
  auto level = [&](int k, int u) {
    load_own(k - 1 - D, o[(u + D) % (D + 1)]);
    load_row(k - D, r[(u + D) % (D + 1)]);
    __builtin_amdgcn_sched_barrier(0);
    T pu[V];
    advance(k - 1, o[u], pu);
    step(k, r[u], pu);
    __builtin_amdgcn_sched_barrier(0);
  };
  int k0 = top - 1;
  for (; k0 > D; k0 -= D + 1) {
#pragma unroll
    for (int u = 0; u <= D; ++u) level(k0 - u, u);
  }
#pragma unroll
  for (int u = 0; u <= D; ++u) {
    if (k0 - u > 0) level(k0 - u, u);
    else if (k0 == u) step(0, r[u], none);
  }
#pragma unroll
  for (int c = 0; c < V; ++c)
    if (!ok[c]) dot[c] = T(0);
  T zero[V];
#pragma unroll
  for (int c = 0; c < V; ++c) zero[c] = T(0);
  publish<T, V>(s, t, vert, dot, zero);
}

template <typename T, int V, int U, bool LKEEP>
hipError_t update(hipStream_t st, const StreamLaunch& l, bool init) {
  const Tile* d = V == 2 ? l.d_pairs : l.d_tiles;
  const int n = V == 2 ? l.npairs : l.ntiles;
  if (n <= 0) return hipSuccess;
  if (init) hipLaunchKernelGGL((k_update<T, V, U, true, LKEEP>), dim3(n), dim3(64 * H), 0, st, l.d_sys, d);
  else hipLaunchKernelGGL((k_update<T, V, U, false, LKEEP>), dim3(n), dim3(64 * H), 0, st, l.d_sys, d);
  return hipGetLastError();
}

template <typename T, int V, int D>
hipError_t matvec(hipStream_t st, const StreamLaunch& l) {
  const Tile* d = V == 2 ? l.d_pairs : l.d_tiles;
  const int n = V == 2 ? l.npairs : l.ntiles;
  if (n <= 0) return hipSuccess;
  if (l.tab && !l.wrap) hipLaunchKernelGGL((k_matvec<T, V, true, false, D>), dim3(n), dim3(64 * H), 0, st, l.d_sys, d);
  else if (l.tab) hipLaunchKernelGGL((k_matvec<T, V, true, true, D>), dim3(n), dim3(64 * H), 0, st, l.d_sys, d);
  else hipLaunchKernelGGL((k_matvec<T, V, false, true, D>), dim3(n), dim3(64 * H), 0, st, l.d_sys, d);
  return hipGetLastError();
}
}  // namespace

hipError_t stream_update(hipStream_t st, const StreamLaunch& l, bool init) {
  if (!l.fp32) return update<double, 1, 4, true>(st, l, init);
  return l.npairs >= kPairs ? update<float, 2, 4, true>(st, l, init) : update<float, 1, 8, false>(st, l, init);
}

hipError_t stream_matvec(hipStream_t st, const StreamLaunch& l) {
  if (!l.fp32) return matvec<double, 1, 2>(st, l);
  return l.npairs >= kPairs ? matvec<float, 2, 2>(st, l) : matvec<float, 1, 3>(st, l);
}

}  // namespace onh
