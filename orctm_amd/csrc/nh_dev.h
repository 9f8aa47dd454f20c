// nh_dev.h -- device code shared by the solver's kernels: memory access, the storage of the line factors,
// wavefront and block sums, and the rows of the operator rebuilt from the compact form.
#pragma once

#include <math.h>

#include <type_traits>

#include "nh_flags.h"
#include "nh_kernels.h"

namespace onh {

__device__ __forceinline__ double fmad(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fmad(float a, float b, float c) { return fmaf(a, b, c); }

// Pointers read from a Sys in memory are generic; casting them to the global address space lets the
// compiler use global_load/global_store and count only vector-memory operations in its waits.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> G(const void* p) {
  return (gptr<T>)(const_cast<void*>(p));
}

// v of lane l ^ OFF, for values that already agree in the lanes whose numbers differ in bits above OFF only
// (as in a sum over falling offsets): lane swaps and row rotations in the vector unit, where a shuffle goes
// through LDS (a sum of two values over the wavefront: 0.1 us against 0.5).
template <int OFF>
__device__ __forceinline__ unsigned fold_bits(unsigned v) {
  if constexpr (OFF == 8) return __builtin_amdgcn_update_dpp(0u, v, 0x128, 0xf, 0xf, false);       // row_ror:8
  else if constexpr (OFF == 4) return __builtin_amdgcn_update_dpp(0u, v, 0x124, 0xf, 0xf, false);  // row_ror:4
  else if constexpr (OFF == 2) return __builtin_amdgcn_update_dpp(0u, v, 0x4e, 0xf, 0xf, false);   // quad_perm 2,3,0,1
  else return __builtin_amdgcn_update_dpp(0u, v, 0xb1, 0xf, 0xf, false);                           // quad_perm 1,0,3,2
}
template <int OFF>
__device__ __forceinline__ float fold_add(float v) {
  if constexpr (OFF >= 16) {
    const unsigned u = __float_as_uint(v);
    const auto p = OFF == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false)
                             : __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
  } else {
    return v + __uint_as_float(fold_bits<OFF>(__float_as_uint(v)));
  }
}
template <int OFF>
__device__ __forceinline__ double fold_add(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  auto join = [](unsigned l, unsigned h) { return __longlong_as_double((long long)((unsigned long long)h << 32 | l)); };
  if constexpr (OFF >= 16) {
    const auto a = OFF == 32 ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                             : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = OFF == 32 ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                             : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return join(a[0], b[0]) + join(a[1], b[1]);
  } else {
    return v + join(fold_bits<OFF>(lo), fold_bits<OFF>(hi));
  }
}

// The sum over the wavefront, lane l paired with l ^ 32, l ^ 16, ..., l ^ 1; the same bits in every lane.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  v = fold_add<32>(v);
  v = fold_add<16>(v);
  v = fold_add<8>(v);
  v = fold_add<4>(v);
  v = fold_add<2>(v);
  return fold_add<1>(v);
}

// Storage of the FP32 line-preconditioner factors: IEEE fp16 bits, normal range only (the rules of
// the oracle's factor_round32): l with |l| < 2^-14 is stored as 0; invD is scaled by a power of two
// per column (largest scaled value in [2^14, 2^15)) with magnitudes raised to at least 2^-14. The
// rounding is done with integer operations (ties to even) so that it is the oracle's to the bit;
// decoding is the exact fp16 -> fp32 conversion.
__device__ __forceinline__ uint16_t half_bits(float v) {
  const uint32_t u0 = __float_as_uint(v);
  const uint32_t sgn = (u0 >> 16) & 0x8000u;
  const float a = fabsf(v);
  if (!(a < 65520.0f)) return isnan(v) ? (uint16_t)0x7E00u : (uint16_t)(sgn | 0x7C00u);
  if (a == 0.0f) return (uint16_t)sgn;
  const uint32_t u = (u0 + 0xFFFu + ((u0 >> 13) & 1u)) & 0xFFFFE000u;
  const uint32_t e = ((u >> 23) & 0xFFu) - 112u;  // fp32 exponent bias 127 -> fp16 bias 15
  return (uint16_t)(sgn | (e << 10) | ((u >> 13) & 0x3FFu));
}

__device__ __forceinline__ float half_val(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }

constexpr float kHalfMin = 6.103515625e-05f;  // 2^-14

// Streaming accesses of the inner kernels: every value is touched once per launch and re-read only
// by the next launch, a gigabyte or more later, so they carry the non-temporal hint (no cache
// residency is expected; the stores do not evict lines other blocks still read).
template <typename T>
__device__ __forceinline__ T ld_nt(gptr<const T> p, size_t i) {
  return __builtin_nontemporal_load(p + i);
}
template <typename T>
__device__ __forceinline__ void st_nt(gptr<T> p, size_t i, T v) {
  __builtin_nontemporal_store(v, p + i);
}

// Buffer-descriptor access (the matvec kernel's column march). A descriptor covers one array; a lane
// addresses it by a 32-bit byte offset (its column's offset plus the level's). A lane that must not
// touch memory takes an offset at or past kOob, beyond every array of at most kBufMaxBytes: the
// hardware's range check then returns 0 for its load and drops its store. A whole wavefront is masked
// by a descriptor of size 0. So every wavefront issues the same memory instructions on every path, and
// the compiler's wait counts keep the loads of the next level in flight instead of draining them where
// branches around loads and stores join.
constexpr uint32_t kOob = 0x80000000u;
static_assert(kBufMaxBytes <= kOob, "offsets of valid lanes stay below kOob");
constexpr int kBufWord3 = 0x00020000;  // gfx9 descriptor word 3: 32-bit data format, untyped access
using Rsrc = __amdgpu_buffer_rsrc_t;
enum : int { kAuxNone = 0, kAuxNt = 2 };  // cache policy bits: none, non-temporal

__device__ __forceinline__ Rsrc buf_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, kBufWord3);
}
template <typename E, int AUX>
__device__ __forceinline__ E bld(Rsrc r, uint32_t vo) {
  if constexpr (sizeof(E) == 2) {
    return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b16(r, vo, 0, AUX));
  } else if constexpr (sizeof(E) == 4) {
    return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(r, vo, 0, AUX));
  } else {
    static_assert(sizeof(E) == 8, "2-, 4- or 8-byte elements");
    return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(r, vo, 0, AUX));
  }
}
template <typename E>
__device__ __forceinline__ void bst_nt(Rsrc r, uint32_t vo, E v) {
  if constexpr (sizeof(E) == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, vo, 0, kAuxNt);
  } else {
    static_assert(sizeof(E) == 8, "4- or 8-byte elements");
    typedef unsigned int U2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, vo, 0, kAuxNt);
  }
}

// Factor storage per inner precision: fp16 bits for FP32, the value itself for FP64.
template <typename T>
struct Fac {
  using S = T;
  __device__ static T dec(T v) { return v; }
  __device__ static T ld(gptr<const S> p, size_t i) { return p[i]; }
  __device__ static T ld_nt(gptr<const S> p, size_t i) { return onh::ld_nt(p, i); }
};
template <>
struct Fac<float> {
  using S = uint16_t;
  __device__ static float dec(uint16_t v) { return half_val(v); }
  __device__ static float ld(gptr<const uint16_t> p, size_t i) { return half_val(p[i]); }
  __device__ static float ld_nt(gptr<const uint16_t> p, size_t i) { return half_val(onh::ld_nt(p, i)); }
};

// Sum of a and b over a block of NW wavefronts; valid in thread 0.
template <typename T, int NW = NT / 64>
__device__ __forceinline__ void block_sum2(T& a, T& b) {
  __shared__ T sh[2 * NW];
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) {
    sh[w] = a;
    sh[NW + w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    T sa = sh[0], sb = sh[NW];
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      sa += sh[q];
      sb += sh[NW + q];
    }
    a = sa;
    b = sb;
  }
}

// Neighbour map of the DMDA: periodic wrap where cyclic, else validity (outside reads +0).
__device__ __forceinline__ bool map_ij(int& i, int& j, int nx, int ny, int cx, int cy) {
  if (cx) {
    if (i < 0)
      i += nx;
    else if (i >= nx)
      i -= nx;
  }
  if (cy) {
    if (j < 0)
      j += ny;
    else if (j >= ny)
      j -= ny;
  }
  return i >= 0 && i < nx && j >= 0 && j < ny;
}

// One row of compute_matrix rebuilt from the compact form, in T arithmetic (double: the operations
// of the assembly, bit for bit; float: the inner operator). c7: centre, W, E, N, S, U, D.
// flags: bit 0 wet; bits 1-6 coupling present W E N S U D; bits 7-8 X_C variant (full, XUe*XP,
// XUw*XP, 0); bits 9-10 Y_C variant (full, YVs*YP, YVn*YP, 0); bit 11 Z_C variant (full, ZW*ZP).
// FLAT: one select after the other; a chain of ?: becomes branches, which empty the load pipeline of kernels that keep
// many loads in flight. The same value either way.
template <typename T, bool FLAT = false>
__device__ __forceinline__ void row_coef(const T* cc, T zwk, T zwk1, T zpk, unsigned f, T* c7) {
  const T xw = cc[0], xe = cc[1], yn = cc[2], ys = cc[3];
  const unsigned xc = (f >> 7) & 3u, yc = (f >> 9) & 3u;
  T X_C, Y_C;
  if constexpr (FLAT) {
    X_C = xc == 2 ? xw : T(0), Y_C = yc == 2 ? yn : T(0);
    X_C = xc == 1 ? xe : X_C;
    X_C = xc == 0 ? cc[4] : X_C;
    Y_C = yc == 1 ? ys : Y_C;
    Y_C = yc == 0 ? cc[5] : Y_C;
  } else {
    X_C = xc == 0 ? cc[4] : xc == 1 ? xe : xc == 2 ? xw : T(0);
    Y_C = yc == 0 ? cc[5] : yc == 1 ? ys : yc == 2 ? yn : T(0);
  }
  const T Z_C = ((f >> 11) & 1u) ? zwk * zpk : (zwk + zwk1) * zpk;
  c7[0] = -(X_C + Y_C + Z_C);
  c7[1] = (f & (1u << 1)) ? xw : T(0);
  c7[2] = (f & (1u << 2)) ? xe : T(0);
  c7[3] = (f & (1u << 3)) ? yn : T(0);
  c7[4] = (f & (1u << 4)) ? ys : T(0);
  c7[5] = (f & (1u << 5)) ? zwk * zpk : T(0);
  c7[6] = (f & (1u << 6)) ? zwk1 * zpk : T(0);
}

// ZW/ZP of one column from the per-level table and the column's 3-level window, and the column's flag
// bits from its wet depths (Sys::tab).
template <typename T>
struct ZCol {
  gptr<const T> tw, tp;
  int kx;
  T w0, w1, w2, p0, p1, p2;
  int kc, kw, ke, kn, ks;
  unsigned edge;
  __device__ void load(gptr<const T> tw_, gptr<const T> tp_, const int* xk, gptr<const T> xw, gptr<const T> xp,
                       const uint32_t* xf, size_t P, size_t off) {
    tw = tw_;
    tp = tp_;
    kx = xk[off];
    w0 = xw[off];
    w1 = xw[P + off];
    w2 = xw[2 * P + off];
    p0 = xp[off];
    p1 = xp[P + off];
    p2 = xp[2 * P + off];
    const uint32_t a = xf[off], b = xf[P + off], c = xf[2 * P + off];
    kc = (int)(a & 0xffffu);
    kw = (int)(a >> 16);
    ke = (int)(b & 0xffffu);
    kn = (int)(b >> 16);
    ks = (int)(c & 0xffffu);
    edge = c >> 16;
  }
  // flag bits of level m (0-based) of a column of nz levels
  __device__ unsigned flag(int m, int nz) const { return derive_flags(m + 1, nz, kc, kw, ke, kn, ks, edge); }
  // Prepared for coef(): beyond the column's own wet depth a neighbour's plays no part.
  __device__ void clamp() {
    kw = min(kw, kc);
    ke = min(ke, kc);
    kn = min(kn, kc);
    ks = min(ks, kc);
  }
  // row_coef() of level m from the wet depths themselves, without the flag word: the same values.
  __device__ void coef(int m, const T* cc, T zwk, T zwk1, T zpk, T* c7) const {
    const bool wet = m < kc, w = m < kw, e = m < ke, n = m < kn, s = m < ks, below = m + 1 < kc;
    T X_C = e ? cc[1] : T(0), Y_C = s ? cc[3] : T(0);
    const T xw = e ? cc[4] : cc[0], yn = s ? cc[5] : cc[2];
    X_C = w ? xw : X_C;
    Y_C = n ? yn : Y_C;
    X_C = wet ? X_C : cc[4];
    Y_C = wet ? Y_C : cc[5];
    const T zs = zwk + zwk1, Z_C = (m > 0 && wet && !below ? zwk : zs) * zpk;
    c7[0] = -(X_C + Y_C + Z_C);
    c7[1] = w && (edge & 1u) ? cc[0] : T(0);
    c7[2] = e && (edge & 2u) ? cc[1] : T(0);
    c7[3] = n && (edge & 4u) ? cc[2] : T(0);
    c7[4] = s && (edge & 8u) ? cc[3] : T(0);
    c7[5] = m > 0 && wet ? zwk * zpk : T(0);
    c7[6] = below ? zwk1 * zpk : T(0);
  }
  __device__ T zw(int m) const {
    const int d = m - kx;
    return d == 0 ? w0 : d == 1 ? w1 : d == 2 ? w2 : tw[m];
  }
  __device__ T zp(int m) const {
    const int d = m - kx;
    return d == 0 ? p0 : d == 1 ? p1 : d == 2 ? p2 : tp[m];
  }
  // the window's value at level m where the window covers m, else t (the table's entry)
  template <bool FLAT = false>
  __device__ T zw_or(int m, T t) const {
    return pick<FLAT>(m - kx, w0, w1, w2, t);
  }
  template <bool FLAT = false>
  __device__ T zp_or(int m, T t) const {
    return pick<FLAT>(m - kx, p0, p1, p2, t);
  }
  template <bool FLAT>
  __device__ static T pick(int d, T v0, T v1, T v2, T t) {
    if constexpr (FLAT) {
      t = d == 2 ? v2 : t;
      t = d == 1 ? v1 : t;
      return d == 0 ? v0 : t;
    } else {
      return d == 0 ? v0 : d == 1 ? v1 : d == 2 ? v2 : t;
    }
  }
};

// Inner operator row C = S * (-A), S = DLXP*DLYP/ZP, in T arithmetic from the T copies.
template <typename T, bool FLAT = false>
__device__ __forceinline__ void inner_row(const T* cc, T zwk, T zwk1, T zpk, unsigned f, T* c7) {
  row_coef<T, FLAT>(cc, zwk, zwk1, zpk, f, c7);
  const T S = cc[6] / zpk;
#pragma unroll
  for (int q = 0; q < 7; ++q) c7[q] = S * (-c7[q]);
}
// The same from the wet depths (ZCol::clamp() applied).
template <typename T>
__device__ __forceinline__ void inner_row(const T* cc, T zwk, T zwk1, T zpk, int m, const ZCol<T>& z, T* c7) {
  z.coef(m, cc, zwk, zwk1, zpk, c7);
  const T S = cc[6] / zpk;
#pragma unroll
  for (int q = 0; q < 7; ++q) c7[q] = S * (-c7[q]);
}

// ------------------------------------------------------------------------------------------------
// The scalar recurrences of the inner PCG, from the system totals of a phase.

// After the first column update of an inner solve (totals r.z, r.r).
template <typename T>
__device__ __forceinline__ void inner_begin(Inner<T>& in, T rho, T rr) {
  in.rho = rho;
  in.rr0 = rr;
  in.rr = rr;
  in.iter = 0;
  in.first = 1;
  in.pbuf = 0;
  in.xpend = 0;
  in.beta = T(0);
  if (rr == T(0))
    in.done = CONVERGED;
  else if (!(rho > T(0)) || !isfinite((double)rho) || !isfinite((double)rr))
    in.done = BREAKDOWN;
  else
    in.done = RUN;
}

// After an iteration's matvec (total p.q).
template <typename T>
__device__ __forceinline__ void inner_after_matvec(Inner<T>& in, T pq) {
  const T alpha = in.rho / pq;
  in.pq = pq;
  in.alpha = alpha;
  in.xpend = 0;  // the matvec just applied the previous iteration's update
  if (!(pq > T(0)) || !isfinite((double)alpha)) in.done = BREAKDOWN;
}

// After an iteration's column update (totals r.z, r.r).
template <typename T>
__device__ __forceinline__ void inner_after_update(Inner<T>& in, T rho, T rr) {
  in.iter += 1;
  in.rr = rr;
  int d = RUN;
  if (rr <= in.tol2 * in.rr0)
    d = CONVERGED;
  else if (!(rho > T(0)) || !isfinite((double)rho) || !isfinite((double)rr))
    d = BREAKDOWN;
  else if (in.iter >= in.maxit)
    d = NOTCONV;
  else {
    in.beta = rho / in.rho;
    in.rho = rho;
  }
  in.first = 0;
  in.pbuf ^= 1;
  in.xpend = 1;  // x += alpha p of this iteration: applied by the next matvec or by k_refine
  in.done = d;
}

}  // namespace onh
