// Packed rows: the off-diagonal elements of a matrix-free operator in the
// gather form, four bytes each, evaluated once and read back by every product.
//
// Slices of 64 rows (one wavefront); entry e of row r at
//   off[r / 64] + 64 e + r % 64 :  column | id << idx_bits,
// id pointing into a table of the operator's distinct coefficients (id 0 = 0,
// the padding of rows shorter than their slice, which carries the row's own
// index as its column; the products take its x for 0, so that a vector element
// that is not finite stays out of the rows it has no element in).  A symmetry-reduced operator has few distinct
// coefficients (couplings x characters x ratios of stabiliser sizes), so the
// table sits in LDS and an element costs four streamed bytes and its gather.
//
// The sector table (one word per state of the particle sector) needs |G|
// words per basis state and a divergent read per element; packed rows need
// one word per element and stream it.  Heisenberg L = 28, k = 0, p = z = +1:
// 24 MB against 160 MB.
#pragma once
#include "sparse_impl.h"

constexpr int PK_SLOTS = 4096;   // hash slots of the coefficient dictionary
constexpr int PK_LUT_MAX = 1024; // distinct coefficients (16 KB of LDS)
// Probes of a lookup: with at most a quarter of the slots taken, linear
// probing's longest chain is about 13, so 64 are only reached once more values
// came in than the form takes.
constexpr int PK_PROBES = 64;

// dictionary scratch of a build, in device memory
struct PackDict {
  unsigned long long key[PK_SLOTS];  // hash of the value, 0 = free
  double2 val[PK_SLOTS];
  int32_t id[PK_SLOTS];
  int32_t n_lut;      // entries with id 0
  int32_t bad;        // refused: too many values, or two with one hash
  int64_t total;      // entries of all slices
  int32_t used;       // slots taken
};

__device__ __forceinline__ unsigned long long pk_hash(double2 v) {
  unsigned long long a = (unsigned long long)__double_as_longlong(v.x);
  unsigned long long b = (unsigned long long)__double_as_longlong(v.y);
  unsigned long long h = a * 0x9E3779B97F4A7C15ull + (b ^ (b >> 29)) * 0xC2B2AE3D27D4EB4Full;
  h ^= h >> 31;
  h *= 0xD6E8FEB86659FD93ull;
  h ^= h >> 32;
  return h | 1ull;
}

// Slot of value v, entered when it is new; -1 when the build is refused
// already, or by this value.  An operator of many distinct couplings would
// otherwise pay a walk over the full table for every further element.
__device__ __forceinline__ int pk_slot(PackDict* D, double2 v) {
  const unsigned long long h = pk_hash(v);
  int s = (int)(h >> 1) & (PK_SLOTS - 1);
  if (__hip_atomic_load(&D->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return -1;
  for (int p = 0; p < PK_PROBES; ++p) {
    unsigned long long k = __hip_atomic_load(&D->key[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k == 0) {
      k = atomicCAS(&D->key[s], 0ull, h);
      if (k == 0) {
        D->val[s] = v;
        if (atomicAdd(&D->used, 1) < PK_LUT_MAX - 1) return s;  // id 0 is the padding's
        break;
      }
    }
    if (k == h) return s;
    s = (s + 1) & (PK_SLOTS - 1);
  }
  __hip_atomic_store(&D->bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return -1;
}

// The packed rows an H.v context is bound to and their number of entries
// (hv.hip); false when its product takes another form.
bool qsx_hv_ctx_packed(const void* hv_ctx, HvArgs* A, int* dtype, int64_t* entries);

template <typename VT>
using PkLut = typename std::conditional<VTr<VT>::cplx, double2, double>::type;

template <typename VT>
__device__ __forceinline__ void pk_stage_lut(const HvArgs& A, PkLut<VT>* lut) {
  for (int i = threadIdx.x; i < A.pk_nlut; i += 256) {
    if constexpr (VTr<VT>::cplx) lut[i] = A.pk_lut[i];
    else lut[i] = A.pk_lut[i].x;
  }
}

__device__ __forceinline__ double2 pk_diag(const HvArgs& A, int64_t r) {
  if (!A.diag_arr) return make_double2(0.0, 0.0);
  return A.diag_arr_cplx ? ld_stream<double2>((const double2*)A.diag_arr + r)
                         : ld_stream<double>((const double*)A.diag_arr + r);
}

// The gathered element of an entry, next to 0 for a row's padding (id 0, whose
// weight 0 would make a NaN of an element that is not finite): clearing the
// upper word of a double leaves a subnormal, one select instead of two.
__device__ __forceinline__ double pk_keep(double v, uint32_t id) {
  return __hiloint2double(id ? __double2hiint(v) : 0, __double2loint(v));
}
__device__ __forceinline__ double2 pk_x(const float* x, uint32_t id) { return make_double2(id ? *x : 0.0f, 0.0); }
__device__ __forceinline__ double2 pk_x(const double* x, uint32_t id) { return make_double2(pk_keep(*x, id), 0.0); }
__device__ __forceinline__ double2 pk_x(const float2* x, uint32_t id) {
  return make_double2(id ? x->x : 0.0f, id ? x->y : 0.0f);
}
__device__ __forceinline__ double2 pk_x(const double2* x, uint32_t id) {
  return make_double2(pk_keep(x->x, id), pk_keep(x->y, id));
}

// Off-diagonal sum of row rc = 64 sl + lane (the last row for lanes past it):
// the row's four-byte entries with U gathers in flight.  The rows of a slice
// are consecutive lanes, so entry loads are 256-byte segments.
template <typename VT>
__device__ __forceinline__ double2 pk_row(const HvArgs& A, const PkLut<VT>* lut, const VT* __restrict__ vin, int64_t sl,
                                          int lane, int64_t rc) {
  constexpr int U = 8;
  const int bits = A.pk_bits;
  const uint32_t cmask = (1u << bits) - 1u;
  const int64_t o0 = A.pk_off[sl];
  const int wid = (int)((A.pk_off[sl + 1] - o0) >> 6);
  const uint32_t* __restrict__ en = A.pk_ent + o0 + lane;
  double2 acc = make_double2(0.0, 0.0);
  for (int e0 = 0; e0 < wid; e0 += U) {
    uint32_t ev[U];
#pragma unroll
    for (int u = 0; u < U; ++u) ev[u] = e0 + u < wid ? en[(int64_t)(e0 + u) * 64] : (uint32_t)rc;
    VT xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = vin[ev[u] & cmask];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t id = ev[u] >> bits;
      const double2 x = pk_x(&xv[u], id);
      const PkLut<VT> c = lut[id];
      if constexpr (VTr<VT>::cplx) acc = cadd(acc, cmul(c, x));
      else acc.x += c * x.x;
    }
  }
  return acc;
}

// One vector, one lane per row.
//
// Bound by the gathers of x (an L2 line per lane and element where the columns
// of neighbouring rows differ) and the stream of entries.  Heisenberg L = 28
// k = 0 p = z = +1, float64: 13.1 us against 27.3 us through the sector table;
// L = 34 827 against 1,162 us.  Eight gathers in flight (16: 14.9 us, 24: 14.0;
// 4: 13.1); entries through the caches (non-temporal 15.6 us); blocks in runs
// per XCD inside a shared window (dispatch order 13.4 us, one run per XCD
// 14.2); entries in term order (sorted by column 13.8).  EPI: the launch is a
// Taylor term: truncation test of the previous term, F += the stored term,
// norms into the slots.
template <typename VT, bool EPI>
__global__ void __launch_bounds__(256) k_packed_rows(HvArgs A) {
  constexpr bool CPLX = VTr<VT>::cplx;
  __shared__ PkLut<VT> lut[PK_LUT_MAX];
  if (A.skip && *A.skip) return;
  if constexpr (EPI) {
    if (A.chk_c1 && *A.chk_c1 + *A.chk_c2 <= A.tol * *A.chk_F) {
      if (blockIdx.x == 0 && threadIdx.x == 0) *A.done = 1;
      return;
    }
  }
  pk_stage_lut<VT>(A, lut);
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t nsl = (A.Ns + 63) >> 6;
  const VT* __restrict__ vin = (const VT*)A.v_in;
  VT* __restrict__ vout = (VT*)A.v_out;
  double maxB = 0.0, maxF = 0.0;
  const int64_t bi = xcd_chunked(blockIdx.x, gridDim.x, gridDim.x >= 16384 ? 256 : 64);
  const int64_t sl = bi * 4 + w;
  const int64_t r = sl * 64 + lane;
  if (sl < nsl) {
    const int64_t rc = r < A.Ns ? r : A.Ns - 1;  // lanes past the last row read in bounds, store nothing
    const double2 dg = pk_diag(A, rc);
    const double2 xr = VTr<VT>::ld(vin + rc);
    const double2 acc = pk_row<VT>(A, lut, vin, sl, lane, rc);
    if (r < A.Ns) {
      const double2 dsum = cadd(cmul(dg, A.alpha_diag), A.shift);
      double2 res;
      if constexpr (CPLX) res = cadd(cmul(A.alpha_off, acc), cmul(dsum, xr));
      else res = make_double2(A.alpha_off.x * acc.x + dsum.x * xr.x, 0.0);
      if (A.beta) res = cadd(res, VTr<VT>::ld(vout + r));
      VTr<VT>::st(vout + r, res);
      if constexpr (EPI) {
        VT* __restrict__ F = (VT*)A.epi_F;
        const double2 rs = VTr<VT>::rnd(res);  // the stored (rounded) term enters F
        const double2 f = VTr<VT>::rnd(cadd(VTr<VT>::ld(F + r), rs));
        VTr<VT>::st(F + r, f);
        maxB = norm_key<CPLX>(rs);
        maxF = norm_key<CPLX>(f);
      }
    }
  }
  if constexpr (EPI) epi_norms_out(A, norm_of_key<CPLX>(maxB), norm_of_key<CPLX>(maxF));
}

// One Lanczos step up to its dot, from the residual r of the step before
// (not normalised) and the nb partials of ||r||^2:
//   b = ||r||, q = r / b (stored), s = H q - b q_prev (stored),
//   the block's partial of Re <q, s>.
// H q is formed as (H r) / b, so the division and the gathers share one
// launch: the partials are summed after the gathers, hidden behind the other
// blocks' loads.  first: r is the start vector, divided only when its norm is
// off 1 by more than eps, and no b is recorded.
// Bound by the gathers of r and, below a few hundred thousand rows, by the two
// launches of a step.  Heisenberg L = 28 k = 0 p = z = +1, float64, 40 steps:
// 1,056 us against 1,432 us for product, division and two updates apart.
template <typename VT>
__global__ void __launch_bounds__(256) k_packed_lz(HvArgs A, const double* __restrict__ pnrm, int nb,
                                                   VT* __restrict__ q, const VT* __restrict__ qprev, double* bout,
                                                   double eps, int first, double* __restrict__ pdot) {
  constexpr bool CPLX = VTr<VT>::cplx;
  __shared__ PkLut<VT> lut[PK_LUT_MAX];
  pk_stage_lut<VT>(A, lut);
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t nsl = (A.Ns + 63) >> 6;
  const VT* __restrict__ vin = (const VT*)A.v_in;
  VT* __restrict__ vout = (VT*)A.v_out;
  const int64_t bi = xcd_chunked(blockIdx.x, gridDim.x, 64);
  double b = 0.0, dot = 0.0;
  bool have = false;
  // every block makes the same number of rounds, so the sum's barriers match
  const int64_t rounds = (nsl + 4 * (int64_t)gridDim.x - 1) / (4 * (int64_t)gridDim.x);
  for (int64_t it = 0; it < rounds; ++it) {
    const int64_t sl = (it * gridDim.x + bi) * 4 + w;
    const int64_t r = sl * 64 + lane;
    const bool live = r < A.Ns;
    double2 xr = make_double2(0.0, 0.0), h = make_double2(0.0, 0.0), qp = make_double2(0.0, 0.0);
    if (sl < nsl) {
      const int64_t rc = live ? r : A.Ns - 1;
      const double2 dg = pk_diag(A, rc);
      xr = VTr<VT>::ld(vin + rc);
      if (qprev) qp = VTr<VT>::ld(qprev + rc);
      h = pk_row<VT>(A, lut, vin, sl, lane, rc);
      if constexpr (CPLX) h = cadd(h, cmul(dg, xr));
      else h.x += dg.x * xr.x;
    }
    if (!have) {
      b = sqrt(sum_partials(pnrm, nb));
      have = true;
      if (blockIdx.x == 0 && threadIdx.x == 0 && bout) bout[0] = b;
      if (first && fabs(b - 1.0) <= eps) b = 1.0;
    }
    if (live) {
      const double2 qq = VTr<VT>::rnd(make_double2(xr.x / b, xr.y / b));
      VTr<VT>::st(q + r, qq);
      double2 s = VTr<VT>::rnd(make_double2(h.x / b, h.y / b));
      if (qprev) s = VTr<VT>::rnd(make_double2(s.x - b * qp.x, s.y - b * qp.y));
      VTr<VT>::st(vout + r, s);
      dot += qq.x * s.x + qq.y * s.y;
    }
  }
  block_partial(dot, pdot);
}

// Several vectors, (Ns, nvec) row-major: a block takes one slice, its entries
// staged in LDS, 256 / G rows at a time with G lanes per row and CW columns
// per lane (as k_csr_mm); gridDim.y splits a slice's rows over blocks when
// there are few slices.
constexpr int PK_STAGE = 32;  // entries per row staged; wider slices read from memory

template <typename VT, int G, int CW, bool EPI>
__global__ void __launch_bounds__(256) k_packed_mm(HvArgs A) {
  constexpr bool CPLX = VTr<VT>::cplx;
  using LT = PkLut<VT>;
  constexpr int U = CW * sizeof(VT) >= 16 ? 4 : 8;
  constexpr int RB = 256 / G;
  __shared__ LT lut[PK_LUT_MAX];
  __shared__ uint32_t s_ent[PK_STAGE * 64];
  if (A.skip && *A.skip) return;
  if constexpr (EPI) {
    if (A.chk_c1 && *A.chk_c1 + *A.chk_c2 <= A.tol * *A.chk_F) {
      if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *A.done = 1;
      return;
    }
  }
  const int64_t sl = xcd_chunked(blockIdx.x, gridDim.x, gridDim.x >= 16384 ? 256 : 64);
  const int64_t o0 = A.pk_off[sl];
  const int wid = (int)((A.pk_off[sl + 1] - o0) >> 6);
  const uint32_t* __restrict__ ent = A.pk_ent + o0;
  const bool staged = wid <= PK_STAGE;
  if (staged)
    for (int i = threadIdx.x; i < wid * 64; i += 256) s_ent[i] = ent[i];
  pk_stage_lut<VT>(A, lut);
  __syncthreads();
  const VT* __restrict__ vin = (const VT*)A.v_in;
  VT* __restrict__ vout = (VT*)A.v_out;
  const int bits = A.pk_bits;
  const uint32_t cmask = (1u << bits) - 1u;
  const int64_t nv = A.nvec;
  const int lane = threadIdx.x % G;
  double maxB = 0.0, maxF = 0.0;
  for (int q0 = (int)blockIdx.y * RB; q0 < 64; q0 += (int)gridDim.y * RB) {
    const int q = q0 + (int)(threadIdx.x / G);  // row of the slice
    const int64_t r = sl * 64 + q;
    const bool live = q < 64 && r < A.Ns;
    const int qc = live ? q : 0;
    const int64_t rc = sl * 64 + qc;
    double2 dg = make_double2(0.0, 0.0);
    if (A.diag_arr) {
      if (A.diag_arr_cplx) dg = ((const double2*)A.diag_arr)[rc];
      else dg.x = ((const double*)A.diag_arr)[rc];
    }
    const double2 dsum = cadd(cmul(dg, A.alpha_diag), A.shift);
    double curB = 0.0, curF = 0.0;
    for (int64_t j0 = 0; j0 < nv; j0 += G * CW) {
      const bool ok = live && j0 + lane * CW < nv;
      const int64_t j = ok ? j0 + lane * CW : 0;
      double2 acc[CW];
#pragma unroll
      for (int c = 0; c < CW; ++c) acc[c] = make_double2(0.0, 0.0);
      for (int e0 = 0; e0 < wid; e0 += U) {
        uint32_t ev[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          ev[u] = e0 + u < wid ? (staged ? s_ent[(e0 + u) * 64 + qc] : ent[(int64_t)(e0 + u) * 64 + qc]) : (uint32_t)rc;
        VecRun<VT, CW> xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = *(const VecRun<VT, CW>*)(vin + (int64_t)(ev[u] & cmask) * nv + j);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t id = ev[u] >> bits;
          const LT m = lut[id];
#pragma unroll
          for (int c = 0; c < CW; ++c) {
            const double2 x = pk_x(&xv[u].a[c], id);
            if constexpr (CPLX) acc[c] = cadd(acc[c], cmul(m, x));
            else acc[c].x += m * x.x;
          }
        }
      }
      if (ok) {
#pragma unroll
        for (int c = 0; c < CW; ++c) {
          const int64_t o = r * nv + j + c;
          const double2 xr = VTr<VT>::ld(vin + o);
          double2 res;
          if constexpr (CPLX) res = cadd(cmul(A.alpha_off, acc[c]), cmul(dsum, xr));
          else res = make_double2(A.alpha_off.x * acc[c].x + dsum.x * xr.x, 0.0);
          if (A.beta) res = cadd(res, VTr<VT>::ld(vout + o));
          VTr<VT>::st(vout + o, res);
          if constexpr (EPI) {
            VT* __restrict__ F = (VT*)A.epi_F;
            const double2 rs = VTr<VT>::rnd(res);
            const double2 f = VTr<VT>::rnd(cadd(VTr<VT>::ld(F + o), rs));
            VTr<VT>::st(F + o, f);
            curB += CPLX ? cabs2(rs) : fabs(rs.x);
            curF += CPLX ? cabs2(f) : fabs(f.x);
          }
        }
      }
    }
    if constexpr (EPI) {
      maxB = fmax(maxB, grp_sum<G>(curB));
      maxF = fmax(maxF, grp_sum<G>(curF));
    }
  }
  if constexpr (EPI) epi_norms_out(A, maxB, maxF);
}

// Lanes per row: as k_csr_mm's rule, four at least (64 rows fill a block).
inline int pk_group(int64_t n) {
  int best = 64;
  int64_t cost = INT64_MAX;
  for (int g = 64; g >= 8; g >>= 1) {
    const int64_t c = (n + g - 1) / g * (g + 4);
    if (c < cost) { cost = c; best = g; }
  }
  return best == 8 && n <= 4 ? 4 : best;
}

template <typename VT, int CW, bool EPI>
void launch_packed_mm(const HvArgs& A, hipStream_t st) {
  const int G = pk_group(A.nvec / CW);
  const int64_t nsl = (A.Ns + 63) / 64;
  // a slice's row rounds over several blocks until about four blocks per CU
  const int rounds = 64 * G / 256;
  int64_t gy = nsl > 0 ? (1024 + nsl - 1) / nsl : 1;
  if (gy > rounds) gy = rounds;
  const dim3 grid((unsigned)nsl, (unsigned)(gy < 1 ? 1 : gy)), blk(256);
  switch (G) {
    case 4: hipLaunchKernelGGL((k_packed_mm<VT, 4, CW, EPI>), grid, blk, 0, st, A); break;
    case 8: hipLaunchKernelGGL((k_packed_mm<VT, 8, CW, EPI>), grid, blk, 0, st, A); break;
    case 16: hipLaunchKernelGGL((k_packed_mm<VT, 16, CW, EPI>), grid, blk, 0, st, A); break;
    case 32: hipLaunchKernelGGL((k_packed_mm<VT, 32, CW, EPI>), grid, blk, 0, st, A); break;
    default: hipLaunchKernelGGL((k_packed_mm<VT, 64, CW, EPI>), grid, blk, 0, st, A); break;
  }
}

template <typename VT, bool EPI>
void launch_packed_t(const HvArgs& A, hipStream_t st) {
  if (A.nvec == 1) {
    hipLaunchKernelGGL((k_packed_rows<VT, EPI>), dim3((unsigned)qsx_grid(A.Ns, 256)), dim3(256), 0, st, A);
    return;
  }
  if constexpr (sizeof(VT) == 8) {
    if (A.nvec % 2 == 0 && (uintptr_t)A.v_in % 16 == 0) { launch_packed_mm<VT, 2, EPI>(A, st); return; }
  }
  launch_packed_mm<VT, 1, EPI>(A, st);
}
