// Small operators: the whole Taylor loop, or the whole Lanczos recurrence, in
// one workgroup.
//
// Below a few thousand states a term or a step is a fraction of a launch, so
// the loops of sparse.hip spend their time between launches.  Here the vector
// that the products gather from lives in LDS, every thread owns up to SMALL_E
// rows whose other vectors stay in its registers, and the norms and dots are
// block reductions: two or three barriers per term or step instead of two to
// four launches.  Same recurrences, roundings and truncation test as there.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "packed_impl.h"

namespace {

constexpr int SMALL_T = 1024;  // threads
// Sizes up to which one workgroup wins over a launch per term or two per step;
// a row beyond a thread's second leaves too few registers for its elements
// (assembled matrices: small_csr besides).
// Measured on sectors without symmetries, t = 1 steps (about 65 terms) and 30
// Lanczos steps, launches -> one workgroup:
//   assembled     924 rows 593 -> 215 us, 1,716 rows 607 -> 424, 3,432 rows 617 -> 985
//   packed rows   924 rows 423 -> 225 us, 1,716 rows 450 -> 292, 3,432 rows 450 -> 642
//   Lanczos, packed, rows / entries, float64 and complex128:
//     924 / 9,216     302 -> 109 us, 310 -> 118     2,002 / 34,560  337 -> 178, 336 -> 211
//     3,876 / 30,592  255 -> 202,    254 -> 268     4,060 / 24,576  251 -> 177, 285 -> 236
//     3,432 / 36,224  262 -> 249,    268 -> 312     3,060 / 46,848  318 -> 309, 308 -> 365
//   float32 and complex64 at the last three: 255 -> 192 us, 290 -> 310;
//   266 -> 278, 288 -> 425; 309 -> 338, 328 -> 499 (two rows per thread, 2,002
//   / 34,560: 309 -> 193, 368 -> 258)
constexpr int SMALL_N = 2048, SMALL_NNZ = 24576;
// Lanczos on packed rows: up to two rows per thread, and up to four
constexpr int SMALL_N_LZ = 4096, SMALL_NNZ_LZ = 49152, SMALL_NNZ_LZ4 = 32768, SMALL_NNZ_LZ4_CPLX = 20480;

struct SmallArgs {
  // CSR form
  const void* indptr;
  const void* indices;
  const void* data;
  int idx64;
  // packed form
  const int64_t* off;
  const uint32_t* ent;
  const double2* lut;
  int n_lut, bits;
  const void* diag;
  int diag_cplx;
  int n;
  // Taylor loop
  void* F;
  int s, m;
  double tol;
  double2 a, mu, eta;
  // Lanczos
  const void* v0;
  double eps;
  void* Q;
  double* ab;
  int steps;
};

// Row products against the vector xs in LDS.  A row's extent and its first KR
// elements are read once and stay in registers (the lanes of a CSR row start
// on lines of their own: re-reading them every term took 5 us of 6.5 at 924
// rows); longer rows read the rest from memory.
template <typename MT, typename VT, int E>
struct CsrRows {
  static constexpr int KR = E == 1 ? (sizeof(MT) >= 16 ? 8 : 16) : 4;
  static constexpr int LUT = 1;
  using LT = double;
  struct Row {
    int64_t k0;
    int len;
    uint16_t c[KR];
    MT v[KR];
  };
  __device__ static void mac(double2& acc, MT v, const VT* x) {
    const double2 xx = VTr<VT>::ld(x), mm = MTr<MT>::ld(&v);
    if constexpr (VTr<VT>::cplx) {
      if constexpr (MTr<MT>::cplx) acc = cadd(acc, cmul(mm, xx));
      else acc = make_double2(acc.x + mm.x * xx.x, acc.y + mm.x * xx.y);
    } else {
      acc.x += mm.x * xx.x;
    }
  }
  __device__ static void open(Row& R, const SmallArgs& A, int r) {
    R.k0 = ld_idx(A.indptr, A.idx64, r);
    R.len = (int)(ld_idx(A.indptr, A.idx64, r + 1) - R.k0);
    const MT* __restrict__ val = (const MT*)A.data + R.k0;
#pragma unroll
    for (int u = 0; u < KR; ++u) {
      const bool on = u < R.len;
      R.c[u] = on ? (uint16_t)ld_idx(A.indices, A.idx64, R.k0 + u) : (uint16_t)r;
      if (on) R.v[u] = val[u];
    }
  }
  __device__ static double2 dot(const SmallArgs& A, const Row& R, int r, const VT* xs, const LT*) {
    double2 acc = make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < KR; ++u)
      if (u < R.len) mac(acc, R.v[u], xs + R.c[u]);
    const MT* __restrict__ val = (const MT*)A.data + R.k0;
    for (int k = KR; k < R.len; ++k) mac(acc, val[k], xs + (int)ld_idx(A.indices, A.idx64, R.k0 + k));
    return acc;
  }
};

template <typename VT, int E>
struct PackedRows {
  static constexpr int KR = E == 1 ? 24 : E == 2 ? 12 : 4;
  static constexpr int LUT = PK_LUT_MAX;
  using LT = typename std::conditional<VTr<VT>::cplx, double2, double>::type;
  struct Row {
    const uint32_t* e;
    int wid;  // one value per wave: its rows are one slice
    double2 d;
    uint32_t v[KR];  // column | id << 16; the padding's column is n, where xs holds a 0
  };
  __device__ static void mac(double2& acc, LT c, double2 x) {
    if constexpr (VTr<VT>::cplx) acc = cadd(acc, cmul(c, x));
    else acc.x += c * x.x;
  }
  __device__ static void open(Row& R, const SmallArgs& A, int r) {
    const int64_t o0 = A.off[r >> 6];
    R.e = A.ent + o0 + (r & 63);
    R.wid = __builtin_amdgcn_readfirstlane((int)((A.off[(r >> 6) + 1] - o0) >> 6));
    R.d = make_double2(0.0, 0.0);
    if (A.diag) {
      if (A.diag_cplx) R.d = ((const double2*)A.diag)[r];
      else R.d.x = ((const double*)A.diag)[r];
    }
#pragma unroll
    for (int u = 0; u < KR; ++u) {
      const uint32_t ev = u < R.wid ? R.e[u * 64] : 0u, id = ev >> A.bits;
      R.v[u] = (id ? ev & ((1u << A.bits) - 1u) : (uint32_t)A.n) | id << 16;
    }
  }
  __device__ static double2 dot(const SmallArgs& A, const Row& R, int r, const VT* xs, const LT* lut) {
    constexpr bool CPLX = VTr<VT>::cplx;
    const double2 xr = VTr<VT>::ld(xs + r);
    double2 acc;
    if constexpr (CPLX) acc = cmul(R.d, xr);
    else acc = make_double2(R.d.x * xr.x, 0.0);
#pragma unroll
    for (int u = 0; u < KR; ++u)
      if (u < R.wid) mac(acc, lut[R.v[u] >> 16], VTr<VT>::ld(xs + (R.v[u] & 0xffffu)));
    const uint32_t cmask = (1u << A.bits) - 1u;
    for (int u = KR; u < R.wid; ++u) {
      const uint32_t ev = R.e[u * 64], id = ev >> A.bits;
      mac(acc, lut[id], pk_x(xs + (ev & cmask), id));
    }
    return acc;
  }
};

template <typename OP>
__device__ __forceinline__ void small_lut(const SmallArgs& A, typename OP::LT* lut) {
  if constexpr (OP::LUT > 1) {
    for (int i = threadIdx.x; i < A.n_lut; i += blockDim.x) {
      if constexpr (sizeof(typename OP::LT) == 16) lut[i] = A.lut[i];
      else lut[i] = A.lut[i].x;
    }
  }
}

// One workgroup: F <- e^{aA} F with the partition (s, m) of A.
template <typename OP, typename VT, int E>
__global__ void __launch_bounds__(SMALL_T) k_small_expm(SmallArgs A) {
  extern __shared__ unsigned char small_smem[];
  VT* xs = (VT*)small_smem;
  __shared__ typename OP::LT lut[OP::LUT];
  __shared__ double red[2][2][SMALL_T / 64];
  constexpr bool CPLX = VTr<VT>::cplx;
  const int n = A.n, nt = blockDim.x, nw = nt >> 6;
  VT* F = (VT*)A.F;
  typename OP::Row row[E];
  double2 f[E];
  small_lut<OP>(A, lut);
  if (threadIdx.x == 0) VTr<VT>::st(xs + n, make_double2(0.0, 0.0));
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + e * nt;
    const int ic = i < n ? i : n - 1;
    OP::open(row[e], A, ic);
    f[e] = VTr<VT>::ld(F + ic);
    if (i < n) VTr<VT>::st(xs + i, f[e]);
  }
  int par = 0;
  // block maxima of two non-negative values (all threads get them); orders the
  // LDS accesses before it against those after it
  auto max2 = [&](double& p, double& q) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      p = fmax(p, __shfl_xor(p, o, 64));
      q = fmax(q, __shfl_xor(q, o, 64));
    }
    if ((threadIdx.x & 63) == 0) { red[par][0][threadIdx.x >> 6] = p; red[par][1][threadIdx.x >> 6] = q; }
    __syncthreads();
    p = red[par][0][0];
    q = red[par][1][0];
    for (int i = 1; i < nw; ++i) { p = fmax(p, red[par][0][i]); q = fmax(q, red[par][1][i]); }
    par ^= 1;
  };
  auto vabs1 = [](double2 v) { return CPLX ? sqrt(v.x * v.x + v.y * v.y) : fabs(v.x); };
  for (int st = 0; st < A.s; ++st) {
    double c1 = 0.0, dummy = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) c1 = fmax(c1, vabs1(f[e]));
    max2(c1, dummy);  // also: xs is complete
    for (int j = 0; j < A.m; ++j) {
      const double cf = 1.0 / ((double)A.s * (double)(j + 1));
      const double2 at = make_double2(A.a.x * cf, A.a.y * cf);
      double mb = 0.0, mf = 0.0;
      double2 nb[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = threadIdx.x + e * nt;
        const int ic = i < n ? i : n - 1;
        double2 acc = OP::dot(A, row[e], ic, xs, lut);
        const double2 xr = VTr<VT>::ld(xs + ic);
        double2 res;
        if constexpr (CPLX) {
          acc = cadd(acc, make_double2(-(A.mu.x * xr.x - A.mu.y * xr.y), -(A.mu.x * xr.y + A.mu.y * xr.x)));
          res = cmul(at, acc);
        } else {
          res = make_double2(at.x * (acc.x - A.mu.x * xr.x), 0.0);
        }
        nb[e] = VTr<VT>::rnd(res);
        f[e] = VTr<VT>::rnd(cadd(f[e], nb[e]));
        mb = fmax(mb, vabs1(nb[e]));  // rows past the end repeat the last one
        mf = fmax(mf, vabs1(f[e]));
      }
      max2(mb, mf);  // every read of xs is done
      if (c1 + mb <= A.tol * mf) break;
      c1 = mb;
      if (j + 1 < A.m) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int i = threadIdx.x + e * nt;
          if (i < n) VTr<VT>::st(xs + i, nb[e]);
        }
        __syncthreads();
      }
    }
    // next stage: F *= e^{a mu / s}, B = F
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = threadIdx.x + e * nt;
      if constexpr (CPLX) f[e] = VTr<VT>::rnd(cmul(A.eta, f[e]));
      else f[e] = VTr<VT>::rnd(make_double2(f[e].x * A.eta.x, 0.0));
      if (i < n && st + 1 < A.s) VTr<VT>::st(xs + i, f[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + e * nt;
    if (i < n) VTr<VT>::st(F + i, f[e]);
  }
}

// One workgroup: the Lanczos recurrence from v0 (normalised first when its
// norm is off 1 by more than eps), a_i and b_i into ab, q_i into Q (or none).
template <typename OP, typename VT, int E>
__global__ void __launch_bounds__(SMALL_T) k_small_lanczos(SmallArgs A) {
  extern __shared__ unsigned char small_smem[];
  VT* xs = (VT*)small_smem;
  __shared__ typename OP::LT lut[OP::LUT];
  __shared__ double red[2][SMALL_T / 64];
  const int n = A.n, nt = blockDim.x, nw = nt >> 6;
  VT* Q = (VT*)A.Q;
  typename OP::Row row[E];
  double2 q[E], qp[E], r[E];
  small_lut<OP>(A, lut);
  if (threadIdx.x == 0) VTr<VT>::st(xs + n, make_double2(0.0, 0.0));
  int par = 0;
  // block sum in a fixed order; a barrier as max2 above
  auto sum1 = [&](double p) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o, 64);
    if ((threadIdx.x & 63) == 0) red[par][threadIdx.x >> 6] = p;
    __syncthreads();
    p = red[par][0];
    for (int i = 1; i < nw; ++i) p += red[par][i];
    par ^= 1;
    return p;
  };
  double s2 = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = threadIdx.x + e * nt;
    const bool live = i < n;
    OP::open(row[e], A, live ? i : n - 1);
    q[e] = live ? VTr<VT>::ld((const VT*)A.v0 + i) : make_double2(0.0, 0.0);
    qp[e] = make_double2(0.0, 0.0);
    s2 += q[e].x * q[e].x + q[e].y * q[e].y;
  }
  const double nrm = sqrt(sum1(s2));
  const bool scale = fabs(nrm - 1.0) > A.eps;
  double b = 0.0;
  for (int st = 0; st < A.steps; ++st) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = threadIdx.x + e * nt;
      if (st > 0) {
        qp[e] = q[e];
        q[e] = VTr<VT>::rnd(make_double2(r[e].x / b, r[e].y / b));
      } else if (scale) {
        q[e] = VTr<VT>::rnd(make_double2(q[e].x / nrm, q[e].y / nrm));
      }
      if (i < n) {
        VTr<VT>::st(xs + i, q[e]);
        if (Q) VTr<VT>::st(Q + (int64_t)st * n + i, q[e]);
      } else {
        q[e] = make_double2(0.0, 0.0);  // rows past the end add nothing
      }
    }
    __syncthreads();
    double d = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = threadIdx.x + e * nt;
      if (i < n) {
        r[e] = VTr<VT>::rnd(OP::dot(A, row[e], i, xs, lut));
        if (st > 0) r[e] = VTr<VT>::rnd(make_double2(r[e].x - b * qp[e].x, r[e].y - b * qp[e].y));
        d += q[e].x * r[e].x + q[e].y * r[e].y;
      } else {
        r[e] = make_double2(0.0, 0.0);
      }
    }
    const double a = sum1(d);
    double w = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      r[e] = VTr<VT>::rnd(make_double2(r[e].x - a * q[e].x, r[e].y - a * q[e].y));
      w += r[e].x * r[e].x + r[e].y * r[e].y;
    }
    b = sqrt(sum1(w));
    if (threadIdx.x == 0) {
      A.ab[4 * (int64_t)st] = a;
      A.ab[4 * (int64_t)st + 2] = b;
    }
  }
}

// LDS a workgroup of the current device may take: complex128 Lanczos above
// 3,056 rows asks for more than 64 KB.
size_t lds_limit() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
    return 65536;
  return (size_t)v;
}

// False, nothing launched: more LDS than the device has for a workgroup, or
// more rows than the form takes.
template <template <int> class OPE, typename VT, bool LZ, bool FOUR>
bool launch_small(const SmallArgs& A, hipStream_t st) {
  const int E = A.n <= SMALL_T ? 1 : A.n <= 2 * SMALL_T ? 2 : 4;
  int nt = ((A.n + E - 1) / E + 63) / 64 * 64;
  if (nt > SMALL_T) nt = SMALL_T;
  const size_t lds = (size_t)(A.n + 1) * sizeof(VT);  // the vector and the padding's 0
  constexpr size_t fixed = sizeof(typename OPE<1>::LT) * OPE<1>::LUT + (LZ ? 2 : 4) * sizeof(double) * (SMALL_T / 64);
  if (lds + fixed > 65536 && lds + fixed > lds_limit()) return false;
#define QSX_SMALL(EE)                                                                             \
  if constexpr (LZ) hipLaunchKernelGGL((k_small_lanczos<OPE<EE>, VT, EE>), dim3(1), dim3(nt), lds, st, A); \
  else hipLaunchKernelGGL((k_small_expm<OPE<EE>, VT, EE>), dim3(1), dim3(nt), lds, st, A)
  if (E == 1) { QSX_SMALL(1); }
  else if (E == 2) { QSX_SMALL(2); }
  else if constexpr (FOUR) { QSX_SMALL(4); }
  else return false;
#undef QSX_SMALL
  return true;
}

template <typename MT, typename VT>
struct CsrOf {
  template <int E> using Op = CsrRows<MT, VT, E>;
};
template <typename VT>
struct PackedOf {
  template <int E> using Op = PackedRows<VT, E>;
};

template <bool LZ>
bool launch_small_csr(const SmallArgs& A, int mdt, int vdt, hipStream_t st) {
  if (vdt == QSX_F32 && mdt == QSX_F32) return launch_small<CsrOf<float, float>::template Op, float, LZ, false>(A, st);
  if (vdt == QSX_F64 && mdt == QSX_F64) return launch_small<CsrOf<double, double>::template Op, double, LZ, false>(A, st);
  if (vdt == QSX_C64 && mdt == QSX_F32) return launch_small<CsrOf<float, float2>::template Op, float2, LZ, false>(A, st);
  if (vdt == QSX_C64 && mdt == QSX_C64) return launch_small<CsrOf<float2, float2>::template Op, float2, LZ, false>(A, st);
  if (vdt == QSX_C128 && mdt == QSX_F64) return launch_small<CsrOf<double, double2>::template Op, double2, LZ, false>(A, st);
  if (vdt == QSX_C128 && mdt == QSX_C128) return launch_small<CsrOf<double2, double2>::template Op, double2, LZ, false>(A, st);
  return false;
}

template <bool LZ>
bool launch_small_packed(const SmallArgs& A, int vdt, hipStream_t st) {
  switch (vdt) {
    case QSX_F32: return launch_small<PackedOf<float>::template Op, float, LZ, LZ>(A, st);
    case QSX_F64: return launch_small<PackedOf<double>::template Op, double, LZ, LZ>(A, st);
    case QSX_C64: return launch_small<PackedOf<float2>::template Op, float2, LZ, LZ>(A, st);
    case QSX_C128: return launch_small<PackedOf<double2>::template Op, double2, LZ, LZ>(A, st);
    default: return false;
  }
}

bool small_size(int64_t n, int64_t entries) { return n >= 1 && n <= SMALL_N && entries <= SMALL_NNZ; }

// Whether one workgroup wins on an assembled matrix: a term's time here, in
// microseconds, is that of n rows plus what the entries beyond a thread's
// registers cost, which are read from memory on every term (fitted to 744 loops
// over 20 to 2,000 rows of 2 to 200 entries, random and banded, of every
// dtype).  A launch per term takes 6 to 8 us there, a Lanczos step of launches
// 13 to 18 (here 3 more than a term).  200 rows of 100 entries 16.8 us here and
// 7.7 there, 500 of 48 15.7 and 7.2, 500 of 16 2.4 and 7.4.
bool small_csr(int64_t n, int64_t nnz, int mat_dtype, bool lanczos) {
  if (!small_size(n, nnz)) return false;
  const double k = (double)nnz / (double)n;
  if (n <= SMALL_T) {
    const double us = 1.0 + 2e-3 * n + (0.08 + 6e-4 * n) * std::max(0.0, k - (mat_dtype == QSX_C128 ? 8 : 16));
    return us <= (lanczos ? 11.5 : 6.5);
  }
  return k <= 12.5 && 1.8e-3 * n + 4e-4 * n * std::max(0.0, k - 4.0) <= (lanczos ? 11.5 : 7.4);
}

SmallArgs csr_args(const void* indptr, const void* indices, const void* data, int idx64, int64_t n) {
  SmallArgs A;
  std::memset(&A, 0, sizeof(A));
  A.indptr = indptr; A.indices = indices; A.data = data; A.idx64 = idx64; A.n = (int)n;
  return A;
}

// packed rows of an H.v context; false when its product takes another form
bool ctx_args(const void* hv_ctx, bool lanczos, SmallArgs& A, int& dtype) {
  HvArgs H;
  int64_t entries = 0;
  if (!qsx_hv_ctx_packed(hv_ctx, &H, &dtype, &entries)) return false;
  if (lanczos) {
    const bool cplx = dtype == QSX_C64 || dtype == QSX_C128;
    const int64_t most = H.Ns <= 2 * SMALL_T ? SMALL_NNZ_LZ : cplx ? SMALL_NNZ_LZ4_CPLX : SMALL_NNZ_LZ4;
    if (H.Ns < 1 || H.Ns > SMALL_N_LZ || entries > most) return false;
  } else if (!small_size(H.Ns, entries)) {
    return false;
  }
  std::memset(&A, 0, sizeof(A));
  A.off = H.pk_off; A.ent = H.pk_ent; A.lut = H.pk_lut; A.n_lut = H.pk_nlut; A.bits = H.pk_bits;
  A.diag = H.diag_arr; A.diag_cplx = H.diag_arr_cplx;
  A.n = (int)H.Ns;
  return true;
}

void taylor_args(SmallArgs& A, const SmallTaylor& T) {
  A.F = T.v; A.s = T.s; A.m = T.m; A.tol = T.tol; A.a = T.a; A.mu = T.mu;
  const double er = T.a.x * T.mu.x - T.a.y * T.mu.y, ei = T.a.x * T.mu.y + T.a.y * T.mu.x;
  const double mag = std::exp(er / T.s);
  A.eta = make_double2(mag * std::cos(ei / T.s), mag * std::sin(ei / T.s));
}

}  // namespace

bool qsx_small_expm_csr(const void* indptr, const void* indices, const void* data, int idx64, int mat_dtype, int64_t n,
                        int64_t nnz, int vec_dtype, int64_t nvec, const SmallTaylor& T, hipStream_t st) {
  if (nvec != 1 || !small_csr(n, nnz, mat_dtype, false)) return false;
  SmallArgs A = csr_args(indptr, indices, data, idx64, n);
  taylor_args(A, T);
  return launch_small_csr<false>(A, mat_dtype, vec_dtype, st);
}

bool qsx_small_expm_mf(const void* hv_ctx, int vec_dtype, int64_t nvec, const SmallTaylor& T, hipStream_t st) {
  SmallArgs A;
  int dt = -1;
  if (nvec != 1 || !ctx_args(hv_ctx, false, A, dt) || dt != vec_dtype) return false;
  taylor_args(A, T);
  return launch_small_packed<false>(A, vec_dtype, st);
}

// The whole recurrence of qsx_lanczos_run for a small operator in one launch,
// from v0 (normalised when its norm is off 1 by more than eps): a_i and b_i
// into ab (m x 2 x 2 doubles as there), q_0 .. q_{m-1} into Q (m, n) unless it
// is null.  QSX_ERR_UNSUPPORTED, nothing launched: above the sizes at the top,
// or a matrix-free operator without packed rows.
extern "C" int qsx_lanczos_small(int op_kind, const void* hv_ctx, const void* indptr, const void* indices,
                                 const void* data, int idx64, int mat_dtype, int64_t nnz, int dtype, int64_t n, int m,
                                 const void* v0, double eps, void* Q, double* ab, void* stream) {
  if (n < 1 || m < 1 || !v0 || !ab || (op_kind == 0 && !hv_ctx) || (op_kind == 1 && (!indptr || !data))) {
    qsx_set_error("qsx_lanczos_small: bad arguments");
    return QSX_ERR_ARG;
  }
  SmallArgs A;
  int dt = dtype;
  bool ok = false;
  if (op_kind == 0) {
    ok = ctx_args(hv_ctx, true, A, dt) && dt == dtype && A.n == n;
  } else if (small_csr(n, nnz, mat_dtype, true)) {
    A = csr_args(indptr, indices, data, idx64, n);
    ok = true;
  }
  if (ok) {
    A.v0 = v0; A.eps = eps; A.Q = Q; A.ab = ab; A.steps = m;
    ok = op_kind == 0 ? launch_small_packed<true>(A, dtype, (hipStream_t)stream)
                      : launch_small_csr<true>(A, mat_dtype, dtype, (hipStream_t)stream);
  }
  if (!ok) { qsx_set_error("qsx_lanczos_small: not a small operator"); return QSX_ERR_UNSUPPORTED; }
  QSX_LAUNCH_CHECK();
  return QSX_OK;
}
