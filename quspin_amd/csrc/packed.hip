// Packed rows of a matrix-free operator: build and product (packed_impl.h).
// The products are those of ``_core.inplace_op`` over a term list
// (src/quspin/basis/basis_general/base_general.py:392-408).
#include <hipcub/hipcub.hpp>

#include <cstddef>
#include <string>

#include "packed_impl.h"

// per-row element evaluation of the H.v context (hv.hip)
int qsx_hv_ctx_pack_args(const qsx_hv_ctx* X, HvArgs* A, int* N, int* nmaps, int* fermion, int* lookup);

__global__ void __launch_bounds__(256) k_pack_clear(PackDict* D) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < PK_SLOTS) D->key[i] = 0ull;
  if (i == 0) { D->n_lut = 0; D->bad = 0; D->total = 0; D->used = 0; }
}

// What pass 0 keeps of every element where the work buffer has room: its
// coefficient, column and dictionary slot (-1 ends a row), element e of row r
// at (r / 64 * n_off + e) * 64 + r % 64.  Null: pass 1 evaluates them again.
struct PackStash {
  double2* v;
  int2* cs;
};

// PASS 0: enter every coefficient into the dictionary, off[slice] = 64 x the
// slice's widest row.  PASS 1: write the entries (ids assigned).  A row stops
// at its first element after the build is refused.
template <typename I, int M, bool FERM, int LK, int PASS>
__global__ void __launch_bounds__(256) k_pack_rows(HvArgs A, PackDict* D, int64_t* __restrict__ off,
                                                   uint32_t* __restrict__ ent, int bits, PackStash S) {
  __shared__ int64_t sb[(LK == LOOKUP_TABLE || LK == LOOKUP_RANK) ? QSX_SB : 1];
  stage_binom<LK>(A.R, sb);
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t sl = r >> 6;
  if (sl >= (A.Ns + 63) >> 6) return;  // whole waves
  const int lane = threadIdx.x & 63;
  const bool live = r < A.Ns;
  int k = 0;
  const int64_t o0 = PASS == 1 ? off[sl] : 0;
  const int wid = PASS == 1 ? (int)((off[sl + 1] - o0) >> 6) : 0;
  if (live) {
    const I s = ((const I*)A.basis)[r];
    double rsq = 1.0;
    if constexpr (M != 0) rsq = 1.0 / sqrt(load_n(A.nrm, A.n_bytes, r));
    const RowRank rr = row_rank_if<I, LK>(A, sb, s);
    double2 last = make_double2(0.0, 0.0);
    int slot = -1;
    bool go = true;
    for (int t = 0; t < A.n_off && go; ++t) {
      term_element<I, M, FERM, LK, true>(A, sb, rr, A.off + t, s, rsq, A.off_conj, [&](int64_t c, double2 coef) {
        if (slot < 0 || coef.x != last.x || coef.y != last.y) {  // neighbouring terms often share the value
          slot = pk_slot(D, coef);
          last = coef;
        }
        if (slot < 0) { go = false; return; }
        if constexpr (PASS == 1) {
          const double2 v = D->val[slot];
          if (v.x != coef.x || v.y != coef.y) D->bad = 1;
          if (k < wid) ent[o0 + (int64_t)k * 64 + lane] = (uint32_t)c | ((uint32_t)D->id[slot] << bits);
        } else if (S.v) {
          if (k >= A.n_off) { D->bad = 1; go = false; return; }
          const int64_t o = (sl * A.n_off + k) * 64 + lane;
          S.v[o] = coef;
          S.cs[o] = make_int2((int)c, slot);
        }
        ++k;
      });
    }
  }
  if constexpr (PASS == 0) {
    if (S.v && live && k < A.n_off) S.cs[(sl * A.n_off + k) * 64 + lane] = make_int2(0, -1);
    int m = k;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    if (lane == 0) off[sl] = (int64_t)m * 64;
  } else {
    // padding: the row itself (the last row for lanes past the end), weight 0
    const uint32_t pad = (uint32_t)(live ? r : A.Ns - 1);
    for (; k < wid; ++k) ent[o0 + (int64_t)k * 64 + lane] = pad;
  }
}

// Pass 1 from the kept elements: the same entries without evaluating the
// operator again.  First product of a new operator, build included: momentum
// sector of L = 22 912 -> 701 us, of L = 24 with 16 vectors 1,292 -> 1,083;
// 40 Lanczos steps of L = 16, k = 5 890 -> 774.
__global__ void __launch_bounds__(256) k_pack_kept(PackStash S, int n_off, int64_t Ns, PackDict* D,
                                                   const int64_t* __restrict__ off, uint32_t* __restrict__ ent,
                                                   int bits) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t sl = r >> 6;
  if (sl >= (Ns + 63) >> 6) return;
  const int lane = threadIdx.x & 63;
  const int64_t o0 = off[sl];
  const int wid = (int)((off[sl + 1] - o0) >> 6);
  const uint32_t pad = (uint32_t)(r < Ns ? r : Ns - 1);
  bool more = r < Ns;
  for (int k = 0; k < wid; ++k) {
    uint32_t e = pad;
    if (more) {
      const int64_t o = (sl * n_off + k) * 64 + lane;
      const int2 cs = k < n_off ? S.cs[o] : make_int2(0, -1);
      more = cs.y >= 0;
      if (more) {
        const double2 v = D->val[cs.y], c = S.v[o];
        if (v.x != c.x || v.y != c.y) D->bad = 1;
        e = (uint32_t)cs.x | ((uint32_t)D->id[cs.y] << bits);
      }
    }
    ent[o0 + (int64_t)k * 64 + lane] = e;
  }
}

// ids 1 .. n of the occupied slots in slot order, and the total of the scan
__global__ void __launch_bounds__(1024) k_pack_ids(PackDict* D, const int64_t* __restrict__ off, int64_t nsl) {
  __shared__ int s[1024];
  constexpr int PER = PK_SLOTS / 1024;
  const int t = threadIdx.x;
  int n = 0;
  for (int q = 0; q < PER; ++q) n += D->key[t * PER + q] != 0;
  s[t] = n;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? s[t - o] : 0;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  int id = s[t] - n + 1;
  for (int q = 0; q < PER; ++q)
    if (D->key[t * PER + q] != 0) D->id[t * PER + q] = id++;
  if (t == 1023) D->n_lut = s[t] + 1;
  if (t == 0) D->total = off[nsl];
}

__global__ void __launch_bounds__(256) k_pack_lut(const PackDict* __restrict__ D, double2* __restrict__ lut) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i == 0) lut[0] = make_double2(0.0, 0.0);
  if (i < PK_SLOTS && D->key[i] != 0) lut[D->id[i]] = D->val[i];
}

template <typename I, int M, bool FERM, int LK>
static void launch_pack(const HvArgs& A, int pass, PackDict* D, int64_t* off, uint32_t* ent, int bits,
                        PackStash S, hipStream_t st) {
  const dim3 grid((unsigned)qsx_grid(A.Ns, 256)), blk(256);
  if (pass == 0) hipLaunchKernelGGL((k_pack_rows<I, M, FERM, LK, 0>), grid, blk, 0, st, A, D, off, ent, bits, S);
  else hipLaunchKernelGGL((k_pack_rows<I, M, FERM, LK, 1>), grid, blk, 0, st, A, D, off, ent, bits, S);
}

template <typename I>
static void pack_dispatch(const HvArgs& A, int nmaps, bool fm, int lk, int pass, PackDict* D, int64_t* off,
                          uint32_t* ent, int bits, PackStash S, hipStream_t st) {
  if (lk == LOOKUP_TABLE) {
    if (fm) launch_pack<I, 1, true, LOOKUP_TABLE>(A, pass, D, off, ent, bits, S, st);
    else launch_pack<I, 1, false, LOOKUP_TABLE>(A, pass, D, off, ent, bits, S, st);
  } else if (nmaps == 0) {
    if (lk == LOOKUP_RANK) launch_pack<I, 0, false, LOOKUP_RANK>(A, pass, D, off, ent, bits, S, st);
    else launch_pack<I, 0, false, LOOKUP_SEARCH>(A, pass, D, off, ent, bits, S, st);
  } else if (fm) {
    QSX_HV_MSWITCH(nmaps, (launch_pack<I, MM, true, LOOKUP_SEARCH>(A, pass, D, off, ent, bits, S, st)));
  } else {
    QSX_HV_MSWITCH(nmaps, (launch_pack<I, MM, false, LOOKUP_SEARCH>(A, pass, D, off, ent, bits, S, st)));
  }
}

static int bits_for(int64_t Ns) {
  int b = 1;
  while (((int64_t)1 << b) < Ns) ++b;
  return b;
}

static size_t scan_bytes(int64_t n) {
  size_t tb = 0;
  (void)hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (const int64_t*)nullptr, (int64_t*)nullptr, (int)n, 0);
  return (tb + 255) / 256 * 256;
}

// Most bytes of kept elements (24 each).  Above it they are evaluated twice: a
// pass takes about 1.7 ms at L = 28 (243 MB of elements), for
// which a build does not take a buffer ten times its result.
constexpr int64_t PK_STASH_MAX = 64 << 20;

// The parts of the work buffer
struct PackWork {
  size_t tb;              // scan scratch
  int64_t tmp, wid, v, cs, bytes;  // offsets; v = 0: no elements kept
  PackWork(int64_t Ns, int n_off) {
    const int64_t nsl = (Ns + 63) / 64, kept = nsl * 64 * n_off;
    tb = scan_bytes(nsl + 1);
    tmp = (int64_t)(sizeof(PackDict) + 255) / 256 * 256;
    wid = tmp + (int64_t)tb;
    bytes = (wid + 8 * (nsl + 1) + 255) / 256 * 256;
    v = cs = 0;
    if (kept * 24 <= PK_STASH_MAX) {
      v = bytes;
      cs = v + kept * 16;
      bytes = cs + kept * 8;
    }
  }
  PackStash stash(void* work) const {
    return v ? PackStash{(double2*)((char*)work + v), (int2*)((char*)work + cs)} : PackStash{nullptr, nullptr};
  }
};

extern "C" int64_t qsx_hv_pack_work_bytes(const qsx_hv_ctx* X) {
  HvArgs A;
  int N, nm, fm, lk;
  if (!X || qsx_hv_ctx_pack_args(X, &A, &N, &nm, &fm, &lk)) return 0;
  return PackWork(A.Ns, A.n_off).bytes;
}

// First pass: slice offsets into off (device, (Ns + 63) / 64 + 1 entries), the
// dictionary into work, and the sizes the second pass needs.
// QSX_ERR_UNSUPPORTED: the operator has no packed form (no off-diagonal terms,
// a list that does not commute with the group, unfolded diagonal terms, too
// many distinct coefficients for four-byte entries).
extern "C" int qsx_hv_pack_count(const qsx_hv_ctx* X, int64_t* off, void* work, int64_t work_bytes, int64_t* entries,
                                 int* n_lut, int* idx_bits, void* stream) {
  HvArgs A;
  int N, nm, fm, lk;
  if (!X || !off || !work || !entries || !n_lut || !idx_bits) { qsx_set_error("qsx_hv_pack_count: bad arguments"); return QSX_ERR_ARG; }
  int rc = qsx_hv_ctx_pack_args(X, &A, &N, &nm, &fm, &lk);
  if (rc) return rc;
  const PackWork W(A.Ns, A.n_off);
  if (work_bytes < W.bytes) { qsx_set_error("qsx_hv_pack_count: work buffer too small"); return QSX_ERR_ARG; }
  hipStream_t st = (hipStream_t)stream;
  const int64_t nsl = (A.Ns + 63) / 64;
  PackDict* D = (PackDict*)work;
  char* tmp = (char*)work + W.tmp;
  size_t tb = W.tb;
  int64_t* wid = (int64_t*)((char*)work + W.wid);
  const int bits = bits_for(A.Ns);
  hipLaunchKernelGGL(k_pack_clear, dim3(PK_SLOTS / 256), dim3(256), 0, st, D);
  if (N <= 32) pack_dispatch<uint32_t>(A, nm, fm, lk, 0, D, wid, nullptr, bits, W.stash(work), st);
  else pack_dispatch<uint64_t>(A, nm, fm, lk, 0, D, wid, nullptr, bits, W.stash(work), st);
  QSX_LAUNCH_CHECK();
  QSX_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, wid, off, (int)(nsl + 1), st));
  hipLaunchKernelGGL(k_pack_ids, dim3(1), dim3(1024), 0, st, D, off, nsl);
  QSX_LAUNCH_CHECK();
  struct { int32_t n_lut, bad; int64_t total; } h;
  static_assert(offsetof(PackDict, total) - offsetof(PackDict, n_lut) == 8, "tail layout");
  QSX_CHECK_HIP(hipMemcpyAsync(&h, (char*)work + offsetof(PackDict, n_lut), sizeof(h), hipMemcpyDeviceToHost, st));
  QSX_CHECK_HIP(hipStreamSynchronize(st));
  int idb = 1;
  while ((1 << idb) < h.n_lut) ++idb;
  if (h.bad || h.n_lut > PK_LUT_MAX || bits + idb > 32) {
    qsx_set_error("packed rows: too many distinct coefficients for four-byte entries");
    return QSX_ERR_UNSUPPORTED;
  }
  *entries = h.total;
  *n_lut = h.n_lut;
  *idx_bits = bits;
  return QSX_OK;
}

// Second pass: the entries (uint32, `entries` of them) and the coefficients
// (n_lut complex128 values).  Returns with the buffers complete.
extern "C" int qsx_hv_pack_fill(const qsx_hv_ctx* X, int64_t* off, void* work, void* ent, void* lut, void* stream) {
  HvArgs A;
  int N, nm, fm, lk;
  if (!X || !off || !work || !ent || !lut) { qsx_set_error("qsx_hv_pack_fill: bad arguments"); return QSX_ERR_ARG; }
  int rc = qsx_hv_ctx_pack_args(X, &A, &N, &nm, &fm, &lk);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  PackDict* D = (PackDict*)work;
  const int bits = bits_for(A.Ns);
  const PackStash S = PackWork(A.Ns, A.n_off).stash(work);
  if (S.v)
    hipLaunchKernelGGL(k_pack_kept, dim3((unsigned)qsx_grid(A.Ns, 256)), dim3(256), 0, st, S, A.n_off, A.Ns, D, off,
                       (uint32_t*)ent, bits);
  else if (N <= 32) pack_dispatch<uint32_t>(A, nm, fm, lk, 1, D, off, (uint32_t*)ent, bits, S, st);
  else pack_dispatch<uint64_t>(A, nm, fm, lk, 1, D, off, (uint32_t*)ent, bits, S, st);
  hipLaunchKernelGGL(k_pack_lut, dim3(PK_SLOTS / 256), dim3(256), 0, st, D, (double2*)lut);
  QSX_LAUNCH_CHECK();
  int32_t bad = 0;
  QSX_CHECK_HIP(hipMemcpyAsync(&bad, (char*)work + offsetof(PackDict, bad), sizeof(bad), hipMemcpyDeviceToHost, st));
  QSX_CHECK_HIP(hipStreamSynchronize(st));
  if (bad) { qsx_set_error("packed rows: two coefficients share a dictionary key"); return QSX_ERR_UNSUPPORTED; }
  return QSX_OK;
}

// One product (A.epi_F set: one Taylor term) on the packed rows of A.
int qsx_packed_launch(const HvArgs& A, int dtype, hipStream_t st) {
  const bool epi = A.epi_F != nullptr;
  switch (dtype) {
    case QSX_F32: epi ? launch_packed_t<float, true>(A, st) : launch_packed_t<float, false>(A, st); break;
    case QSX_F64: epi ? launch_packed_t<double, true>(A, st) : launch_packed_t<double, false>(A, st); break;
    case QSX_C64: epi ? launch_packed_t<float2, true>(A, st) : launch_packed_t<float2, false>(A, st); break;
    case QSX_C128: epi ? launch_packed_t<double2, true>(A, st) : launch_packed_t<double2, false>(A, st); break;
    default: qsx_set_error("unknown dtype code"); return QSX_ERR_ARG;
  }
  QSX_LAUNCH_CHECK();
  return QSX_OK;
}
