// Connected elements <x|H|x'> of the two operator families on the VMC path.
//
// nka_ising_conn   : IsingJax.get_conn_padded (netket/operator/_ising/jax.py:125-165)
// nka_localop_conn : LocalOperatorJax.get_conn_padded
//                    (netket/operator/_local_operator/jax.py:74-201)
//
// Both write the padded layout of the reference bit for bit: xp (B, K, N)
// int8 spin values and mels (B, K) in the operator dtype.
#include <stdarg.h>
#include <stdio.h>

#include "nka_common.hpp"
#include "netket_amd.h"

namespace nka {

static thread_local char g_err[512];
void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}
const char* last_error() { return g_err; }

// ---------------------------------------------------------------------------
// Ising.  Row 0: x, mel J * sum_e (2*[x_u == x_v] - 1) (an exact integer sum
// times J).  Row r >= 1: x with site r-1 flipped, mel -h.
// ---------------------------------------------------------------------------
__global__ void ising_xp_kernel(const int8_t* __restrict__ x, int64_t B, int N, int K,
                                int8_t* __restrict__ xp) {
  const int64_t total = B * (int64_t)K * N;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int i = (int)(idx % N);
    const int64_t br = idx / N;
    const int r = (int)(br % K);
    const int64_t b = br / K;
    const int8_t v = x[b * N + i];
    xp[idx] = (r >= 1 && i == r - 1) ? (int8_t)(-v) : v;
  }
}

template <class T>
__global__ void ising_mel_kernel(const int8_t* __restrict__ x, int64_t B, int N, int K,
                                 const int32_t* __restrict__ edges, int E, T h, T J,
                                 T* __restrict__ mels) {
  for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < B;
       b += (int64_t)gridDim.x * blockDim.x) {
    const int8_t* xb = x + b * N;
    int s = 0;
    for (int e = 0; e < E; ++e) s += (xb[edges[2 * e]] == xb[edges[2 * e + 1]]) ? 1 : -1;
    T* m = mels + b * K;
    m[0] = J * (T)s;
    for (int r = 1; r < K; ++r) m[r] = -h;
  }
}

// ---------------------------------------------------------------------------
// Local operators.  One wavefront per sample.
//
// Entry order of the reference (before compaction): [diagonal if the operator
// has a nonzero diagonal], then for each term (grouped by acting size, which
// the host already did) the off-diagonal elements of the row selected by x.
// Compaction keeps entries with |mel| > mel_cutoff in order and pads with
// (x, 0) up to max_conn_size (jax.py:189-199).  Every stored off-diagonal
// element already satisfies |mel| > cutoff, so only the diagonal can drop.
// ---------------------------------------------------------------------------
template <class T>
__device__ inline int term_row(const int8_t* xs, const int32_t* sites, int ns) {
  int r = 0;
  for (int k = 0; k < ns; ++k) r = 2 * r + (xs[sites[k]] < 0 ? 1 : 0);
  return r;
}

template <class T>
__global__ void localop_conn_kernel(const int8_t* __restrict__ x, int64_t B, int N,
                                    nka_localop op, int8_t* __restrict__ xp,
                                    T* __restrict__ mels, int32_t* __restrict__ n_conn_out) {
  extern __shared__ unsigned char smem[];
  const int wid = threadIdx.x / NKA_WAVE;
  const int lane = lane_id();
  const int waves = blockDim.x / NKA_WAVE;
  const int K = op.max_conn_size;
  // per-wave LDS: x (N bytes, padded to 16), entry table (K ints)
  const int xbytes = (N + 15) & ~15;
  unsigned char* base = smem + (size_t)wid * (xbytes + 4 * (size_t)K);
  int8_t* xs = (int8_t*)base;
  int32_t* entry = (int32_t*)(base + xbytes);  // encoded (term, k) or -1 = diag

  const int32_t* op_sites = op.op_sites;
  const T* row_diag = (const T*)op.row_diag;
  const T* conn_mel = (const T*)op.conn_mel;

  for (int64_t b = (int64_t)blockIdx.x * waves + wid; b < B; b += (int64_t)gridDim.x * waves) {
    for (int i = lane; i < N; i += NKA_WAVE) xs[i] = x[b * N + i];
    wave_lds_sync();

    // diagonal: constant + (sum over groups of the in-order sum of the group's
    // terms), jax.py:117-122
    int count = 0;
    if (lane == 0) {
      double d = 0.0, gsum = 0.0;
      int gsize = op.n_ops > 0 ? op.op_nsites[0] : 0;
      for (int t = 0; t < op.n_ops; ++t) {
        if (op.op_nsites[t] != gsize) {
          d += gsum;
          gsum = 0.0;
          gsize = op.op_nsites[t];
        }
        const int r = term_row<T>(xs, op_sites + 4 * t, op.op_nsites[t]);
        gsum += (double)row_diag[op.op_row_off[t] + r];
      }
      d += gsum;
      const T diag = (T)(op.constant + d);
      int e = 0;
      if (op.nonzero_diagonal && fabs((double)diag) > op.mel_cutoff) {
        entry[e++] = -1;
        mels[b * K] = diag;
      }
      // off-diagonal entries in term order
      for (int t = 0; t < op.n_ops; ++t) {
        const int r = term_row<T>(xs, op_sites + 4 * t, op.op_nsites[t]);
        const int row = op.op_row_off[t] + r;
        const int nc = op.row_nconn[row];
        const int off = op.row_conn_off[row];
        for (int k = 0; k < nc && e < K; ++k) {
          entry[e] = off + k;
          mels[b * K + e] = conn_mel[off + k];
          ++e;
        }
      }
      for (int p = e; p < K; ++p) {
        entry[p] = -2;
        mels[b * K + p] = (T)0;
      }
      if (n_conn_out) n_conn_out[b] = e;
      count = e;
    }
    count = __shfl(count, 0, NKA_WAVE);
    wave_lds_sync();

    // rows: x with the sites of the selected term set to the column's states
    for (int e = 0; e < K; ++e) {
      const int code = entry[e];
      int8_t* row = xp + (b * K + e) * (int64_t)N;
      int t = -1, newidx = 0, ns = 0;
      int s0 = -1, s1 = -1, s2 = -1, s3 = -1;
      if (code >= 0) {
        // find the term owning conn index `code` (binary search on row_conn_off is
        // avoided: the host stores the owning term's sites in op_sites via conn2term)
        t = op.conn_term[code];
        newidx = op.conn_newidx[code];
        ns = op.op_nsites[t];
        s0 = op_sites[4 * t + 0];
        s1 = op_sites[4 * t + 1];
        s2 = op_sites[4 * t + 2];
        s3 = op_sites[4 * t + 3];
      }
      for (int i = lane; i < N; i += NKA_WAVE) {
        int8_t v = xs[i];
        if (code >= 0) {
          int k = -1;
          if (i == s0) k = 0;
          else if (i == s1) k = 1;
          else if (i == s2) k = 2;
          else if (i == s3) k = 3;
          if (k >= 0 && k < ns) {
            const int li = (newidx >> (ns - 1 - k)) & 1;
            v = li ? (int8_t)-1 : (int8_t)1;
          }
        }
        row[i] = v;
      }
    }
    (void)count;
    wave_lds_sync();
  }
}

// ---------------------------------------------------------------------------
// The same connected elements as a list, for estimators that update a
// neighbour's amplitude and never need x' itself: mels (B, K) as above, and for
// every nonzero one (its slot counted in *count, in no fixed order of the
// samples) its row b K + k and the at most four sites where x' differs from x,
// ascending, 16 bits each: site | (x'_site > 0) << 15, 0xffff for none.  8
// bytes per element instead of the N of a configuration.  One wavefront per
// sample; the terms of a sample are looked up 64 at a time (16384 samples of the
// 10x10 J1-J2 model, 401 elements each: 0.26 ms; the padded configurations, one
// lane walking the terms, and their compaction took 2.57 ms).
// ---------------------------------------------------------------------------
// Slot of this wavefront's n list entries.
__device__ inline int list_slots(int* __restrict__ count, int n) {
  int at = 0;
  if (lane_id() == 0) at = atomicAdd(count, n);
  return __builtin_amdgcn_readfirstlane(at);
}

template <class T>
__global__ void __launch_bounds__(256) ising_list_kernel(const int8_t* __restrict__ x, int64_t B, int N, int K,
                                                         const int32_t* __restrict__ edges, int E, T h, T J,
                                                         T* __restrict__ mels, int* __restrict__ rows,
                                                         uint64_t* __restrict__ sites, int* __restrict__ count) {
  const int lane = lane_id();
  for (int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); b < B; b += (int64_t)gridDim.x * 4) {
    const int8_t* xb = x + b * N;
    int s = 0;
    for (int e = lane; e < E; e += 64) s += (xb[edges[2 * e]] == xb[edges[2 * e + 1]]) ? 1 : -1;
    s = (int)wave_sum_u32((uint32_t)s);
    const T diag = J * (T)s;
    const int nd = diag != (T)0 ? 1 : 0, nf = K > 1 && -h != (T)0 ? K - 1 : 0;
    const int at = list_slots(count, nd + nf);
    if (lane == 0) {
      mels[b * K] = diag;
      if (nd) {
        rows[at] = (int)(b * K);
        sites[at] = ~0ull;
      }
    }
    for (int r = 1 + lane; r < K; r += 64) {
      mels[b * K + r] = -h;
      if (nf) {
        rows[at + nd + r - 1] = (int)(b * K + r);
        sites[at + nd + r - 1] = (~0ull << 16) | (uint64_t)(r - 1) | (xb[r - 1] > 0 ? 0ull : 0x8000ull);
      }
    }
  }
}

template <class T>
__global__ void __launch_bounds__(256) localop_list_kernel(const int8_t* __restrict__ x, int64_t B, int N,
                                                           nka_localop op, T* __restrict__ mels,
                                                           int* __restrict__ rows, uint64_t* __restrict__ sites,
                                                           int* __restrict__ count) {
  extern __shared__ unsigned char smem[];
  const int lane = lane_id(), K = op.max_conn_size;
  int8_t* xs = (int8_t*)smem + (size_t)(threadIdx.x >> 6) * ((N + 15) & ~15);
  const T* row_diag = (const T*)op.row_diag;
  const T* conn_mel = (const T*)op.conn_mel;
  for (int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); b < B; b += (int64_t)gridDim.x * 4) {
    for (int i = lane; i < N; i += 64) xs[i] = x[b * N + i];
    wave_lds_sync();
    // the diagonal, summed in term order within each group of equal acting
    // size, and the number of off-diagonal elements
    double d = 0.0, gsum = 0.0;
    int gsize = op.n_ops > 0 ? op.op_nsites[0] : 0;
    uint32_t nnz = 0;
    for (int t0 = 0; t0 < op.n_ops; t0 += 64) {
      const int t = t0 + lane;
      double dt = 0.0;
      int ns = 0;
      if (t < op.n_ops) {
        ns = op.op_nsites[t];
        const int row = op.op_row_off[t] + term_row<T>(xs, op.op_sites + 4 * t, ns);
        dt = (double)row_diag[row];
        nnz += (uint32_t)op.row_nconn[row];
      }
      const int cnt = min(64, op.n_ops - t0);
      const int lo = __double2loint(dt), hi = __double2hiint(dt);
      for (int l = 0; l < cnt; ++l) {
        const int sz = __builtin_amdgcn_readlane(ns, l);
        if (sz != gsize) {
          d += gsum;
          gsum = 0.0;
          gsize = sz;
        }
        gsum += __hiloint2double(__builtin_amdgcn_readlane(hi, l), __builtin_amdgcn_readlane(lo, l));
      }
    }
    d += gsum;
    const T diag = (T)(op.constant + d);
    const bool has_diag = op.nonzero_diagonal && fabs((double)diag) > op.mel_cutoff;
    int e = has_diag ? 1 : 0;
    const int total = min(K, e + (int)wave_sum_u32(nnz));
    const int at = list_slots(count, total);
    if (has_diag && lane == 0) {
      mels[b * K] = diag;
      rows[at] = (int)(b * K);
      sites[at] = ~0ull;
    }
    for (int t0 = 0; t0 < op.n_ops; t0 += 64) {
      const int t = t0 + lane;
      int nc = 0, off = 0, ns = 0, r = 0;
      if (t < op.n_ops) {
        ns = op.op_nsites[t];
        r = term_row<T>(xs, op.op_sites + 4 * t, ns);
        nc = op.row_nconn[op.op_row_off[t] + r];
        off = op.row_conn_off[op.op_row_off[t] + r];
      }
      int inc = nc;  // inclusive prefix sum over the lanes
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o);
        if (lane >= o) inc += v;
      }
      for (int k = 0; k < nc; ++k) {
        const int p = e + inc - nc + k;
        if (p >= K) break;
        const int newidx = op.conn_newidx[off + k];
        uint64_t code = ~0ull;
        for (int q = ns - 1; q >= 0; --q) {
          const int was = (r >> (ns - 1 - q)) & 1, now = (newidx >> (ns - 1 - q)) & 1;
          if (was != now) code = (code << 16) | (uint64_t)op.op_sites[4 * t + q] | (now ? 0ull : 0x8000ull);
        }
        mels[b * K + p] = conn_mel[off + k];
        rows[at + p] = (int)(b * K + p);
        sites[at + p] = code;
      }
      e += __shfl(inc, 63);
    }
    for (int p = min(e, K) + lane; p < K; p += 64) mels[b * K + p] = (T)0;
    wave_lds_sync();
  }
}

// The lists of B samples (op_kind and op as for the local-energy entry points;
// op_K elements per sample).  Sites have to fit 15 bits.
int launch_conn_list(int op_kind, const void* op, const int8_t* x, int64_t B, int N, int K, void* mels, int* rows,
                     uint64_t* sites, int* count, hipStream_t s) {
  NKA_CHECK_ARG(N < 32768, "connected elements: more than 32767 sites");
  const unsigned g = (unsigned)std::min<int64_t>((B + 3) / 4, 16384);
  if (op_kind == NKA_OP_ISING) {
    const nka_ising* o = (const nka_ising*)op;
    NKA_CHECK_ARG(K == 1 || K == N + 1, "nka_ising_conn: n_rows must be 1 or N+1");
    NKA_CHECK_ARG(o->n_edges >= 0 && (o->n_edges == 0 || o->edges), "nka_ising_conn: bad edges");
    NKA_CHECK_ARG(o->mel_dtype == NKA_F32 || o->mel_dtype == NKA_F64, "nka_ising_conn: bad dtype");
    if (o->mel_dtype == NKA_F64)
      hipLaunchKernelGGL(ising_list_kernel<double>, dim3(g), dim3(256), 0, s, x, B, N, K, o->edges, o->n_edges, o->h,
                         o->J, (double*)mels, rows, sites, count);
    else
      hipLaunchKernelGGL(ising_list_kernel<float>, dim3(g), dim3(256), 0, s, x, B, N, K, o->edges, o->n_edges,
                         (float)o->h, (float)o->J, (float*)mels, rows, sites, count);
  } else {
    const nka_localop* o = (const nka_localop*)op;
    NKA_CHECK_ARG(o->max_conn_size >= 1, "nka_localop_conn: max_conn_size must be >= 1");
    NKA_CHECK_ARG(o->mel_dtype == NKA_F32 || o->mel_dtype == NKA_F64, "nka_localop_conn: bad dtype");
    const size_t lds = 4 * (size_t)((N + 15) & ~15);
    // (the operators that nka_localop_conn takes, whose LDS holds the elements as well)
    NKA_CHECK_ARG(lds + 16 * (size_t)K <= 64 * 1024, "nka_localop_conn: N or max_conn_size too large");
    if (o->mel_dtype == NKA_F64)
      hipLaunchKernelGGL(localop_list_kernel<double>, dim3(g), dim3(256), lds, s, x, B, N, *o, (double*)mels, rows,
                         sites, count);
    else
      hipLaunchKernelGGL(localop_list_kernel<float>, dim3(g), dim3(256), lds, s, x, B, N, *o, (float*)mels, rows,
                         sites, count);
  }
  NKA_CHECK_LAUNCH("connected elements");
  return NKA_OK;
}

}  // namespace nka

using namespace nka;

extern "C" {

const char* nka_last_error(void) { return nka::last_error(); }

const char* nka_version(void) { return "netket_amd 0.1 (gfx950)"; }

int nka_ising_conn(const int8_t* x, int64_t n_batch, int n_sites, const int32_t* edges,
                   int n_edges, double h, double J, int mel_dtype, int n_rows, int8_t* xp,
                   void* mels, void* stream) {
  NKA_CHECK_ARG(n_batch >= 0 && n_sites > 0, "nka_ising_conn: bad sizes");
  NKA_CHECK_ARG(n_rows == 1 || n_rows == n_sites + 1, "nka_ising_conn: n_rows must be 1 or N+1");
  NKA_CHECK_ARG(n_edges >= 0 && (n_edges == 0 || edges), "nka_ising_conn: bad edges");
  NKA_CHECK_ARG(mel_dtype == NKA_F32 || mel_dtype == NKA_F64, "nka_ising_conn: bad dtype");
  if (n_batch == 0) return NKA_OK;
  hipStream_t s = (hipStream_t)stream;
  const int64_t total = n_batch * (int64_t)n_rows * n_sites;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(ising_xp_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, n_batch,
                     n_sites, n_rows, xp);
  int64_t mb = (n_batch + 255) / 256;
  if (mb > 65536) mb = 65536;
  if (mel_dtype == NKA_F64)
    hipLaunchKernelGGL(ising_mel_kernel<double>, dim3((unsigned)mb), dim3(256), 0, s, x,
                       n_batch, n_sites, n_rows, edges, n_edges, h, J, (double*)mels);
  else
    hipLaunchKernelGGL(ising_mel_kernel<float>, dim3((unsigned)mb), dim3(256), 0, s, x,
                       n_batch, n_sites, n_rows, edges, n_edges, (float)h, (float)J,
                       (float*)mels);
  NKA_CHECK_LAUNCH("nka_ising_conn");
  return NKA_OK;
}

int nka_localop_conn(const int8_t* x, int64_t n_batch, int n_sites, const nka_localop* op,
                     int8_t* xp, void* mels, int32_t* n_conn, void* stream) {
  NKA_CHECK_ARG(op != nullptr, "nka_localop_conn: null operator");
  NKA_CHECK_ARG(n_batch >= 0 && n_sites > 0, "nka_localop_conn: bad sizes");
  NKA_CHECK_ARG(op->max_conn_size >= 1, "nka_localop_conn: max_conn_size must be >= 1");
  NKA_CHECK_ARG(op->mel_dtype == NKA_F32 || op->mel_dtype == NKA_F64,
                "nka_localop_conn: bad dtype");
  if (n_batch == 0) return NKA_OK;
  hipStream_t s = (hipStream_t)stream;
  const int waves = 4;
  const size_t per_wave = (size_t)((n_sites + 15) & ~15) + 4 * (size_t)op->max_conn_size;
  const size_t lds = per_wave * waves;
  NKA_CHECK_ARG(lds <= 64 * 1024, "nka_localop_conn: N or max_conn_size too large (%zu B LDS)",
                lds);
  int64_t blocks = (n_batch + waves - 1) / waves;
  if (blocks > 16384) blocks = 16384;
  if (op->mel_dtype == NKA_F64)
    hipLaunchKernelGGL(localop_conn_kernel<double>, dim3((unsigned)blocks), dim3(64 * waves), lds,
                       s, x, n_batch, n_sites, *op, xp, (double*)mels, n_conn);
  else
    hipLaunchKernelGGL(localop_conn_kernel<float>, dim3((unsigned)blocks), dim3(64 * waves), lds,
                       s, x, n_batch, n_sites, *op, xp, (float*)mels, n_conn);
  NKA_CHECK_LAUNCH("nka_localop_conn");
  return NKA_OK;
}

}  // extern "C"
