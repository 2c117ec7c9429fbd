// isph_persist.h -- the FP64 BiCGStab of isph_solver.h as one resident launch:
// every workgroup owns consecutive row blocks for a whole run of iterations
// and the workgroups meet at grid-wide reductions instead of kernel
// boundaries.
//
// What bounds the launch-per-phase form is not the rows but the seven
// dependent launches of an iteration: at 7,485 rows an iteration took 39 us,
// of which the two products' data need less than 2 us.  Here an iteration
// has three grid-wide reductions of ~2 us each.
//
// Rows and sums.  A workgroup of T threads holds up to R rows per thread: the
// row blocks (256 rows) b0 .. b0 + nbw - 1, thread t row t & 255 of blocks
// (t >> 8) + q T / 256.  r, p, t1, s, t2 of its rows stay in registers.  Sums
// follow the fixed trees of block_tree and final_tree2 over the same 256-row
// blocks, so every scalar and every iterate has the bits of the
// launch-per-phase form.
//
// Vectors at other workgroups' rows.  k_ps_setup lists, per workgroup, the
// 64-row chunks that its rows' columns fall into (its window: its own rows
// and a strip on each side, since rows are sorted by cell) and rewrites each
// column as a 16-bit position in that window.  The products gather from the
// window in LDS.  A workgroup's threads keep r, t1 and p of the window's
// elements in registers: r and t1 are read after the reduction that follows
// their production, and p = r + beta (p - omega t1) is formed for the window
// by the same expression as at its owner, so p is never exchanged.  Rows
// whose window does not fit (wlist's capacity) leave the flag set and the
// solve runs launch by launch.
//
// Visibility between workgroups.  Exchanged data (r, t1, the partial sums)
// is written and read with relaxed agent-scope atomics, which write through
// and read past the per-XCD caches; every wave waits for its stores
// (s_waitcnt) before the workgroup's barrier, after which one lane publishes
// the block's partial sums.  A published word carries 32 bits of the value
// and the reduction's number, so a reader polls the data itself: there is no
// counter and no fence (an agent-scope release writes the XCD's L2 back:
// 8.3 us per barrier of 256 workgroups against 2.4 us for this one).  Two
// sets of words alternate: a set is written again only after the reduction
// between has completed, which every reader of it has passed.
//
// Progress.  The launch is cooperative (all workgroups resident); every wait
// is bounded (PS_SPIN polls) and a wait that ends without its data makes the
// launch return with the abort flag set.
#pragma once
#include <type_traits>

#include "isph_device.h"

#define PS_CHUNK 64                 // rows per window chunk
#define PS_MAX_CHUNKS 16384         // chunks of the largest system (2^20 rows)
#define PS_SPIN (1 << 20)           // polls of one wait: about a second

// DevScalars::counter slots of the resident solve
#define PS_FLAG_WIN 0               // a window exceeds its capacity
#define PS_FLAG_ABORT 1             // a wait ran out

struct PersArg {
  unsigned long long* slots;  // two sets of 4 words per row block, 8 per workgroup
  uint32_t* lidx;             // window positions, slots 2w and 2w+1 of row i at [w * cap + i]
  int32_t* wlist;             // per workgroup: its chunks, ascending (wcap entries)
  int32_t* wcnt;              // per workgroup: their count
  int wcap;                   // window capacity in chunks
  int nbw;                    // row blocks per workgroup
};

template <typename V>
__device__ __forceinline__ void st_agent(V* p, V v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ V ld_agent(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Windows of the workgroups' rows (one workgroup each, as the solve), the
// rows' columns as window positions, and the slots cleared.
template <int T>
__global__ void __launch_bounds__(T) k_ps_setup(Dev D, PersArg Q) {
  __shared__ uint16_t map[PS_MAX_CHUNKS];
  __shared__ int cnt[T];
  const int t = threadIdx.x, wg = blockIdx.x, n = D.sc->n, cap = D.cap;
  const int nch = (n + PS_CHUNK - 1) / PS_CHUNK;
  const int i0 = wg * Q.nbw * RED_BLOCK;
  const int i1 = min(n, min(D.nblk, (wg + 1) * Q.nbw) * RED_BLOCK);
  for (int b = wg * Q.nbw + t; b < min(D.nblk, (wg + 1) * Q.nbw); b += T)
    for (int q = 0; q < 4; q++) {
      Q.slots[4 * (size_t)b + q] = 0;
      Q.slots[4 * ((size_t)D.nblk + b) + q] = 0;
    }
  if (t < 8) Q.slots[8 * ((size_t)D.nblk + wg) + t] = 0;
  for (int c = t; c < nch; c += T) map[c] = 0;
  __syncthreads();
  for (int i = i0 + t; i < i1; i += T) {
    const int L = D.alen[i];
    for (int k0 = 0; k0 < L; k0 += 8) {
      int c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = D.acol[((k0 + u < L) ? k0 + u : k0) * cap + i];
#pragma unroll
      for (int u = 0; u < 8; u++) map[c[u] / PS_CHUNK] = 1;  // every writer stores 1
    }
  }
  __syncthreads();
  // positions of the marked chunks in ascending order: thread t counts a
  // run of consecutive chunks, then the runs are scanned
  const int per = (nch + T - 1) / T, c0 = t * per, c1 = min(nch, c0 + per);
  int own = 0;
  for (int c = c0; c < c1; c++) own += map[c];
  cnt[t] = own;
  __syncthreads();
  for (int off = 1; off < T; off <<= 1) {
    const int a = (t >= off) ? cnt[t - off] : 0;
    __syncthreads();
    cnt[t] += a;
    __syncthreads();
  }
  const int total = cnt[T - 1];
  if (total > Q.wcap) {  // the whole workgroup
    if (t == 0) {
      atomicOr(&D.sc->counter[PS_FLAG_WIN], 1u);
      Q.wcnt[wg] = 0;
    }
    return;
  }
  int pos = cnt[t] - own;
  for (int c = c0; c < c1; c++)
    if (map[c]) {
      Q.wlist[(size_t)wg * Q.wcap + pos] = c;
      map[c] = (uint16_t)pos++;
    }
  if (t == 0) Q.wcnt[wg] = total;
  __syncthreads();
  for (int i = i0 + t; i < i1; i += T) {
    const int L = D.alen[i];
    for (int k0 = 0; k0 < L; k0 += 8) {
      int c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = D.acol[((k0 + u < L) ? k0 + u : k0) * cap + i];
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        if (k0 + u >= L) break;
        const uint32_t a = map[c[u] / PS_CHUNK] * PS_CHUNK + c[u] % PS_CHUNK;
        const uint32_t b = map[c[u + 1] / PS_CHUNK] * PS_CHUNK + c[u + 1] % PS_CHUNK;
        Q.lidx[((k0 + u) >> 1) * cap + i] = a | (b << 16);
      }
    }
  }
}

__device__ __forceinline__ double lane0(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)b);
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// LDS of the resident solve in doubles: the window, then an area shared by
// the block trees and the gathered partials, then the column sums, then (R >
// 1) p and t1 of the workgroup's rows
template <int T, int R>
__host__ __device__ constexpr int ps_tree_doubles() { return 2 * R * (T / 256) * 192; }
template <int T, int R, int W>
__host__ __device__ inline int64_t ps_lds_bytes(int nblk) {
  const int64_t a = ps_tree_doubles<T, R>(), b = 2 * (int64_t)nblk;
  return 8 * ((int64_t)W * T + (a > b ? a : b) + 2 * 256 + 2 + (R > 1 ? 2 * R * T : 0)) + 16;
}

// One word of reduction ep, polled until it carries the number; false when
// the wait ran out
__device__ __forceinline__ bool ps_wait(const unsigned long long* p, unsigned ep, uint32_t& lo) {
  for (int spin = 0; spin < PS_SPIN; spin++) {
    const unsigned long long w = ld_agent(p);
    lo = (uint32_t)w;
    if ((unsigned)(w >> 32) == ep) return true;
  }
  return false;
}
// The payloads of `words` consecutive words of reduction ep into out: a
// double is two words, low half first, so out is the doubles' array.  The
// workgroup reads each word once, 64 consecutive ones per wavefront (four
// cache lines), several in flight per thread.
template <int T>
__device__ __forceinline__ bool ps_collect(const unsigned long long* set, int words, unsigned ep,
                                           uint32_t* out) {
  constexpr int G = 4;
  for (int w0 = threadIdx.x; w0 < words; w0 += G * T) {
    uint32_t lo[G];
    unsigned long long w[G];
    bool all = false;
#pragma unroll
    for (int u = 0; u < G; u++) w[u] = ld_agent(&set[min(w0 + u * T, words - 1)]);
    all = true;
#pragma unroll
    for (int u = 0; u < G; u++) {
      lo[u] = (uint32_t)w[u];
      if ((unsigned)(w[u] >> 32) != ep)
        all = ps_wait(&set[min(w0 + u * T, words - 1)], ep, lo[u]) && all;
    }
    if (!all) return false;
#pragma unroll
    for (int u = 0; u < G; u++)
      if (w0 + u * T < words) out[w0 + u * T] = lo[u];
  }
  return true;
}
__device__ __forceinline__ void ps_publish(unsigned long long* p, unsigned ep, double v) {
  const unsigned long long tag = (unsigned long long)ep << 32;
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  st_agent(p, (b & 0xffffffffull) | tag);
  st_agent(p + 1, (b >> 32) | tag);
}

// Grid-wide sums of NV values per row in the order of block_tree and
// final_tree2.  Every vector store of the caller's before this call is
// visible to every workgroup after it.  Returns false when a wait ran out.
//
// Up to 256 row blocks (one per workgroup, T = 256) every workgroup collects
// all partials itself: one exchange.  With more, the readers' requests for
// the same lines would take longer than a second exchange (24 us against 4 at
// 809 blocks): workgroup 0 collects the partials and sends the sums to a line
// of each workgroup's own.
template <int T, int R, int NV>
__device__ __forceinline__ bool ps_reduce(const PersArg& Q, int nblk, int b0, unsigned ep,
                                          const double (&v)[NV][R], double* area, double* col,
                                          int* bad, double (&out)[NV]) {
  constexpr int S = T / 256;
  const int t = threadIdx.x, wv = (t >> 6) & 3, l = t & 63, sub = t >> 8;
  if (wv) {
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
      for (int q = 0; q < R; q++)
        area[((k * R + q) * S + sub) * 192 + (wv - 1) * 64 + l] = v[k][q];
  }
  __syncthreads();
  double s[NV][R];
  if (wv == 0) {
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const double* a = area + ((k * R + q) * S + sub) * 192;
        s[k][q] = wave_tree((v[k][q] + a[64 + l]) + (a[l] + a[128 + l]));
      }
  }
  __builtin_amdgcn_s_waitcnt(0);  // this wave's vector stores have completed
  __syncthreads();                // ... and every wave's; the trees are read
  // two sets of slots of 4 words per block, used with NV doubles each
  unsigned long long* set = Q.slots + (size_t)(ep & 1) * 4 * nblk;
  if (wv == 0 && l == 0) {
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int lb = q * S + sub;
      if (lb < Q.nbw && b0 + lb < nblk) {
#pragma unroll
        for (int k = 0; k < NV; k++)
          ps_publish(&set[2 * (size_t)(NV * (b0 + lb) + k)], ep, s[k][q]);
      }
    }
  }
  if (T == 256) {
    if (!ps_collect<T>(set, 2 * NV * nblk, ep, reinterpret_cast<uint32_t*>(col))) *bad = 1;
    __syncthreads();
    // every wavefront sums for itself: lane l holds columns l, l + 64, ...
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double c[4];
#pragma unroll
      for (int u = 0; u < 4; u++)
        c[u] = (l + 64 * u < nblk) ? 0.0 + col[NV * (l + 64 * u) + k] : 0.0;
      out[k] = lane0(wave_tree((c[0] + c[2]) + (c[1] + c[3])));
    }
    return !*bad;
  }
  unsigned long long* mail = Q.slots + (size_t)8 * nblk;  // 8 words per workgroup
  double* res = col + 512;
  if (blockIdx.x == 0) {
    if (!ps_collect<T>(set, 2 * NV * nblk, ep, reinterpret_cast<uint32_t*>(area))) *bad = 1;
    __syncthreads();
    if (t < 256) {
#pragma unroll
      for (int k = 0; k < NV; k++) {
        double a = 0.0;
        for (int b = t; b < nblk; b += 256) a = a + area[NV * b + k];
        col[k * 256 + t] = a;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const double* c = col + k * 256;
      out[k] = lane0(wave_tree((c[l] + c[l + 128]) + (c[l + 64] + c[l + 192])));
    }
    if (*bad) return false;  // nothing is sent: the other workgroups' waits run out too
    for (int g = t; g < (int)gridDim.x; g += T) {
#pragma unroll
      for (int k = 0; k < NV; k++) ps_publish(&mail[8 * (size_t)g + 2 * k], ep, out[k]);
    }
    return true;
  }
  if (t < 2 * NV) {
    uint32_t lo;
    if (!ps_wait(&mail[8 * (size_t)blockIdx.x + t], ep, lo)) *bad = 1;
    reinterpret_cast<uint32_t*>(res)[t] = lo;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) out[k] = res[k];
  return !*bad;
}

// Element i of an array through its uniform base and a 32-bit byte offset,
// so that every array shares one offset register
template <typename V>
__device__ __forceinline__ V* ps_at(V* base, unsigned i) {
  typedef typename std::conditional<std::is_const<V>::value, const char, char>::type Byte;
  return reinterpret_cast<V*>(reinterpret_cast<Byte*>(base) + (i * (unsigned)sizeof(V)));
}

// A thread's first KR row entries, held in registers for the whole launch
// (KR 0: none); ps_row reads the rest from memory
template <int KR>
struct PsRow {
  double v[KR ? KR : 1];
  uint32_t w[KR ? KR / 2 : 1];
};

// Eight entries k0.. of row i: their positions and values (those below the
// wavefront's longest row Lm; FULL: all eight are), gathers and products
template <bool FULL>
__device__ __forceinline__ double ps_row8(const uint32_t* ip, const double* vp, int cap,
                                          unsigned i, int k0, int L, int Lm, const double* win,
                                          double acc) {
  uint32_t w[4];
  double v[8], g[8];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = 0u;
    if (FULL || k0 + 2 * q < Lm) w[q] = *ps_at(ip + (size_t)q * cap, i);
  }
#pragma unroll
  for (int u = 0; u < 8; u++) {
    v[u] = 0.0;
    if (FULL || k0 + u < Lm) v[u] = *ps_at(vp + (size_t)u * cap, i);
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = (k0 + 2 * q < L) ? w[q] : 0u;  // a shorter row's slots hold no position
    g[2 * q] = win[w[q] & 0xffffu];
    g[2 * q + 1] = win[w[q] >> 16];
  }
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const double a = acc + v[u] * g[u];
    acc = (k0 + u < L) ? a : acc;
  }
  return acc;
}

// y_i = sum_k A_ik win[pos(k)] in row order (the order of ell_row_sum).  The
// loop runs to the wavefront's longest row (Lm, uniform), so the slots' bases
// are scalars.
template <int KR>
__device__ __forceinline__ double ps_row(const PsRow<KR>& M, const uint32_t* idx,
                                         const double* val, int cap, unsigned i, int L, int Lm,
                                         const double* win) {
  double acc = 0.0;
#pragma unroll
  for (int k0 = 0; k0 < KR; k0 += 8) {
    if (k0 >= Lm) break;
    double g[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const uint32_t w = M.w[(k0 + u) / 2];
      g[u] = win[(u & 1) ? (w >> 16) : (w & 0xffffu)];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const double a = acc + M.v[k0 + u] * g[u];
      acc = (k0 + u < L) ? a : acc;
    }
  }
  const uint32_t* ip = idx + (size_t)(KR / 2) * cap;
  const double* vp = val + (size_t)KR * cap;
  int k0 = KR;
#pragma unroll 1
  for (; k0 + 8 <= Lm; k0 += 8) {
    acc = ps_row8<true>(ip, vp, cap, i, k0, L, Lm, win, acc);
    ip += (size_t)4 * cap;
    vp += (size_t)8 * cap;
  }
  if (k0 < Lm) acc = ps_row8<false>(ip, vp, cap, i, k0, L, Lm, win, acc);
  return acc;
}
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) v = max(v, __shfl_xor(v, s, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// up to `iters` BiCGStab iterations from the state in D.sol, D.r, D.rh, D.pp
// and the scalars (k_bicg_init or a previous launch); leaves the state there
template <int T, int R, int W, int KR>
__global__ void __launch_bounds__(T) k_bicg_resident(Dev D, PersArg Q, int iters, unsigned ep) {
  constexpr int S = T / 256;
  // With several rows per thread the 128 registers of a 1024-thread
  // workgroup do not hold every vector: p and t1 of the rows sit in LDS
  // slots of their thread, r, rh and x are read from memory where used (by
  // their own thread only; r past the caches, as it is exchanged).
  constexpr bool XREG = R == 1;
  extern __shared__ double ps_lds[];
  const int t = threadIdx.x, sub = t >> 8, wg = blockIdx.x;
  DevScalars* Sc = D.sc;
  const int n = Sc->n, nblk = D.nblk, cap = D.cap, b0 = wg * Q.nbw;
  const int ta = ps_tree_doubles<T, R>();
  double* win = ps_lds;
  double* area = win + W * T;
  double* col = area + (ta > 2 * nblk ? ta : 2 * nblk);
  double* lp = col + 514;
  double* lt = lp + R * T;
  int* bad = reinterpret_cast<int*>(XREG ? lp : lt + R * T);
  if (t == 0) *bad = 0;
  double rho = Sc->rho;
  const double bnorm = Sc->bnorm, tol = D.P.tol;
  const int max_iter = D.P.max_iter;
  int it = Sc->iters;
  int row[R], len[R], lmx[R];
  double r[R], rh[R], pv[R], x[R], tv[R];
  PsRow<KR> M[R];
  auto P = [&](int q) -> double& {
    if constexpr (XREG) return pv[q];
    else return lp[q * T + t];
  };
  auto T1 = [&](int q) -> double& {
    if constexpr (XREG) return tv[q];
    else return lt[q * T + t];
  };
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int lb = q * S + sub, i = (b0 + lb) * RED_BLOCK + (t & 255);
    const bool in = lb < Q.nbw && i < n;
    row[q] = in ? i : -1;
    len[q] = in ? D.alen[i] : 0;
    lmx[q] = wave_max(len[q]);
    r[q] = (in && XREG) ? D.r[i] : 0.0;
    rh[q] = (in && XREG) ? D.rh[i] : 0.0;
    x[q] = (in && XREG) ? D.sol[i] : 0.0;
    P(q) = in ? D.pp[i] : 0.0;
#pragma unroll
    for (int k = 0; k < KR; k++) {
      M[q].v[k] = (k < len[q]) ? D.aval[k * cap + i] : 0.0;
      if (k % 2 == 0) M[q].w[k / 2] = (k < len[q]) ? Q.lidx[(k / 2) * cap + i] : 0u;
    }
  }
  // the window's elements of this thread: element e = w T + t is row
  // 64 c + (t & 63) with c the chunk of its wavefront (-1: none)
  const int wn = Q.wcnt[wg], l = t & 63;
  int wc[W];
  double rw[W], pw[W], tw[W];
#pragma unroll
  for (int w = 0; w < W; w++) {
    const int s = w * (T / PS_CHUNK) + t / PS_CHUNK;
    wc[w] = __builtin_amdgcn_readfirstlane((s < wn) ? Q.wlist[(size_t)wg * Q.wcap + s] : -1);
    const int g = wc[w] * PS_CHUNK + l;
    const bool in = wc[w] >= 0 && g < n;
    rw[w] = in ? D.r[g] : 0.0;
    pw[w] = in ? D.pp[g] : 0.0;
  }
  __syncthreads();
  int conv = 0, brk = 0, done = 0;
  double alpha = 0.0, omega = 0.0, beta = 0.0, rr = 0.0, rel = 0.0;
  bool ok = true;
  for (int k = 0; k < iters; k++) {
    // (the row numbers are opaque to the compiler here, or it would hold
    // every array's address of every row in registers across iterations)
#pragma unroll
    for (int q = 0; q < R; q++) asm volatile("" : "+v"(row[q]));
    // t1 = A p ; alpha = rho / (t1 . rh)
#pragma unroll
    for (int w = 0; w < W; w++) win[w * T + t] = pw[w];
    __syncthreads();
    double v1[1][R], o1[1];
#pragma unroll
    for (int q = 0; q < R; q++) {
      __builtin_amdgcn_sched_barrier(0);  // one row's loads in registers at a time
      if (!XREG) rh[q] = (row[q] >= 0) ? *ps_at(D.rh, row[q]) : 0.0;
      double t1 = 0.0;
      if (row[q] >= 0) {
        t1 = ps_row<KR>(M[q], Q.lidx, D.aval, cap, row[q], len[q], lmx[q], win);
        st_agent(ps_at(D.t1, row[q]), t1);
      }
      T1(q) = t1;
      v1[0][q] = (row[q] >= 0) ? t1 * rh[q] : 0.0;
    }
    ok = ps_reduce<T, R, 1>(Q, nblk, b0, ep++, v1, area, col, bad, o1);
    if (!ok) break;
    // s = r - alpha t1 ; t2 = A s ; omega = (t2 . s) / (t2 . t2)
#pragma unroll
    for (int w = 0; w < W; w++) {
      // uniform base of the chunk, one lane offset
      const double* c = D.t1 + (int64_t)wc[w] * PS_CHUNK;
      tw[w] = (wc[w] >= 0 && l < n - wc[w] * PS_CHUNK) ? ld_agent(c + (unsigned)l) : 0.0;
    }
    alpha = rho / o1[0];
#pragma unroll
    for (int w = 0; w < W; w++) win[w * T + t] = rw[w] - alpha * tw[w];
    __syncthreads();
    double s[R], t2[R], v2[2][R], o2[2];
#pragma unroll
    for (int q = 0; q < R; q++) {
      __builtin_amdgcn_sched_barrier(0);
      if (!XREG) r[q] = (row[q] >= 0) ? ld_agent(ps_at(D.r, row[q])) : 0.0;
      t2[q] = (row[q] >= 0) ? ps_row<KR>(M[q], Q.lidx, D.aval, cap, row[q], len[q], lmx[q], win) : 0.0;
      s[q] = r[q] - alpha * T1(q);
      v2[0][q] = (row[q] >= 0) ? t2[q] * s[q] : 0.0;
      v2[1][q] = (row[q] >= 0) ? t2[q] * t2[q] : 0.0;
    }
    ok = ps_reduce<T, R, 2>(Q, nblk, b0, ep++, v2, area, col, bad, o2);
    if (!ok) break;
    omega = o2[0] / o2[1];
    // x = (x + alpha p) + omega s ; r = s - omega t2 ; rho' = r . rh ; rr = r . r
#pragma unroll
    for (int q = 0; q < R; q++) {
      if (!XREG) {
        rh[q] = (row[q] >= 0) ? *ps_at(D.rh, row[q]) : 0.0;
        x[q] = (row[q] >= 0) ? *ps_at(D.sol, row[q]) : 0.0;
      }
      x[q] = (x[q] + alpha * P(q)) + omega * s[q];
      r[q] = s[q] - omega * t2[q];
      if (row[q] >= 0) {
        st_agent(ps_at(D.r, row[q]), r[q]);
        if (!XREG) *ps_at(D.sol, row[q]) = x[q];
      }
      v2[0][q] = (row[q] >= 0) ? r[q] * rh[q] : 0.0;
      v2[1][q] = (row[q] >= 0) ? r[q] * r[q] : 0.0;
      P(q) = P(q) - omega * T1(q);
    }
#pragma unroll
    for (int w = 0; w < W; w++) pw[w] = pw[w] - omega * tw[w];
    ok = ps_reduce<T, R, 2>(Q, nblk, b0, ep++, v2, area, col, bad, o2);
    if (!ok) break;
    // FIN_BETA
    it++;
    const double rhon = o2[0];
    rr = o2[1];
    rel = sqrt(rr) / bnorm;
    if (sqrt(rr) <= tol * bnorm) {
      conv = 1;
      done = 1;
    } else if (!(isfinite(alpha) && isfinite(omega)) || omega == 0.0 || rhon == 0.0 ||
               !isfinite(rhon)) {
      brk = 1;
      done = 1;
    } else {
      beta = (rhon / rho) * (alpha / omega);
      rho = rhon;
      if (it >= max_iter) done = 1;
    }
    if (done) break;
    // p = r + beta (p - omega t1), here and over the window
#pragma unroll
    for (int w = 0; w < W; w++) {
      // uniform base of the chunk, one lane offset
      const double* c = D.r + (int64_t)wc[w] * PS_CHUNK;
      rw[w] = (wc[w] >= 0 && l < n - wc[w] * PS_CHUNK) ? ld_agent(c + (unsigned)l) : 0.0;
    }
#pragma unroll
    for (int w = 0; w < W; w++) pw[w] = rw[w] + beta * pw[w];
#pragma unroll
    for (int q = 0; q < R; q++) P(q) = r[q] + beta * P(q);
  }
#pragma unroll
  for (int q = 0; q < R; q++)
    if (row[q] >= 0) {
      if (XREG) *ps_at(D.sol, row[q]) = x[q];
      *ps_at(D.pp, row[q]) = P(q);
    }
  if (t == 0 && !ok) atomicOr(&Sc->counter[PS_FLAG_ABORT], 1u);
  if (wg == 0 && t == 0 && ok) {
    Sc->rho = rho;
    Sc->alpha = alpha;
    Sc->omega = omega;
    Sc->beta = beta;
    Sc->rr = rr;
    Sc->rel = rel;
    Sc->iters = it;
    Sc->conv = conv;
    Sc->brk = brk;
    Sc->done = done;
  }
}
