// isph_persist.h -- the FP64 BiCGStab of isph_solver.h as one resident launch:
// every workgroup owns consecutive row blocks for a whole run of iterations
// and the workgroups meet at grid-wide reductions instead of kernel
// boundaries.
//
// What bounds the launch-per-phase form is not the rows but the seven
// dependent launches of an iteration: at 7,485 rows an iteration took 39 us,
// of which the two products' data need less than 2 us.  Here an iteration
// has three grid-wide reductions of ~2 us each and takes 9.7 us; at 22k rows
// 12.0 (40 before), at 95k 14.8 (42), at 207k 20.9 (50.7), at 653k, where the
// products' streaming is most of it, 59.0 (93.5).
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
// window in LDS.  With one row per thread a workgroup's threads keep r, t1 and p
// of the window's elements in registers: t1 and r of other workgroups' rows are
// read while the reduction after their production is under way, and
// p = r + beta (p - omega t1) is formed for the window by the same expression
// as at its owner, so p is not exchanged.  With several rows per thread those
// registers hold the rows' own vectors, and p and s themselves are exchanged.
//
// What fits.  The columns of a workgroup's rows lie in the cell columns on either
// side, not further up or down than its own rows and a cell more.  Up to seven
// row blocks per workgroup (~458k rows) that fits the window however high the
// cell columns; beyond, they may have some (6,144 - own rows) / 2 - 250 rows:
// basins 360 particles deep fit and 380 do not at eight blocks, 320 and 340 at
// ten, 270 and 280 at twelve.  Other systems (wlist's capacity) leave a flag set,
// and the solve runs launch by launch.
//
// Visibility between workgroups.  Exchanged values (r, t1, the partial sums)
// are doubles in two 64-bit words, each with 32 bits of the value and the
// number of the reduction it belongs to, written and read with relaxed
// agent-scope atomics, which write through and read past the per-XCD caches.
// A reader polls the data itself, so there is no counter, no wait for stores
// and no fence (an agent-scope release writes the XCD's L2 back: 8.3 us per
// barrier of 256 workgroups against 2.4 us for an exchange of words).  A word
// is written again only after a reduction that its readers took part in after
// their reads; the partial sums, read within one, alternate between two sets.
//
// Progress.  The launch is cooperative (all workgroups resident); every wait
// is bounded (PS_SPIN polls) and a wait that ends without its data makes the
// launch return with the abort flag set.  Other work that keeps CUs of the
// device busy for that long does so; the host then solves the system again from
// its start, launch by launch (what the others computed meanwhile may hang on
// values that never came).  k_ps_setup keeps the start for that.
#pragma once
#include <type_traits>

#include "isph_device.h"

#define PS_CHUNK 64                 // rows per window chunk
#define PS_MAX_CHUNKS 16384         // chunks of the largest system (2^20 rows)
#define PS_SPIN (1 << 20)           // polls of one wait: some tenths of a second

// DevScalars::counter slots of the resident solve
#define PS_FLAG_WIN 0               // a window exceeds its capacity
#define PS_FLAG_ABORT 1             // a wait ran out

struct PersArg {
  unsigned long long* slots;  // two sets of 4 words per row block, 8 per workgroup
  // the words of t1 and r (several rows per thread: of s and p), one array
  // per half
  unsigned long long *tlo, *thi, *rlo, *rhi;
  uint32_t* lidx;             // window positions, slots 2w and 2w+1 of row i at [w * ls + i]
  int ls;                     // leading dimension of lidx
  int32_t* wlist;             // per workgroup: its chunks, ascending (wcap entries)
  int32_t* wcnt;              // per workgroup: their count, and the slot of its own first chunk
  int wcap;                   // window capacity in chunks
  int nbw;                    // row blocks per workgroup
  int ended;                  // workgroups whose waits count as run out (0 but in a test)
  double* x0;                 // the solution vector at the start
};

template <typename V>
__device__ __forceinline__ void st_agent(V* p, V v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ V ld_agent(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Element i of an array through its uniform base and a 32-bit byte offset,
// so that every array shares one offset register
template <typename V>
__device__ __forceinline__ V* ps_at(V* base, unsigned i) {
  typedef typename std::conditional<std::is_const<V>::value, const char, char>::type Byte;
  return reinterpret_cast<V*>(reinterpret_cast<Byte*>(base) + (i * (unsigned)sizeof(V)));
}

// An exchanged word polled in a loop: the index is opaque, so the loop holds
// one offset per word and not a 64-bit address
__device__ __forceinline__ unsigned long long ld_word(const unsigned long long* base, unsigned i) {
  asm volatile("" : "+v"(i));
  return ld_agent(ps_at(base, i));
}

// ---- the window of the rows i0 .. i1 - 1 of a workgroup of T threads ----
// Its 64-row chunks: those that the rows are in and those that their columns fall
// into.  map (nch entries) gets 1 for each, cnt the prefix sums of the threads'
// shares of them; `own` is this thread's share.  Returns their number.
template <int T>
__device__ __forceinline__ int ps_window_chunks(const int32_t* acol, const int32_t* alen, int cap,
                                                int i0, int i1, int nch, uint16_t* map, int* cnt,
                                                int& own) {
  const int t = threadIdx.x;
  for (int c = t; c < nch; c += T) map[c] = 0;
  __syncthreads();
  for (int i = i0 + t; i < i1; i += T) {
    const int L = alen[i];
    map[i / PS_CHUNK] = 1;  // its own rows, in order, whatever the columns
    for (int k0 = 0; k0 < L; k0 += 8) {
      int c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = acol[((k0 + u < L) ? k0 + u : k0) * cap + i];
#pragma unroll
      for (int u = 0; u < 8; u++) map[c[u] / PS_CHUNK] = 1;  // every writer stores 1
    }
  }
  __syncthreads();
  // thread t counts a run of consecutive chunks, then the runs are scanned
  const int per = (nch + T - 1) / T, c0 = t * per, c1 = min(nch, c0 + per);
  own = 0;
  for (int c = c0; c < c1; c++) own += map[c];
  cnt[t] = own;
  __syncthreads();
  for (int off = 1; off < T; off <<= 1) {
    const int a = (t >= off) ? cnt[t - off] : 0;
    __syncthreads();
    cnt[t] += a;
    __syncthreads();
  }
  return cnt[T - 1];
}
// The chunks in ascending order (wlist), their count and the slot of the
// workgroup's first own one (wcnt), and in map the slot of each
template <int T>
__device__ __forceinline__ void ps_window_list(int i0, int nch, int own, int total, uint16_t* map,
                                               const int* cnt, int32_t* wlist, int32_t* wcnt) {
  const int t = threadIdx.x;
  const int per = (nch + T - 1) / T, c0 = t * per, c1 = min(nch, c0 + per);
  int pos = cnt[t] - own;
  for (int c = c0; c < c1; c++)
    if (map[c]) {
      wlist[pos] = c;
      if (c == i0 / PS_CHUNK) wcnt[1] = pos;
      map[c] = (uint16_t)pos++;
    }
  if (t == 0) wcnt[0] = total;
}
// The rows' columns as window positions, slots 2w and 2w + 1 of row i in word
// [w * ls + i]; map holds the chunks' slots (after a barrier)
template <int T>
__device__ __forceinline__ void ps_window_positions(const int32_t* acol, const int32_t* alen,
                                                    int cap, int i0, int i1, const uint16_t* map,
                                                    uint32_t* lidx, int ls) {
  for (int i = i0 + threadIdx.x; i < i1; i += T) {
    const int L = alen[i];
    for (int k0 = 0; k0 < L; k0 += 8) {
      int c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = acol[((k0 + u < L) ? k0 + u : k0) * cap + i];
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        if (k0 + u >= L) break;
        const uint32_t a = map[c[u] / PS_CHUNK] * PS_CHUNK + c[u] % PS_CHUNK;
        const uint32_t b = map[c[u + 1] / PS_CHUNK] * PS_CHUNK + c[u + 1] % PS_CHUNK;
        lidx[(size_t)((k0 + u) >> 1) * ls + i] = a | (b << 16);
      }
    }
  }
}

// Windows of the workgroups' rows (one workgroup each, as the solve), the
// rows' columns as window positions, the slots cleared and the start kept
template <int T>
__global__ void __launch_bounds__(T) k_ps_setup(Dev D, PersArg Q) {
  __shared__ uint16_t map[PS_MAX_CHUNKS];
  __shared__ int cnt[T];
  const int t = threadIdx.x, wg = blockIdx.x, n = D.sc->n;
  const int nch = (n + PS_CHUNK - 1) / PS_CHUNK;
  const int i0 = wg * Q.nbw * RED_BLOCK;
  const int i1 = min(n, min(D.nblk, (wg + 1) * Q.nbw) * RED_BLOCK);
  for (int b = wg * Q.nbw + t; b < min(D.nblk, (wg + 1) * Q.nbw); b += T)
    for (int q = 0; q < 4; q++) {
      Q.slots[4 * (size_t)b + q] = 0;
      Q.slots[4 * ((size_t)D.nblk + b) + q] = 0;
    }
  if (t < 8) Q.slots[8 * ((size_t)D.nblk + wg) + t] = 0;
  for (int i = i0 + t; i < i1; i += T) {
    Q.tlo[i] = Q.thi[i] = Q.rlo[i] = Q.rhi[i] = 0;
    Q.x0[i] = D.sol[i];
  }
  int own;
  const int total = ps_window_chunks<T>(D.acol, D.alen, D.cap, i0, i1, nch, map, cnt, own);
  if (total > Q.wcap) {  // the whole workgroup
    if (t == 0) {
      atomicOr(&D.sc->counter[PS_FLAG_WIN], 1u);
      Q.wcnt[2 * wg] = 0;
    }
    return;
  }
  ps_window_list<T>(i0, nch, own, total, map, cnt, Q.wlist + (size_t)wg * Q.wcap,
                    Q.wcnt + 2 * wg);
  __syncthreads();
  ps_window_positions<T>(D.acol, D.alen, D.cap, i0, i1, map, Q.lidx, Q.ls);
}

// a value that is the same in every lane (that of the first), out of the vector
// registers
__device__ __forceinline__ double lane0(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)b);
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// LDS of the resident solve in doubles: the window, then an area shared by
// the block trees and the gathered partials, then the column sums, then (one
// row per thread) t1, later r, of the workgroup's rows
template <int T, int R>
__host__ __device__ constexpr int ps_tree_doubles() { return 2 * R * (T / 256) * 192; }
// row positions and values kept in LDS: what the window leaves of it
constexpr int ps_lds_pos(int T, int R) { return T != 1024 ? 0 : R == 3 ? 16 : 22; }
constexpr int ps_lds_val(int T, int R) { return T == 1024 && R == 1 ? 7 : 0; }
template <int T, int R, int W>
__host__ __device__ inline int64_t ps_lds_bytes(int nblk) {
  const int64_t a = ps_tree_doubles<T, R>(), b = 2 * (int64_t)nblk, w = (int64_t)W * T;
  const int64_t area = a > b ? a : b, own = 2 * 256 + 2 + (R > 1 ? 0 : T);
  if (T == 1024)  // the area shares the window's place; row entries
    return 8 * ((w > area ? w : area) + own + ps_lds_val(T, R) * R * T) +
           4 * (ps_lds_pos(T, R) / 2 * R * T);
  return 8 * (w + area + own);
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
template <int T, int G>
__device__ __forceinline__ bool ps_collect(const unsigned long long* set, int words, unsigned ep,
                                           uint32_t* out) {
  for (int w0 = threadIdx.x; w0 < words; w0 += G * T) {
    uint32_t lo[G];
    unsigned long long w[G];
    bool all = false;
#pragma unroll
    for (int u = 0; u < G; u++) w[u] = ld_word(set, min(w0 + u * T, words - 1));
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
// final_tree2; `mid` runs between the publication of this workgroup's partial
// sums and the wait for the others'.  Returns false when a wait ran out.
//
// Up to 256 row blocks (one per workgroup, T = 256) every workgroup collects
// all partials itself: one exchange.  With more, the readers' requests for
// the same lines would take longer than a second exchange (24 us against 4 at
// 809 blocks): workgroup 0 collects the partials and sends the sums to a line
// of each workgroup's own.
template <int T, int R, int NV, typename MID>
__device__ __forceinline__ bool ps_reduce(const PersArg& Q, int nblk, int b0, unsigned ep,
                                          const double (&v)[NV][R], double* area, double* col,
                                          int* bad, double (&out)[NV], MID mid) {
  constexpr int S = T / 256;
  int t = threadIdx.x;
  if (T == 1024) asm volatile("" : "+v"(t));  // (opaque: no addresses held over the iterations)
  const int wv = (t >> 6) & 3, l = t & 63, sub = t >> 8;
  if (T == 1024) __syncthreads();  // the area is in the window's place
  // tree j = k R + q of a block is summed by wavefront j mod 4 of its four;
  // the other three leave their values in LDS
#pragma unroll
  for (int k = 0; k < NV; k++)
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int j = k * R + q, o = j & 3;
      if (wv != o) area[(j * S + sub) * 192 + (wv < o ? wv : wv - 1) * 64 + l] = v[k][q];
    }
  __syncthreads();
  // two sets of slots of 4 words per block, used with NV doubles each
  unsigned long long* set = Q.slots + (size_t)(ep & 1) * 4 * nblk;
#pragma unroll
  for (int k = 0; k < NV; k++)
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int j = k * R + q, o = j & 3;
      if (wv == o) {
        const double* a = area + (j * S + sub) * 192 + l;
        const double w0 = (o == 0) ? v[k][q] : a[0];
        const double w1 = (o == 1) ? v[k][q] : a[(o < 1 ? 0 : 1) * 64];
        const double w2 = (o == 2) ? v[k][q] : a[(o < 2 ? 1 : 2) * 64];
        const double w3 = (o == 3) ? v[k][q] : a[2 * 64];
        const double s = wave_tree((w0 + w2) + (w1 + w3));
        const int lb = q * S + sub;
        if (l == 0 && lb < Q.nbw && b0 + lb < nblk)
          ps_publish(&set[2 * (size_t)(NV * (b0 + lb) + k)], ep, s);
      }
    }
  mid();
  if (T == 256) {
    if (!ps_collect<T, 4>(set, 2 * NV * nblk, ep, reinterpret_cast<uint32_t*>(col))) *bad = 1;
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
    __syncthreads();  // the trees are read; the area takes the partials
    if (!ps_collect<T, 4>(set, 2 * NV * nblk, ep, reinterpret_cast<uint32_t*>(area)))
      *bad = 1;
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

// A thread's first KR row entries, held in registers for the whole launch
// (KR 0: none); ps_row reads the rest from memory
template <int KR>
struct PsRow {
  double v[KR ? KR : 1];
  uint32_t w[KR ? KR / 2 : 1];
};

// U entries k0.. of row i: their positions and values (those below the
// wavefront's longest row Lm; FULL: all are), gathers and products
template <int U, bool FULL>
__device__ __forceinline__ double ps_entries(const uint32_t*& ip, const double*& vp, int ls,
                                             int cap, unsigned i, int k0, int L, int Lm,
                                             const double* win, double acc) {
  uint32_t w[U / 2];
  double v[U], g[U];
#pragma unroll
  for (int q = 0; q < U / 2; q++) {
    w[q] = 0u;
    if (FULL || k0 + 2 * q < Lm) w[q] = *ps_at(ip, i);
    ip += ls;
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    v[u] = 0.0;
    if (FULL || k0 + u < Lm) v[u] = *ps_at(vp, i);
    vp += cap;
  }
#pragma unroll
  for (int q = 0; q < U / 2; q++) {
    w[q] = (k0 + 2 * q < L) ? w[q] : 0u;  // a shorter row's slots hold no position
    g[2 * q] = win[w[q] & 0xffffu];
    g[2 * q + 1] = win[w[q] >> 16];
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    const double a = acc + v[u] * g[u];
    acc = (k0 + u < L) ? a : acc;
  }
  return acc;
}

// y_i = sum_k A_ik win[pos(k)] in row order (the order of ell_row_sum).  The
// loop runs to the wavefront's longest row (Lm, uniform), so the slots' bases
// are scalars.
template <int U, int KR>
__device__ __forceinline__ double ps_row(const PsRow<KR>& M, const uint32_t* idx, int ls,
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
  const uint32_t* ip = idx + (size_t)(KR / 2) * ls;
  const double* vp = val + (size_t)KR * cap;
  int k0 = KR;
#pragma unroll 1
  for (; k0 + U <= Lm; k0 += U)
    acc = ps_entries<U, true>(ip, vp, ls, cap, i, k0, L, Lm, win, acc);
  if (k0 < Lm) acc = ps_entries<U, false>(ip, vp, ls, cap, i, k0, L, Lm, win, acc);
  return acc;
}
// The same with the first KP positions and KV values of every row in LDS
// (lw, lv: those of this row), where 1,024 threads have no registers for them:
// what an iteration streams is most of its time there.  Without / with them, us
// per iteration: 20.3 / 19.0 at 136k rows, 26.5 / 20.9 at 207k, 39.3 / 36.9 at
// 307k, 44.9 / 40.5 at 409k, 63.0 / 59.0 at 653k.
template <int U, int KP, int KV, int T>
__device__ __forceinline__ double ps_row_lds(const uint32_t* lw, const double* lv, int t,
                                             const uint32_t* idx, int ls, const double* val,
                                             int cap, unsigned i, int L, int Lm,
                                             const double* win) {
  double acc = 0.0;
  const double* vp = val + (size_t)KV * cap;
#pragma unroll
  for (int k0 = 0; k0 < KP; k0 += U) {
    if (k0 >= Lm) break;
    double v[U], g[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (k0 + u >= KP) continue;
      if (k0 + u < KV) {
        v[u] = lv[(k0 + u) * T + t];
      } else {
        v[u] = (k0 + u < Lm) ? *ps_at(vp, i) : 0.0;
        vp += cap;
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (k0 + u >= KP) continue;
      const uint32_t w = lw[((k0 + u) / 2) * T + t];
      g[u] = win[(u & 1) ? (w >> 16) : (w & 0xffffu)];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (k0 + u >= KP) continue;
      const double a = acc + v[u] * g[u];
      acc = (k0 + u < L) ? a : acc;
    }
  }
  const uint32_t* ip = idx + (size_t)(KP / 2) * ls;
  int k0 = KP;
#pragma unroll 1
  for (; k0 + U <= Lm; k0 += U)
    acc = ps_entries<U, true>(ip, vp, ls, cap, i, k0, L, Lm, win, acc);
  if (k0 < Lm) acc = ps_entries<U, false>(ip, vp, ls, cap, i, k0, L, Lm, win, acc);
  return acc;
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) v = max(v, __shfl_xor(v, s, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// up to `iters` BiCGStab iterations from the state in D.sol, D.r, D.rh, D.pp
// and the scalars (k_bicg_init or a previous launch); leaves the state there.
//
// One row per thread: the window's p, r and t1 stay in registers as above.
// Several rows per thread: those registers hold the rows' own vectors, so p
// and s themselves are exchanged, straight into the window in LDS (two more
// hops of ~1.5 us in an iteration of 40 us and more, where 150 spilled
// registers took 20).
template <int T, int R, int W, int KR>
__global__ void __launch_bounds__(T) k_bicg_resident(Dev D, PersArg Q, int iters, unsigned ep) {
  constexpr int S = T / 256;
  constexpr bool ONE = R == 1;
  // row entries in flight per thread (several rows: 4, 6, 8 took 37.8, 36.9,
  // 36.4 us an iteration at 307k rows and 59.0, 59.0, 59.2 at 653k)
  constexpr int U = ONE ? 8 : 6;
  constexpr int WR = ONE ? W : 1;  // window elements in registers
  extern __shared__ double ps_lds[];
  __shared__ int bad_[1];
  int* bad = bad_;
  const int wg = blockIdx.x;
  DevScalars* Sc = D.sc;
  const int n = Sc->n, nblk = D.nblk, cap = D.cap, b0 = wg * Q.nbw;
  const int ta = ps_tree_doubles<T, R>();
  double* win = ps_lds;
  // 1,024 threads: the reductions' area in the window's place, for row entries
  const int tn = ta > 2 * nblk ? ta : 2 * nblk;
  double* area = (T == 1024) ? win : win + W * T;
  double* col = (T == 1024) ? win + (W * T > tn ? W * T : tn) : area + tn;
  double* own = col + 514;  // one row per thread: its t1, then r
  constexpr int KP = ps_lds_pos(T, R), KV = ps_lds_val(T, R);
  double* lv = own + (ONE ? T : 0);
  uint32_t* lw = reinterpret_cast<uint32_t*>(lv + KV * R * T);
  double rho = Sc->rho;
  const double bnorm = Sc->bnorm, tol = D.P.tol;
  const int max_iter = D.P.max_iter;
  int it = Sc->iters;
  int row[R], len[R], lmx[R];
  double r[R], rh[R], p[R], x[R], t1[R];
  PsRow<KR> M[R];
  // the window's elements of this thread: element e = w T + t is row
  // 64 c + (t & 63) with c the chunk of its wavefront (-1: none)
  int wc[W];
  double rw[WR], pw[WR], tw[WR];
  const int oc0 = b0 * (RED_BLOCK / PS_CHUNK), oc1 = oc0 + Q.nbw * (RED_BLOCK / PS_CHUNK);
  const int wn = Q.wcnt[2 * wg], s0 = Q.wcnt[2 * wg + 1];
  {
    const int t = threadIdx.x, sub = t >> 8, l = t & 63;
    if (t == 0) *bad = wg < Q.ended;
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int lb = q * S + sub, i = (b0 + lb) * RED_BLOCK + (t & 255);
      const bool in = lb < Q.nbw && i < n;
      row[q] = in ? i : -1;
      len[q] = in ? D.alen[i] : 0;
      lmx[q] = wave_max(len[q]);
      r[q] = in ? D.r[i] : 0.0;
      p[q] = in ? D.pp[i] : 0.0;
      rh[q] = (in && ONE) ? D.rh[i] : 0.0;
      x[q] = (in && ONE) ? D.sol[i] : 0.0;
#pragma unroll
      for (int k = 0; k < KR; k++) {
        M[q].v[k] = (k < len[q]) ? D.aval[k * cap + i] : 0.0;
        if (k % 2 == 0) M[q].w[k / 2] = (k < len[q]) ? Q.lidx[(size_t)(k / 2) * Q.ls + i] : 0u;
      }
#pragma unroll
      for (int k = 0; k < KP; k += 2)
        lw[(q * KP / 2 + k / 2) * T + t] =
            (k < len[q]) ? Q.lidx[(size_t)(k / 2) * Q.ls + i] : 0u;
#pragma unroll
      for (int k = 0; k < KV; k++)
        lv[(q * KV + k) * T + t] = (k < len[q]) ? D.aval[k * cap + i] : 0.0;
    }
#pragma unroll
    for (int w = 0; w < W; w++) {
      const int s = w * (T / PS_CHUNK) + t / PS_CHUNK;
      wc[w] = __builtin_amdgcn_readfirstlane((s < wn) ? Q.wlist[(size_t)wg * Q.wcap + s] : -1);
      if (ONE) {
        const int g = wc[w] * PS_CHUNK + l;
        const bool in = wc[w] >= 0 && g < n;
        rw[w] = in ? D.r[g] : 0.0;
        pw[w] = in ? D.pp[g] : 0.0;
      }
    }
  }
  __syncthreads();
  int conv = 0, brk = 0, done = 0;
  double alpha = 0.0, omega = 0.0, beta = 0.0, rr = 0.0, rel = 0.0;
  bool ok = true;
  for (int k = 0; k < iters; k++) {
    // (opaque: or the compiler holds every address formed from these in
    // registers over the iterations)
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int q = 0; q < R; q++) asm volatile("" : "+v"(row[q]));
    const int l = t & 63;
    // a value of this thread's row q to the other workgroups, as words of e
    auto put = [&](unsigned long long* lo, unsigned long long* hi, int q, unsigned e, double v) {
      const unsigned long long tag = (unsigned long long)e << 32;
      const unsigned long long b = (unsigned long long)__double_as_longlong(v);
      if (row[q] >= 0) {
        st_agent(ps_at(lo, row[q]), (b & 0xffffffffull) | tag);
        st_agent(ps_at(hi, row[q]), (b >> 32) | tag);
      }
    };
    // N of the window's elements from w0 on: other workgroups' rows from their
    // words of e (o[j]; own rows' entries are left)
    auto get = [&]<int N>(const unsigned long long* lo, const unsigned long long* hi, unsigned e,
                          int w0, double (&o)[N]) {
      for (int spin = 0;;) {
        unsigned long long a[N], b[N];
        bool all = true;
#pragma unroll
        for (int j = 0; j < N; j++) {
          const int c = wc[w0 + j];
          a[j] = b[j] = (unsigned long long)e << 32;
          if (c >= 0 && (c < oc0 || c >= oc1) && l < n - c * PS_CHUNK) {
            a[j] = ld_word(lo + (int64_t)c * PS_CHUNK, l);
            b[j] = ld_word(hi + (int64_t)c * PS_CHUNK, l);
          }
        }
#pragma unroll
        for (int j = 0; j < N; j++) {
          all = all && (unsigned)(a[j] >> 32) == e && (unsigned)(b[j] >> 32) == e;
          o[j] = __longlong_as_double((long long)((a[j] & 0xffffffffull) | (b[j] << 32)));
        }
        if (all) break;
        if (++spin >= PS_SPIN || ((spin & 1023) == 0 && *(volatile int*)bad)) {
          *bad = 1;
          break;
        }
      }
    };
    // several rows per thread: v of every row into the window
    auto exchange = [&](unsigned long long* lo, unsigned long long* hi, unsigned e,
                        const double (&v)[R]) {
#pragma unroll
      for (int q = 0; q < R; q++) {
        put(lo, hi, q, e, v[q]);
        if (row[q] >= 0) win[s0 * PS_CHUNK + q * T + t] = v[q];
      }
#pragma unroll
      for (int w0 = 0; w0 < W; w0 += 2) {
        double o[2];
        static_assert(ONE || W % 2 == 0, "window elements are read two at a time");
        get(lo, hi, e, w0, o);
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int c = wc[w0 + j];
          if (c >= 0 && (c < oc0 || c >= oc1)) win[(w0 + j) * T + t] = o[j];
        }
      }
    };
    // one row per thread: the window's v, own rows' from LDS
    auto window = [&](const unsigned long long* lo, const unsigned long long* hi, unsigned e,
                      double (&o)[WR]) {
      get(lo, hi, e, 0, o);
#pragma unroll
      for (int w = 0; w < WR; w++)
        if (wc[w] >= oc0 && wc[w] < oc1) o[w] = own[(wc[w] - oc0) * PS_CHUNK + l];
    };
    auto product = [&](int q) -> double {
      if constexpr (KP > 0)
        return ps_row_lds<U, KP, KV, T>(lw + q * KP / 2 * T, lv + q * KV * T, t, Q.lidx, Q.ls,
                                        D.aval, cap, row[q], len[q], lmx[q], win);
      else
        return ps_row<U, KR>(M[q], Q.lidx, Q.ls, D.aval, cap, row[q], len[q], lmx[q], win);
    };
    // t1 = A p ; alpha = rho / (t1 . rh)
    if constexpr (ONE) {
#pragma unroll
      for (int w = 0; w < W; w++) win[w * T + t] = pw[w];
    } else {
      exchange(Q.rlo, Q.rhi, ep, p);
    }
    __syncthreads();
    double v1[1][R], o1[1];
#pragma unroll
    for (int q = 0; q < R; q++) {
      __builtin_amdgcn_sched_barrier(0);  // one row's loads in registers at a time
      if (!ONE) rh[q] = (row[q] >= 0) ? *ps_at(D.rh, row[q]) : 0.0;
      t1[q] = (row[q] >= 0) ? product(q) : 0.0;
      if constexpr (ONE) {
        own[t] = t1[q];
        put(Q.tlo, Q.thi, q, ep, t1[q]);
      }
      v1[0][q] = (row[q] >= 0) ? t1[q] * rh[q] : 0.0;
    }
    ok = ps_reduce<T, R, 1>(Q, nblk, b0, ep, v1, area, col, bad, o1, [&]() {
      if constexpr (ONE) window(Q.tlo, Q.thi, ep, tw);
    });
    ep++;
    if (!ok) break;
    // s = r - alpha t1 (in r) ; t2 = A s ; omega = (t2 . s) / (t2 . t2)
    alpha = rho / o1[0];
#pragma unroll
    for (int q = 0; q < R; q++) r[q] = r[q] - alpha * t1[q];
    if constexpr (ONE) {
#pragma unroll
      for (int w = 0; w < W; w++) win[w * T + t] = rw[w] - alpha * tw[w];
    } else {
      exchange(Q.tlo, Q.thi, ep, r);
    }
    __syncthreads();
    double t2[R], v2[2][R], o2[2];
#pragma unroll
    for (int q = 0; q < R; q++) {
      __builtin_amdgcn_sched_barrier(0);
      t2[q] = (row[q] >= 0) ? product(q) : 0.0;
      v2[0][q] = (row[q] >= 0) ? t2[q] * r[q] : 0.0;
      v2[1][q] = (row[q] >= 0) ? t2[q] * t2[q] : 0.0;
    }
    ok = ps_reduce<T, R, 2>(Q, nblk, b0, ep, v2, area, col, bad, o2, [&]() {
      if constexpr (!ONE) {
#pragma unroll
        for (int q = 0; q < R; q++) {
          rh[q] = (row[q] >= 0) ? *ps_at(D.rh, row[q]) : 0.0;
          x[q] = (row[q] >= 0) ? *ps_at(D.sol, row[q]) : 0.0;
        }
      }
    });
    ep++;
    if (!ok) break;
    omega = o2[0] / o2[1];
    // x = (x + alpha p) + omega s ; r = s - omega t2 ; rho' = r . rh ; rr = r . r
#pragma unroll
    for (int q = 0; q < R; q++) {
      x[q] = (x[q] + alpha * p[q]) + omega * r[q];
      if (!ONE && row[q] >= 0) *ps_at(D.sol, row[q]) = x[q];
      r[q] = r[q] - omega * t2[q];
      p[q] = p[q] - omega * t1[q];
      if constexpr (ONE) {
        own[t] = r[q];
        put(Q.rlo, Q.rhi, q, ep, r[q]);
      }
      v2[0][q] = (row[q] >= 0) ? r[q] * rh[q] : 0.0;
      v2[1][q] = (row[q] >= 0) ? r[q] * r[q] : 0.0;
    }
    if constexpr (ONE) {
#pragma unroll
      for (int w = 0; w < W; w++) pw[w] = pw[w] - omega * tw[w];
    }
    ok = ps_reduce<T, R, 2>(Q, nblk, b0, ep, v2, area, col, bad, o2, [&]() {
      if constexpr (ONE) window(Q.rlo, Q.rhi, ep, rw);
    });
    ep++;
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
    if constexpr (ONE) {
#pragma unroll
      for (int w = 0; w < W; w++) pw[w] = rw[w] + beta * pw[w];
    }
#pragma unroll
    for (int q = 0; q < R; q++) p[q] = r[q] + beta * p[q];
  }
  const int t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < R; q++)
    if (row[q] >= 0) {
      if (ONE) D.sol[row[q]] = x[q];
      D.pp[row[q]] = p[q];
      D.r[row[q]] = r[q];
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
