// isph_mgres.h -- the precision-form BiCGStab (isph_mg.h) of any number of
// scenarios as one resident launch.
//
// The launch-per-phase form takes 18 to 26 dependent launches per iteration,
// and below a few hundred thousand rows almost all of an iteration is their
// latency: 92 us at 7,485 rows, 116 us at 22k, 140 us at 137k, where the data
// of an iteration needs 1, 2 and 12 us.  Here the phases of an iteration
// meet through memory words instead: every value that another workgroup
// needs travels as one 64-bit word, the float in its low half and the number
// of the V-cycle in its high half, and the reader polls the word itself.  No
// phase waits for more than the words it reads.
//
// Work split.  A scenario's row blocks (256 rows) lie in runs of nbw blocks on
// its row workgroups (512 threads with a row each, or 1,024 with up to three);
// one more workgroup per scenario runs the coarse levels, with their stencils
// and the dense inverse in registers and LDS for the whole solve, and forms
// the dot products.  An iteration takes 38 us at 7,485 and 22k rows, 56 at
// 137k, 66 at 207k and 133 at 653k: up to ~130k rows the chain of some 20
// exchanges of 1.2 us with the work between them, above that half and more the
// products' streaming.
// Windows, row positions and the polling rules are those of isph_persist.h.
//   level 0   x0 (and ph, sh) of the window's rows by words; the products
//             gather from LDS
//   restrict  a cell's rows are summed by the workgroup holding its first
//             row; rows of the next workgroup arrive by words
//   levels 1..m   aggregates (down) and cells (up) in equal runs per
//             workgroup; right-hand sides and corrections by words (with one
//             row per thread every window forms its level-1 corrections)
//   levels m+1..  the coarse workgroup
// The arithmetic and its order are those of the launch-per-phase bodies, so
// every iterate, scalar and count has the same bits.
//
// A word is rewritten one V-cycle later; the dot product between the two has
// collected partial sums that every reader published after its reads.
#pragma once
#include "isph_batch.h"
#include "isph_cells.h"
#include "isph_persist.h"

#define RS_W 6                      // window elements per thread
#define RS_WCAP (RS_W * 1024 / PS_CHUNK)  // window chunks of a workgroup at most
// Threads of the coarse workgroup's first level at most, four per unknown of
// the next; their stencils stay in registers.  A level more on the row workgroups costs two more hops of
// ~1.2 us a V-cycle, a level of 1-4 unknowns per thread more in the one
// workgroup 2-4 us: 1,024 against 2,560 unknowns took 51.0 against 55.8 us
// per iteration at 7,485 rows and 73.7 against 77.4 at 22k; 300 took 52.4
// and 74.7.
#define RS_CO_MAX 1024
#define RS_PER(T) ((RS_CO_MAX + (T)-1) / (T))
// Cells of its window that a thread forms the level-1 correction of, with one
// row per thread; 0: the cells' own workgroups do, and send it.  Forming it in
// every window repeats work and saves an exchange: 45.7 us an iteration with
// the exchange, 43.4 without at 22k rows, 61.8 and 57.5 at 137k, 72.2 and 67.3
// at 207k; with two and three rows per thread 88.3 and 92.1 at 307k, 133.1 and
// 134.1 at 653k.
constexpr int rs_cells(int R) { return R == 1 ? 2 : 0; }
#define RS_MAIL 16                  // words of a workgroup's mail line
#define RS_TAIL 256                 // rows of the next workgroups in a workgroup's last cell

struct ResDev {
  int wg0, G;                 // first workgroup; row workgroups (the coarse one is wg0 + G)
  int nbw;                    // row blocks per workgroup
  int m;                      // cell levels 1..m on the row workgroups
  int ended;                  // workgroups of the scenario whose waits count as run out
  unsigned long long* slots;  // 10 words per row block
  unsigned long long* mail;   // RS_MAIL words per workgroup
  unsigned long long *x0w, *phw, *r0w;  // a word per row: x0, V-cycle result, r0
  unsigned long long *bw, *ew;          // a word per cell of every level: b, e
  int32_t* wlist;             // per workgroup: RS_WCAP window chunks
  int32_t* wcnt;              // per workgroup: their count, and the slot of its own first chunk
};

// A pointer read from a table, in the global address space (else its
// accesses are flat ones)
template <typename V>
__device__ __forceinline__ V* glob(V* p) {
  return (V*)(__attribute__((address_space(1))) V*)p;
}
template <typename A>
__device__ __forceinline__ A ld_table(const A* p) {
  return *(const A*)(const __attribute__((address_space(1))) A*)p;
}

// One tagged float; the wait is bounded and ends early once a wait of the
// workgroup has run out
__device__ __forceinline__ float rs_wait(const unsigned long long* p, unsigned tag,
                                         volatile int* bad, unsigned long long w) {
  if ((unsigned)(w >> 32) != tag) {
    int spin = 0;
    do {
      w = ld_agent(p);
      if (++spin >= PS_SPIN || ((spin & 1023) == 0 && *bad)) {
        *bad = 1;
        break;
      }
    } while ((unsigned)(w >> 32) != tag);
  }
  return __uint_as_float((uint32_t)w);
}
// N words together: ld(k) reads word k (a word of the tag itself where lane
// needs none); all are read again until every one carries the number
template <int N, typename LD>
__device__ __forceinline__ void rs_poll(unsigned tag, volatile int* bad, LD ld,
                                        float (&out)[N]) {
  for (int spin = 0;;) {
    unsigned long long w[N];
#pragma unroll
    for (int k = 0; k < N; k++) w[k] = ld(k);
    bool all = true;
#pragma unroll
    for (int k = 0; k < N; k++) {
      all = all && (unsigned)(w[k] >> 32) == tag;
      out[k] = __uint_as_float((uint32_t)w[k]);
    }
    if (all) return;
    if (++spin >= PS_SPIN || ((spin & 1023) == 0 && *bad)) {
      *bad = 1;
      return;
    }
  }
}
__device__ __forceinline__ void rs_put(unsigned long long* p, unsigned tag, float v) {
  st_agent(p, ((unsigned long long)tag << 32) | __float_as_uint(v));
}

// The level table in LDS: a level's sizes by one LDS read (from memory every
// use would be a load, a store of the loop before it being in the way)
__device__ __forceinline__ MgLevel rs_level(const MgLevel* lev, int l) {
  MgLevel L = lev[l];
  L.ny = __builtin_amdgcn_readfirstlane(L.ny);
  L.nx = __builtin_amdgcn_readfirstlane(L.nx);
  L.n = __builtin_amdgcn_readfirstlane(L.n);
  L.off = __builtin_amdgcn_readfirstlane(L.off);
  return L;
}

// scenario of this workgroup
__device__ __forceinline__ int rs_locate(const ResDev* rs, int S, int wg) {
  int s = 0;
  while (s + 1 < S && rs[s + 1].wg0 <= wg) s++;
  return s;
}

// Windows, window positions (into D.aoff) and cleared words, one workgroup
// per row workgroup of the solve
template <int T, int R>
__global__ void __launch_bounds__(T) kb_rs_setup(BatchDev B, const ResDev* rs) {
  __shared__ uint16_t map[PS_MAX_CHUNKS];
  __shared__ int cnt[T];
  const int wcap = RS_W * T / PS_CHUNK;
  const int s = rs_locate(rs, B.S, blockIdx.x), t = threadIdx.x;
  const ResDev& Q = rs[s];
  const Dev& D = B.devs[s];
  const MgDev& G = B.mgs[s];
  const int wg = blockIdx.x - Q.wg0;
  if (wg >= Q.G) {  // the coarse workgroup's place
    return;
  }
  const int n = D.sc->n, cap = D.cap, nblk = D.nblk;
  const int nch = (n + PS_CHUNK - 1) / PS_CHUNK;
  const int i0 = wg * Q.nbw * RED_BLOCK;
  const int i1 = min(n, min(nblk, (wg + 1) * Q.nbw) * RED_BLOCK);
  const int32_t* acol = glob(D.acol);
  const int32_t* alen = glob(D.alen);
  uint32_t* lidx = glob(D.aoff);
  for (int b = wg * Q.nbw * 10 + t; b < min(nblk, (wg + 1) * Q.nbw) * 10; b += T)
    Q.slots[b] = 0;
  if (t < RS_MAIL) Q.mail[wg * RS_MAIL + t] = 0;
  for (int i = i0 + t; i < i1; i += T) {
    Q.x0w[i] = 0;
    Q.phw[i] = 0;
    Q.r0w[i] = 0;
  }
  const int tot = G.lev[G.nlev].off + G.lev[G.nlev].n;
  for (int c = (int)((int64_t)tot * wg / Q.G) + t; c < (int)((int64_t)tot * (wg + 1) / Q.G);
       c += T) {
    Q.bw[c] = 0;
    Q.ew[c] = 0;
  }
  int own;
  const int total = ps_window_chunks<T>(acol, alen, cap, i0, i1, nch, map, cnt, own);
  // rows of the last cell in later workgroups (rs_rows_solve's tail)
  int tail = 0;
  if (i1 > i0 && i1 < n) {
    const int k = D.cell[i1 - 1];
    tail = D.cstart[k + 1] - i1;
  }
  if (total > wcap || tail > RS_TAIL) {  // the whole workgroup
    if (t == 0) atomicOr(&D.sc->counter[PS_FLAG_WIN], 1u);
    return;
  }
  int32_t* wlist = Q.wlist + (size_t)wg * RS_WCAP;
  ps_window_list<T>(i0, nch, own, total, map, cnt, wlist, Q.wcnt + 2 * wg);
  if (rs_cells(R) > 0) {
    // the window's cells (a chunk's rows lie in cell order), of which
    // rs_rows_solve takes rs_cells per thread
    if (t == 0) cnt[0] = 0;
    __syncthreads();
    int mine = 0;
    for (int p = t; p < total * PS_CHUNK; p += T) {
      const int g = wlist[p / PS_CHUNK] * PS_CHUNK + p % PS_CHUNK;
      if (g < n && (g % PS_CHUNK == 0 || D.cell[g] != D.cell[g - 1])) mine++;
    }
    atomicAdd(&cnt[0], mine);
    __syncthreads();
    if (cnt[0] > rs_cells(R) * T && t == 0) atomicOr(&D.sc->counter[PS_FLAG_WIN], 1u);
  }
  __syncthreads();
  ps_window_positions<T>(acol, alen, cap, i0, i1, map, lidx, cap);
}

// ---------------------------------------------------------------------
// rows
// ---------------------------------------------------------------------
// The first entries of a workgroup's rows stay on the chip for the launch: read
// from memory, a row's three batches of entries are three dependent trips of
// ~0.5 us in each of the six products of an iteration, and above ~250k rows
// the traffic itself is what bounds them.  512 threads with a row each have
// the registers (for the FP64 values too); 1,024 threads keep positions and
// FP16 values in the LDS that the window leaves: 22, 14 and 8 entries of each
// row at 1, 2 and 3 rows per thread.  An iteration took 42.0 us before and
// 38.0 after at 7,485 rows, 42.6 and 37.5 at 22k, 64.6 and 61.7 at 137k, 93.7
// and 87.4 at 310k, 104.8 and 95.7 at 413k, 139.8 and 133.2 at 653k.
constexpr int rs_reg_entries(int T, int R) { return T == 512 && R == 1 ? 24 : 0; }
constexpr int rs_lds_entries(int T, int R) {
  return T != 1024 ? 0 : R == 1 ? 22 : R == 2 ? 14 : 8;
}
// words of the window with the rows' r0, which the reductions' area shares
constexpr int rs_work_words(int T, int R) {
  const int area = 2 * 5 * (T / 256) * 192, window = RS_W * T + R * T + RS_TAIL;
  return area > window ? area : window;
}
template <int T, int R>
struct RsEntries {
  static constexpr int KR = rs_reg_entries(T, R), KL = rs_lds_entries(T, R), K = KR + KL;
  uint32_t rw[KR ? KR / 2 : 1], rv[KR ? KR / 2 : 1];  // positions, FP16 values
  double rd[KR ? KR : 1];                             // FP64 values
  uint32_t* lw;                                       // positions, then FP16 values
  __device__ __forceinline__ void load(const uint32_t* ip, const uint32_t* hp, const double* vp,
                                       int cap, unsigned i, int L, int t, uint32_t* lds) {
    lw = lds;
#pragma unroll
    for (int q = 0; q < K / 2; q++) {
      const bool in = 2 * q < L;
      const uint32_t w = in ? *ps_at(ip + (size_t)q * cap, i) : 0u;
      const uint32_t h = in ? *ps_at(hp + (size_t)q * cap, i) : 0u;
      if (KR) {
        rw[KR ? q : 0] = w;
        rv[KR ? q : 0] = h;
      } else {
        lw[q * T + t] = w;
        lw[(KL / 2 + q) * T + t] = h;
      }
    }
    if (KR)
#pragma unroll
      for (int k = 0; k < KR; k++) rd[k] = k < L ? *ps_at(vp + (size_t)k * cap, i) : 0.0;
  }
  __device__ __forceinline__ uint32_t w(int q, int t) const {
    return KR ? rw[KR ? q : 0] : lw[q * T + t];
  }
  __device__ __forceinline__ uint32_t h(int q, int t) const {
    return KR ? rv[KR ? q : 0] : lw[(KL / 2 + q) * T + t];
  }
};

__device__ __forceinline__ float rs_half(uint32_t h, int u) {
  const unsigned short b = (unsigned short)((u & 1) ? (h >> 16) : (h & 0xffffu));
  return __half2float(__ushort_as_half(b));
}
// sum of the row's FP16 values times the window's floats, in entry order
// (the order of ell_row_sum_h)
template <bool FULL>
__device__ __forceinline__ float rs_row_h8(const uint32_t*& ip, const uint32_t*& hp, int cap,
                                           unsigned i, int k0, int L, int Lm, const float* X,
                                           float acc) {
  uint32_t w[4], h[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = h[q] = 0u;
    if (FULL || k0 + 2 * q < Lm) {
      w[q] = *ps_at(ip, i);
      h[q] = *ps_at(hp, i);
    }
    ip += cap;
    hp += cap;
  }
  float g[8];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = (k0 + 2 * q < L) ? w[q] : 0u;
    g[2 * q] = X[w[q] & 0xffffu];
    g[2 * q + 1] = X[w[q] >> 16];
  }
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const float a = acc + rs_half(h[u / 2], u) * g[u];
    acc = (k0 + u < L) ? a : acc;
  }
  return acc;
}
template <int T, int R>
__device__ __forceinline__ float rs_row_h(const RsEntries<T, R>& E, const uint32_t* ip,
                                          const uint32_t* hp, int cap, unsigned i, int t, int L,
                                          int Lm, const float* X) {
  constexpr int K = RsEntries<T, R>::K;
  float acc = 0.0f;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 8) {
    if (k0 >= Lm) break;
    float g[8], a[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (k0 + u >= K) continue;
      const uint32_t w = E.w((k0 + u) / 2, t);
      g[u] = X[(u & 1) ? w >> 16 : w & 0xffffu];
      a[u] = rs_half(E.h((k0 + u) / 2, t), u);
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (k0 + u >= K) continue;
      const float s = acc + a[u] * g[u];
      acc = (k0 + u < L) ? s : acc;
    }
  }
  ip += (size_t)(K / 2) * cap;
  hp += (size_t)(K / 2) * cap;
  int k0 = K;
#pragma unroll 1
  for (; k0 + 8 <= Lm; k0 += 8) {
    acc = rs_row_h8<true>(ip, hp, cap, i, k0, L, Lm, X, acc);
  }
  if (k0 < Lm) acc = rs_row_h8<false>(ip, hp, cap, i, k0, L, Lm, X, acc);
  return acc;
}
// sum of the row's FP64 values times the window's floats, in entry order
template <bool FULL>
__device__ __forceinline__ double rs_row_d8(const uint32_t*& ip, const double*& vp, int cap,
                                            unsigned i, int k0, int L, int Lm, const float* X,
                                            double acc) {
  uint32_t w[4];
  double v[8];
  float g[8];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = 0u;
    if (FULL || k0 + 2 * q < Lm) w[q] = *ps_at(ip, i);
    ip += cap;
  }
#pragma unroll
  for (int u = 0; u < 8; u++) {
    v[u] = 0.0;
    if (FULL || k0 + u < Lm) v[u] = *ps_at(vp, i);
    vp += cap;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = (k0 + 2 * q < L) ? w[q] : 0u;
    g[2 * q] = X[w[q] & 0xffffu];
    g[2 * q + 1] = X[w[q] >> 16];
  }
#pragma unroll
  for (int u = 0; u < 8; u++) {
    const double a = acc + v[u] * (double)g[u];
    acc = (k0 + u < L) ? a : acc;
  }
  return acc;
}
template <int T, int R>
__device__ __forceinline__ double rs_row_d(const RsEntries<T, R>& E, const uint32_t* ip,
                                           const double* vp, int cap, unsigned i, int t, int L,
                                           int Lm, const float* X) {
  constexpr int K = RsEntries<T, R>::K, KR = RsEntries<T, R>::KR;
  double acc = 0.0;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 8) {
    if (k0 >= Lm) break;
    float g[8];
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (k0 + u >= K) continue;
      if (KR) v[u] = E.rd[KR ? k0 + u : 0];
      else v[u] = (k0 + u < Lm) ? *ps_at(vp, i) : 0.0;
      vp += cap;
      const uint32_t w = E.w((k0 + u) / 2, t);
      g[u] = X[(u & 1) ? w >> 16 : w & 0xffffu];
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (k0 + u >= K) continue;
      const double s = acc + v[u] * (double)g[u];
      acc = (k0 + u < L) ? s : acc;
    }
  }
  ip += (size_t)(K / 2) * cap;
  int k0 = K;
  if (K >= Lm) return acc;
#pragma unroll 1
  for (; k0 + 8 <= Lm; k0 += 8) {
    acc = rs_row_d8<true>(ip, vp, cap, i, k0, L, Lm, X, acc);
  }
  if (k0 < Lm) acc = rs_row_d8<false>(ip, vp, cap, i, k0, L, Lm, X, acc);
  return acc;
}

// ---------------------------------------------------------------------
// dot products: the row workgroups publish their blocks' partial sums, the
// coarse workgroup sums them in the order of final_tree2 and sends the sums
// to each workgroup's mail line
// ---------------------------------------------------------------------
template <int T, int NV>
__device__ __forceinline__ bool rs_collect(const ResDev& Q, int nblk, unsigned ep,
                                                double* col, double* res, volatile int* bad,
                                                double (&out)[NV]) {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  const int l = t & 63, wave = t >> 6;
  const unsigned long long* slots = glob(Q.slots);
  // thread t sums column t & 255 (blocks c, c + 256, ...) of one or two values
  for (int e = t; e < NV * 256; e += T) {
    const int k = e >> 8, c = e & 255;
    const unsigned long long* p = slots + 2 * (size_t)k * nblk;
    double a = 0.0;
    for (int b0 = c; b0 < nblk; b0 += 4 * 256) {
      unsigned long long w[4][2];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int b = min(b0 + 256 * u, nblk - 1);
        w[u][0] = ld_agent(p + 2 * (size_t)b);
        w[u][1] = ld_agent(p + 2 * (size_t)b + 1);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int b = b0 + 256 * u;
        if (b < nblk) {
          const uint32_t lo = __float_as_uint(rs_wait(p + 2 * (size_t)b, ep, bad, w[u][0]));
          const uint32_t hi = __float_as_uint(rs_wait(p + 2 * (size_t)b + 1, ep, bad, w[u][1]));
          a = a + __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
        }
      }
    }
    col[e] = a;
  }
  __syncthreads();
  if (wave < NV) {
    const double* c = col + wave * 256;
    const double s = wave_tree((c[l] + c[l + 128]) + (c[l + 64] + c[l + 192]));
    if (l == 0) res[wave] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) out[k] = res[k];
  return !*bad;
}

template <int T, int R, int NV>
__device__ __forceinline__ bool rs_publish_wait(const ResDev& Q, int wg, int nblk, unsigned ep,
                                                const double (&v)[NV][R], double* area,
                                                double* res, volatile int* bad,
                                                double (&out)[NV]) {
  constexpr int S4 = T / 256;
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  const int wv = (t >> 6) & 3, l = t & 63, sub = t >> 8;
  // A block's trees are summed by its four wavefronts in turn, the other three
  // leaving their values in LDS, the rows of a thread one after the other: the
  // area (5 KB per four wavefronts for the five products) takes the place of
  // the window, and what it leaves free holds row entries.
  unsigned long long* slots = glob(Q.slots);
  const int b0 = wg * Q.nbw;
#pragma unroll
  for (int q = 0; q < R; q++) {
    __syncthreads();  // the window's or the last values' readers are through
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int o = (k * R + q) & 3;
      if (wv != o) area[(k * S4 + sub) * 192 + (wv < o ? wv : wv - 1) * 64 + l] = v[k][q];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int o = (k * R + q) & 3;
      if (wv == o) {
        const double* a = area + (k * S4 + sub) * 192 + l;
        const double w0 = (o == 0) ? v[k][q] : a[0];
        const double w1 = (o == 1) ? v[k][q] : a[(o < 1 ? 0 : 1) * 64];
        const double w2 = (o == 2) ? v[k][q] : a[(o < 2 ? 1 : 2) * 64];
        const double w3 = (o == 3) ? v[k][q] : a[2 * 64];
        const double s = wave_tree((w0 + w2) + (w1 + w3));
        const int lb = q * S4 + sub;
        if (l == 0 && lb < Q.nbw && b0 + lb < nblk)
          ps_publish(&slots[2 * ((size_t)k * nblk + b0 + lb)], ep, s);
      }
    }
  }
  if (t < 2 * NV) {
    const unsigned long long* p = glob(Q.mail) + wg * RS_MAIL + t;
    const float f = rs_wait(p, ep, bad, 0ull);
    reinterpret_cast<uint32_t*>(res)[t] = __float_as_uint(f);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) out[k] = res[k];
  return !*bad;
}

template <int T, int NV>
__device__ __forceinline__ bool rs_collect_send(const ResDev& Q, int nblk, unsigned ep,
                                                double* col, double* res, volatile int* bad,
                                                double (&out)[NV]) {
  if (!rs_collect<T, NV>(Q, nblk, ep, col, res, bad, out)) return false;
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  unsigned long long* mail = glob(Q.mail);
  for (int e = t; e < Q.G * 2 * NV; e += T) {
    const int g = e / (2 * NV), j = e - g * 2 * NV;
    st_agent(&mail[g * RS_MAIL + j], ((unsigned long long)ep << 32) |
                                         reinterpret_cast<const uint32_t*>(res)[j]);
  }
  return true;
}

// A scenario's hierarchy: the level table in LDS, uniform pointers
struct RsMg {
  const MgLevel* lev;
  const float *sten, *rdg;
  float w, c;
};

// The scalars of an iteration, formed alike by every workgroup of the scenario
// (pb_finalize: PFIN_ALPHA, PFIN_OMEGA)
struct RsScalars {
  double rho, alpha, omega, beta, rr, rel;
  int iters, conv, brk, done;
  bool update;  // the stopped iteration's x and r update still applies
};
__device__ __forceinline__ void rs_alpha(RsScalars& z, double s0) {
  z.alpha = lane0(z.rho / s0);
  if (!isfinite(z.alpha)) {
    z.brk = 1;
    z.done = 1;
  }
}
__device__ __forceinline__ void rs_omega(RsScalars& z, const double (&s)[5], double stop,
                                         double bnorm, int max_iter) {
  const double om = lane0(s[0] / s[1]);
  z.omega = om;
  z.update = false;
  if (!isfinite(om) || om == 0.0) {
    z.brk = 1;
    z.done = 1;
    return;
  }
  z.update = true;
  const double rr0 = s[4] - om * s[0], rr = (rr0 < 0.0) ? 0.0 : rr0;
  const double rhon = s[3] - om * s[2];
  z.iters++;
  z.rr = rr;
  z.rel = sqrt(rr) / bnorm;
  if (sqrt(rr) <= stop) {
    z.conv = 1;
    z.done = 1;
  } else if (rhon == 0.0 || !isfinite(rhon) || !isfinite(rr)) {
    z.brk = 1;
    z.done = 1;
  } else {
    z.beta = lane0((rhon / z.rho) * (z.alpha / om));
    z.rho = lane0(rhon);
    if (z.iters >= max_iter) z.done = 1;
  }
}

// ---------------------------------------------------------------------
// cell levels on the row workgroups (mg_lvl_down, mg_lvl_up)
// ---------------------------------------------------------------------
// first item of workgroup w of G's equal runs over n items
__device__ __forceinline__ int rs_part(int n, int w, int G) { return (int)((int64_t)n * w / G); }

// neighbours of cell (ci, cj): a bit for each that exists
__device__ __forceinline__ unsigned rs_has(const MgLevel& L, int ci, int cj) {
  const unsigned row = (ci > 0 ? 1u : 0u) | 2u | (ci + 1 < L.ny ? 4u : 0u);
  return (cj > 0 ? row : 0u) | (row << 3) | (cj + 1 < L.nx ? row << 6 : 0u);
}
// neighbour k, the cell itself in place of a missing one (its term is not
// added); formed anew at each use, for nine of them held over the polls are
// nine registers
__device__ __forceinline__ int rs_nbr(unsigned has, int I, int ny, int k) {
  return I + (((has >> k) & 1) ? (k / 3 - 1) * ny + (k % 3 - 1) : 0);
}
// the coarser cell holding neighbour k of a cell at place q (row q & 1, column
// q >> 1) of cell P
__device__ __forceinline__ int rs_par(unsigned has, int P, int q, int ny, int k) {
  const int di = ((q & 1) + k % 3 - 1) >> 1, dj = ((q >> 1) + k / 3 - 1) >> 1;
  return P + (((has >> k) & 1) ? dj * ny + di : 0);
}

template <int T>
__device__ __forceinline__ void rs_down(const RsMg& M, const ResDev& Q, int wg, int t,
                                        int l, unsigned tag, volatile int* bad) {
  const MgLevel L = rs_level(M.lev, l), C = rs_level(M.lev, l + 1);
  const float w = M.w;
  const float* st = M.sten + 9 * (size_t)L.off;
  const float* rd = M.rdg + L.off;
  unsigned long long* bw = glob(Q.bw);
  const unsigned long long* bl = bw + L.off;
  const int J0 = rs_part(C.n, wg, Q.G), J1 = rs_part(C.n, wg + 1, Q.G);
  for (int e = t; e < 4 * (J1 - J0); e += T) {
    const int J = J0 + (e >> 2), q = e & 3;
    const int CJ = J / C.ny, CI = J - CJ * C.ny;
    const int ci = 2 * CI + (q & 1), cj = 2 * CJ + (q >> 1);
    const bool in = ci < L.ny && cj < L.nx;
    const int I = in ? cj * L.ny + ci : 0;
    const unsigned has = in ? rs_has(L, ci, cj) : 0u;
    float sv[9], rv[9], bv[9];
#pragma unroll
    for (int k = 0; k < 9; k++) {
      sv[k] = *ps_at(st + (size_t)k * L.n, I);
      rv[k] = *ps_at(rd, rs_nbr(has, I, L.ny, k));
    }
    rs_poll<9>(tag, bad, [&](int k) { return ld_word(bl, rs_nbr(has, I, L.ny, k)); }, bv);
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const float tk = sv[k] * ((w * bv[k]) * rv[k]);
      if ((has >> k) & 1) acc = acc + tk;
    }
    const float bI = bv[4];
    const float res = in ? bI - acc : 0.0f;
    const int lane = t & 63, base = lane & ~3;
    const float r1 = __shfl(res, base + 1, 64), r2 = __shfl(res, base + 2, 64),
                r3 = __shfl(res, base + 3, 64);
    const int in_mask = __shfl((int)in, base + 1, 64) | (__shfl((int)in, base + 2, 64) << 1) |
                        (__shfl((int)in, base + 3, 64) << 2);
    if (q == 0) {
      float s = 0.0f;
      if (in) s = s + res;
      if (in_mask & 1) s = s + r1;
      if (in_mask & 2) s = s + r2;
      if (in_mask & 4) s = s + r3;
      rs_put(ps_at(bw + C.off, J), tag, s);
    }
  }
}

// value of level-L cell I after the correction from level C and the
// post-smoothing sweep, from the words of both levels
__device__ __forceinline__ float rs_up_cell(const RsMg& M, const ResDev& Q, const MgLevel& L,
                                            const MgLevel& C, int I, unsigned tag,
                                            volatile int* bad) {
  const float w = M.w, c = M.c;
  const float* st = M.sten + 9 * (size_t)L.off;
  const float* rd = M.rdg + L.off;
  const unsigned long long* bw = glob(Q.bw) + L.off;
  const unsigned long long* ec = glob(Q.ew) + C.off;
  const int cj = I / L.ny, ci = I - cj * L.ny;
  const int P = (cj >> 1) * C.ny + (ci >> 1), q = (ci & 1) | ((cj & 1) << 1);
  const unsigned has = rs_has(L, ci, cj);
  float xv[9], xc[9];
  // (the words of this level are those that the way down polled)
  rs_poll<9>(tag, bad, [&](int k) { return ld_word(bw, rs_nbr(has, I, L.ny, k)); }, xv);
  const float bI = xv[4], rI = *ps_at(rd, I);
#pragma unroll
  for (int k = 0; k < 9; k++) xv[k] = (w * xv[k]) * *ps_at(rd, rs_nbr(has, I, L.ny, k));
  float sv[9];
#pragma unroll
  for (int k = 0; k < 9; k++) sv[k] = *ps_at(st + (size_t)k * L.n, I);
  rs_poll<9>(tag, bad, [&](int k) { return ld_word(ec, rs_par(has, P, q, C.ny, k)); }, xc);
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    xv[k] = xv[k] + c * xc[k];
    const float tk = sv[k] * xv[k];
    if ((has >> k) & 1) acc = acc + tk;
  }
  return xv[4] + (w * (bI - acc)) * rI;
}

template <int T>
__device__ __forceinline__ void rs_up(const RsMg& M, const ResDev& Q, int wg, int t,
                                      int l, unsigned tag, volatile int* bad) {
  const MgLevel L = rs_level(M.lev, l), C = rs_level(M.lev, l + 1);
  unsigned long long* ew = glob(Q.ew) + L.off;
  const int I0 = rs_part(L.n, wg, Q.G), I1 = rs_part(L.n, wg + 1, Q.G);
  for (int I = I0 + t; I < I1; I += T)
    rs_put(ps_at(ew, I), tag, rs_up_cell(M, Q, L, C, I, tag, bad));
}

// ---------------------------------------------------------------------
// the coarse workgroup (mg_coarse_block with its data kept in LDS and
// registers over the solve)
//
// Every V-cycle waits for this workgroup, so what counts is the length of its
// chain.  A level takes one barrier down and one up: thread e has unknown
// e & 3 of aggregate e >> 2, and the aggregate's residuals are summed by
// shuffles.  Which unknown that is and which neighbours it has is worked out
// once per solve (a word per thread and level), the first level's stencil,
// diagonals and smoothed values stay in registers, and the pre-smoothed
// values of the levels below are formed from b by their readers.
// ---------------------------------------------------------------------
// unknown of level L (coarsened to C) of thread e, and its neighbours: bits 0-9
// and 10-18 (0 where the aggregate has no such unknown)
__device__ __forceinline__ int rs_co_info(const MgLevel& L, const MgLevel& C, int e) {
  const int J = e >> 2;
  if (J >= C.n) return 0;
  const int CJ = J / C.ny, CI = J - CJ * C.ny;
  const int ci = 2 * CI + (e & 1), cj = 2 * CJ + ((e >> 1) & 1);
  if (ci >= L.ny || cj >= L.nx) return 0;
  const int I = cj * L.ny + ci;
  int Nb[9], has = 0;
  mg_nbr9(L, ci, cj, I, Nb);
#pragma unroll
  for (int k = 0; k < 9; k++) has |= (Nb[k] >= 0) << k;
  return I | (has << 10);
}
// neighbour k of the unknown, itself in place of a missing one
__device__ __forceinline__ int rs_co_nbr(int info, int ny, int k) {
  const int I = info & 1023;
  return ((info >> (10 + k)) & 1) ? I + (k / 3 - 1) * ny + (k % 3 - 1) : I;
}
// the level-C unknown holding neighbour k, for thread e
__device__ __forceinline__ int rs_co_par(int info, int e, int cny, int k) {
  const int di = ((e & 1) + k % 3 - 1) >> 1, dj = (((e >> 1) & 1) + k / 3 - 1) >> 1;
  return ((info >> (10 + k)) & 1) ? (e >> 2) + dj * cny + di : e >> 2;
}
// x of the pre-smoothing sweep at the unknown and its neighbours
__device__ __forceinline__ void rs_co_x(int info, int ny, float w, const float* b,
                                        const float (&rd)[9], float (&x)[9], float& bI) {
  float bv[9];
#pragma unroll
  for (int k = 0; k < 9; k++) bv[k] = b[rs_co_nbr(info, ny, k)];
#pragma unroll
  for (int k = 0; k < 9; k++) x[k] = (w * bv[k]) * rd[k];
  bI = bv[4];
}
// residual of x, summed over the aggregate by its first thread
__device__ __forceinline__ float rs_co_down(int info, int t, const float (&st)[9],
                                            const float (&x)[9], float bI) {
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const float tk = st[k] * x[k];
    if ((info >> (10 + k)) & 1) acc = acc + tk;
  }
  const int in = (info >> 14) & 1;
  const float res = in ? bI - acc : 0.0f;
  const int base = t & 60;
  const float r1 = __shfl(res, base + 1, 64), r2 = __shfl(res, base + 2, 64),
              r3 = __shfl(res, base + 3, 64);
  const int i1 = __shfl(in, base + 1, 64), i2 = __shfl(in, base + 2, 64),
            i3 = __shfl(in, base + 3, 64);
  float s = 0.0f;
  if (in) s = s + res;
  if (i1) s = s + r1;
  if (i2) s = s + r2;
  if (i3) s = s + r3;
  return s;
}
// the unknown's value after the correction and the post-smoothing sweep
__device__ __forceinline__ float rs_co_up(int info, int e, int cny, float w, float c,
                                          const float* xc, const float (&st)[9],
                                          const float (&x)[9], float bI, float rI) {
  float xv[9];
#pragma unroll
  for (int k = 0; k < 9; k++) xv[k] = x[k] + c * xc[rs_co_par(info, e, cny, k)];
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const float tk = st[k] * xv[k];
    if ((info >> (10 + k)) & 1) acc = acc + tk;
  }
  return xv[4] + (w * (bI - acc)) * rI;
}

template <int T>
__device__ __forceinline__ void rs_coarse_solve(const Dev& D, const MgDev& M, const ResDev& Q,
                                                const MgLevel* lev,
                                                int iters, unsigned v0, unsigned ep,
                                                double* lds) {
  constexpr int PER = RS_PER(T);
  const int t0 = threadIdx.x;
  DevScalars* Sc = glob(D.sc);
  const int nblk = D.nblk, nl = M.nlev, l0 = Q.m + 1;
  const float w = M.w, c = M.cscale;
  double* col = lds;
  double* res = lds + 5 * 256;
  volatile int* bad = reinterpret_cast<int*>(res + 6);
  const MgLevel L0 = rs_level(lev, l0), LD = rs_level(lev, nl);
  const MgLevel C0 = rs_level(lev, l0 < nl ? l0 + 1 : nl);
  const int base = L0.off;
  const int S = LD.off + LD.n - base;
  const int stb = C0.off;
  const int nst = l0 < nl ? 9 * (LD.off - stb) : 0, nrd = nst / 9;
  const int nd8 = (LD.n + 7) & ~7;  // rows of the inverse, to a multiple of 8 with zeros
  double* DI = res + 8;
  float* Bv = reinterpret_cast<float*>(DI + nd8 * LD.n);  // S, and zeros after the last level
  float* R = Bv + S + 8;
  float* ST = R + S;
  float* RD = ST + nst;
  int* IN = reinterpret_cast<int*>(RD + nrd);
  const float* sten = glob(M.sten);
  const float* rdg = glob(M.rdg);
  const double* dinv = glob(M.dense_inv);
  if (t0 == 0) *bad = Q.G < Q.ended;
  if (t0 < 8) Bv[S + t0] = 0.0f;
  for (int e = t0; e < nd8 * LD.n; e += T) DI[e] = e < LD.n * LD.n ? dinv[e] : 0.0;
  for (int e = t0; e < nst; e += T) ST[e] = sten[9 * (size_t)stb + e];
  for (int e = t0; e < nrd; e += T) RD[e] = rdg[stb + e];
  {
    int* in = IN;
    for (int l = l0 + 1; l < nl; l++) {
      const MgLevel L = rs_level(lev, l), C = rs_level(lev, l + 1);
      for (int e = t0; e < 4 * C.n; e += T) in[e] = rs_co_info(L, C, e);
      in += 4 * C.n;
    }
  }
  float st0[PER][9], rd0[PER][9];
  int inf0[PER];
#pragma unroll
  for (int q = 0; q < PER; q++) {
    inf0[q] = l0 < nl ? rs_co_info(L0, C0, t0 + q * T) : 0;
    const float* sg = sten + 9 * (size_t)L0.off;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      st0[q][k] = sg[k * L0.n + (inf0[q] & 1023)];
      rd0[q][k] = rdg[base + rs_co_nbr(inf0[q], L0.ny, k)];
    }
  }
  const unsigned long long* bw = glob(Q.bw) + base;
  unsigned long long* ew = glob(Q.ew) + base;
  RsScalars z;
  z.rho = Sc->rho;
  z.iters = Sc->iters;
  z.conv = z.brk = z.done = 0;
  z.alpha = z.omega = z.beta = z.rr = z.rel = 0.0;
  const double bnorm = Sc->bnorm;
  const double frac = (D.P.inner_tol > 0.0) ? D.P.inner_tol : PB_STOP_FRAC;
  const double stop = frac * D.P.tol * bnorm;
  const int max_iter = D.P.max_iter;
  __syncthreads();
  for (int it = 0; it < iters; it++) {
#pragma unroll 1
    for (int half = 0; half < 2; half++) {
      const unsigned tag = v0 + 2 * it + half;
      // (opaque: or the compiler holds every address formed from these in
      // registers over the iterations)
      int t = threadIdx.x;
      asm volatile("" : "+v"(t));
#pragma unroll
      for (int q = 0; q < PER; q++) asm volatile("" : "+v"(inf0[q]));
      // right-hand side of the first level
      float x0[PER][9], b0[PER];
      if (l0 < nl) {
        rs_poll<PER>(tag, bad, [&](int q) {
          return (inf0[q] >> 14) & 1 ? ld_word(bw, inf0[q] & 1023)
                                     : (unsigned long long)tag << 32;
        }, b0);
#pragma unroll
        for (int q = 0; q < PER; q++)
          if ((inf0[q] >> 14) & 1) Bv[inf0[q] & 1023] = b0[q];
      } else if (t < LD.n) {
        Bv[t] = rs_wait(bw + t, tag, bad, 0ull);
      }
      __syncthreads();
      if (l0 < nl) {
        float* bc = Bv + (C0.off - base);
#pragma unroll
        for (int q = 0; q < PER; q++) {
          const int e = t + q * T;
          rs_co_x(inf0[q], L0.ny, w, Bv, rd0[q], x0[q], b0[q]);
          const float s = rs_co_down(inf0[q], t, st0[q], x0[q], b0[q]);
          if (!(e & 3) && (e >> 2) < C0.n) bc[e >> 2] = s;
        }
        __syncthreads();
      }
      const int* in = IN;
      for (int l = l0 + 1; l < nl; l++) {
        const MgLevel L = rs_level(lev, l), C = rs_level(lev, l + 1);
        const float* st = ST + 9 * (L.off - stb);
        float* bc = Bv + (C.off - base);
        for (int e = t; e < 4 * C.n; e += T) {
          const int info = in[e];
          float sv[9], rv[9], x[9], bI;
#pragma unroll
          for (int k = 0; k < 9; k++) {
            sv[k] = st[k * L.n + (info & 1023)];
            rv[k] = RD[L.off - stb + rs_co_nbr(info, L.ny, k)];
          }
          rs_co_x(info, L.ny, w, Bv + (L.off - base), rv, x, bI);
          const float s = rs_co_down(info, t, sv, x, bI);
          if (!(e & 3)) bc[e >> 2] = s;
        }
        in += 4 * C.n;
        __syncthreads();
      }
      if (t < LD.n) {
        // eight rows of the inverse requested before the last eight are used
        const float* b = Bv + (LD.off - base);
        const double* di = DI + t;
        double acc = 0.0, dv[8];
        float bv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          dv[u] = di[u * LD.n];
          bv[u] = b[u];
        }
        for (int J = 8; J < nd8; J += 8) {
          double dn[8];
          float bn[8];
#pragma unroll
          for (int u = 0; u < 8; u++) {
            dn[u] = di[(J + u) * LD.n];
            bn[u] = b[J + u];
          }
#pragma unroll
          for (int u = 0; u < 8; u++) {
            acc = acc + dv[u] * (double)bv[u];
            dv[u] = dn[u];
            bv[u] = bn[u];
          }
        }
#pragma unroll
        for (int u = 0; u < 8; u++) acc = acc + dv[u] * (double)bv[u];
        if (l0 == nl) rs_put(&ew[t], tag, (float)acc);
        R[LD.off - base + t] = (float)acc;
      }
      __syncthreads();
      for (int l = nl - 1; l > l0; l--) {
        const MgLevel L = rs_level(lev, l), C = rs_level(lev, l + 1);
        const float* st = ST + 9 * (L.off - stb);
        const float* xc = R + (C.off - base);
        float* out = R + (L.off - base);
        in -= 4 * C.n;
        for (int e = t; e < 4 * C.n; e += T) {
          const int info = in[e];
          if (!((info >> 14) & 1)) continue;
          float sv[9], rv[9], x[9], bI;
#pragma unroll
          for (int k = 0; k < 9; k++) {
            sv[k] = st[k * L.n + (info & 1023)];
            rv[k] = RD[L.off - stb + rs_co_nbr(info, L.ny, k)];
          }
          rs_co_x(info, L.ny, w, Bv + (L.off - base), rv, x, bI);
          out[info & 1023] = rs_co_up(info, e, C.ny, w, c, xc, sv, x, bI, rv[4]);
        }
        __syncthreads();
      }
      if (l0 < nl) {
        const float* xc = R + (C0.off - base);
#pragma unroll
        for (int q = 0; q < PER; q++)
          if ((inf0[q] >> 14) & 1)
            rs_put(&ew[inf0[q] & 1023], tag,
                   rs_co_up(inf0[q], t + q * T, C0.ny, w, c, xc, st0[q], x0[q], b0[q],
                            rd0[q][4]));
        __syncthreads();
      }
      if (half == 0) {
        double o[1];
        if (!rs_collect_send<T, 1>(Q, nblk, ep++, col, res, bad, o)) return;
        rs_alpha(z, o[0]);
        if (z.done) break;
      } else {
        double o[5];
        if (!rs_collect_send<T, 5>(Q, nblk, ep++, col, res, bad, o)) return;
        rs_omega(z, o, stop, bnorm, max_iter);
      }
    }
    if (z.done) break;
  }
  if (t0 == 0) {
    Sc->rho = z.rho;
    Sc->alpha = z.alpha;
    Sc->omega = z.omega;
    Sc->beta = z.beta;
    Sc->rr = z.rr;
    Sc->rel = z.rel;
    Sc->iters = z.iters;
    Sc->conv = z.conv;
    Sc->brk = z.brk;
    Sc->done = z.done;
  }
}

// ---------------------------------------------------------------------
// the row workgroups
// ---------------------------------------------------------------------
template <int T, int R>
__device__ __forceinline__ void rs_rows_solve(const Dev& D, const MgDev& M, const ResDev& Q,
                                              const MgLevel* lev,
                                              int wg, int iters, unsigned v0, unsigned ep,
                                              double* lds) {
  constexpr int S4 = T / 256, W = RS_W;
  const int t = threadIdx.x, l = t & 63;
  DevScalars* Sc = glob(D.sc);
  const int n = Sc->n, nblk = D.nblk, cap = D.cap;
  const int i0 = wg * Q.nbw * RED_BLOCK, i1 = min(n, min(nblk, (wg + 1) * Q.nbw) * RED_BLOCK);
  double* res = lds;
  volatile int* bad = reinterpret_cast<int*>(res + 6);
  double* area = res + 8;  // 5 S4 192 doubles, in the window's place
  float* X = reinterpret_cast<float*>(res + 8);  // the window
  float* r0s = X + W * T;                  // r0 of the workgroup's rows
  if (t == 0) *bad = wg < Q.ended;
  float* E1 = X + rs_work_words(T, R) + rs_lds_entries(T, R) * R * T;  // corrections of the window's cells
  unsigned long long* x0w = glob(Q.x0w);
  unsigned long long* phw = glob(Q.phw);
  unsigned long long* r0w = glob(Q.r0w);
  const MgLevel L1 = rs_level(lev, 1);
  unsigned long long* b1w = glob(Q.bw) + L1.off;
  const unsigned long long* e1w = glob(Q.ew) + L1.off;
  const RsMg H{lev, glob(M.sten), glob(M.rdg), M.w, M.cscale};
  const uint32_t* lidx = glob(D.aoff);
  const uint32_t* av16 = glob(D.av16);
  const double* aval = glob(D.aval);
  const int32_t* cstart = glob(D.cstart);
  const int32_t* cell = glob(D.cell);
  double* sol = glob(D.sol);
  const float mw = M.w, mc = M.cscale;
  // this thread's rows: local row q T + t
  const int32_t* wl = glob(Q.wlist) + (size_t)wg * RS_WCAP;
  const int wn = glob(Q.wcnt)[2 * wg], s0 = glob(Q.wcnt)[2 * wg + 1];
  int row[R], len[R], lmx[R];
  float p[R], rh[R], d0[R];
  double r[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int i = i0 + q * T + t;
    const bool in = i < i1;
    row[q] = in ? i : -1;
    len[q] = in ? glob(D.alen)[i] : 0;
    lmx[q] = wave_max(len[q]);
    p[q] = in ? glob(D.pp32)[i] : 0.0f;
    rh[q] = in ? glob(D.rh32)[i] : 0.0f;
    d0[q] = in ? glob(M.d0)[i] : 0.0f;
    r[q] = in ? glob(D.r)[i] : 0.0;
  }
  RsEntries<T, R> E[R];
#pragma unroll
  for (int q = 0; q < R; q++)
    E[q].load(lidx, av16, aval, cap, max(row[q], 0), len[q], t,
              reinterpret_cast<uint32_t*>(X) + rs_work_words(T, R) + q * E[0].KL * T);
  // window elements: chunk (uniform per wavefront), cell of the row; own
  // chunks hold the workgroup's rows at positions s0 * 64 + local row
  const int oc0 = i0 / PS_CHUNK, oc1 = (i1 + PS_CHUNK - 1) / PS_CHUNK;
  int wc[W], wk[W];
#pragma unroll
  for (int w = 0; w < W; w++) {
    const int s = w * (T / PS_CHUNK) + t / PS_CHUNK;
    wc[w] = __builtin_amdgcn_readfirstlane((s < wn) ? wl[s] : -1);
    const int g = wc[w] * PS_CHUNK + l;
    wk[w] = (wc[w] >= 0 && g < n) ? cell[g] : -1;
  }
  // One row per thread: the level-1 corrections of the window's cells are formed
  // here rather than by the cells' workgroups, which saves an exchange.  Thread
  // t has cells t, t + T, ... of the window's; a window element keeps its
  // cell's number (in wk).
  constexpr int NC = rs_cells(R);
  int uc[NC ? NC : 1];
  if constexpr (NC > 0) {
    static_assert(rs_number_words<T, W, NC>() <= rs_work_words(T, R), "no room in the window");
    __syncthreads();
    rs_number_cells<T, W, NC>(t, wk, uc, reinterpret_cast<int*>(X));
  }
  // cells whose first row is here, with the empty ones up to the next
  // workgroup's first; rows of a cell begun earlier are sent to its workgroup
  auto first_owned = [&](int i) {
    const int k = cell[i];
    return cstart[k] == i ? k : k + 1;
  };
  const int K0 = wg == 0 ? 0 : (i0 >= n ? L1.n : first_owned(i0));
  const int K1 = i1 >= n ? L1.n : first_owned(i1);
  int head = 0;
  if (i0 < n) {
    const int k = cell[i0];
    if (cstart[k] < i0) head = min(cstart[k + 1], i1) - i0;
  }
  const int tail = (K1 > K0 && i0 < i1 && i1 < n) ? cstart[K1] - i1 : 0;
  int ca0 = 0, ca1 = 0;  // local rows of this thread's first cell
  if (K0 + t < K1) {
    ca0 = cstart[K0 + t] - i0;
    ca1 = cstart[K0 + t + 1] - i0;
  }
  RsScalars z;
  z.rho = Sc->rho;
  z.iters = Sc->iters;
  z.conv = z.brk = z.done = 0;
  z.alpha = z.omega = z.beta = z.rr = z.rel = 0.0;
  const double bnorm = Sc->bnorm;
  const double frac = (D.P.inner_tol > 0.0) ? D.P.inner_tol : PB_STOP_FRAC;
  const double stop = frac * D.P.tol * bnorm;
  const int max_iter = D.P.max_iter;
  double t1[R];
  float ph[R], sh[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    t1[q] = 0.0;
    ph[q] = 0.0f;
  }
  __syncthreads();
  bool ok = true, pend = false;  // pend: the x update of the iteration before is to come
  for (int it = 0; it < iters && ok; it++) {
#pragma unroll 1
    for (int half = 0; half < 2; half++) {
      const unsigned tag = v0 + 2 * it + half;
      // (opaque: or the compiler holds every address formed from these in
      // registers over the iterations)
      int t = threadIdx.x;
      asm volatile("" : "+v"(t));
#pragma unroll
      for (int q = 0; q < R; q++) asm volatile("" : "+v"(row[q]));
#pragma unroll
      for (int w = 0; w < W; w++) asm volatile("" : "+v"(wk[w]));
#pragma unroll
      for (int j = 0; j < NC; j++) asm volatile("" : "+v"(uc[j]));
      const int l = t & 63;
      // ---- V-cycle of v = p (half 0) or s, which is in r (half 1)
      float v[R];
#pragma unroll
      for (int q = 0; q < R; q++) {
        v[q] = half ? (float)r[q] : p[q];
        if (row[q] >= 0) {
          const float x0 = (mw * v[q]) * d0[q];
          rs_put(ps_at(x0w, row[q]), tag, x0);
          X[s0 * PS_CHUNK + q * T + t] = x0;
        }
      }
      auto window = [&](const unsigned long long* words) {
        auto other = [&](int w) {
          return wc[w] >= 0 && (wc[w] < oc0 || wc[w] >= oc1) && wk[w] >= 0;
        };
        float e[W];
        rs_poll<W>(tag, bad, [&](int w) {
          return other(w) ? ld_word(words + (int64_t)wc[w] * PS_CHUNK, l)
                          : (unsigned long long)tag << 32;
        }, e);
#pragma unroll
        for (int w = 0; w < W; w++)
          if (other(w)) X[w * T + t] = e[w];
      };
      // x += alpha ph + omega sh of the iteration before, while x0 is on its
      // way (nothing of the iteration waits for it)
      double xs[R];
      if (pend) {
#pragma unroll
        for (int q = 0; q < R; q++)
          if (row[q] >= 0) xs[q] = *ps_at(sol, row[q]);
      }
      window(x0w);
      if (pend) {
#pragma unroll
        for (int q = 0; q < R; q++)
          if (row[q] >= 0)
            *ps_at(sol, row[q]) = (xs[q] + z.alpha * (double)ph[q]) + z.omega * (double)sh[q];
        pend = false;
      }
      __syncthreads();
      // r0 = v - A x0
#pragma unroll
      for (int q = 0; q < R; q++) {
        __builtin_amdgcn_sched_barrier(0);
        if (row[q] >= 0) {
          const float acc = rs_row_h<T, R>(E[q], lidx, av16, cap, row[q], t, len[q], lmx[q], X);
          const float r0 = v[q] - acc;
          r0s[q * T + t] = r0;
          if (q * T + t < head) rs_put(ps_at(r0w, row[q]), tag, r0);
        }
      }
      // the last cell's rows of the next workgroups follow this one's
      if (t < tail) r0s[i1 - i0 + t] = rs_wait(ps_at(r0w + i1, t), tag, bad, 0ull);
      __syncthreads();
      // restriction to level 1, a cell per thread, rows in order
      {
        int a0 = ca0, a1 = ca1;
        for (int K = K0 + t; K < K1; K += T) {
          if (K != K0 + t) {
            a0 = cstart[K] - i0;
            a1 = cstart[K + 1] - i0;
          }
          float s = 0.0f;
          for (int b0 = a0; b0 < a1; b0 += 8) {
            float u8[8];
#pragma unroll
            for (int u = 0; u < 8; u++) u8[u] = r0s[min(b0 + u, a1 - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++)
              if (b0 + u < a1) s = s + u8[u];
          }
          rs_put(ps_at(b1w, K), tag, s);
        }
      }
      for (int lv = 1; lv <= Q.m; lv++) rs_down<T>(H, Q, wg, t, lv, tag, bad);
      for (int lv = Q.m; lv > (NC ? 1 : 0); lv--) rs_up<T>(H, Q, wg, t, lv, tag, bad);
      // x1 = x0 + c e1 over the window
      if constexpr (NC > 0) {
        const MgLevel C1 = rs_level(lev, Q.m ? 2 : 1);
#pragma unroll
        for (int j = 0; j < NC; j++)
          if (uc[j] >= 0)
            E1[t + j * T] = Q.m ? rs_up_cell(H, Q, L1, C1, uc[j], tag, bad)
                                : rs_wait(ps_at(e1w, uc[j]), tag, bad, 0ull);
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; w++)
          if (wk[w] >= 0) X[w * T + t] = X[w * T + t] + mc * E1[wk[w]];
      } else {
        // one wavefront waits for the first corrections before the others read
        // theirs
        if (t < 64 && wk[0] >= 0) (void)rs_wait(ps_at(e1w, wk[0]), tag, bad, 0ull);
        __syncthreads();
        float e[W];
        rs_poll<W>(tag, bad, [&](int w) {
          return wk[w] >= 0 ? ld_word(e1w, wk[w]) : (unsigned long long)tag << 32;
        }, e);
#pragma unroll
        for (int w = 0; w < W; w++)
          if (wk[w] >= 0) X[w * T + t] = X[w * T + t] + mc * e[w];
      }
      __syncthreads();
      // x = x1 + w (v - A x1) d
      float y[R];
#pragma unroll
      for (int q = 0; q < R; q++) {
        __builtin_amdgcn_sched_barrier(0);
        y[q] = 0.0f;
        if (row[q] >= 0) {
          const float acc = rs_row_h<T, R>(E[q], lidx, av16, cap, row[q], t, len[q], lmx[q], X);
          y[q] = X[s0 * PS_CHUNK + q * T + t] + mw * (v[q] - acc) * d0[q];
          rs_put(ps_at(phw, row[q]), tag, y[q]);
        }
      }
      __syncthreads();  // the gathers of x1 are done
#pragma unroll
      for (int q = 0; q < R; q++)
        if (row[q] >= 0) X[s0 * PS_CHUNK + q * T + t] = y[q];
      window(phw);
      __syncthreads();
      // ---- the product, FP64
      double acc[R];
#pragma unroll
      for (int q = 0; q < R; q++) {
        __builtin_amdgcn_sched_barrier(0);
        acc[q] = (row[q] >= 0) ? rs_row_d<T, R>(E[q], lidx, aval, cap, row[q], t, len[q], lmx[q], X) : 0.0;
      }
      if (half == 0) {
        double o[1], pv[1][R];
#pragma unroll
        for (int q = 0; q < R; q++) {
          t1[q] = acc[q];
          ph[q] = y[q];
          pv[0][q] = (row[q] >= 0) ? acc[q] * (double)rh[q] : 0.0;
        }
        ok = rs_publish_wait<T, R, 1>(Q, wg, nblk, ep++, pv, area, res, bad, o);
        if (!ok) break;
        rs_alpha(z, o[0]);
        if (z.done) break;
        // s = r - alpha t1
#pragma unroll
        for (int q = 0; q < R; q++) r[q] = r[q] - z.alpha * t1[q];
      } else {
        double o[5], pv[5][R];
#pragma unroll
        for (int q = 0; q < R; q++) {
          const bool in = row[q] >= 0;
          const double sv = r[q], rd = (double)rh[q];
          sh[q] = y[q];
          pv[0][q] = in ? acc[q] * sv : 0.0;
          pv[1][q] = in ? acc[q] * acc[q] : 0.0;
          pv[2][q] = in ? acc[q] * rd : 0.0;
          pv[3][q] = in ? sv * rd : 0.0;
          pv[4][q] = in ? sv * sv : 0.0;
        }
        ok = rs_publish_wait<T, R, 5>(Q, wg, nblk, ep++, pv, area, res, bad, o);
        if (!ok) break;
        rs_omega(z, o, stop, bnorm, max_iter);
        if (z.done && !z.update) break;
        pend = true;
        // r = s - omega t2 ; p = r + beta (p - omega t1)
#pragma unroll
        for (int q = 0; q < R; q++)
          if (row[q] >= 0) {
            r[q] = r[q] - z.omega * acc[q];
            if (!z.done) p[q] = (float)(r[q] + z.beta * ((double)p[q] - z.omega * t1[q]));
          }
      }
    }
    if (z.done) break;
  }
  if (!ok) {
    if (t == 0) atomicOr(&Sc->counter[PS_FLAG_ABORT], 1u);
    return;
  }
#pragma unroll
  for (int q = 0; q < R; q++)
    if (row[q] >= 0) {
      if (pend) {
        double* xp = ps_at(sol, row[q]);
        *xp = (*xp + z.alpha * (double)ph[q]) + z.omega * (double)sh[q];
      }
      *ps_at(glob(D.r), row[q]) = r[q];
      *ps_at(glob(D.pp32), row[q]) = p[q];
    }
}

template <int T, int R>
__host__ __device__ inline int64_t rs_row_lds() {
  return 8 * 8 + 4 * (rs_work_words(T, R) + rs_lds_entries(T, R) * R * T + rs_cells(R) * T);
}
// whether the coarse workgroup can take level l0 and those below
__host__ __device__ inline bool rs_coarse_fits(const MgDev& G, int l0) {
  return l0 == G.nlev || (4 * G.lev[l0 + 1].n <= RS_CO_MAX && G.lev[l0].n <= 1024);
}
__host__ __device__ inline int64_t rs_coarse_lds(const MgDev& G, int l0) {
  int64_t v = 8, st = 0, in = 0;
  for (int l = l0; l <= G.nlev; l++) {
    v += 2 * (int64_t)G.lev[l].n;
    if (l > l0 && l < G.nlev) {
      st += 10 * (int64_t)G.lev[l].n;
      in += 4 * (int64_t)G.lev[l + 1].n;
    }
  }
  const int64_t nd = G.lev[G.nlev].n;
  return 8 * (5 * 256 + 8 + ((nd + 7) & ~7) * nd) + 4 * (v + st + in);
}

// up to `iters` iterations of every unfinished scenario
template <int T, int R>
__global__ void __launch_bounds__(T) kb_pb_resident(BatchDev B, const ResDev* rs, int iters,
                                                       unsigned v0, unsigned ep) {
  extern __shared__ double rs_lds[];
  const int s = rs_locate(rs, B.S, blockIdx.x);
  __shared__ MgLevel lev[MG_MAX_LEVELS];
  const ResDev Q = rs[s];  // copies: fields of a table in memory are read anew after every store
  const Dev& D = B.devs[s];
  const MgDev& M = B.mgs[s];
  const int wg = blockIdx.x - Q.wg0;
  if (threadIdx.x < MG_MAX_LEVELS) lev[threadIdx.x] = M.lev[threadIdx.x];
  __syncthreads();
  if (D.sc->done) return;  // every workgroup of the scenario
  if (wg == Q.G) rs_coarse_solve<T>(D, M, Q, lev, iters, v0, ep, rs_lds);
  else rs_rows_solve<T, R>(D, M, Q, lev, wg, iters, v0, ep, rs_lds);
}
