// isph_cells.h -- numbering of the cells behind a resident workgroup's window.
//
// Thread t of T holds the cells of window elements t, t + T, ... (wk; -1: no
// row).  A chunk is 64 consecutive elements, one wavefront's in one of the W
// rounds, and its rows lie in cell order: a cell begins at each element whose
// cell differs from the one before, and at a chunk's first row (a cell that
// spans two chunks has two numbers).  On return an element's wk is its cell's
// number, in window order, and uc holds the cells numbered t, t + T, ... (-1:
// none).  Nothing but wavefront operations and barriers, so the same text also
// runs on a host emulation of a workgroup.
#pragma once

// words of LDS: the numbers' end, cells begun per chunk, the cells
template <int T, int W, int NC>
constexpr int rs_number_words() { return 1 + W * T / 64 + NC * T; }

template <int T, int W, int NC>
__device__ __forceinline__ void rs_number_cells(int t, int (&wk)[W], int (&uc)[NC], int* lds) {
  const int l = t & 63;
  // (the end has a word of its own: a wavefront that is through with the counts
  // must not write over them while another still sums them)
  int *end = lds, *begun = end + 1, *list = begun + W * T / 64;
  bool first[W];
  if (t == 0) *end = 0;
#pragma unroll
  for (int w = 0; w < W; w++) {
    const int before = __shfl_up(wk[w], 1, 64);
    first[w] = wk[w] >= 0 && (l == 0 || before != wk[w]);
    const unsigned long long m = __ballot(first[w]);
    if (l == 0) begun[w * (T / 64) + t / 64] = (int)__popcll(m);
  }
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int w = 0; w < W; w++) {
    const int s = w * (T / 64) + t / 64;
    int base = 0;
    for (int k = 0; k < s; k++) base += begun[k];
    const unsigned long long m = __ballot(first[w]);
    const int u = base + (int)__popcll(m & (~0ull >> (63 - l))) - 1;
    if (first[w]) list[u] = wk[w];
    if (wk[w] >= 0) {
      wk[w] = u;
      total = u + 1;
    }
  }
  atomicMax(end, total);
  __syncthreads();
  total = *end;
#pragma unroll
  for (int j = 0; j < NC; j++) uc[j] = (t + j * T < total) ? list[t + j * T] : -1;
  __syncthreads();
}
