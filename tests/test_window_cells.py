"""Numbering of the cells behind a resident workgroup's window (isph_cells.h),
run on the host: its text compiled with g++ over an emulation of a workgroup
whose lanes are coroutines.  A wavefront runs from one barrier to the next
while the others wait, in an order that each run chooses, so a wavefront that
gets far ahead of the others, or stays far behind, is an ordinary run here.  The
result may not depend on that order."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "beach-slope_amd" / "csrc"

EMULATOR = r"""
#include <ucontext.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline

constexpr int STACK = 32 * 1024;
enum Op { RUN, SHFL, BALLOT, BARRIER, END };
struct Lane {
  ucontext_t ctx;
  Op op = RUN;
  int in = 0;
  unsigned long long out = 0;
};
static std::vector<Lane> lanes;
static std::vector<char> stacks;
static ucontext_t scheduler;
static int cur;

static unsigned long long stop(Op op, int in) {
  Lane& me = lanes[cur];
  me.op = op;
  me.in = in;
  swapcontext(&me.ctx, &scheduler);
  return me.out;
}
static int __shfl_up(int v, int, int) { return (int)stop(SHFL, v); }
static unsigned long long __ballot(bool v) { return stop(BALLOT, v); }
static void __syncthreads() { stop(BARRIER, 0); }
static int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
static void atomicMax(int* p, int v) { *p = std::max(*p, v); }

#include SOURCE

constexpr int W = 6, NC = 2;
constexpr int GUARD = -1000000;
static std::vector<int> lds;
static int wk[1024][W], uc[1024][NC];

template <int T>
static void lane_main() {
  const int t = cur;
  int k[W], u[NC];
  for (int w = 0; w < W; w++) k[w] = wk[t][w];
  rs_number_cells<T, W, NC>(t, k, u, lds.data());
  for (int w = 0; w < W; w++) wk[t][w] = k[w];
  for (int j = 0; j < NC; j++) uc[t][j] = u[j];
  stop(END, 0);
}

// a wavefront up to its next barrier (or its end); its lanes meet at every
// wavefront operation
static void run_wave(int wave) {
  for (;;) {
    for (int l = 0; l < 64; l++) {
      cur = wave * 64 + l;
      swapcontext(&scheduler, &lanes[cur].ctx);
    }
    Lane* v = &lanes[wave * 64];
    unsigned long long mask = 0;
    for (int l = 0; l < 64; l++) {
      if (v[l].op != v[0].op) { std::puts("lanes of a wavefront diverged"); std::exit(1); }
      if (v[l].in) mask |= 1ull << l;
    }
    if (v[0].op == BARRIER || v[0].op == END) return;
    for (int l = 63; l >= 0; l--)
      v[l].out = v[0].op == BALLOT ? mask : (unsigned long long)(unsigned)v[l ? l - 1 : 0].in;
  }
}

template <int T>
static void run(std::vector<int> order, std::mt19937& rng, bool shuffled) {
  lanes.assign(T, Lane());
  stacks.resize((size_t)T * STACK);
  for (int t = 0; t < T; t++) {
    getcontext(&lanes[t].ctx);
    lanes[t].ctx.uc_stack.ss_sp = &stacks[(size_t)t * STACK];
    lanes[t].ctx.uc_stack.ss_size = STACK;
    lanes[t].ctx.uc_link = nullptr;
    makecontext(&lanes[t].ctx, lane_main<T>, 0);
  }
  for (bool end = false; !end;) {
    if (shuffled) std::shuffle(order.begin(), order.end(), rng);
    for (int wave : order) run_wave(wave);
    end = lanes[0].op == END;
    for (const Lane& l : lanes)
      if ((l.op == END) != end) { std::puts("a barrier not met by all"); std::exit(1); }
  }
}

template <int T>
static int check(unsigned seed) {
  std::mt19937 rng(seed);
  int bad = 0;
  for (int shape = 0; shape < 5; shape++) {
    // chunks of the window (the last one ragged), rows per cell
    const int chunks = shape == 0 ? W * T / 64 : shape == 1 ? W * T / 64 - 1 : shape == 2 ? 1
                     : shape == 3 ? 0 : 1 + (int)(rng() % (W * T / 64));
    const int rows = shape == 1 ? 3 * W * T : chunks * 64 - (chunks ? (int)(rng() % 63) : 0);
    int in[1024][W], want_wk[1024][W];
    std::vector<int> cells;
    int cell = 7;
    for (int s = 0; s < W * T / 64; s++)
      for (int l = 0; l < 64; l++) {
        const int e = s * 64 + l, t = e % T, w = e / T;
        in[t][w] = want_wk[t][w] = -1;
        if (s >= chunks || e >= rows) continue;
        if (l == 0) cell += 1 + (int)(rng() % 90);       // chunks need not be adjacent
        else if (rng() % 4 == 0) cell += 1 + (int)(rng() % 3);  // ~4 rows and up per cell
        in[t][w] = cell;
        if (l == 0 || cells.back() != cell) cells.push_back(cell);
        want_wk[t][w] = (int)cells.size() - 1;
      }
    if ((int)cells.size() > NC * T) { std::printf("%d cells\n", (int)cells.size()); return 1; }
    for (int way = 0; way < 5; way++) {
      std::vector<int> order(T / 64);
      for (int k = 0; k < T / 64; k++) order[k] = way == 1 ? T / 64 - 1 - k : k;
      std::copy(&in[0][0], &in[0][0] + 1024 * W, &wk[0][0]);
      lds.assign(rs_number_words<T, W, NC>() + 16, GUARD);
      run<T>(order, rng, way >= 2);
      for (size_t k = lds.size() - 16; k < lds.size(); k++) bad += lds[k] != GUARD;
      for (int t = 0; t < T; t++) {
        for (int w = 0; w < W; w++) bad += wk[t][w] != want_wk[t][w];
        for (int j = 0; j < NC; j++) {
          const int u = t + j * T;
          bad += uc[t][j] != (u < (int)cells.size() ? cells[u] : -1);
        }
      }
      if (bad) {
        std::printf("T %d, window %d, order %d: %d wrong\n", T, shape, way, bad);
        return 1;
      }
    }
  }
  return 0;
}

int main(int, char** argv) {
  const int T = std::atoi(argv[1]);
  for (unsigned seed = 1; seed <= 3; seed++)
    if (T == 512 ? check<512>(seed) : check<1024>(seed)) return 1;
  return 0;
}
"""


@pytest.fixture(scope="module")
def emulated(tmp_path_factory):
    d = tmp_path_factory.mktemp("cells")
    (d / "emu.cpp").write_text(EMULATOR)
    exe = d / "emu"
    subprocess.run(["g++", "-O1", "-std=c++17", f'-DSOURCE="{CSRC / "isph_cells.h"}"',
                    "-o", str(exe), str(d / "emu.cpp")], check=True, timeout=120)
    return exe


@pytest.mark.parametrize("threads", [512, 1024])
def test_numbers_do_not_depend_on_the_wavefronts_order(emulated, threads):
    r = subprocess.run([str(emulated), str(threads)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
