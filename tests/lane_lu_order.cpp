// Runs eliminate_by_lanes' four lanes one after another between its syncs, in
// every order of the lanes, and compares each result with a serial elimination:
// a phase whose outcome depends on which lane goes first lacks a sync.
#include <stdio.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <vector>

#include "../mole_amd/csrc/lane_lu.hpp"

namespace {

constexpr int kLanes = 4;
ucontext_t scheduler, lane_ctx[kLanes];
std::vector<char> stacks[kLanes];
bool finished[kLanes];
int syncs[kLanes];
std::function<void(int)> body;

void entry(int lane) {
  body(lane);
  finished[lane] = true;
}

// Every lane's body, a phase at a time, the lanes of a phase in `order`.
void run_lanes(const int *order) {
  for (int l = 0; l < kLanes; ++l) {
    stacks[l].resize(1 << 16);
    finished[l] = false;
    syncs[l] = 0;
    getcontext(&lane_ctx[l]);
    lane_ctx[l].uc_stack.ss_sp = stacks[l].data();
    lane_ctx[l].uc_stack.ss_size = stacks[l].size();
    lane_ctx[l].uc_link = &scheduler;
    makecontext(&lane_ctx[l], (void (*)())entry, 1, l);
  }
  while (!std::all_of(finished, finished + kLanes, [](bool f) { return f; }))
    for (int k = 0; k < kLanes; ++k)
      if (!finished[order[k]]) swapcontext(&scheduler, &lane_ctx[order[k]]);
}

void serial(double *A, double *y, int n) {
  for (int p = 0; p < n; ++p) {
    int piv = p;
    for (int r = p + 1; r < n; ++r)
      if (fabs(A[r * n + p]) > fabs(A[piv * n + p])) piv = r;
    if (piv != p) {
      for (int k = 0; k < n; ++k) std::swap(A[p * n + k], A[piv * n + k]);
      std::swap(y[p], y[piv]);
    }
    for (int r = p + 1; r < n; ++r) {
      const double f = A[r * n + p] / A[p * n + p];
      for (int k = p; k < n; ++k) A[r * n + k] = fma(-f, A[p * n + k], A[r * n + k]);
      y[r] = fma(-f, y[p], y[r]);
    }
  }
}

uint64_t rng = 1;
double uniform() {
  rng = rng * 6364136223846793005ull + 1442695040888963407ull;
  return (double)(int64_t)rng * 0x1p-63;
}

}  // namespace

int main() {
  int bad = 0, orders = 0;
  for (int n = 1; n <= 8; ++n)
    for (int steps : {n, 8})
      for (int rep = 0; rep < 4; ++rep) {
        std::vector<double> A0(n * n), y0(n);
        for (double &v : A0) v = uniform();
        for (int r = 0; r < n; ++r) y0[r] = r == rep % n ? 1.0 : 0.0;
        if (rep == 0)  // a swap in every column but the last
          for (int r = 0; r < n; ++r)
            for (int k = 0; k < n; ++k) A0[r * n + k] += (k == (r + n - 1) % n) ? 4.0 * n : 0.0;
        if (rep == 1 && n > 1) A0[0] = 0.0;
        std::vector<double> A1 = A0, y1 = y0;
        serial(A1.data(), y1.data(), n);
        int order[kLanes] = {0, 1, 2, 3};
        do {
          std::vector<double> A = A0, y = y0;
          body = [&](int lane) {
            mole::eliminate_by_lanes(A.data(), y.data(), n, steps, lane, [lane] {
              ++syncs[lane];
              swapcontext(&lane_ctx[lane], &scheduler);
            });
          };
          run_lanes(order);
          bool same = !memcmp(y.data(), y1.data(), sizeof(double) * n);
          for (int r = 0; r < n; ++r)
            for (int k = r; k < n; ++k) same = same && !memcmp(&A[r * n + k], &A1[r * n + k], sizeof(double));
          for (int l = 0; l < kLanes; ++l) same = same && syncs[l] == 3 * steps;
          if (!same && bad++ < 5)
            printf("n %d steps %d matrix %d lanes %d%d%d%d: not the serial elimination\n", n, steps, rep, order[0],
                   order[1], order[2], order[3]);
          ++orders;
        } while (std::next_permutation(order, order + kLanes));
      }
  printf("%d of %d orders differ\n", bad, orders);
  return bad != 0;
}
