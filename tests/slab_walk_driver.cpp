// Host-side check of the bounded-load kernels' slab walk (walk_slabs and
// SlabOffsets in tensorforge_amd/csrc/staged_gemm.hpp), compiled with hipcc for the
// host only by tests/test_slab_walk.py.  A model of one workgroup: two register sets,
// two LDS buffers, A and B resources of the sizes the kernel gives them.  For every K
// (one row of A in the tile: the smallest resource), tile-k, split and window it
// checks that each load's scalar offset is below its resource's size, that slab t is
// computed from the bytes of slab t, and that each slab is computed once, in order.
#include <cstdio>

#include "staged_gemm.hpp"

struct Model {
  int nk, bk, ldb, k, kb, n0;  // kb: first k of this workgroup's range; n0: its first column
  int kt = 0, base = 0, loads = 0;
  long size_a = 0, size_b = 0;
  int reg_a[2] = {-1, -1}, reg_b[2] = {-1, -1}, lds_a[2] = {-1, -1}, lds_b[2] = {-1, -1};
  tfk::SlabOffsets at;
  bool ok = true;

  int a_step() const { return bk * 4; }
  int b_step() const { return bk * ldb * 4; }
  void rebase(int first) {
    const long rest = ((k - kb < nk * bk ? k - kb : nk * bk) - (long)first * bk) * ldb - n0;
    size_b = 4 * (rest > 0 ? rest : 0);
    base = first;
    at.rebase(first, nk, a_step(), b_step());
  }
  void load(int set) {
    // With nothing to load the resources are empty and the offsets zero.
    if (nk > 0 ? at.a < 0 || at.a >= size_a || at.b < 0 || at.b >= size_b : at.a != 0 || at.b != 0) ok = false;
    reg_a[set] = at.a / a_step();
    reg_b[set] = base + at.b / b_step();
    ++loads;
  }
  void store(int set) {
    lds_a[set] = reg_a[set];
    lds_b[set] = reg_b[set];
  }
  void compute(int t) {
    if (lds_a[t & 1] != t || lds_b[t & 1] != t) ok = false;
  }
  template <int P>
  void slab(int t, bool loading, bool storing) {
    if (storing) store(P ^ 1);
    if (loading) load(P ^ 1);
    compute(t);
    if (loading) at.next<P>(a_step(), b_step());
  }
  bool run(int window) {
    int done = 0;
    size_a = 4L * (k - kb);
    tfk::walk_slabs(
        nk, kt, [&]() { return window; }, [&](int first) { rebase(first); },
        [&](auto set) {
          load(decltype(set)::value);
          at.next<0>(a_step(), b_step());
        },
        [&]() { store(0); }, [&]() {},
        [&](int stop) {
          for (; kt < stop; kt += 2) {
            slab<0>(kt, true, true);
            slab<1>(kt + 1, true, true);
            done += 2;
          }
        },
        [&]() {
          slab<0>(kt, false, true);
          slab<1>(kt + 1, false, true);
          done += 2;
        },
        [&]() {
          slab<0>(kt, false, false);
          ++done;
        });
    return ok && done == nk;
  }
};

int main() {
  long cases = 0;
  for (int bk : {8, 16, 32, 64})
    for (int k = 0; k <= 24 * bk; k += (k < 4 * bk ? 1 : bk / 8))
      for (int splits = 1; splits <= 3; ++splits)
        for (int split = 0; split < splits; ++split)
          for (int n0 : {0, 64, 99}) {
            const int slabs = (k + bk - 1) / bk;
            if (splits > 1 && slabs < splits) continue;
            const int first = slabs * split / splits, nk = slabs * (split + 1) / splits - first;
            for (int window = 2; window <= nk + 2; window += 2) {
              Model m{nk, bk, 100, k, first * bk, n0};
              ++cases;
              if (!m.run(window < nk ? window : nk)) {
                std::printf("tile-k %d K %d split %d of %d column %d window %d: FAILED\n", bk, k, split, splits, n0, window);
                return 1;
              }
            }
          }
  // B past 2 GiB: the offsets of the last slab do not fit 31 bits until the last window.
  tfk::SlabOffsets o;
  o.rebase(0, 1000, 64, 1 << 28);
  if (o.last_b != 0x7fffffff || o.last_a != 999 * 64) return 1;
  o.rebase(997, 1000, 64, 1 << 28);
  if (o.last_b != 2 << 28) return 1;
  std::printf("%ld walks ok\n", cases);
  return 0;
}
