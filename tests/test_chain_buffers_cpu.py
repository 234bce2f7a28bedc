"""The buffers of whole chains in limited memory (csrc/chain_buffers.h, against
an allocator of a given capacity): whatever fits with the filtered projections
in the plain layout is accepted, for a plan and for a batch of several, and row
pairs are taken only where they leave what later calls need.  No buffer is held
that its owner does not know of.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "chain_buffers.h"
// capacity later refused-call (other pairs plain)... in bytes
int main(int argc, char** argv) {
  size_t cap = atoll(argv[1]), later = atoll(argv[2]), used = 0;
  int refuse = atoi(argv[3]), n = (argc - 4) / 3, calls = 0;
  void *other[8] = {}, *filt[8] = {};
  fct::Buffer o[8];
  fct::FilteredBuffer f[8];
  for (int j = 0; j < n; ++j) {
    o[j] = {&other[j], (size_t)atoll(argv[4 + 3 * j])};
    f[j] = {&filt[j], (size_t)atoll(argv[5 + 3 * j]), (size_t)atoll(argv[6 + 3 * j])};
  }
  std::map<void*, size_t> held;
  bool pairs = true;
  int e = fct::alloc_chain(
      o, n, f, n, &pairs,
      [&](void** at, size_t b) {
        *at = nullptr;
        if (used + b > cap || ++calls == refuse) return 2;
        used += b;
        *at = (void*)(size_t)(0x1000 + 16 * held.size() + calls * 4096);
        held[*at] = b;
        return 0;
      },
      [&](void* p) {
        if (!held.count(p)) abort();
        used -= held[p];
        held.erase(p);
      },
      [&] { return cap - used > later ? cap - used - later : (size_t)0; });
  size_t known = 0;
  for (int j = 0; j < n; ++j) {
    if (other[j]) known += held.at(other[j]);
    if (filt[j]) known += held.at(filt[j]);
  }
  printf("%d %d %zu %zu\n", e, (int)pairs, used, known);
}
"""


@pytest.fixture(scope="module")
def chain(tmp_path_factory):
    d = tmp_path_factory.mktemp("chain")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "freect_amd", "csrc"),
                    str(d / "t.cpp"), "-o", str(d / "t")], check=True)

    def run(capacity, later, jobs, refuse=0):
        args = [str(v) for v in (capacity, later, refuse, *sum(jobs, ()))]
        out = subprocess.run([str(d / "t"), *args], capture_output=True, text=True, check=True)
        e, pairs, used, known = map(int, out.stdout.split())
        assert used == known   # nothing is lost
        return e, pairs, used

    return run


FP32 = [(30, 200, 100), (50, 80, 40), (10, 400, 200)]   # others 90, pairs 680, plain 340
FP16 = [(30, 50, 100), (50, 20, 40), (10, 100, 200)]    # others 90, pairs 170, plain 340


@pytest.mark.parametrize("capacity,later,result",
                         [(770, 0, (0, 1, 770)), (769, 0, (0, 0, 430)), (430, 0, (0, 0, 430)),
                          (800, 31, (0, 0, 430)), (801, 31, (0, 1, 770)), (430, 500, (0, 0, 430)),
                          (429, 0, (2, 0, None))])
def test_fp32_batch(chain, capacity, later, result):
    e, pairs, used = chain(capacity, later, FP32)
    assert (e, pairs) == result[:2] and result[2] in (None, used)


@pytest.mark.parametrize("capacity,later", [(230, 0), (229, 0), (430, 1000)])
def test_one_plan(chain, capacity, later):
    e, pairs, used = chain(capacity, later, FP32[:1])
    assert (e, pairs, used) == ((0, 1, 230) if capacity - 30 - later >= 200 else (0, 0, 130))


def test_fp16_pairs_are_the_smaller_layout(chain):
    assert chain(260, 1000, FP16) == (0, 1, 260)
    assert chain(259, 0, FP16)[0] == 2


@pytest.mark.parametrize("refuse", [4, 5, 6])
def test_pairs_refused_with_room(chain, refuse):
    # (Fragmented memory: one of the pairs' allocations fails all the same.)
    assert chain(10000, 0, FP32, refuse) == (0, 0, 430)
