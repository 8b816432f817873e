"""Places of an element's nodes in the line stage's LDS slots, checked at compile time for every (P, Q) pair: every thread of an
element's points gets a place inside a slot, also where the element has fewer nodes than points; the nodes' places differ, and the
other threads' is none of them."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "honee-4aiad_amd", "csrc")

SOURCE = """
#include "basis3d.hpp"
template <int P, int Q, int NST>
constexpr bool places() {
  using L = basis3::LineStage<P, Q, 1, NST>;
  bool taken[L::Q3] = {};
  for (int t = 0; t < L::Q3; t++) {
    const int at = L::node(t);
    if (at < 0 || at >= L::Q3 || taken[at]) return false;
    if (t < P * P * P) taken[at] = true;
  }
  return true;
}
static_assert(places<%d, %d, 5>(), "places of nodes");
"""


@pytest.mark.parametrize("P,Q", [(2, 2), (2, 3), (2, 4), (3, 3), (3, 4), (3, 5), (4, 5), (4, 6), (5, 5), (5, 6)])
def test_places_of_nodes(P, Q, tmp_path):
    src = tmp_path / "places.hip"
    src.write_text(SOURCE % (P, Q))
    r = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
