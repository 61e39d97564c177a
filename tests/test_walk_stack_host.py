"""How deep a walk's stack gets that is spread to be handed on, finds no room and goes on (hand_spread,
WalkTree::deep_need): over the walk trees of deep meshes with every child reached, as next to a sphere's
centre, it stays within the capacity that the tree's mesh is given, which the full spread does not. And
which trees' walks can use up a budget (WalkTree::visits)."""
import os
import shutil
import subprocess

import pytest

from test_host_sanitizers import CSRC, DRIVER

MAIN = r"""
#include "walk_schedule.hpp"

#include <algorithm>

using Item = std::pair<uint32_t, uint32_t>; // (ref, cnt)

struct TreeWalk
{
  const WalkTree&   t;
  std::vector<Item> st; // the top last
  size_t            deepest = 0, visits = 0;

  void start(Item e) { st.assign(1, e); }
  void push_children(uint32_t node)
  {
    for (int k = 0; k < 4; k++)
      if (t.nodes[node].cnt[k] != kInvalid) st.push_back({t.nodes[node].ref[k], t.nodes[node].cnt[k] & (kBoxChild - 1u)});
    deepest = std::max(deepest, st.size());
  }
  void walk(uint32_t budget)
  {
    while (!st.empty() && budget--) {
      const Item e = st.back();
      st.pop_back();
      visits++;
      if (e.second == 0u) push_children(e.first);
    }
  }
  // as the device's spread_walk
  void spread(int s)
  {
    for (int i = 0; i < int(st.size()) && int(st.size()) < s; i++) {
      const Item e = st[i];
      if (e.second != 0u) continue;
      st[i] = st.back();
      st.pop_back();
      push_children(e.first);
    }
  }
};

// The deepest stack of walks from e that are out of budget, spread, and go on; and of those of the items
// they would have handed on.
static size_t deepest(const WalkTree& t, Item e, const int spread[2], int stage)
{
  size_t d = 0;
  for (uint32_t b : {1u, 2u, 15u, 40u, 60u, 150u, 151u, 152u, 153u, 1000u}) {
    TreeWalk w{t};
    w.start(e);
    w.walk(b);
    if (w.st.empty()) break;
    w.spread(spread[stage]);
    const auto items = w.st;
    w.walk(~0u);
    d = std::max(d, w.deepest);
    if (stage == 0)
      for (size_t i = 0; i < items.size(); i += 5) d = std::max(d, deepest(t, items[i], spread, 1));
  }
  return d;
}

int main()
{
  std::vector<float>    v;
  std::vector<uint32_t> f;
  icosphere(7, v, f);
  PseudoNormals pn;
  std::string   err;
  CHECK(compute_pseudo_normals(v.data(), v.size() / 3, f.data(), f.size() / 3, pn, err));
  size_t over = 0; // trees on which the full spread does not fit
  for (auto [K, leaf] : {std::pair{4, 1}, {4, 2}, {4, 16}, {8, 1}, {8, 4}}) {
    PackedMesh pm;
    CHECK(build_sah_mesh(v.data(), v.size() / 3, f.data(), f.size() / 3, K, leaf, pn, pm, err));
    WalkTree t;
    build_walk_tree(pm, 1.0f, t);
    const int    capacity = 64 * ((t.stack_need + 63) / 64);
    const int    spread[2] = {hand_spread(0, capacity, t.deep_need), hand_spread(1, capacity, t.deep_need)};
    const size_t d = deepest(t, {0u, 0u}, spread, 0), full = deepest(t, {0u, 0u}, kHandSpread, 0);
    std::printf("K=%d leaf=%d: stack_need %d deep_need %d spread %d %d: %zu (full spread %zu) of %d\n", K, leaf,
                t.stack_need, t.deep_need, spread[0], spread[1], d, full, capacity);
    CHECK(t.deep_need <= t.stack_need && spread[0] > 0);
    TreeWalk all{t};
    all.start({0u, 0u});
    all.walk(~0u);
    CHECK(all.visits == t.visits && all.deepest <= size_t(t.stack_need));
    CHECK(can_hand_on(t.visits, uint32_t(t.visits) - 1) && !can_hand_on(t.visits, uint32_t(t.visits)));
    CHECK(d <= size_t(capacity));
    over += full > size_t(capacity);
  }
  CHECK(over >= 2); // the trees are deep enough to tell
  CHECK(hand_spread(0, 64, 64) == 0 && hand_spread(0, 64, 1) == kHandSpread[0]);
  CHECK(hand_counts_fit(0xFFFFFFFFull) && !hand_counts_fit(0x100000000ull)); // 2^32 points in 64 instances
  std::printf("stack bound checked\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ absent")
def test_stack_of_handed_on_walks(tmp_path):
    src = tmp_path / "walks.cpp"
    src.write_text(DRIVER[:DRIVER.index("static void build_all")] + MAIN)
    exe = tmp_path / "walks"
    cmd = ["g++", "-std=c++17", "-O2", "-pthread", "-I" + CSRC, str(src), os.path.join(CSRC, "mesh_build.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, (run.stdout[-2000:], run.stderr[-4000:])
    assert "stack bound checked" in run.stdout
