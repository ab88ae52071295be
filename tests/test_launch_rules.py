"""The broad phase's grid leaves room for the simulations that may be stepped at once."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "lsdem2.0_amd" / "csrc"


def _blocks(tmp_path, cases):
    src = tmp_path / "rules.cpp"
    src.write_text('#include "launch_rules.h"\n#include <cstdio>\nint main() {\n'
                   + "".join(f'  std::printf("%d\\n", lsd::broadPhaseBlocks({n}ll, {c}ll, {cu}));\n' for n, c, cu in cases)
                   + "}\n")
    exe = tmp_path / "rules"
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]


def test_simulations_stepped_at_once_fit(tmp_path):
    at_once = [(32, n) for n in (1, 27, 511, 513, 1000, 3001, 4000, 4096)] + [(6, 20_000), (4, 32_000), (1, 200_000)]
    blocks = _blocks(tmp_path, [(n, n, 256) for _, n in at_once])
    for (count, n), b in zip(at_once, blocks):
        assert 8 <= b and count * b <= 256, f"{count} of {n} particles: {b} blocks each"  # (a CU holds one block)


def test_sparse_domains_and_small_gpus(tmp_path):
    assert _blocks(tmp_path, [(1000, 2_400_000, 256), (1000, 2_400_000, 64), (0, 1, 256), (10_000_000, 1, 256)]) == [147, 64, 8, 256]


def test_the_library_uses_the_rule():
    assert "c->coopBlocks = broadPhaseBlocks(nP, P.sg.ncell, c->numCU);" in (CSRC / "api.hip").read_text()


def test_masters_are_shared_once_and_evenly(tmp_path):
    src = tmp_path / "share.cpp"
    src.write_text(r'''
#include "launch_rules.h"
#include <cstdio>
#include <vector>
template <int GROUPS>
void run(int n, int blocks) {
  std::vector<int> seen(n, 0);
  int busy = 0, most = 0;
  for (int b = 0; b < blocks; ++b) {
    const lsd::MasterShare<GROUPS> s(n, blocks, b);
    std::vector<int> of(GROUPS, 0);
    for (int i = 0; i < s.chunk; ++i)
      if (s.at(i) < n) {
        ++seen[s.at(i)];
        ++of[i % GROUPS];
      }
    int top = 0, sum = 0;
    for (int v : of) { top = v > top ? v : top; sum += v; }
    busy += sum > 0;
    most = top > most ? top : most;
  }
  bool once = true;
  for (int v : seen) once = once && v == 1;
  std::printf("%d %d %d\n", once ? 1 : 0, blocks - busy, most);
}
int main() {
  for (int n : {1, 7, 8, 9, 31, 33, 1000, 4001}) {
    run<lsd::kFindThreads / lsd::kFindLanes>(n, lsd::pairsFindBlocks(n));  // separate launches
    run<32>(n, 8);                                                          // the single launch
  }
}
''')
    exe = tmp_path / "share"
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    rows = [tuple(map(int, r.split())) for r in
            subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()]
    assert all(once == 1 for once, _, _ in rows)
    assert all(idle == 0 and most == 1 for _, idle, most in rows[::2])  # every block busy, a master per group
