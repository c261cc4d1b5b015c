"""The step down to a smaller workspace where the device has no room for one (error.h, host code):
only a failed allocation is answered with a smaller request, any other error reaches the caller."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]
SOURCE = r"""
#include <cstdio>
#include "symforce_amd/csrc/error.h"
using namespace symhip;
// reserve(m) throws `kind` while m > room; prints the sizes asked for and the outcome
static void run(int want, int room, const char* kind) {
  std::printf("%d %d %s:", want, room, kind);
  try {
    const int got = reserve_at_most(want, [&](int m) {
      std::printf(" %d", m);
      if (m <= room) return;
      if (kind[0] == 'm') throw OutOfMemory("memory");
      if (kind[0] == 'e') throw Error("device");
      throw 1;
    });
    std::printf(" = %d\n", got);
  } catch (const OutOfMemory&) { std::printf(" memory\n");
  } catch (const Error&) { std::printf(" error\n");
  } catch (int) { std::printf(" other\n"); }
}
int main() {
  for (const char* kind : {"memory", "error", "other"})
    for (int room : {0, 1, 5, 13}) run(13, room, kind);
  run(1, 0, "memory");
}
"""
WANT = """\
13 0 memory: 13 6 3 1 memory
13 1 memory: 13 6 3 1 = 1
13 5 memory: 13 6 3 = 3
13 13 memory: 13 = 13
13 0 error: 13 error
13 1 error: 13 error
13 5 error: 13 error
13 13 error: 13 = 13
13 0 other: 13 other
13 1 other: 13 other
13 5 other: 13 other
13 13 other: 13 = 13
1 0 memory: 1 memory
"""


def test_only_a_failed_allocation_asks_for_less(tmp_path):
    src = tmp_path / "reserve.cc"
    src.write_text(SOURCE)
    exe = tmp_path / "reserve"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(REPO), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert out == WANT
