"""A staging slot whose event could not be recorded is not free before the work that
reads it is done."""
import os
import subprocess

import highuvlith_amd as H

HOST = os.path.join(os.path.dirname(os.path.abspath(H.__file__)), "csrc", "host")

MARKS = r"""
#include <initializer_list>
#include "slot_mark.hpp"
struct Slot { bool busy = false; };
int main() {
  for (bool recorded : {false, true}) {
    Slot s;
    int order = 0, at_record = 0, at_wait = 0;
    auto call = [&](bool fails) {
      const huvi::SlotMark mark(&s, [&] { at_record = ++order; return recorded; },
                                [&] { at_wait = ++order; });
      if (order) return 1;  // nothing before the call returns
      if (fails) return 2;
      return 3;
    };
    if (call(recorded) != (recorded ? 2 : 3)) return 1;
    if (at_record != 1 || at_wait != (recorded ? 0 : 2) || s.busy != recorded) return 2;
  }
  return 0;
}
"""


def test_marks(tmp_path):
    src, exe = tmp_path / "marks.cpp", tmp_path / "marks"
    src.write_text(MARKS)
    subprocess.run(["g++", "-std=c++17", "-I", HOST, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
