"""The planners' memory (plan_memo.h): nested questions, as the workspace of a layer on padded channels
asks, and what is forgotten first."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "paralleltnnlayers_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include "plan_memo.h"
using Key = std::array<int, 1>;
cp4::PlanMemo<Key, int> memo;
int made = 0;
int ask(int k) { return memo.get(Key{k}, [&] { ++made; return 10 * k; }); }
#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }
int main() {
  for (int i = 0; i < 4; ++i) memo.answers[i] = -1, memo.keys[i] = Key{-7};   // (not what zeros would hide)
  // a question inside a question: both are remembered, and no slot counts that was never written
  CHECK(memo.get(Key{1}, [&] { ++made; return ask(2) + 1; }) == 21);
  CHECK(made == 2 && memo.used == 2);
  for (int i = 0; i < memo.used; ++i) CHECK(memo.keys[i] == Key{1} || memo.keys[i] == Key{2});
  CHECK(ask(1) == 21 && ask(2) == 20 && made == 2);
  // an answer that was given out does not change under its holder, whatever is asked then
  auto&& held = memo.get(Key{1}, [&] { return 0; });
  for (int k = 3; k < 9; ++k) CHECK(ask(k) == 10 * k);
  CHECK(held == 21);
  // the last four are kept
  made = 0;
  for (int k = 5; k < 9; ++k) CHECK(ask(k) == 10 * k);
  CHECK(made == 0 && ask(4) == 40 && made == 1);
  // nested at a full memory, three deep
  CHECK(memo.get(Key{20}, [&] { return memo.get(Key{21}, [&] { return ask(22) + 1; }) + 1; }) == 222);
  made = 0;
  CHECK(ask(20) == 222 && ask(21) == 221 && ask(22) == 220 && made == 0);
  return 0;
}
"""


def test_plan_memo(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no host compiler here")
    source, program = tmp_path / "memo.cpp", tmp_path / "memo"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(source), "-o", str(program)], check=True)
    r = subprocess.run([str(program)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
