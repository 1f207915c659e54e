"""The kernels' LDS layouts (csrc/kdn_lds_layout.hpp) against their bank conflicts, counted on the host.

The layouts are constexpr index functions; a small host program asks them for the word of every lane of every access the
kernels make and counts, for the widths the hardware serves at once (4 bytes: half a wave over 32 banks; 16 bytes: 16
lanes over 64), the most distinct words that meet on one bank.  Each layout must also place its elements one to one.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kernel-deltanet_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <set>
#include "kdn_lds_layout.hpp"
using namespace kdn;

// The most distinct pieces on one bank over groups of `lanes` lanes: pieces of `width` words, `banks` banks of a word.
template <class F>
int ways(F word, int lanes, int width, int banks) {
  int worst = 0;
  for (int l0 = 0; l0 < 64; l0 += lanes) {
    std::set<int> seen[64];
    for (int l = l0; l < l0 + lanes; ++l) seen[word(l) / width % (banks / width)].insert(word(l));
    for (auto& s : seen) worst = (int)s.size() > worst ? (int)s.size() : worst;
  }
  return worst;
}
template <class F> int ways4(F f) { return ways(f, 32, 1, 32); }
template <class F> int ways16(F f) { return ways(f, 16, 4, 64); }
void up(int& worst, int v) { worst = v > worst ? v : worst; }

int main() {
  // the fp32 state kernel's K copy
  int rd = 0, wr = 0;
  std::set<int> kf;
  for (int half = 0; half < 2; ++half) {
    up(wr, ways16([&](int l) { return kf32_write(l, half); }));
    for (int e = 0; e < 4; ++e) up(rd, ways4([&](int l) { return kf32_read(l, e, half); }));
    for (int g = 0; g < 4; ++g)
      for (int e = 0; e < 4; ++e)
        for (int q = 0; q < 4; ++q)
          for (int i = 0; i < 4; ++i) {
            const int w = kf32_word(g, e, q, half) + i;
            if (w < 0 || w >= 512 || w != kf32_write(4 * g + e + 16 * q, half) + i || w != kf32_read(4 * q + i + 16 * g, e, half) ||
                w != ((kf32_word(g, e, q, 0) ^ (4 * half)) + i)) return 1;
            kf.insert(w);
          }
  }
  printf("kf32_places %d\nkf32_read %d\nkf32_write %d\n", (int)kf.size(), rd, wr);

  // A of the blocked inverse: rows over the lanes (prep_kernel's stores, the column walk's reads), columns over the
  // lanes with four rows each (prep8_kernel's stores), the substitution's reads
  int ar = 0, ac = 0, sub = 0;
  std::set<int> as;
  for (int i = 0; i < 4; ++i)
    for (int k = 0; k < 4; ++k) {
      up(ac, ways16([&](int l) { return a_word(16 * i + 4 * (l >> 4), 16 * k + (l & 15)); }));
      for (int e = 0; e < 4; ++e) {
        up(ar, ways4([&](int l) { return a_word(16 * i + (l & 15), 16 * k + 4 * (l >> 4) + e); }));
        if (k == i)
          for (int c = 4 * e; c < 4 * e + 4; ++c) up(sub, ways16([&](int l) { return a_word(16 * i + 4 * (l & 3), 16 * i + c); }));
      }
    }
  for (int r = 0; r < 64; ++r)
    for (int c = 0; c < 64; ++c) {
      const int w = a_word(r, c);
      if (w < 0 || w >= 4096 || w != a_word(r & ~3, c) + (r & 3) || a_word(r & ~3, c) % 4) return 1;
      as.insert(w);
    }
  printf("a_places %d\na_rows %d\na_cols %d\na_substitution %d\n", (int)as.size(), ar, ac, sub);

  // T: the substitution's stores (the block and the zeros to its right), the accumulator-layout accesses, 16-byte rows
  int td = 0, ta = 0, tr = 0;
  std::set<int> ts;
  auto t_word = [](int r, int c) { return r * 64 + t_swizzle(r, c); };
  for (int b = 0; b < 4; ++b)
    for (int k = 0; k < 4; ++k) {
      up(tr, ways16([&](int l) { return t_word(16 * b + (l & 15), 16 * k + 4 * (l >> 4)); }));
      for (int e = 0; e < 4; ++e) {
        up(ta, ways4([&](int l) { return t_word(16 * b + 4 * (l >> 4) + e, 16 * k + (l & 15)); }));
        if (k >= b)
          up(td, ways4([&](int l) { return t_word(16 * b + 4 * (l & 3) + e, 16 * k + (l >> 2)); }));
      }
    }
  for (int r = 0; r < 64; ++r)
    for (int c = 0; c < 64; ++c) {
      if (t_word(r, c) != t_word(r, c & ~3) + (c & 3)) return 1;
      ts.insert(t_word(r, c));
    }
  printf("t_places %d\nt_substitution %d\nt_tiles %d\nt_rows %d\n", (int)ts.size(), td, ta, tr);
  return 0;
}
"""


@pytest.fixture(scope="module")
def counts(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("lds")
    (d / "layouts.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "layouts"), str(d / "layouts.cpp")], check=True)
    out = subprocess.run([str(d / "layouts")], capture_output=True, text=True, check=True).stdout
    return {k: int(v) for k, v in (line.split() for line in out.splitlines())}


@pytest.mark.parametrize("access", ["kf32_read", "kf32_write", "a_rows", "a_cols", "a_substitution",
                                    "t_substitution", "t_tiles", "t_rows"])
def test_no_bank_conflicts(counts, access):
    assert counts[access] == 1


@pytest.mark.parametrize("layout,words", [("kf32_places", 512), ("a_places", 4096), ("t_places", 4096)])
def test_one_word_per_element(counts, layout, words):
    assert counts[layout] == words
