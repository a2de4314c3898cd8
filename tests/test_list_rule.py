"""When a remeshed mesh's edge lists are stored (samoa_amd/csrc/swe_list_rule.hpp),
compiled for the host with g++: a run that remeshes too often for them never
stores any, one that remeshes rarely stores them at once, and no run pays more
for lists than their traversals save by more than one storing's cost."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <initializer_list>
#include "swe_list_rule.hpp"
using namespace swe;
static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL line %d: %s\n", __LINE__, #c); ++bad; } } while (0)
int main() {
    for (long cells : {1L, 1000L, (1L << 18) - 1, 1L << 18, 1L << 22, 1L << 29}) {
        const long pay = lists_break_even(cells);
        // calls of `per` steps each, `interval` steps between remeshings
        for (long interval = 1; interval <= 200; ++interval)
            for (long per : {1L, 2L, 3L, interval}) {
                if (interval % per) continue;
                long before = 0, balance = 0;  // in steps' savings: storing costs `pay`
                for (long mesh = 0; mesh < 6; ++mesh) {
                    long uses = 0, stored_at = -1;
                    for (; uses < interval; uses += per)
                        if (stored_at < 0 && lists_pay(cells, uses, per, before)) stored_at = uses;
                    if (interval < pay) CHECK(stored_at < 0);
                    if (interval >= pay && (mesh > 0 || per >= pay)) CHECK(stored_at == 0);
                    if (interval > 2 * pay) CHECK(stored_at >= 0);
                    if (stored_at >= 0) balance += (interval - stored_at) - pay;
                    CHECK(balance >= -pay);
                    before = interval;
                }
            }
        // a run in one call, from a graph's 48 steps on
        CHECK(lists_pay(cells, 0, 48, 0));
        // a mesh that came after a long one and is remeshed early pays once
        CHECK(lists_pay(cells, 0, 1, 1000));
        CHECK(!lists_pay(cells, 0, 1, 1));
    }
    std::printf(bad ? "BAD\n" : "OK\n");
    return bad != 0;
}
"""


def test_rule(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(DRIVER)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "samoa_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
