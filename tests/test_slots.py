"""The rule by which a context's optional device buffers grow (csrc/slots.h),
compiled for the host with an allocator that refuses sizes."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "slots.h"

static std::map<void*, size_t> live;
static size_t largest;  // an allocation past it is refused
static size_t unused = 1 << 20;
static int asked;

static void* get(size_t n) {
    ++asked;
    if (n > largest) return nullptr;
    void* p = malloc(1);
    live[p] = n;
    return p;
}
static void drop(void* p) {
    if (!live.count(p)) abort();
    live.erase(p);
    free(p);
}
static void grow(sl::Slots* s, size_t bytes, size_t least) { sl::grow(s, bytes, least, get, drop, [] { return unused; }); }
static void show(const sl::Slots& s) {
    if (s.p && live.at(s.p) != s.bytes) abort();
    printf("%zu %zu %d\n", s.bytes, live.size(), asked);
    asked = 0;
}

int main() {
    sl::Slots s;
    largest = 1000;
    grow(&s, 256, 64), show(s);    // given
    grow(&s, 200, 64), show(s);    // there already
    largest = 100;
    grow(&s, 4000, 2000), show(s);  // refused down to the least: the 256 stay
    grow(&s, 4000, 2000), show(s);  // not asked again
    sl::Slots t;
    largest = 600;
    grow(&t, 4000, 64), show(t);   // halved until given, beside s
    largest = 5000;
    grow(&t, 4000, 64), show(t);   // what was refused is not asked again
    sl::Slots u;
    grow(&u, 4000, 64), show(u);
    grow(&u, 5000, 64), show(u);   // replaced: the old one is released
    sl::Slots v;
    unused = 8000;
    grow(&v, 4000, 64), show(v);   // cut to an eighth of the free memory
    unused = 1 << 20;
    grow(&v, 4000, 64), show(v);   // and stays so
    sl::Slots w;
    unused = 8000;
    grow(&w, 4000, 2000), show(w);  // not asked for below the least
    largest = 300;
    void* a = sl::take(&u, 200, get, drop);  // given: u (5000) stays
    printf("%d %zu\n", a != nullptr, u.bytes);
    largest = 100;
    void* b = sl::take(&u, 200, [](size_t n) { if (live.size() < 5) largest = 200; return get(n); }, drop);
    printf("%d %zu\n", b != nullptr, u.bytes);  // refused at first: u is released
    void* c = sl::take(&u, 300, get, drop);
    printf("%d %zu\n", c != nullptr, u.bytes);  // nothing left to release
    char* buf = nullptr;
    size_t cap = 0;
    const auto alloc = [](char** p, size_t n) { return (*p = (char*)get(n)) ? 0 : -3; };
    const auto replace = [&](size_t n) {
        const int rc = sl::replace(&buf, &cap, n, alloc, [](char* p) { drop(p); });
        printf("%d %d %zu\n", rc, buf != nullptr, cap);
    };
    largest = 100;
    replace(50);
    replace(200);  // refused: no buffer, and none is said to be there
    replace(40);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_growth(tmp_path):
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "swiftlink_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
    assert [tuple(map(int, x.split())) for x in out.splitlines()] == [
        (256, 1, 1), (256, 1, 0), (256, 1, 2), (256, 1, 0), (500, 2, 4), (500, 2, 0), (4000, 3, 1), (5000, 3, 1),
        (1000, 4, 1), (1000, 4, 0), (0, 4, 0),
        (1, 5000), (1, 0), (0, 0),
        (0, 1, 50), (-3, 0, 0), (0, 1, 40)]
