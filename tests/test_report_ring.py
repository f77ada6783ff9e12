"""The ring of reports that launches leave in host memory (csrc/report_ring.h), host code only: order, reports that never
come, a full ring, slots used again.  Compiled with the host compiler and run here."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zk-deepseek_amd", "csrc")

SOURCE = r"""
#include "report_ring.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
typedef zk::ReportRing<int, 8, 4> Ring;
static unsigned long long storage[8 * 4];
struct Open { unsigned long long *at; unsigned seq; int parts; };
static Open send(Ring &r, int tag, int parts)
{
    Open o = { nullptr, 0, parts };
    o.at = r.open(&o.seq);
    if (o.at) r.push(tag, o.seq, parts);
    return o;
}
static void deliver(const Open &o, int parts)
{
    for (int i = 0; i < parts; i++) o.at[i] = (unsigned long long)o.seq << 32 | (unsigned)i;
}
int main()
{
    Ring r;
    unsigned none;
    CHECK(!r.open(&none));                              // no memory: no reports
    r.words = storage;
    std::vector<int> got;
    auto drain = [&]() { got.clear(); r.drain([&](int tag, const volatile unsigned long long *w, int parts) { CHECK((unsigned)w[parts - 1] == (unsigned)(parts - 1)); got.push_back(tag); }); };
    auto is = [&](std::vector<int> want) { return got == want; };
    // in order, and only whole ones
    Open a = send(r, 1, 2), b = send(r, 2, 4), c = send(r, 3, 1);
    drain(); CHECK(is({}));
    deliver(a, 1); drain(); CHECK(is({}));
    deliver(a, 2); deliver(b, 3); drain(); CHECK(is({ 1 }));
    deliver(b, 4); deliver(c, 1); drain(); CHECK(is({ 2, 3 }));
    // one that never comes does not hold up those behind it
    Open d = send(r, 4, 2), e = send(r, 5, 2), f = send(r, 6, 2);
    (void)d;
    drain(); CHECK(is({}));
    deliver(e, 2); drain(); CHECK(is({ 5 }));
    deliver(f, 2); drain(); CHECK(is({ 6 }));
    // several of them, the last of all missing for now
    Open g[4];
    for (int i = 0; i < 4; i++) g[i] = send(r, 10 + i, 1);
    deliver(g[2], 1); drain(); CHECK(is({ 12 }));
    deliver(g[3], 1); drain(); CHECK(is({ 13 }));
    // a full ring takes no more, and its slots come back
    for (int i = 0; i < 8; i++) { Open o = send(r, 20 + i, 1); CHECK(o.at); g[i & 3] = o; }
    CHECK(!send(r, 99, 1).at);
    deliver(g[3], 1); drain(); CHECK(is({ 27 }));
    for (int n = 0; n < 100; n++) { Open o = send(r, n, 3); CHECK(o.at); deliver(o, 3); drain(); CHECK(is({ n })); }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_report_ring(tmp_path):
    src, exe = tmp_path / "ring.cpp", tmp_path / "ring"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
