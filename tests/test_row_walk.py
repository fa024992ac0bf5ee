"""In-edge loops at the top of an edge type's range (2^32 - 2 edges): the
device headers' own functions, compiled for the host (CPU only)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# every row ends at `e`, up to 2^32 - 2, and has `d` in-edges; a loop that
# passes 2^32 is stopped after more rounds than the row can need. Reserved
# address space without memory stands in for the 17 GB of sources.
PROG = r"""
#include <stdio.h>
#include <stdlib.h>
#include <sys/mman.h>
#include "vh_common.h"

static void fail(const char* what, uint32_t b, uint32_t e) {
    printf("%s: row [%u, %u)\n", what, b, e);
    exit(1);
}
template <int STEP>
static void walk(uint32_t b, uint32_t e) {
    uint64_t rounds = 0, seen = 0;
    for (uint32_t k = b; k < e; k = vh_row_next(k, e, STEP)) {
        if (k < b || ++rounds > (uint64_t)(e - b) / STEP + 1) fail("walk", b, e);
        for (uint32_t q = 0; q < STEP; q++) seen += q < e - k ? 1 : 0;
    }
    if (seen != e - b) fail("walk: edges", b, e);
}
// the in-edges asked about: those whose own draw is below
static void any(uint32_t b, uint32_t e) {
    const uint64_t pre = vh_hash_pre(7, e, b), below[2] = {~0ull, vh_u01_below(0.3)};
    for (uint64_t pt : below) {
        bool want[128] = {}, got[128] = {};
        uint64_t calls = 0;
        for (uint32_t q = 0; q < e - b; q++) want[q] = (vh_hash_fin(pre, q + 1) >> 11) < pt;
        const bool none = vh_any_infecting(pre, pt, b, e, [&](uint32_t k) {
            if (k < b || k >= e || ++calls > 2ull * (e - b)) fail("any", b, e);
            got[k - b] = true;
            return false;
        });
        if (none || memcmp(want, got, sizeof want)) fail("any: in-edges", b, e);
        for (uint32_t q = 0; q < e - b; q++)
            if (vh_any_infecting(pre, pt, b, e, [&](uint32_t k) { return k - b == q; }) != want[q])
                fail("any: one infected", b, e);
    }
}
// lane l's in-edges of a row: every 64th from its own on, in order
static void lanes(uint32_t b, uint32_t e) {
    for (uint32_t l = 0; l < 64; l++) {
        uint64_t next = (uint64_t)b + l;
        auto one = [&](uint32_t k) {
            if (k != next || next >= e) fail("lane", b, e);
            next += 64;
        };
        vh_lane_edges(b, e, l, [&](uint32_t k) { for (uint32_t q = 0; q < 4; q++) one(k + 64 * q); }, one);
        if (next < e) fail("lane: ends early", b, e);
    }
}
int main() {
    const size_t bytes = (size_t)1 << 34;
    uint32_t* src = (uint32_t*)mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (src == MAP_FAILED) return 2;
    static DCtx c;
    static uint8_t states[8 * 512];
    c.a[1].rstate = states;
    c.a[1].nslots = 512;
    c.a[1].bytes = 8;
    c.a[1].readable = 1;
    c.e[0].src = src;
    c.e[0].src_type = 1;
    const uint64_t top = (1ull << 32) - 2;
    for (uint64_t k = top - 400; k < top; k++) src[k] = (uint32_t)(k % 512) + 1;
    const Neighbors nb(&c, 0);
    for (uint32_t gap = 0; gap < 40; gap += gap < 8 ? 1 : 5)
        for (uint32_t d = 0; d <= 100; d++) {
            const uint32_t e = (uint32_t)(top - gap), b = e - d;
            walk<4>(b, e);
            walk<8>(b, e);
            walk<16>(b, e);
            walk<32>(b, e);
            walk<64>(b, e);
            walk<256>(b, e);
            any(b, e);
            lanes(b, e);
            lanes(b - 5 * d, e);
            const uint8_t* p[8];
            for (uint32_t k = b; k < e; k = vh_row_next(k, e, 8)) {
                if (!nb.some(k, e, p)) fail("some", b, e);
                for (uint32_t q = 0; q < 8; q++) {
                    const uint64_t j = q < e - k ? (uint64_t)k + q : e - 1u;
                    if (p[q] != states + 8 * (j % 512)) fail("some: state", b, e);
                }
            }
        }
    // a row that takes the whole range, stepped over in large strides
    uint64_t rounds = 0;
    for (uint32_t k = 5; k < (uint32_t)top; k = vh_row_next(k, (uint32_t)top, 1u << 20)) rounds++;
    if (rounds != (top - 5 + (1 << 20) - 1) >> 20) fail("whole range", 5, (uint32_t)top);
    puts("ok");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("hipcc"):
        pytest.skip("no hipcc to compile the device headers with")
    d = tmp_path_factory.mktemp("row_walk")
    src = d / "row_walk.hip"
    src.write_text(PROG)
    exe = d / "row_walk"
    subprocess.run(["hipcc", "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-result",
                    "-I", os.path.join(ROOT, "vahana.jl_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe)], check=True)
    return str(exe)


def test_rows_up_to_the_last_edge(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert r.stdout == "ok\n"
