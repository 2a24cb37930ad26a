"""Index arithmetic of the tangent's storage (csrc/gf_index.h), compiled for the host,
against exact integers at sizes whose storage holds more entries than 32 bits count."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "giraffe_amd", "csrc")

_PAIR = r'''
#include <cstdint>
#include <cstdio>
#include "gf_index.h"
int main(int argc, char **argv)
{
    long long a[18];
    while (true) {
        for (int i = 0; i < 18; i++) if (scanf("%lld", a + i) != 1) return 0;
        gf_gmat g{};
        g.layout = (int)a[0]; g.m = (int)a[1]; g.hb = (int)a[4]; g.ld = (int)a[5];
        g.B = g.A + a[1] * a[2];
        g.C = g.B + a[1] * a[2];
        int R[6], C[6];
        for (int i = 0; i < 6; i++) { R[i] = (int)a[6 + i]; C[i] = (int)a[12 + i]; }
        size_t row[6]; unsigned step[36];
        gm_pair(g, R, C, row, step);
        for (int k = 0; k < 36; k++) printf("%llu ", (unsigned long long)(row[k / 6] + step[k]));
        printf("\n");
    }
}
'''


@pytest.fixture(scope="module")
def pair(tmp_path_factory):
    d = tmp_path_factory.mktemp("index")
    src, exe = d / "pair.cpp", d / "pair"
    src.write_text(_PAIR)
    subprocess.check_call(["g++", "-std=c++17", "-Wno-unknown-pragmas", "-I", CSRC, str(src), "-o", str(exe)])

    def run(layout, m, npad, hb, ld, R, C):
        line = " ".join(str(v) for v in [layout, m, npad, 0, hb, ld, *R, *C])
        out = subprocess.run([str(exe)], input=line, capture_output=True, text=True, check=True).stdout
        return [int(v) for v in out.split()]

    return run


def test_wide_band_rows(pair):
    """A plate of 172 x 172 elements with beams along it: 618,684 free DOFs, a half-band of
    3,623 entries and 1.04 x 2^32 entries in all; its first and last rows, and a node
    pair with constrained DOFs (only the free ones have an address of their own)."""
    nf, hb = 618684, 3623
    ld = 2 * hb
    assert nf * (ld + 1) > 2 ** 32
    for r0, c0 in ((0, 0), (0, hb - 5), (nf - 6, nf - 6), (nf - 6, nf - 6 - hb + 5), (nf - 1 - hb, nf - 6)):
        R, C = list(range(r0, r0 + 6)), list(range(c0, c0 + 6))
        assert pair(1, 0, 0, hb, ld, R, C) == [r * ld + c + hb for r in R for c in C]
    R, C = [nf - 6, -1, nf - 5, -1, -1, nf - 4], [-1, nf - 9, -1, nf - 8, nf - 7, -1]
    got = pair(1, 0, 0, hb, ld, R, C)
    for k in range(36):
        r, c = R[k // 6], C[k % 6]
        if r >= 0 and c >= 0:
            assert got[k] == r * ld + c + hb
        else:
            assert 0 <= got[k] < nf * (ld + 1)


@pytest.mark.parametrize("m,nf", [(6, 60), (16, 4096), (17, 12005), (32, 2 ** 24 - 32), (1, 12), (31, 31 * 541200)])
def test_block_rows(pair, m, nf):
    """The block-tridiagonal form up to its largest order: 2^24 rows of 32-row blocks,
    1.5 x 10^9 entries."""
    npad = -(-nf // m) * m
    n6 = min(6, m)
    for r0, c0 in ((0, 0), (0, n6), (nf - 6, nf - 6), (nf - 6, nf - 6 - n6), (nf // 2, nf // 2 + n6)):
        R, C = list(range(r0, r0 + 6)), list(range(c0, c0 + 6))
        got = pair(0, m, npad, 0, 0, R, C)
        for k in range(36):
            r, c = R[k // 6], C[k % 6]
            kind = 1 + (c // m > r // m) - (c // m < r // m)
            if abs(c // m - r // m) <= 1:
                assert got[k] == kind * npad * m + r * m + c % m


_FRONT = r'''
#include <cstdio>
#include "gf_index.h"
int main()
{
    int i, j, mp;
    while (scanf("%d %d %d", &i, &j, &mp) == 3) printf("%llu\n", (unsigned long long)(8 * gf_front_at(i, j, mp)));
}
'''


def test_front_entries(tmp_path):
    """Byte offsets of FP64 entries around 2^32 bytes (23,170 rows) and 2^32 entries."""
    src, exe = tmp_path / "front.cpp", tmp_path / "front"
    src.write_text(_FRONT)
    subprocess.check_call(["g++", "-std=c++17", "-Wno-unknown-pragmas", "-I", CSRC, str(src), "-o", str(exe)])
    cases = [(i, j, mp) for mp in (64, 23168, 23232, 25472, 65472, 65536, 70016) for i in (0, 63, mp // 2, mp - 1)
             for j in (0, mp - 1)]
    out = subprocess.run([str(exe)], input="\n".join("%d %d %d" % c for c in cases), capture_output=True, text=True,
                         check=True).stdout
    assert [int(v) for v in out.split()] == [8 * (i * mp + j) for i, j, mp in cases]
