"""Host rules that pick a kernel's shape from the sizes of a call (csrc/dmla_rules.h), on the CPU.

The header is plain C++: a small driver compiled here answers questions about it, so the rules are
checked over many sizes against independent restatements, without a GPU."""
import heapq
import os
import random
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "ds-flashdmla-moe_amd", "csrc")
CXX = shutil.which("g++")
pytestmark = pytest.mark.skipif(CXX is None, reason="g++ is needed")

DRIVER = r"""
#include <cstdio>
#include <cstring>
#include "dmla_rules.h"
int main() {
  char what[16];
  while (std::scanf("%15s", what) == 1) {
    if (!std::strcmp(what, "otf")) {
      long cus, bh, sq, sk, causal;
      if (std::scanf("%ld %ld %ld %ld %ld", &cus, &bh, &sq, &sk, &causal) != 5) return 1;
      std::printf("%d", dmla::otf_rows((int)cus, bh, sq, sk, (int)causal));
      for (const auto& s : dmla::kOtfShapes)
        std::printf(" %.9g", dmla::otf_estimate_us(s, (int)cus, bh, sq, sk, (int)causal));
      std::printf("\n");
    } else {
      long cus, b, h, sq, sk, causal;
      if (std::scanf("%ld %ld %ld %ld %ld %ld", &cus, &b, &h, &sq, &sk, &causal) != 6) return 1;
      const dmla::PrefillSplit sp = dmla::prefill_split(cus, b, h, sq, sk, (int)causal);
      std::printf("%d %ld %ld", sp.n_layers, (long)sp.workgroups(), (long)sp.slots());
      for (int j = 0; j < sp.n_layers; ++j) std::printf(" %d", sp.first_rt[j]);
      for (int j = 0; j <= sp.n_layers; ++j) std::printf(" %d", sp.layer_base[j]);
      std::printf("\n");
    }
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src = d / "driver.cpp"
    src.write_text(DRIVER)
    run = subprocess.run([CXX, "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined",
                          "-fno-sanitize-recover=undefined", "-I" + CSRC, str(src), "-o", str(d / "driver")],
                         capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stderr[-2000:]

    def _ask(lines):
        r = subprocess.run([str(d / "driver")], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        return [line.split() for line in r.stdout.splitlines()]

    return _ask


def _otf(ask, sizes, cus=256):
    """(B * H, Sq, Sk, causal) -> (rows, {rows: estimate})"""
    out = ask([f"otf {cus} {bh} {sq} {sk} {int(c)}" for bh, sq, sk, c in sizes])
    return [(int(a[0]), dict(zip((512, 256, 128), map(float, a[1:])))) for a in out]


@pytest.mark.parametrize(
    "bh,sq,sk,causal,rows",
    [
        # Grids just past a multiple of the CU count, equally long workgroups: the shape that measured best.
        (32, 2100, 2100, False, 512),    # 160 workgroups; 288 of 256 rows would run two rounds
        (64, 1100, 1100, False, 512),
        (128, 600, 4000, True, 512),     # a chunk of a long context
        (16, 4313, 7385, False, 512),
        (24, 3639, 8036, False, 512),
        (160, 463, 463, False, 512),
        (144, 2028, 4254, True, 512),
        (96, 2048, 8056, True, 512),     # K and V past the last cache: more row tiles, more HBM traffic
        (32, 1100, 1100, False, 256),    # 160 workgroups; 288 of 128 rows would run two rounds
        (64, 513, 513, False, 256),
        # The listed sizes of the forward's measurements keep their shapes.
        (32, 500, 500, True, 128),
        (64, 4096, 4096, True, 512),
        (32, 777, 777, True, 128),
        (32, 2000, 2000, False, 256),
    ],
)
def test_otf_rows_count_whole_rounds(ask, bh, sq, sk, causal, rows):
    assert _otf(ask, [(bh, sq, sk, causal)])[0][0] == rows


# The sizes of test_otf_gpu.py::test_otf_row_tiles by the shape that runs them.
@pytest.mark.parametrize("rows,sizes", [
    (128, [(6, 257, 129, True), (64, 700, 700, True), (96, 513, 700, True), (2, 300, 357, False), (3, 130, 165, True)]),
    (256, [(2, 20, 20, True), (2, 129, 95, False), (512, 130, 130, True)]),
    (512, [(512, 257, 600, False), (512, 257, 257, True), (256, 300, 300, False), (512, 500, 1000, True)]),
])
def test_otf_test_sizes_reach_their_shape(ask, rows, sizes):
    assert [r for r, _ in _otf(ask, sizes)] == [rows] * len(sizes)


def test_otf_estimate_is_the_schedule(ask):
    """Up to eight workgroups per CU the estimate is the makespan of the row tiles in launch order on CUs
    that take the next workgroup when they are free; with equally long workgroups it is whole rounds at
    any size; it never falls below the mean load."""
    shapes = {512: (6.0, 2.75, 0.4), 256: (3.7, 1.7, 0.3), 128: (4.6, 1.25, 0.2)}
    rng = random.Random(3)
    sizes = []
    while len(sizes) < 300:
        bh, sq = rng.randint(8, 300), rng.randint(1, 6000)
        sk = sq if rng.random() < 0.5 else rng.randint(1, 8192)
        if bh * sk * 512 <= 256e6:   # past that the estimate counts HBM traffic too
            sizes.append((bh, sq, sk, rng.random() < 0.5))
    cus = 256
    for (bh, sq, sk, causal), (rows, est) in zip(sizes, _otf(ask, sizes, cus)):
        biased = {r: e * (0.95 if r == 512 else 1.0) for r, e in est.items()}
        assert biased[rows] == min(biased.values())
        for r, (fixed, tile, busy) in shapes.items():
            nq = -(-sq // r)
            n = nq * bh
            per_tile = tile + busy * min(1.0, n / cus)
            lens = []
            for qt in range(nq - 1, -1, -1):
                kend = min(sk, min(sq, (qt + 1) * r) + sk - sq) if causal else sk
                lens.append(fixed + per_tile * (-(-max(kend, 0) // 64)))
            if n <= 8 * cus:
                free = [0.0] * cus
                for w in lens:
                    for _ in range(bh):
                        heapq.heapreplace(free, free[0] + w)
                assert est[r] == pytest.approx(max(free), rel=1e-6), (bh, sq, sk, causal, r)
            elif not causal and n <= 64 * cus:
                assert est[r] == pytest.approx(-(-n // cus) * lens[0], rel=1e-6), (bh, sq, sk, causal, r)
            assert est[r] >= 0.98 * sum(lens) * bh / cus, (bh, sq, sk, causal, r)


def test_otf_rows_over_all_sizes_and_devices(ask):
    """Any size and CU count gives one of the three shapes (run under UBSan)."""
    sizes = [(1, 1, 0, True), (1, 1, 1, False), (1, 1 << 30, 1 << 30, True), (1 << 31, 1 << 30, 1 << 30, False),
             (1 << 31, 1, 1, True), (7, 300, 20, True), (1, 1 << 24, 5, True), (1024, 1, 1 << 30, False), (3, 40000, 40000, True)]
    for cus in (1, 32, 64, 256, 304, 1000):
        assert all(r in (128, 256, 512) for r, _ in _otf(ask, sizes, cus))


def test_prefill_split_layout_and_bound(ask):
    """Every part of a row tile with several parts has a slot of its own, row tiles with one part have
    none, and the workgroups (with them the workspace) are bounded by sixteen per CU."""
    rng = random.Random(4)
    sizes = [(5, 5, 2047, 137187, 1), (1, 1, 700, 700, 1), (1, 16, 512, 8192, 1), (16, 128, 3, 41, 1), (1, 8, 6148, 8182, 0)]
    while len(sizes) < 400:
        b, h, sq = rng.randint(1, 16), 1 << rng.randint(0, 7), int(2 ** rng.uniform(0, 13))
        sizes.append((b, h, sq, sq if rng.random() < 0.3 else int(2 ** rng.uniform(0, 18)), rng.randint(0, 1)))
    splits = ragged = 0
    for cus in (256, 64):
        out = ask([f"prefill {cus} {b} {h} {sq} {sk} {c}" for b, h, sq, sk, c in sizes])
        for (b, h, sq, sk, c), line in zip(sizes, out):
            n, wgs, slots, *rest = map(int, line)
            n_rt = -(-h * sq // 64)
            if n == 1:
                assert (wgs, slots) == (n_rt, 0)
                continue
            splits += 1
            first, base = rest[:n], rest[n:]
            assert wgs * b <= 16 * cus and first == sorted(first) and first[0] == 0 and base[0] == 0
            used = []
            for rt in range(n_rt):
                parts = sum(rt >= f for f in first)
                tiles = -(-(min(sk, (min((rt + 1) * 64, h * sq) - 1) // h + 1 + sk - sq) if c else sk) // 32)
                assert 1 <= parts <= max(tiles, 1)
                if parts > 1:
                    used += [base[j] - (first[1] if j else 0) + n_rt - 1 - rt for j in range(parts)]
                ragged += parts == 1
            assert sorted(used) == list(range(slots)), (b, h, sq, sk, c)
            assert wgs == slots + first[1]
    assert splits > 100 and ragged > 0
