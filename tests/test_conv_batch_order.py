"""Convolution batches whose requests of different bandwidths share memory.

The groups of a batch run as branches of one graph unless one writes memory
that another reads or writes; such a batch runs its groups one after another in
ascending bandwidth.  The rule is compared with a pairwise search on the CPU;
on the GPU batches with shared buffers match the plans' convolutions one after
another, bit for bit.
"""
import contextlib
import itertools
import os
import random
import subprocess

import pytest

from conftest import ROOT

DRIVER = """
#include <cstdio>
#include "s2_overlap.h"
int main() {
    int n;
    while (std::scanf("%d", &n) == 1) {
        std::vector<s2::MemRange> v(n);
        for (auto& r : v) {
            unsigned long lo, hi;
            int g, w;
            if (std::scanf("%lu %lu %d %d", &lo, &hi, &g, &w) != 4) return 1;
            r = {lo, hi, g, w != 0};
        }
        std::printf("%d\\n", (int)s2::groups_conflict(v));
    }
}
"""


def pairwise(ranges):
    return any(a[2] != b[2] and (a[3] or b[3]) and a[0] < b[1] and b[0] < a[1]
               for a, b in itertools.combinations(ranges, 2))


def test_groups_conflict_matches_a_pairwise_search(tmp_path):
    src, exe = tmp_path / "d.cc", tmp_path / "d"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "s2kit_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    rng = random.Random(1)
    sets = [[], [(0, 8, 0, 1), (8, 16, 1, 1)], [(0, 9, 0, 1), (8, 16, 1, 0)], [(0, 9, 0, 0), (8, 16, 1, 0)],
            [(0, 9, 0, 1), (8, 16, 0, 1)]]
    for _ in range(4000):
        n, span = rng.randint(1, 9), rng.choice([6, 20, 200])
        s = []
        for _ in range(n):
            lo = rng.randrange(span)
            s.append((lo, lo + rng.randint(1, 5), rng.randrange(rng.randint(1, 4)), int(rng.random() < 0.4)))
        sets.append(s)
    text = "\n".join(" ".join(str(x) for x in itertools.chain([len(s)], *s)) for s in sets)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split()
    want = [str(int(pairwise(s))) for s in sets]
    assert out == want and 0.1 < want.count("1") / len(want) < 0.9


@pytest.fixture(scope="module")
def env():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import s2kit_amd
    s2kit_amd.lib()
    return s2kit_amd, torch, torch.device("cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("shared", ["output_to_signal", "filter_overwritten", "outputs"])
@pytest.mark.parametrize("prec", [0, 2])
def test_shared_buffers_keep_the_order_of_bandwidths(env, shared, prec):
    S, torch, dev = env
    bws, F = (32, 48, 96), 3
    gen = torch.Generator(device=dev)
    gen.manual_seed(7 * len(shared) + prec)
    start = {bw: [torch.randn((F, 2 * bw, 2 * bw), generator=gen, dtype=torch.float64, device=dev) for _ in range(6)]
             for bw in bws}

    def buffers():
        t = {bw: [x.clone() for x in start[bw]] for bw in bws}
        lo, hi = bws[0], bws[2]
        if shared == "output_to_signal":  # the small group's real plane lies in the large group's signal
            t[lo][4] = t[hi][0].view(-1)[:F * 4 * lo * lo].view(F, 2 * lo, 2 * lo)
        elif shared == "filter_overwritten":  # the large group's real plane runs over the small group's filter
            t[lo][2] = t[hi][4].view(-1)[64:64 + F * 4 * lo * lo].view(F, 2 * lo, 2 * lo)
        else:  # both write the same memory
            t[lo][4] = t[hi][4].view(-1)[:F * 4 * lo * lo].view(F, 2 * lo, 2 * lo)
        return t

    got, want = buffers(), buffers()
    reqs = [(bw, *[x[f] for x in got[bw]]) for bw in reversed(bws) for f in range(F)]
    with contextlib.closing(S.ConvBatch(reqs, precision=prec)) as batch:
        plans = [(bw, S.Plan(bw, F, precision=prec)) for bw in bws]
        for _ in range(3):  # the shared planes change from replay to replay
            batch.run()
            for bw, p in plans:
                p.conv(*want[bw])
            torch.cuda.synchronize()
            for bw in bws:
                assert all(torch.equal(a, b) for a, b in zip(got[bw], want[bw])), (shared, bw)
        for _, p in plans:
            p.close()
