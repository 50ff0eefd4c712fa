"""Which kernels a plan's calls run changes no result of the plan."""
import contextlib

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import s2kit_amd
    s2kit_amd.lib()
    return s2kit_amd, torch, torch.device("cuda:0")


def grids(torch, dev, bw, F, seed, planes=2):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    return [torch.randn((F, 2 * bw, 2 * bw), generator=gen, dtype=torch.float64, device=dev) for _ in range(planes)]


def pair(torch, plan, g, h, fmt):
    """Coefficients of the grids, and the grids of those coefficients."""
    F, n = g.shape[:2]
    a, b = (torch.empty((F, n * n // 4), dtype=torch.float64, device=g.device) for _ in range(2))
    x, y = torch.empty_like(g), torch.empty_like(g)
    plan.forward(g, h, a, b, data_format=fmt)
    plan.inverse(a, b, x, y, data_format=fmt)
    return a, b, x, y


@pytest.mark.parametrize("bw,F", [(257, 4), (257, 5), (257, 16), (300, 4), (320, 17), (321, 5), (321, 16), (400, 17),
                                  (511, 4), (512, 5)])
@pytest.mark.parametrize("fmt", [0, 1])
def test_results_do_not_depend_on_the_field_count(env, bw, F, fmt):
    # FP64 plans from bw = 257 to 512, at the field counts where calls change
    # kernels: the fields of a call have the same bits in calls of one, two and
    # three fields on the same plan, and after it was autotuned.
    S, torch, dev = env
    print(f"field counts bw={bw} F={F} fmt={fmt}", flush=True)
    g, h = grids(torch, dev, bw, F, bw + F)
    with contextlib.closing(S.Plan(bw, F)) as plan:
        whole = pair(torch, plan, g, h, fmt)
        for k in (1, 2, 3):
            for u, v in zip(pair(torch, plan, g[:k], h[:k], fmt), whole):
                assert torch.equal(u, v[:k]), k
        plan.autotune(F)
        for k in (F, 1):
            for u, v in zip(pair(torch, plan, g[:k], h[:k], fmt), whole):
                assert torch.equal(u, v[:k]), k


@pytest.mark.parametrize("bw", [321, 512])
def test_convolutions_do_not_depend_on_the_field_count(env, bw):
    S, torch, dev = env
    F = 5
    print(f"conv field counts bw={bw}", flush=True)
    t = grids(torch, dev, bw, F, bw, 4)
    a, b, x, y = (torch.empty_like(t[0]) for _ in range(4))
    with contextlib.closing(S.Plan(bw, F)) as plan:
        plan.conv(*t, a, b)
        for f in range(F):
            plan.conv(*[v[f:f + 1] for v in t], x[f:f + 1], y[f:f + 1])
    assert torch.equal(a, x) and torch.equal(b, y)


@pytest.mark.parametrize("bw,F,want", [
    (256, 8, {(32, 1)}), (256, 64, {(64, 1)}), (300, 16, {(64, 1)}), (512, 4, {(32, 1)}),  # K-chunked: one shape
    (512, 1, {(16, 1), (32, 1)}),  # K-chunked forward, direct inverse
    (64, 3, {(16, 1), (16, 2), (32, 1), (32, 2)}), (64, 80, {(16, 1), (16, 2), (32, 1), (32, 2)})])
def test_autotune_of_dense_plans(env, bw, F, want):
    # The choice reported is one that the call runs, and calls of every size
    # keep their bits.
    S, torch, dev = env
    print(f"autotune bw={bw} F={F}", flush=True)
    top = max(F, 4)
    g, h = grids(torch, dev, bw, top, bw + F)
    with contextlib.closing(S.Plan(bw, top)) as plan:
        before = {(k, fmt): pair(torch, plan, g[:k], h[:k], fmt) for k in {1, F, top} for fmt in (0, 1)}
        assert plan.tuning() == (0, 0, 0)
        plan.autotune(F)
        cols, tiles, rings = plan.tuning()
        assert (cols, tiles) in want and rings == 0
        for (k, fmt), outs in before.items():
            assert all(torch.equal(u, v) for u, v in zip(pair(torch, plan, g[:k], h[:k], fmt), outs)), (k, fmt)


@pytest.mark.parametrize("bw,F,prec,cutoff", [
    (8, 2, 0, 8), (8, 2, 0, 3), (11, 3, 0, 11), (64, 1, 0, 64), (64, 9, 0, 64), (100, 5, 0, 100), (131, 2, 0, 131),
    (128, 65, 0, 128), (512, 1, 0, 512), (512, 3, 0, 200), (600, 1, 0, 100), (600, 2, 0, 600), (128, 65, 1, 128),
    (64, 5, 1, 20), (32, 3, 2, 32), (100, 5, 2, 100), (131, 2, 2, 131), (128, 65, 2, 128), (64, 9, 3, 64)])
def test_real_calls_read_no_stale_row(env, bw, F, prec, cutoff):
    # REAL calls neither write nor read the order rows m >= bw of the
    # intermediate, in every ring FFT and Legendre instance: NaN left there by a
    # COMPLEX call does not reach them.
    S, torch, dev = env
    print(f"stale rows bw={bw} F={F} prec={prec} cutoff={cutoff}", flush=True)
    g, h = grids(torch, dev, bw, F, bw)
    bad = torch.full_like(g, float("nan"))
    out = []
    for poison in (False, True):
        with contextlib.closing(S.Plan(bw, F, precision=prec, cutoff=cutoff)) as plan:
            a, b = (torch.empty((F, bw * bw), dtype=torch.float64, device=dev) for _ in range(2))
            x, y = torch.empty_like(g), torch.empty_like(g)
            if poison:
                pair(torch, plan, bad, bad, 0)
            plan.forward(g, h, a, b, data_format=1)
            if poison:
                pair(torch, plan, bad, bad, 0)
            plan.inverse(a, b, x, y, data_format=1)
            out.append((a, b, x, y))
    for u, v in zip(*out):
        assert bool(torch.isfinite(v).all()) and torch.equal(u, v)


@pytest.mark.parametrize("bw,F,prec", [(64, 481, 2), (200, 129, 2), (255, 97, 2), (64, 481, 3), (128, 225, 3)])
def test_real_pair_workgroups_match_order_workgroups(env, bw, F, prec):
    # Mixed and split REAL calls on both sides of the line between workgroups of
    # one order (fewer than 512 order-pair workgroups) and of order pairs.
    S, torch, dev = env
    pairs = ((bw + 1) // 2 + 7) // 8 * 8

    def workgroups(n):  # of the forward; 64 data columns each, two per REAL field
        return pairs * -(-2 * n // 64)

    assert workgroups(F) >= 512 > workgroups(3)
    print(f"REAL pair workgroups bw={bw} F={F} prec={prec}", flush=True)
    g, h = grids(torch, dev, bw, F, bw + F)
    with contextlib.closing(S.Plan(bw, F, precision=prec)) as plan:
        whole = pair(torch, plan, g, h, 1)
        for f in (0, F - 3):
            for u, v in zip(pair(torch, plan, g[f:f + 3], h[f:f + 3], 1), whole):
                assert torch.equal(u, v[f:f + 3])


@pytest.mark.parametrize("bw,F,k,fmt", [
    (194, 9, 8, 1), (256, 9, 8, 1), (257, 5, 4, 0), (274, 5, 4, 0), (316, 5, 4, 0), (317, 5, 4, 0), (340, 9, 7, 1),
    (384, 9, 5, 1), (385, 5, 4, 0), (447, 9, 8, 1), (479, 5, 4, 0), (480, 5, 4, 0)])
def test_calls_of_one_column_tile(env, bw, F, k, fmt):
    # Calls of at most 16 data columns run the direct dense kernels where larger
    # ones run K-chunked (forward and inverse to lines of their own): the same bits.
    S, torch, dev = env
    print(f"one column tile bw={bw} F={F} k={k} fmt={fmt}", flush=True)
    g, h = grids(torch, dev, bw, F, bw)
    assert k * (2 if fmt else 4) <= 16 < F * (2 if fmt else 4)
    with contextlib.closing(S.Plan(bw, F)) as plan:
        whole = pair(torch, plan, g, h, fmt)
        for f in (0, F - k):
            for u, v in zip(pair(torch, plan, g[f:f + k], h[f:f + k], fmt), whole):
                assert torch.equal(u, v[f:f + k]), f


def test_zonal_needs_a_seminaive_order(env):
    S, torch, dev = env
    g, h = grids(torch, dev, 16, 2, 1)
    z = [torch.empty((2, 16), dtype=torch.float64, device=dev) for _ in range(2)]
    with contextlib.closing(S.Plan(16, 2, cutoff=0)) as plan:
        with pytest.raises(S.S2Error, match="cosine table"):
            plan.zonal(g, h, *z)
