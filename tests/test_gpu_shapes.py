"""The sizes at which the kernels' shapes change: the slabs of the small all-pairs
evaluation, four-wave M2L blocks with idle waves, and evaluations that follow
others on one context (which write their arrays instead of clearing them).

Tolerances (FP64): the all-pairs sums differ from the reference sum in their
order only, n terms of relative round-off 2^-53 each against the sum of their
magnitudes; the FMM against the oracle as in test_gpu_parity."""
import numpy as np
import pytest

from conftest import relerr_vec

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _flags(n, seed, sinks, sources):
    rng = np.random.default_rng(seed)
    return ((rng.random(n) < sinks) | ((rng.random(n) < sources).astype(np.uint8) << 1)
            ).astype(np.uint8)


def _eval(torch, f, x, v, m, flags=None):
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, v, m)]
    fl = None if flags is None else torch.from_numpy(flags).cuda()
    out = f.eval(*d, flags=fl)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in out]


def _direct(x, v, m, flags):
    """Sums and sums of magnitudes over all pairs, one target at a time."""
    n = m.size
    q = m * ((flags >> 1) & 1)
    out, mag = [], []
    for a in (np.zeros(n), np.zeros((n, 3)), np.zeros((n, 3))):
        out.append(a)
        mag.append(np.zeros(n))
    for i in range(n):
        if not flags[i] & 1:
            continue
        d, w = x - x[i], v - v[i]
        r2 = (d * d).sum(1)
        ri = np.where(r2 > 0, 1.0 / np.sqrt(np.where(r2 > 0, r2, 1.0)), 0.0)
        f = q * ri ** 3
        k = 3.0 * f * (d * w).sum(1) * ri * ri
        out[0][i], mag[0][i] = (q * ri).sum(), (q * ri).sum()
        out[1][i], mag[1][i] = (f[:, None] * d).sum(0), (f * np.sqrt(r2)).sum()
        out[2][i] = (f[:, None] * w - k[:, None] * d).sum(0)
        mag[2][i] = (f * np.linalg.norm(w, axis=1) + np.abs(k) * np.sqrt(r2)).sum()
    return out, mag


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 255, 256, 257, 1009, 8192, 8193])
@pytest.mark.parametrize("masked", [False, True])
def test_gpu_small_direct_slabs(torch_cuda, n, masked):
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    x, v, m = ics.plummer(n, seed=n)
    if n > 2:
        x[n // 2] = x[0]  # a coincident pair does not interact
    flags = _flags(n, n, 0.7, 0.8) if masked else np.full(n, 3, np.uint8)
    got = _eval(torch_cuda, tca.Fmm(p=4, direct_below=10 ** 6), x, v, m,
                flags if masked else None)
    want, mag = _direct(x, v, m, flags)
    # a pair's own term: some ten roundings; then n additions of partial sums
    tol = (10 + n) * 2.0 ** -53
    for g, w, a in zip(got, want, mag):
        err = np.abs(g - w) if g.ndim == 1 else np.linalg.norm(g - w, axis=1)
        assert np.all(err <= 4 * tol * a), float(np.max(err / np.maximum(a, 1e-300)))


@pytest.mark.parametrize("p", [13, 14, 15, 19, 20])
def test_gpu_m2l_blocks_with_idle_waves(torch_cuda, oracle_lib, p):
    """One body in forty takes a force: most targets have no sink, so the
    four-wave blocks of orders 14 and up hold waves that write nothing, and the
    last block is not full."""
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    n, u = 4001, [0.2, -0.3, 0.1]
    x, v, m = ics.plummer(n, seed=p)
    flags = _flags(n, p, 0.025, 0.9)
    f = tca.Fmm(p=p, ncrit=32, theta=0.6, direct_below=0)
    f.set_shift(u)
    gp, ga, gj = _eval(torch_cuda, f, x, v, m, flags)
    o = oracle_lib.Oracle(p, ncrit=32, theta=0.6, shift_frac=u)
    op, oa, oj, _ = o.eval(x, v, m, issink=flags & 1, issource=(flags >> 1) & 1)
    on = (flags & 1) == 1
    assert relerr_vec(ga[on], oa[on])[1] < 1e-10
    assert relerr_vec(gj[on], oj[on])[1] < 1e-9
    assert not gp[~on].any() and not ga[~on].any() and not gj[~on].any()


@pytest.mark.parametrize("mac", [0, 1])
def test_gpu_nothing_left_from_the_evaluation_before(torch_cuda, mac):
    """A context's second evaluation (fewer bodies, other masks) equals a fresh
    context's: the rows, results and flags that it does not clear are written."""
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics

    def ctx():
        f = tca.Fmm(p=6, ncrit=24, theta=0.5, mac=mac, direct_below=0)
        f.set_shift([0.1, 0.2, -0.3])
        return f

    f = ctx()
    _eval(torch_cuda, f, *ics.plummer(20000, seed=1))
    x, v, m = ics.dehnen(9001, seed=2)
    flags = _flags(9001, 3, 0.3, 0.6)
    again, fresh = _eval(torch_cuda, f, x, v, m, flags), _eval(torch_cuda, ctx(), x, v, m, flags)
    # the same lists and sums; the atomics' order is the only difference
    for g, w in zip(again, fresh):
        assert np.max(np.abs(g - w)) <= 1e-12 * np.max(np.abs(w))


@pytest.mark.parametrize("ncand", [1, 2, 5, 21, 33, 64])
def test_gpu_leaf_choice(torch_cuda, ncand):
    """A wave holds 64, 32, 12, 3, 1 and 1 leaves: every leaf gets the cheapest
    candidate predicted to meet the target, and where none does the most accurate
    one."""
    import mlp_oracle as mo
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    rng = np.random.default_rng(ncand)
    P = (mo.init_params(1) + rng.normal(scale=0.05, size=mo.NPARAM)).astype(np.float32)
    q = rng.integers(2, 7, ncand)
    theta = np.linspace(0.3, 0.9, ncand).astype(np.float32)
    cost = rng.permutation(ncand).astype(np.float32) + 1

    def run(target):
        f = tca.Fmm(p=6, ncrit=16, theta=0.5, direct_below=0)
        f.set_shift([0.1, 0.2, -0.3])
        f.set_order_model(P, q, theta, cost, [-10] * 9, [10] * 9, target)
        f.set_adaptive(2)
        _eval(torch_cuda, f, *ics.plummer(3001, seed=7))
        feat, _, pred = f.leaf_data()
        return feat.cpu().numpy().clip(-10, 10), pred.cpu().numpy()

    feat, _ = run(1.0)
    nl = len(feat)
    X = np.empty((nl, ncand, mo.NIN))
    X[..., :9] = feat[:, None]
    X[..., 9] = q / 20.0
    X[..., 10] = theta
    y = mo.forward(P.astype(np.float64), X.reshape(-1, mo.NIN)).reshape(nl, ncand)
    tol = 1e-4 * max(1.0, np.max(np.abs(y)))  # the network's, as for its own kernel
    for level in (y.min() - 1, np.median(y), y.max() + 1):
        _, pred = run(10.0 ** level)
        met = y <= level
        choice = np.where(met.any(1), np.where(met, cost, np.inf).argmin(1), y.argmin(1))
        want = y[np.arange(nl), choice]
        clear = np.all(np.abs(y - level) > 2 * tol, axis=1)
        assert clear.sum() >= nl // 4
        # (another of almost the same error may be taken: its prediction is as good)
        assert np.all(np.abs(pred - want)[clear] <= tol)


def test_gpu_leaf_calls_need_the_last_evaluations_tree(torch_cuda):
    """After an evaluation without a tree (all pairs) or with another one (the
    master sum's), the leaf calls and the tuner refuse: the leaves of the tree
    before it index bodies that the smaller system does not have."""
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    torch = torch_cuda
    f = tca.Fmm(p=4, ncrit=32, theta=0.6, direct_below=1000)
    f.set_adaptive(1, 4, 0.6)
    big, small = ics.plummer(5000, seed=3), ics.plummer(300, seed=4)

    def refused(n):
        a = torch.ones(n, 3, dtype=torch.float64, device="cuda")
        for call in (f.leaf_data, lambda: f.leaf_errors(a, a), f.tune_p2p):
            with pytest.raises(RuntimeError):
                call()

    def tree():  # (the master sum takes the shift back to zero)
        f.set_shift([0.1, 0.2, -0.3])
        _eval(torch, f, *big)

    tree()
    feat, lob, _ = f.leaf_data()
    assert feat.shape[0] == f.stats()["nleaves"] and int(lob.max()) == feat.shape[0] - 1
    _eval(torch, f, *small)
    refused(300)
    tree()
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in small]
    f.master_eval(*d, get_steps=True)
    refused(300)
    tree()
    assert f.leaf_errors(*[torch.ones(5000, 3, dtype=torch.float64, device="cuda")] * 2).shape
    assert torch.equal(f.leaf_data()[1], lob)


@pytest.mark.parametrize("p", [13, 14])
def test_gpu_l2l_beside_a_long_p2p(torch_cuda, oracle_lib, p):
    """Beside a long P2P list L2L takes one wave per child up to order 13 and
    512 threads above."""
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    n, u = 9001, [0.2, -0.3, 0.1]
    x, v, m = ics.plummer(n, seed=p)
    f = tca.Fmm(p=p, ncrit=5, theta=0.28, direct_below=0)
    f.set_shift(u)
    _, ga, gj = _eval(torch_cuda, f, x, v, m)
    assert f.stats()["n_p2p_cells"] > 1 << 18
    o = oracle_lib.Oracle(p, ncrit=5, theta=0.28, shift_frac=u)
    _, oa, oj, _ = o.eval(x, v, m)
    assert relerr_vec(ga, oa)[1] < 1e-10 and relerr_vec(gj, oj)[1] < 1e-9


@pytest.mark.parametrize("n,ncrit,theta", [(4096, 1, 0.3), (5000, 2, 0.3), (4097, 3, 0.3)])
def test_gpu_levels_and_steps_of_many_tiles(torch_cuda, oracle_lib, n, ncrit, theta):
    """Levels of more cells than the launch's blocks hold at once (64 each, n / 512
    but at least 8 blocks) and walk steps of several rounds per block (256 pairs a
    round, n / 32 but at least 64 blocks): the oracle's tree and lists."""
    import taichi_collisional_amd as tca
    u = [0.2, -0.3, 0.1]
    rng = np.random.default_rng(n)
    x, v, m = rng.random((n, 3)), rng.normal(size=(n, 3)), np.full(n, 1.0 / n)
    f = tca.Fmm(p=6, ncrit=ncrit, theta=theta, direct_below=0)
    f.set_shift(u)
    _, ga, gj = _eval(torch_cuda, f, x, v, m)
    o = oracle_lib.Oracle(6, ncrit=ncrit, theta=theta, shift_frac=u)
    _, oa, oj, _ = o.eval(x, v, m)
    st = f.stats()
    for k in ("ncells", "nleaves", "depth", "n_m2l", "n_p2p_cells", "n_p2p_pairs"):
        assert st[k] == o.stats[k], k
    # the widest level holds at least the average one's cells, the widest of at
    # most 2 depth + 1 steps at least that share of the lists' pairs
    assert st["ncells"] / (st["depth"] + 1) > 64 * max(8, n // 512)
    assert (st["n_m2l"] + st["n_p2p_cells"]) / (2 * st["depth"] + 1) > 256 * max(64, n // 32)
    assert relerr_vec(ga, oa)[1] < 1e-10 and relerr_vec(gj, oj)[1] < 1e-9


def test_gpu_many_evaluations_on_one_context(torch_cuda):
    """The scans' tags start again after some hundred evaluations: all of them give
    the first one's forces (the atomics' order is the only difference)."""
    import taichi_collisional_amd as tca
    from taichi_collisional_amd import ics
    torch = torch_cuda
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in ics.plummer(2001, seed=1)]
    f = tca.Fmm(p=4, ncrit=16, theta=0.6, direct_below=0)
    f.set_shift([0.1, 0.2, -0.3])
    first = [t.clone() for t in f.eval(*d)]
    for _ in range(400):
        for g, w in zip(f.eval(*d), first):
            assert float((g - w).abs().max()) <= 1e-12 * float(w.abs().max())
