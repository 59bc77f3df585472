"""GPU checks of the batched 20-state BF16-MFMA pruning against the FP64
oracle.

BF16 operands carry an 8-bit significand, so the per-tree lnL is compared
with a relative tolerance of 2e-3 (the measured error is reported by
bench.py); every tree in a batch of uneven trees must meet it, which also
checks the persistent work queue and the per-tree bookkeeping."""
import os

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    from phylocaml_amd import device as D

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return D.Context(0)


def _oracle(t):
    from phylocaml_amd import aa

    v, _ = O.lnl(t.n_leaves, t.children, t.root, t.blen, t.pi, t.q, t.rates, t.probs,
                 aa.tips_bitmask(t.tips), t.weights, threads=min(16, os.cpu_count() or 1))
    return v


@pytest.mark.parametrize("waves", [1, 2, 4, 8])
def test_batch_matches_oracle(ctx, waves):
    from phylocaml_amd import aa

    print(f"aa batch waves={waves}", flush=True)
    rng = np.random.default_rng(7)
    trees = []
    for k in range(9):
        N = int(rng.integers(2, 70))
        P = int(rng.integers(1, 900))
        trees.append(aa.synth_tree(1000 + k, N, P, n_sim=300))
    # ambiguous/missing tips
    trees[3].tips[:, ::7] = 255
    b = aa.AABatch(ctx, trees, waves=waves)
    b.run()
    ctx.sync()
    got = b.lnl.cpu().numpy()
    for k, t in enumerate(trees):
        ov = _oracle(t)
        rel = abs(got[k] - ov) / abs(ov)
        print(f"tree {k}: N={t.n_leaves} P={t.n_patterns} oracle {ov:.6f} gpu {got[k]:.6f} "
              f"rel {rel:.2e}", flush=True)
        assert rel <= 2e-3, (k, got[k], ov)
    # a second run on the same batch gives the same answer (queue reset)
    b.run()
    ctx.sync()
    assert np.array_equal(b.lnl.cpu().numpy(), got)


@pytest.mark.parametrize("waves", [4, 8])
def test_register_stack_levels_give_the_same_bits(ctx, monkeypatch, waves):
    # the bottom stack levels held in registers carry the same BF16 operands
    # as the LDS rows: identical results with and without them
    from phylocaml_amd import aa

    rng = np.random.default_rng(11)
    trees = [aa.synth_tree(2000 + k, int(rng.integers(40, 140)), int(rng.integers(100, 700)),
                           n_sim=200) for k in range(6)]
    out = {}
    for reg in ("0", "3"):
        monkeypatch.setenv("PHY_AA_REG", reg)
        print(f"aa register levels {reg} waves={waves}", flush=True)
        b = aa.AABatch(ctx, trees, waves=waves)
        b.run()
        ctx.sync()
        out[reg] = b.lnl.cpu().numpy()
    assert np.array_equal(out["0"], out["3"])
    ov = _oracle(trees[0])
    assert abs(out["3"][0] - ov) <= 2e-3 * abs(ov)


def test_tiny_exact_cases(ctx):
    # constant tips and a two-taxon tree: L = sum_i pi_i P_ij(t1 + t2)
    from phylocaml_amd import aa

    t = aa.synth_tree(5, 2, 40, n_sim=40)
    b = aa.AABatch(ctx, [t], waves=1)
    b.run()
    ctx.sync()
    ov = _oracle(t)
    assert abs(b.lnl.cpu().numpy()[0] - ov) <= 2e-3 * abs(ov)


@pytest.mark.parametrize("waves", [1, 4, 8])
def test_large_trees_cross_leaf_id_chunks(ctx, waves):
    # the kernel holds the leaf-id stream 128 ids at a time and advances it by
    # 64: trees of 129-300 leaves cross several such refills
    from phylocaml_amd import aa

    print(f"aa large trees waves={waves}", flush=True)
    trees = [aa.synth_tree(3000 + k, N, P, n_sim=150)
             for k, (N, P) in enumerate([(129, 70), (200, 130), (300, 40), (257, 17)])]
    trees[1].tips[:, ::5] = 255
    b = aa.AABatch(ctx, trees, waves=waves)
    b.run()
    ctx.sync()
    got = b.lnl.cpu().numpy()
    for k, t in enumerate(trees):
        ov = _oracle(t)
        rel = abs(got[k] - ov) / abs(ov)
        print(f"tree {k}: N={t.n_leaves} P={t.n_patterns} rel {rel:.2e}", flush=True)
        assert rel <= 2e-3, (k, got[k], ov)


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("waves", [1, 4, 8])
def test_one_and_two_rate_classes(ctx, R, waves):
    # the R = 1 and R = 2 kernels (the other tests use four Gamma classes)
    from dataclasses import replace

    from phylocaml_amd import aa

    print(f"aa rate classes R={R} waves={waves}", flush=True)
    rates = {1: [1.0], 2: [0.35, 1.65]}[R]
    rng = np.random.default_rng(31 + R)
    trees = []
    for k in range(6):
        t = aa.synth_tree(5000 + 10 * R + k, int(rng.integers(2, 150)), int(rng.integers(1, 600)),
                          n_sim=120)
        trees.append(replace(t, rates=np.array(rates), probs=np.full(R, 1.0 / R)))
    b = aa.AABatch(ctx, trees, waves=waves)
    b.run()
    ctx.sync()
    got = b.lnl.cpu().numpy()
    for k, t in enumerate(trees):
        ov = _oracle(t)
        assert abs(got[k] - ov) <= 2e-3 * abs(ov), (k, got[k], ov)


def _balanced(n):
    """Children of a balanced tree of n = 2^k leaves (the deepest stack)."""
    ch, level, nxt = [], list(range(n)), n
    while len(level) > 1:
        level2 = []
        for a, b in zip(level[::2], level[1::2]):
            ch += [a, b]
            level2.append(nxt)
            nxt += 1
        level = level2
    return np.array(ch, np.int32), nxt - 1


@pytest.mark.parametrize("R", [1, 2, 4])
def test_every_tile_gives_the_same_trees(ctx, R):
    # one or two groups of 16 patterns per wave, 0 / 3 / 4 stack levels in
    # registers (by the deepest tree of a batch) and the rest in LDS: the same
    # operations per pattern, so the lnL differ by the order of an FP64 sum of
    # <= 1,000 terms (1,000 x 2^-53 ~ 1e-13)
    from dataclasses import replace

    from phylocaml_amd import aa

    rng = np.random.default_rng(61 + R)
    rates = np.array({1: [1.0], 2: [0.3, 1.7], 4: [0.05, 0.4, 0.9, 2.65]}[R])
    for name, shapes in (("shallow", [(2, 1), (3, 17), (5, 300)]),
                         ("deep", [(128, 129), (2, 16), (64, 1), (33, 257), (16, 1000)])):
        trees = []
        for k, (n, p) in enumerate(shapes):
            t = aa.synth_tree(7000 + 10 * R + k, n, p, n_sim=100)
            if name == "deep" and n & (n - 1) == 0:
                ch, root = _balanced(n)
                t = replace(t, children=ch, root=root)
            t.tips[rng.random(t.tips.shape) < 0.05] = 255
            trees.append(replace(t, rates=rates, probs=np.full(R, 1.0 / R)))
        got = {}
        for waves in (1, 2, 4, 8):
            print(f"aa {name} R={R} waves={waves}", flush=True)
            b = aa.AABatch(ctx, trees, waves=waves)
            b.run()
            ctx.sync()
            got[waves] = b.lnl.cpu().numpy()
        for waves in (1, 2, 8):
            assert np.allclose(got[waves], got[4], rtol=1e-12, atol=0)
        for k, t in enumerate(trees):
            ov = _oracle(t)
            assert abs(got[4][k] - ov) <= 2e-3 * abs(ov), (k, got[4][k], ov)


@pytest.mark.parametrize("t", [2e-10, 5e-10, 1e-8])
def test_sister_cherries_of_short_branches(ctx, t):
    # ((a, b), (c, d)) with no direct exchange between the four states: each
    # cherry's values are ~1e-21, and without a rescale there their product at
    # the parent (branches of length 0) leaves FP32's range.  The same tree with a missing leaf beside
    # a and c on branches of length 0 (P = 1) has the same values at every node
    # and no node of two leaves that needs a rescale.
    from phylocaml_amd import aa

    rng = np.random.default_rng(5)
    pi = rng.dirichlet(np.full(20, 20.0))
    ex = rng.uniform(0.5, 2.0, (20, 20))
    ex[:4, :4] = 0.0
    ex = np.triu(ex, 1)
    q = (ex + ex.T) * pi[None, :]
    np.fill_diagonal(q, -q.sum(1))
    q /= -(pi * np.diag(q)).sum()
    one, w = np.ones(1), np.ones(1, np.uint32)

    def tree(n, children, blen, codes):
        return aa.AATree(n, np.array(children, np.int32), 2 * n - 2, np.array(blen), pi, q, one, one,
                         np.array(codes, np.uint8)[:, None], w)

    plain, padded = [], []
    for p in ([0, 1, 2, 3], [1, 3, 0, 2], [2, 0, 3, 1], [3, 2, 1, 0], [0, 1, 5, 3], [7, 8, 9, 10]):
        plain.append(tree(4, [0, 1, 2, 3, 4, 5], [t] * 4 + [0.0] * 3, p))
        # leaves a b c d ? ?: 6 = (a, ?), 7 = (6, b), 8 = (c, ?), 9 = (8, d), 10 = (7, 9)
        padded.append(tree(6, [0, 4, 6, 1, 2, 5, 8, 3, 7, 9],
                           [0.0, t, 0.0, t, 0.0, 0.0, t, 0.0, t, 0.0, 0.0], p + [255, 255]))
    print(f"aa sister cherries t={t}", flush=True)
    b = aa.AABatch(ctx, plain + padded, waves=4)
    b.run()
    ctx.sync()
    got, want = np.split(b.lnl.cpu().numpy(), 2)
    print(got, want, flush=True)
    ok = np.isfinite(want)  # a negative entry of P (rounding of its eigen sum) may leave no value
    assert ok.sum() >= 3
    assert np.all(np.abs(got[ok] - want[ok]) <= 1e-6 * np.abs(want[ok]))


@pytest.mark.parametrize("R", [1, 2, 4])
def test_groups_of_a_wave_give_the_same_bits(ctx, R):
    # at 8 waves a wave takes two groups of 16 patterns where the tiles are more
    # than the CUs, one otherwise (always at R = 2): the same trees alone and
    # among many
    from dataclasses import replace

    from phylocaml_amd import aa

    rng = np.random.default_rng(13)
    trees = []
    for k in range(5):
        t = aa.synth_tree(3000 + k, int(rng.integers(4, 90)), int(rng.integers(200, 900)), n_sim=200)
        if R != 4:
            t = replace(t, rates=np.array([0.4, 1.6])[:R] if R > 1 else np.ones(1),
                        probs=np.full(R, 1.0 / R))
        trees.append(t)
    print(f"aa groups R={R}", flush=True)
    got = []
    for copies in (1, 40):
        b = aa.AABatch(ctx, trees * copies, waves=8)
        assert (b.n_items > 512) == (copies > 1) and (copies > 1 or b.n_items <= 64)
        b.run()
        ctx.sync()
        got.append(b.lnl.cpu().numpy().reshape(copies, -1))
        b.close()
    assert np.array_equal(got[1], np.repeat(got[0], 40, 0))
    for k, t in enumerate(trees):
        ov = _oracle(t)
        assert abs(got[0][0, k] - ov) <= 2e-3 * abs(ov)
