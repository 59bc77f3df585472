"""GPU parity of the Fitch kernels against the oracle: bit-exact sets, per-site
costs, per-node costs and totals, through the C ABI."""
import os
import sys
import time

import numpy as np
import pytest

from conftest import caterpillar, random_tree
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    from phylocaml_amd import device as D

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return D.Context(0)


def _sets(rng, n, amb=True):
    if amb:
        return rng.integers(1, 16, n).astype(np.uint8)
    return (1 << rng.integers(0, 4, n)).astype(np.uint8)


@pytest.mark.parametrize("S", [1, 15, 16, 17, 1000, 100003])
@pytest.mark.parametrize("weighted", [False, True])
def test_node_ops_match_oracle(ctx, rng, S, weighted):
    from phylocaml_amd import nonadditive as NA

    _say(f"node ops S={S} weighted={weighted}")
    w = rng.integers(1, 7, S).astype(np.uint32) if weighted else None
    wf = None if w is None else w.astype(np.float64)
    a, b, c = (_sets(rng, S) for _ in range(3))
    x, y, z = (NA.of_sets(ctx, s, w) for s in (a, b, c))
    m = NA.median_2(ctx, None, None, x, y)
    om, oc = O.fitch_median2(a, b, wf)
    assert np.array_equal(NA.to_sets(m), om) and m.cost == oc
    assert NA.distance_1(ctx, None, x, y) == oc
    m3 = NA.median_3(ctx, None, None, x, y, z)
    o3, oc3 = O.fitch_median3(a, b, c, wf)
    assert np.array_equal(NA.to_sets(m3), o3) and m3.cost == oc3
    d2 = NA.distance_2(ctx, None, x, y, z)
    assert d2 == O.fitch_median2(O.fitch_median2(a, b)[0], c, wf)[1]
    fp = _sets(rng, S)
    f = NA.of_sets(ctx, fp, w)
    adj, changed = NA.adjust_3(ctx, None, None, x, y, z, f)
    assert np.array_equal(NA.to_sets(adj), O.fitch_adjust3(a, b, c, fp))
    # in-place reuse of the previous value's block (the `t option` argument)
    prev = NA.of_sets(ctx, _sets(rng, S), w)
    m2 = NA.median_2(ctx, None, prev, x, y)
    assert m2.states.data_ptr() == prev.states.data_ptr()
    assert np.array_equal(NA.to_sets(m2), om)


def _tree_case(ctx, N, ch, root, leaves_u8, weights):
    from phylocaml_amd import device as D, nonadditive as NA

    S = leaves_u8.shape[1]
    topo = D.Topology(N, ch, root, ctx)
    ft = NA.alloc_tree(ctx, topo, S, D.pack_nibbles(leaves_u8), with_final=True,
                       with_node_cost=True)
    wd = None if weights is None else D.to_device(weights, ctx.device)
    NA.downpass(ctx, topo, ft, wd)
    NA.uppass(ctx, topo, ft)
    ctx.sync()
    osets, osc, onc, otot = O.fitch_downpass(N, ch, root, leaves_u8, weights, threads=8)
    ofin = O.fitch_uppass(N, ch, root, osets)
    got_sets = ft.sets.cpu().numpy()
    assert np.array_equal(got_sets[N:], D.pack_nibbles(osets[N:])), "prelim sets differ"
    assert np.array_equal(ft.final.cpu().numpy(), D.pack_nibbles(ofin)), "final sets differ"
    assert np.array_equal(ft.site_cost.cpu().numpy()[:S], osc), "site costs differ"
    assert np.array_equal(ft.node_cost.cpu().numpy(), onc), "node costs differ"
    assert int(ft.total.cpu().numpy()[0]) == otot


@pytest.mark.parametrize("N", [2, 3, 17, 128, 1024])
@pytest.mark.parametrize("S", [1, 17, 5000])
def test_tree_passes_match_oracle(ctx, rng, N, S):
    for kind in ("random", "caterpillar"):
        _say(f"tree passes N={N} S={S} {kind}")
        ch, root = random_tree(rng, N) if kind == "random" else caterpillar(N)
        leaves = rng.integers(1, 16, (N, S)).astype(np.uint8)
        w = rng.integers(1, 5, S).astype(np.uint32) if kind == "random" else None
        _tree_case(ctx, N, ch, root, leaves, w)


@pytest.mark.parametrize("nt", ["0", "1"])
@pytest.mark.parametrize("words", ["1", "2", "4"])
@pytest.mark.parametrize("batch", ["4", "8", "16", "32"])
@pytest.mark.parametrize("split", ["0", "1"])
def test_prefetch_depth_and_split_forms(ctx, rng, monkeypatch, batch, split, words, nt):
    # the whole-tree and the split (parts side by side, then the top) forms,
    # at every operand prefetch depth and lane width, with cached or
    # non-temporal row accesses, give the oracle's bits
    monkeypatch.setenv("PHY_FITCH_BATCH", batch)
    monkeypatch.setenv("PHY_FITCH_SPLIT", split)
    monkeypatch.setenv("PHY_FITCH_WORDS", words)
    monkeypatch.setenv("PHY_FITCH_NT", nt)
    N, S = 300, 3001
    _say(f"fitch forms batch={batch} split={split} words={words} nt={nt}")
    ch, root = random_tree(rng, N)
    leaves = rng.integers(1, 16, (N, S)).astype(np.uint8)
    w = rng.integers(1, 5, S).astype(np.uint32)
    if batch == "32" and words == "4":
        # (2 x 32 + depth) sets of 16 B per thread exceed one block's LDS even
        # at 64 threads: the launch is refused with PHY_ERANGE
        from phylocaml_amd._lib import PhyError

        with pytest.raises(PhyError) as e:
            _tree_case(ctx, N, ch, root, leaves, w)
        assert e.value.code == 5
        return
    _tree_case(ctx, N, ch, root, leaves, w)


@pytest.mark.parametrize("N,narrow", [(1000, "1"), (1000, "0"), (8192, "1")])
def test_split_part_counts_as_bytes_or_words(ctx, rng, monkeypatch, N, narrow):
    # the parts hand their per-site counts to the top as bytes when every part
    # has at most 255 internal nodes (1,000 leaves: parts of <= 103), else as
    # 32-bit words (8,192 leaves: parts of up to ~1,500); PHY_FITCH_NARROW=0
    # forces words
    monkeypatch.setenv("PHY_FITCH_NARROW", narrow)
    S = 517
    _say(f"fitch split counts N={N} narrow={narrow}")
    ch, root = random_tree(rng, N)
    leaves = rng.integers(1, 16, (N, S)).astype(np.uint8)
    w = rng.integers(1, 5, S).astype(np.uint32)
    _tree_case(ctx, N, ch, root, leaves, w)


def test_1024_taxa_1e6_sites_bit_exact(ctx):
    """1,024-taxon Yule tree, 10^6 IUPAC sites (the parsimony benchmark
    workload): every preliminary and final set, every site cost and the total
    against the oracle."""
    from phylocaml_amd import device as D, nonadditive as NA, synth

    N, S = 1024, 1_000_000
    _say("1,024 taxa x 10^6 sites: generating")
    tree = synth.yule(N, 1, 0.1)
    lv = synth.fitch_leaves(N, S, 1)
    topo = D.Topology(N, tree.children, tree.root, ctx)
    ft = NA.alloc_tree(ctx, topo, S, lv, with_final=True, with_node_cost=True)
    NA.downpass(ctx, topo, ft)
    NA.uppass(ctx, topo, ft)
    ctx.sync()
    _say("1,024 taxa x 10^6 sites: oracle")
    t0 = time.time()
    leaves = D.unpack_nibbles(lv, S)
    osets, osc, onc, otot = O.fitch_downpass(N, tree.children, tree.root, leaves,
                                             threads=min(16, os.cpu_count() or 1))
    _say(f"oracle downpass {time.time() - t0:.1f}s")
    assert int(ft.total.cpu().numpy()[0]) == otot
    assert np.array_equal(ft.site_cost.cpu().numpy(), osc)
    assert np.array_equal(ft.node_cost.cpu().numpy(), onc)
    assert int(onc.sum()) == otot
    assert np.array_equal(ft.sets.cpu().numpy()[N:], D.pack_nibbles(osets[N:]))
    ofin = O.fitch_uppass(N, tree.children, tree.root, osets)
    assert np.array_equal(ft.final.cpu().numpy(), D.pack_nibbles(ofin))
    _say(f"1,024 taxa x 10^6 sites: total cost {otot}")


def test_empty_and_bad_arguments(ctx):
    from phylocaml_amd import _lib, device as D

    lib = _lib.lib
    buf = torch.zeros(4, dtype=torch.uint64, device="cuda:0")
    cost = torch.ones(1, dtype=torch.uint64, device="cuda:0")
    # zero sites: cost 0, no launch
    assert lib.phy_fitch_median2(ctx.handle, D.dptr(buf), D.dptr(buf), D.dptr(buf), 0, None,
                                 D.dptr(cost)) == 0
    ctx.sync()
    assert int(cost.cpu()[0]) == 0
    assert lib.phy_fitch_median2(ctx.handle, D.dptr(buf), D.dptr(buf), D.dptr(buf), -1, None,
                                 None) == 1
    topo = D.Topology(3, np.array([0, 1, 2, 3], np.int32), 4, ctx)
    # stride smaller than the block
    assert lib.phy_fitch_downpass(ctx.handle, topo.handle, D.dptr(buf), 1, 100, None,
                                  D.dptr(buf), None, D.dptr(cost)) == 1
    # host-only topology cannot run on the device
    host_topo = D.Topology(3, np.array([0, 1, 2, 3], np.int32), 4)
    assert lib.phy_fitch_uppass(ctx.handle, host_topo.handle, D.dptr(buf), D.dptr(buf), 1,
                                1) == 1


@pytest.mark.parametrize("N,S", [(23, 700), (24, 700), (31, 2100), (32, 2100), (40, 1), (40, 513),
                                 (301, 20_011), (24, 530_001), (130, 200_003), (130, 400_003),
                                 (256, 4099), (256, 5000), (257, 4103), (257, 4700)])
@pytest.mark.parametrize("weights", ["unit", "small", "heavy"])
def test_pass_shapes_and_node_costs(ctx, rng, N, S, weights):
    # both sides of the dispatch lines (whole tree below 24 leaves up and 32
    # down, fine split with narrow lanes, its part counts in 8 bits up to 256
    # leaves and in 16 beyond, or one a word in a last block of few sites, whole
    # tree or coarse split and wide lanes at many sites) with node costs counted,
    # weighed by bit planes (up to 8 bits) or walked (one site of 2^20 makes its
    # wave do so)
    _say(f"fitch shapes N={N} S={S} weights={weights}")
    ch, root = random_tree(rng, N)
    leaves = rng.integers(1, 16, (N, S)).astype(np.uint8)
    w = None if weights == "unit" else rng.integers(0, 256, S).astype(np.uint32)
    if weights == "heavy":
        w[S // 2] = 1 << 20
    _tree_case(ctx, N, ch, root, leaves, w)


@pytest.mark.parametrize("S", [1, 1025, 4111, 70_003])
@pytest.mark.parametrize("weights", ["unit", "small", "heavy"])
def test_insertion_costs_match_oracle(ctx, rng, monkeypatch, S, weights):
    # one wave to several chunks of words a query, runs that share or change
    # the inserted node, one query and more than a run, weights by bit planes
    # or walked; a block per query, runs, and the choice between them on both
    # sides of its line (many queries)
    from phylocaml_amd import device as D
    from phylocaml_amd._lib import lib

    rows = 9
    sets = rng.integers(1, 16, (2, rows, S)).astype(np.uint8)
    pre, fin = (D.to_device(D.pack_nibbles(x), ctx.device) for x in sets)
    w = None if weights == "unit" else rng.integers(0, 256, S).astype(np.uint32)
    if weights == "heavy":
        w[S // 2] = 1 << 20
    wd = None if w is None else D.to_device(w, ctx.device)
    allq = np.stack([np.repeat(np.arange(rows), 81), np.tile(np.repeat(np.arange(rows), 9), rows),
                     np.tile(np.arange(rows), 81)], 1).astype(np.int32)
    pairs = {(a, b): O.fitch_median2(sets[1][a], sets[1][b])[0] for a in range(rows)
             for b in range(rows)}
    ww = np.ones(S, np.int64) if w is None else w.astype(np.int64)
    want = [int(ww[(sets[0][c] & pairs[a, b]) == 0].sum()) for c, a, b in allq.tolist()]
    many = np.tile(allq, (25, 1))
    for n, form in ((1, "0"), (1, "1"), (65, "0"), (65, "1"), (729, "0"), (729, "1"), (729, None),
                    (25 * 729, None), (25 * 729 - 3, "1")):
        monkeypatch.delenv("PHY_FITCH_INSERT", raising=False)
        if form:
            monkeypatch.setenv("PHY_FITCH_INSERT", form)
        _say(f"insertion costs S={S} {weights} n={n} form {form}")
        dq = D.to_device(np.ascontiguousarray(many[:n]), ctx.device)
        out = torch.full((n,), 7, dtype=torch.int64, device="cuda")
        ctx.check(lib.phy_fitch_insertion_costs(ctx.handle, D.dptr(pre), D.dptr(fin), D.words(S), S,
                                                D.dptr(wd), n, D.dptr(dq), D.dptr(out)), "insertion")
        assert out.cpu().tolist() == (want * 25)[:n]


@pytest.mark.parametrize("N", [24, 64, 127])
def test_passes_of_one_small_topology_on_two_streams(rng, N):
    # below 128 leaves a pass shares nothing with another one of its topology:
    # two alignments of different lengths, passes in flight side by side
    from phylocaml_amd import device as D, nonadditive as NA

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _say(f"fitch two streams N={N}")
    ch, root = random_tree(rng, N)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ctxs = [D.Context(0, stream=s.cuda_stream) for s in streams]
    topo = D.Topology(N, ch, root, ctxs[0])
    leaves = [rng.integers(1, 16, (N, S)).astype(np.uint8) for S in (3001, 60_007)]
    fts = [NA.alloc_tree(c, topo, lv.shape[1], D.pack_nibbles(lv), with_node_cost=True)
           for c, lv in zip(ctxs, leaves)]
    torch.cuda.synchronize()
    for _ in range(30):
        for c, ft in zip(ctxs, fts):
            NA.downpass(c, topo, ft, None)
    torch.cuda.synchronize()
    for ft, lv in zip(fts, leaves):
        osets, osc, onc, otot = O.fitch_downpass(N, ch, root, lv, None, threads=8)
        assert np.array_equal(ft.sets.cpu().numpy()[N:], D.pack_nibbles(osets[N:]))
        assert np.array_equal(ft.site_cost.cpu().numpy()[:lv.shape[1]], osc)
        assert np.array_equal(ft.node_cost.cpu().numpy(), onc)
        assert int(ft.total.cpu().numpy()[0]) == otot


@pytest.mark.parametrize("N", [24, 200, 300])
def test_site_costs_at_a_word_aligned_address(ctx, rng, N):
    from phylocaml_amd import device as D, nonadditive as NA

    S = 4099
    _say(f"fitch unaligned site costs N={N}")
    ch, root = random_tree(rng, N)
    leaves = rng.integers(1, 16, (N, S)).astype(np.uint8)
    topo = D.Topology(N, ch, root, ctx)
    ft = NA.alloc_tree(ctx, topo, S, D.pack_nibbles(leaves), with_node_cost=True)
    buf = torch.full((S + 3,), 7, dtype=torch.int32, device="cuda")
    ft.site_cost = buf[1:S + 1].view(torch.uint32)
    NA.downpass(ctx, topo, ft, None)
    osets, osc, onc, otot = O.fitch_downpass(N, ch, root, leaves, None, threads=8)
    assert np.array_equal(ft.site_cost.cpu().numpy(), osc)
    assert int(ft.total.cpu().numpy()[0]) == otot
    assert buf.cpu().tolist()[0] == 7 and buf.cpu().tolist()[S + 1:] == [7, 7]
