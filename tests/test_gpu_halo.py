"""GPU parity of halo extraction (lstc_halo_sizes / lstc_halo_extract).

Bit-exact CSR equality with the oracle's restatement of round_clean_subgraph.cu,
and the invariant that the parts' owned-row counts sum to the whole count.
"""
import numpy as np
import pytest
import torch

import graphs as G

pytestmark = pytest.mark.gpu


def _device_graph(lstc, n, s, d):
    ds = torch.from_numpy(np.ascontiguousarray(s, np.uint32).view(np.int32)).cuda()
    dd = torch.from_numpy(np.ascontiguousarray(d, np.uint32).view(np.int32)).cuda()
    return lstc.clean_orient(n, ds, dd, keep_symmetric=True)


@pytest.mark.parametrize("name,builder,k", [
    ("multigraph", lambda O: G.random_multigraph(2000, 12000, seed=3), 3),
    ("rmat_s12", lambda O: O.gen_rmat(12, 16, seed=2), 8),
    ("grid", lambda O: O.gen_grid(30, 30, 0.3, 4), 4),
    ("K100", lambda O: G.complete(100), 2),
])
@pytest.mark.parametrize("mode", [0, 1])
def test_halo_bit_exact(lstc, oracle, name, builder, k, mode):
    n, s, d = builder(oracle)
    g = _device_graph(lstc, n, s, d)
    sym, og = oracle.clean_orient(n, s, d)
    part = lstc.partition_random(g.n, k, seed=5)
    opart = oracle.partition_random(sym.n, k, seed=5)
    for p in range(k):
        h = lstc.halo_extract(g, part, p, mode=mode, with_l2g=True)
        oh = oracle.halo_extract(sym, opart, p, mode)
        assert h.n_owned == oh.n_owned and h.n == oh.csr.n and h.m == oh.csr.m, (name, p)
        off, col = h.to_numpy()
        assert np.array_equal(off, oh.csr.off), (name, p)
        assert np.array_equal(col, oh.csr.col), (name, p)
        assert np.array_equal(h.meta["l2g"].cpu().numpy().view(np.uint32), oh.l2g), (name, p)


@pytest.mark.parametrize("k,mode", [(2, 0), (8, 0), (8, 1)])
def test_halo_parts_sum_to_unpartitioned(lstc, oracle, k, mode):
    n, s, d = lstc.generate_rmat(15, 16, seed=3)
    g = lstc.clean_orient(n, s, d, keep_symmetric=True)
    total = lstc.count(g)
    part = lstc.partition_random(g.n, k, seed=1)
    acc = 0
    for p in range(k):
        h = lstc.halo_extract(g, part, p, mode=mode)
        acc += lstc.count(h)  # counts owned rows [0, n_owned)
    assert acc == total


def test_halo_empty_part(lstc, oracle):
    n, s, d = G.complete(20)
    g = _device_graph(lstc, n, s, d)
    part = torch.zeros(g.n, dtype=torch.int32, device="cuda")
    h = lstc.halo_extract(g, part, 1)  # nobody is in part 1
    assert h.n == 0 and h.m == 0 and h.n_owned == 0
    h = lstc.halo_extract(g, part, 0)
    assert h.n == 20 and h.n_owned == 20 and lstc.count(h) == 20 * 19 * 18 // 6


@pytest.mark.parametrize("name,builder,k", [
    ("rmat_s13", lambda O: O.gen_rmat(13, 16, seed=6), 8),
    ("grid", lambda O: O.gen_grid(40, 40, 0.3, 4), 4),
    ("chung_lu", lambda O: O.gen_chung_lu(20000, 2.1, 30, 4e3, seed=3), 3),
])
@pytest.mark.parametrize("mode", [0, 1])
def test_halo_split_parts_match_oracle(lstc, oracle, name, builder, k, mode):
    """Halo parts with owned-source in-lists (lstc_in_lists) counted split, part by part and batched."""
    n, s, d = builder(oracle)
    g = _device_graph(lstc, n, s, d)
    sym, og = oracle.clean_orient(n, s, d)
    whole = oracle.count(og)
    part = lstc.partition_random(g.n, k, seed=7)
    opart = oracle.partition_random(sym.n, k, seed=7)
    parts, acc = [], 0
    for p in range(k):
        h = lstc.halo_extract(g, part, p, mode=mode, split=True)
        oh = oracle.halo_extract(sym, opart, p, mode)
        want_off, want_col = G.owned_in_lists(oh.csr.off, oh.csr.col, oh.n_owned)
        assert np.array_equal(h.in_off.cpu().numpy().view(np.uint64), want_off), (name, p)
        assert h.meta["in_entries"] == len(want_col)
        assert np.array_equal(h.in_col[: len(want_col)].cpu().numpy().view(np.uint32), want_col), (name, p)
        want = oracle.count(oh.csr, n_owned=oh.n_owned)
        assert lstc.count(h) == want, (name, p)
        assert lstc.count(h, split=False) == want, (name, p)
        for t in (lstc.Tune(tiny_max=1), lstc.Tune(tiny_max=4), lstc.Tune(unroll=8, table_scale=2)):
            assert lstc.count(h, tune=t) == want, (name, p, t.as_dict())
        parts.append(h)
        acc += want
    assert acc == whole
    assert lstc.count_batch(parts) == [lstc.count(h) for h in parts]


@pytest.mark.parametrize("name,builder,k", [
    ("rmat_s13", lambda O: O.gen_rmat(13, 16, seed=6), 8),
    ("grid", lambda O: O.gen_grid(40, 40, 0.3, 4), 4),
])
@pytest.mark.parametrize("mode", [0, 1])
def test_halo_parts_stream_copy(lstc, oracle, name, builder, k, mode):
    """lstc_stream_copy on split halo parts (words only for the owned rows' arcs): every row again
    at its 32-entry aligned start, each word with a list pointing there, and the counts (alone,
    batched, under tunings) equal the oracle's per part."""
    n, s, d = builder(oracle)
    g = _device_graph(lstc, n, s, d)
    sym, og = oracle.clean_orient(n, s, d)
    part = lstc.partition_random(g.n, k, seed=7)
    opart = oracle.partition_random(sym.n, k, seed=7)
    parts, wants = [], []
    for p in range(k):
        h = lstc.halo_extract(g, part, p, mode=mode, split=True)
        oh = oracle.halo_extract(sym, opart, p, mode)
        nw = int(oh.csr.off[oh.n_owned])
        before = h.col_seg[:nw].cpu().numpy().view(np.uint64).copy()
        lstc.stream_copy(h)
        deg = np.diff(oh.csr.off.astype(np.int64))
        start = np.concatenate([[0], np.cumsum((deg + 31) // 32 * 32)]).astype(np.int64)
        assert int(h.scol.numel()) == max(int(start[-1]), 1)
        scol = h.scol.cpu().numpy().view(np.uint32)
        for v in np.flatnonzero(deg):
            assert np.array_equal(scol[start[v]: start[v] + deg[v]], oh.csr.col[oh.csr.off[v]: oh.csr.off[v + 1]])
        words = h.col_seg[:nw].cpu().numpy().view(np.uint64)
        assert np.array_equal(words >> np.uint64(32), before >> np.uint64(32))  # lengths kept
        has = (words >> np.uint64(32)) != 0
        ids = oh.csr.col[:nw]
        assert np.array_equal((words & np.uint64(0xFFFFFFFF))[has], start[ids][has].astype(np.uint64))
        want = oracle.count(oh.csr, n_owned=oh.n_owned)
        assert lstc.count(h) == want, (name, p)
        for t in (lstc.Tune(tiny_max=1), lstc.Tune(unroll=8, table_scale=2)):
            assert lstc.count(h, tune=t) == want, (name, p, t.as_dict())
        parts.append(h)
        wants.append(want)
    assert lstc.count_batch(parts) == wants
    assert sum(wants) == oracle.count(og)


def test_bare_csr_stream_copy(lstc, oracle):
    """A bare oriented CSR (no preprocessing outputs): in-lists and words (lstc_in_lists_segments),
    then the streaming copy; the count and the batched count equal the oracle's."""
    n, s, d = oracle.gen_rmat(14, 16, seed=9)
    _, og = oracle.clean_orient(n, s, d)
    bare = lstc.Graph.from_numpy(og.off, og.col)
    lstc.in_lists(bare)
    lstc.stream_copy(bare)
    want = oracle.count(og)
    assert bare.scol is not None and lstc.count(bare) == want
    assert lstc.count_batch([bare]) == [want]


def _parts_equal_oracle(lstc, oracle, g, sym, part_dev, part_host, k, mode, tag, one_pass=True):
    parts = lstc.halo_extract_parts(g, part_dev, k, mode=mode, with_l2g=True,
                                    one_pass_limit_bytes=(8 << 30) if one_pass else 0)
    assert len(parts) == k
    for p, h in enumerate(parts):
        oh = oracle.halo_extract(sym, part_host, p, mode)
        assert (h.n_owned, h.n, h.m) == (oh.n_owned, oh.csr.n, oh.csr.m), (tag, p)
        off, col = h.to_numpy()
        assert np.array_equal(off, oh.csr.off), (tag, p)
        assert np.array_equal(col, oh.csr.col), (tag, p)
        assert np.array_equal(h.meta["l2g"].cpu().numpy().view(np.uint32), oh.l2g), (tag, p)
    return parts


@pytest.mark.parametrize("name,builder,k", [
    ("multigraph", lambda O: G.random_multigraph(2000, 12000, seed=3), 3),
    ("rmat_s12", lambda O: O.gen_rmat(12, 16, seed=2), 8),
    ("rmat_s12_k64", lambda O: O.gen_rmat(12, 16, seed=2), 64),
    ("rmat_s13_k13", lambda O: O.gen_rmat(13, 8, seed=6), 13),
    ("rmat_s13_k17", lambda O: O.gen_rmat(13, 8, seed=7), 17),
    ("rmat_s12_k32", lambda O: O.gen_rmat(12, 8, seed=8), 32),
    ("grid", lambda O: O.gen_grid(30, 30, 0.3, 4), 4),
    ("K100", lambda O: G.complete(100), 2),
    ("K100_k1", lambda O: G.complete(100), 1),
    ("star", lambda O: G.star(300), 5),
])
@pytest.mark.parametrize("mode", [0, 1])
def test_halo_parts_bit_exact(lstc, oracle, name, builder, k, mode):
    """All k parts from one call equal the oracle's part-by-part extraction."""
    n, s, d = builder(oracle)
    g = _device_graph(lstc, n, s, d)
    sym, _ = oracle.clean_orient(n, s, d)
    part = lstc.partition_random(g.n, k, seed=5)
    opart = oracle.partition_random(sym.n, k, seed=5)
    _parts_equal_oracle(lstc, oracle, g, sym, part, opart, k, mode, name)


@pytest.mark.parametrize("mode", [0, 1])
def test_halo_parts_unowned_and_empty_parts(lstc, oracle, mode):
    """Vertices assigned to a part >= k are owned by no part but may be halo vertices; empty parts
    give empty owned blocks.  Same result as the single-part call and the oracle."""
    n, s, d = oracle.gen_rmat(11, 16, seed=8)
    g = _device_graph(lstc, n, s, d)
    sym, _ = oracle.clean_orient(n, s, d)
    rng = np.random.default_rng(4)
    k = 6
    host = rng.choice(np.array([0, 2, 3, 5, 7, 99], np.uint32), size=sym.n)  # parts 1 and 4 empty, 7 and 99 unowned
    dev = torch.from_numpy(host.view(np.int32)).cuda()
    parts = _parts_equal_oracle(lstc, oracle, g, sym, dev, host, k, mode, "unowned")
    for p in range(k):
        one = lstc.halo_extract(g, dev, p, mode=mode)
        assert one.n == parts[p].n and one.m == parts[p].m
        assert all(np.array_equal(a, b) for a, b in zip(one.to_numpy(), parts[p].to_numpy()))
    assert parts[1].owned == 0 and parts[4].owned == 0


def test_halo_parts_sum_and_capacity_errors(lstc, oracle):
    from trianglecount_amd._lib import HaloOut
    import ctypes as C
    n, s, d = lstc.generate_rmat(15, 16, seed=3)
    g = lstc.clean_orient(n, s, d, keep_symmetric=True)
    total = lstc.count(g)
    part = lstc.partition_random(g.n, 8, seed=1)
    parts = lstc.halo_extract_parts(g, part, 8, mode=0, split=True)
    assert sum(lstc.count_batch(parts)) == total
    # a part whose output capacity is too small is refused before anything is written
    L = lstc.load()
    outs = (HaloOut * 8)()
    bufs = []
    for p, h in enumerate(parts):
        off = torch.full((h.n + 1,), -7, dtype=torch.int64, device="cuda")
        col = torch.empty(max(h.m, 1), dtype=torch.int32, device="cuda")
        bufs.append((off, col))
        outs[p].off, outs[p].col = off.data_ptr(), col.data_ptr()
        outs[p].n_local_cap, outs[p].m_local_cap = h.n, h.m - (1 if p == 3 else 0)
    nb = C.c_size_t()
    lstc.check(L.lstc_halo_parts_workspace(g.n, 8, C.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    st = L.lstc_halo_parts_extract(C.c_void_p(g.sym_off.data_ptr()), C.c_void_p(g.sym_col.data_ptr()), g.n,
                                   C.c_void_p(part.data_ptr()), 8, 0, outs, C.c_void_p(ws.data_ptr()), nb.value,
                                   C.c_void_p(lstc.stream_handle()))
    assert st == -1  # LSTC_ERR_INVALID
    assert all(int(off[0].item()) == -7 for off, _ in bufs)
    assert L.lstc_halo_parts_workspace(g.n, 65, C.byref(nb)) == -1


@pytest.mark.parametrize("n,k", [(1000, 3), (1000, 8), (7, 8), (1, 1), (4096, 64)])
def test_partition_contig(lstc, n, k):
    """Contiguous blocks (Halo_creation_preprocess.py:292-300): n // k vertices per part,
    the remainder (everything when n < k) in part 0."""
    want = np.zeros(n, np.uint32)
    l = n // k
    for i in range(k):
        want[i * l:(i + 1) * l] = i
    got = lstc.partition_contig(n, k).cpu().numpy().view(np.uint32)
    assert np.array_equal(got, want)


def test_partition_from_file_drives_halo(lstc, oracle, tmp_path):
    """An externally computed assignment (here: blocks of a BFS order, as a METIS-like stand-in)
    read from a node-parts file gives the same halo parts as the oracle with that assignment."""
    n, s, d = oracle.gen_rmat(12, 16, seed=14)
    g = _device_graph(lstc, n, s, d)
    sym, _ = oracle.clean_orient(n, s, d)
    # BFS order from vertex 0 over the symmetric CSR, cut into k blocks
    k = 5
    seen = np.zeros(sym.n, bool)
    order = []
    for root in range(sym.n):
        if seen[root]:
            continue
        seen[root] = True
        q = [root]
        while q:
            v = q.pop(0)
            order.append(v)
            for w in sym.col[sym.off[v]:sym.off[v + 1]]:
                if not seen[w]:
                    seen[w] = True
                    q.append(int(w))
    host = np.zeros(sym.n, np.uint32)
    host[np.array(order)] = (np.arange(sym.n) * k // sym.n).astype(np.uint32)
    path = tmp_path / "g_part.csr_node_parts_metis_5"
    path.write_text(" ".join(str(int(x)) for x in host) + "\n")
    dev = lstc.partition_from_file(str(path), sym.n, k)
    assert np.array_equal(dev.cpu().numpy().view(np.uint32), host)
    _parts_equal_oracle(lstc, oracle, g, sym, dev, host, k, 0, "metis-like")
    # the parts still sum to the whole
    parts = lstc.halo_extract_parts(g, dev, k)
    assert sum(lstc.count_batch(parts)) == lstc.count(g)


def test_partition_file_errors(lstc, tmp_path):
    short = tmp_path / "short"
    short.write_text("0 1 2\n")
    with pytest.raises(lstc.LstcError, match="holds 3 values"):
        lstc.partition_from_file(str(short), 10, 4)
    big = tmp_path / "big"
    big.write_text("0 1 7 2\n")
    with pytest.raises(lstc.LstcError, match="part 7 >= k"):
        lstc.partition_from_file(str(big), 4, 4)
    with pytest.raises(lstc.LstcError, match="cannot open"):
        lstc.partition_from_file(str(tmp_path / "missing"), 4, 4)


@pytest.mark.parametrize("mode", [0, 1])
def test_halo_parts_sized_then_extracted(lstc, oracle, mode):
    """The two-call path (exact sizes first, lstc_halo_parts_sizes + lstc_halo_parts_extract) gives the
    same parts as the one-pass build."""
    n, s, d = oracle.gen_rmat(12, 16, seed=21)
    g = _device_graph(lstc, n, s, d)
    sym, _ = oracle.clean_orient(n, s, d)
    part = lstc.partition_random(g.n, 6, seed=4)
    opart = oracle.partition_random(sym.n, 6, seed=4)
    _parts_equal_oracle(lstc, oracle, g, sym, part, opart, 6, mode, "two-call", one_pass=False)


def test_halo_parts_build_reports_sizes_when_too_small(lstc, oracle):
    import ctypes as C
    from trianglecount_amd._lib import HaloOut
    n, s, d = oracle.gen_rmat(11, 16, seed=2)
    g = _device_graph(lstc, n, s, d)
    part = lstc.partition_random(g.n, 3, seed=1)
    want = lstc.halo_extract_parts(g, part, 3)
    L = lstc.load()
    outs = (HaloOut * 3)()
    keep = []
    for p in range(3):
        off = torch.full((4,), -7, dtype=torch.int64, device="cuda")
        col = torch.empty(4, dtype=torch.int32, device="cuda")
        keep.append((off, col))
        outs[p].off, outs[p].col, outs[p].n_local_cap, outs[p].m_local_cap = off.data_ptr(), col.data_ptr(), 3, 4
    nl, no, ml = (C.c_uint32 * 3)(), (C.c_uint32 * 3)(), (C.c_uint64 * 3)()
    nb = C.c_size_t()
    lstc.check(L.lstc_halo_parts_workspace(g.n, 3, C.byref(nb)))
    ws = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    st = L.lstc_halo_parts_build(C.c_void_p(g.sym_off.data_ptr()), C.c_void_p(g.sym_col.data_ptr()), g.n,
                                 C.c_void_p(part.data_ptr()), 3, 0, outs, nl, no, ml, C.c_void_p(ws.data_ptr()),
                                 nb.value, C.c_void_p(lstc.stream_handle()))
    assert st == -1
    assert [(nl[p], no[p], ml[p]) for p in range(3)] == [(h.n, h.owned, h.m) for h in want]
    assert all(int(off[0].item()) == -7 for off, _ in keep)


@pytest.mark.parametrize("degree", [2047, 2048, 2049, 5000])
@pytest.mark.parametrize("k,mode", [(1, 0), (5, 1), (8, 0), (11, 0)])
def test_halo_parts_long_rows(lstc, oracle, degree, k, mode):
    """Hub rows on both sides of the length from which a workgroup walks them, joined to each other."""
    rng = np.random.default_rng(degree)
    n, hubs = 6000, 4
    far = [rng.choice(np.arange(hubs, n), degree - (hubs - 1), replace=False) for _ in range(hubs)]
    pairs = [(h, o) for h in range(hubs) for o in range(h)]
    s = np.concatenate([np.full(len(f), h) for h, f in enumerate(far)] + [[a for a, _ in pairs], rng.integers(0, n, 3000)])
    d = np.concatenate(far + [[b for _, b in pairs], rng.integers(0, n, 3000)])
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    g = _device_graph(lstc, n, s, d)
    sym, _ = oracle.clean_orient(n, s, d)
    part = lstc.partition_random(g.n, k, seed=7)
    _parts_equal_oracle(lstc, oracle, g, sym, part, oracle.partition_random(sym.n, k, seed=7), k, mode, degree)
