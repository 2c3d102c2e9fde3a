"""GPU parity of spike compaction and of the two delivery kernels."""
import numpy as np
import pytest
import torch

from oracle import glif3_oracle as orc
from bmtk_amd import network as net, ops
from gpu_util import bits_of, rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 16384, 16385, (1 << 20) + 3])
@pytest.mark.parametrize("p", [0.0, 0.003, 0.3, 1.0])
def test_compaction_is_flatnonzero(n, p):
    rng = np.random.default_rng(n % 1000 + int(p * 1000))
    z = (rng.random(n) < p).astype(np.uint8) if p < 1.0 else np.ones(n, np.uint8)
    want = np.flatnonzero(z).astype(np.int32)
    comp = ops.SpikeCompactor(n)
    for src in (to_dev(z), to_dev(bits_of(z))):
        ids, count = comp(src)
        c = int(count.item())
        assert c == want.size
        np.testing.assert_array_equal(ids[:c].cpu().numpy(), want)


@pytest.mark.parametrize("n", [1, 64, 65, 4095, 4097, 65535, 65536, 65537, 131071, 131072, 131073])
@pytest.mark.parametrize("p", [0.0, 0.03, 0.2, 1.0])
def test_compaction_of_bits_on_either_side_of_one_launch(n, p):
    """Words of a wavefront's lanes, two words a lane and the size from which two launches take over; bits beyond n are set."""
    rng = np.random.default_rng(n)
    z = (rng.random(n) < p).astype(np.uint8)
    words = np.zeros(ops.n_words(n) + 1, np.uint64)
    words[:-1] = np.packbits(np.concatenate([z, np.ones(ops.n_words(n) * 64 - n, np.uint8)]), bitorder="little").view(np.uint64)
    c = ops.SpikeCompactor(n)
    ids, count = c(to_dev(words.view(np.int64)))
    assert int(count) == int(z.sum())
    np.testing.assert_array_equal(ids[:int(count)].cpu().numpy(), np.flatnonzero(z))


def test_compaction_other_paths():
    """Flags that do not start on a 16-byte boundary (the packing then goes through the one-flag-per-thread kernel),
    non-zero flags other than 1, and an input beyond the size the fused two-launch form takes."""
    rng = np.random.default_rng(77)
    z = (rng.random(100_001) < 0.01).astype(np.uint8) * rng.integers(1, 256, 100_001).astype(np.uint8)
    dev = to_dev(z)
    for off in (1, 5, 16):
        comp = ops.SpikeCompactor(z.size - off)
        ids, count = comp(dev[off:])
        want = np.flatnonzero(z[off:]).astype(np.int32)
        assert int(count.item()) == want.size
        np.testing.assert_array_equal(ids[:want.size].cpu().numpy(), want)
    n = (1 << 26) + 5
    big = torch.zeros(n, dtype=torch.uint8, device=dev.device)
    hot = torch.as_tensor(np.sort(rng.choice(n, 50_000, replace=False)), device=dev.device)
    big[hot] = 1
    ids, count = ops.SpikeCompactor(n)(big)
    assert int(count.item()) == 50_000 and torch.equal(ids[:50_000].long(), hot)


def test_compaction_ignores_bits_beyond_n():
    z = np.zeros(100, np.uint8)
    z[[3, 99]] = 1
    bits = bits_of(z).copy()
    bits[1] |= np.int64(-1) << 40          # garbage above element 100 in the last word
    comp = ops.SpikeCompactor(100)
    ids, count = comp(to_dev(bits))
    assert ids[:int(count.item())].cpu().tolist() == [3, 99]


def _edges(rng, n_src, n_tgt, nnz, max_delay=5):
    src = rng.integers(0, n_src, nnz).astype(np.int32)
    tgt = rng.integers(0, n_tgt, nnz).astype(np.int32)
    w = (rng.lognormal(0, 1, nnz) * rng.choice([-1, 1], nnz)).astype(np.float32)
    d = rng.integers(1, max_delay + 1, nnz).astype(np.uint8)
    r = rng.integers(0, 4, nnz).astype(np.uint8)
    return src, tgt, w, d, r


@pytest.mark.parametrize("batch,p", [(1, 0.05), (1, 1.0), (5, 0.2), (64, 0.02), (100, 0.1)])
def test_scatter_matches_oracle(batch, p):
    """fp32 atomics add in an arbitrary order, so the comparison is against the
    fp64 oracle: |diff| <= 1e-5 * max(|want|, sum of |w| into the cell * 1e-2)
    -- the floor is the magnitude rounding errors scale with when signed
    weights cancel."""
    rng = np.random.default_rng(30)
    n_src, n_tgt, L = 300, 257, 6
    src, tgt, w, d, r = _edges(rng, n_src, n_tgt, 20000)
    csr = net.coo_to_csr(src, tgt, w, d, r, n_rows=n_src, major="source")
    table = ops.SynapseTable.from_numpy(csr)
    ring_d = torch.zeros(L, 4, n_tgt * batch, device="cuda")
    ring_c = np.zeros((L, 4, n_tgt * batch))
    mag_c = np.zeros((L, 4, n_tgt * batch))
    csr_abs = (csr[0], csr[1], np.abs(csr[2]), csr[3], csr[4])
    comp = ops.SpikeCompactor(n_src * batch)
    for step in (0, 4, 11):
        z = (rng.random(n_src * batch) < p).astype(np.uint8)
        ids, count = comp(to_dev(z))
        ops.csr_propagate_scatter(ids, count, table, ring_d, n_tgt, batch, step)
        orc.deliver_events(np.flatnonzero(z), batch, csr, ring_c, n_tgt, step)
        orc.deliver_events(np.flatnonzero(z), batch, csr_abs, mag_c, n_tgt, step)
    got = ring_d.cpu().numpy()
    assert np.abs(ring_c).max() > 0
    assert np.max(np.abs(got - ring_c) / np.maximum(np.abs(ring_c), 1e-2 * mag_c + 1e-30)) < 1e-5
    assert np.all(got[mag_c == 0] == 0)


@pytest.mark.parametrize("batch,p", [(1, 0.1), (5, 0.2), (32, 0.05), (64, 0.02), (64, 0.6), (100, 0.1), (130, 0.05)])
def test_gather_bit_exact_vs_fp32_oracle(batch, p):
    """Each ring cell is updated by one wavefront in stored synapse order
    starting from the value already there: identical to the scalar fp32 loop,
    including on a ring that already holds values."""
    rng = np.random.default_rng(31)
    n_src, n_tgt, L = 211, 190, 6
    src, tgt, w, d, r = _edges(rng, n_src, n_tgt, 15000)
    csr = net.coo_to_csr(src, tgt, w, d, r, n_rows=n_tgt, major="target")
    table = ops.SynapseTable.from_numpy(csr)
    ring_c = rng.normal(0, 1, (L, 4, n_tgt * batch)).astype(np.float32)
    ring_d = to_dev(ring_c)
    for step in (0, 5, 9):
        z = (rng.random(n_src * batch) < p).astype(np.uint8)
        ops.csr_propagate_gather(to_dev(bits_of(z)), n_src, table, ring_d, n_tgt, batch, step)
        orc.gather_rows(z, batch, csr, ring_c, n_tgt, step)
        np.testing.assert_array_equal(ring_d.cpu().numpy(), ring_c)


def test_gather_equals_scatter_and_dense_bruteforce():
    rng = np.random.default_rng(32)
    n, L, batch = 150, 6, 64
    src, tgt, w, d, r = _edges(rng, n, n, 9000)
    by_src = net.coo_to_csr(src, tgt, w, d, r, n_rows=n, major="source")
    by_tgt = net.csr_transpose(by_src, n)
    z = (rng.random(n * batch) < 0.05).astype(np.uint8)
    want = orc.dense_deliver_bruteforce(z, batch, src, tgt, w, d, r, L, n, 7)
    ring_g = torch.zeros(L, 4, n * batch, device="cuda")
    ring_s = torch.zeros(L, 4, n * batch, device="cuda")
    ops.csr_propagate_fwd("gather", ops.SynapseTable.from_numpy(by_tgt), ring_g, n, batch, 7,
                          zbits=to_dev(bits_of(z)), n_src=n)
    ids, count = ops.SpikeCompactor(n * batch)(to_dev(z))
    ops.csr_propagate_fwd("scatter", ops.SynapseTable.from_numpy(by_src), ring_s, n, batch, 7,
                          active=ids, n_active=count)
    # floor 1e-2: a hundredth of the unit weight scale (lognormal(0,1) pA), sums of a few signed terms
    assert rel_err(ring_g.cpu().numpy(), want, 1e-2) < 1e-5
    assert rel_err(ring_s.cpu().numpy(), want, 1e-2) < 1e-5


@pytest.mark.parametrize("n_active", [0, 1, 127, 128, 129, 4096, 4097, 8193])
@pytest.mark.parametrize("bound", [None, "exact"])
def test_scatter_rows_shared_by_wavefronts(n_active, bound):
    """Few active elements: up to 64 wavefronts to a row, the rows of every length around a chunk and around all chunks of
    a round.  Weights are small whole numbers, so that the sums are exact in any order."""
    rng = np.random.default_rng(n_active)
    n, L = 9000, 5
    lengths = rng.choice([0, 1, 63, 64, 65, 129], n)
    lengths[:6] = (64 * 64 - 1, 64 * 64, 64 * 64 + 1, 2 * 64 * 64 + 1, 0, 1)
    src = np.repeat(np.arange(n, dtype=np.int32), lengths)
    tgt = rng.integers(0, n, src.size).astype(np.int32)
    w = rng.integers(1, 9, src.size).astype(np.float32)
    d, r = rng.integers(1, L, src.size).astype(np.uint8), rng.integers(0, 4, src.size).astype(np.uint8)
    csr = net.coo_to_csr(src, tgt, w, d, r, n_rows=n, major="source")
    active = np.arange(n_active, dtype=np.int32)
    want = np.zeros((L, 4, n))
    orc.deliver_events(active, 1, csr, want, n, 3)
    ring = torch.zeros(L, 4, n, device="cuda")
    ids = torch.zeros(n, dtype=torch.int32, device="cuda")
    ids[:n_active] = to_dev(active)
    ops.csr_propagate_scatter(ids, to_dev(np.array([n_active], np.int32)), ops.SynapseTable.from_numpy(csr), ring, n, 1, 3,
                              max_active=None if bound is None else n_active)
    np.testing.assert_array_equal(ring.cpu().numpy(), want)


def test_empty_rows_and_no_spikes():
    n, L = 70, 4
    csr = net.coo_to_csr(np.array([5], np.int32), np.array([9], np.int32), np.array([2.0], np.float32),
                         np.array([3], np.uint8), np.array([1], np.uint8), n_rows=n, major="source")
    ring = torch.zeros(L, 4, n, device="cuda")
    comp = ops.SpikeCompactor(n)
    z = np.zeros(n, np.uint8)
    ids, count = comp(to_dev(z))
    ops.csr_propagate_scatter(ids, count, ops.SynapseTable.from_numpy(csr), ring, n, 1, 2)
    assert not ring.any()
    z[[5, 6]] = 1
    ids, count = comp(to_dev(z))
    ops.csr_propagate_scatter(ids, count, ops.SynapseTable.from_numpy(csr), ring, n, 1, 2)
    assert ring[(2 + 3) % L, 1, 9].item() == 2.0 and ring.sum().item() == 2.0


def test_propagate_argument_errors():
    from bmtk_amd._lib import BmtkAmdError
    n = 10
    csr = net.coo_to_csr(np.array([1], np.int32), np.array([2], np.int32), np.array([1.0], np.float32),
                         np.array([1], np.uint8), np.array([0], np.uint8), n_rows=n, major="target")
    t = ops.SynapseTable.from_numpy(csr)
    zb = torch.zeros(2, dtype=torch.int64, device="cuda")
    with pytest.raises(BmtkAmdError):
        ops.csr_propagate_gather(zb, n, t, torch.zeros(17, 4, n, device="cuda"), n, 1, 0)   # L > 16
    with pytest.raises(ValueError):
        ops.csr_propagate_gather(zb, n, t, torch.zeros(4, 4, n + 1, device="cuda"), n, 1, 0)
    with pytest.raises(ValueError):
        net.check_csr(csr, n, n, 1)         # delay 1 needs at least 2 slots


@pytest.mark.parametrize("batch,p", [(1, 0.3), (5, 0.2), (32, 0.05), (64, 0.01), (64, 0.3), (100, 0.1), (130, 0.05)])
def test_pull_matches_oracle(batch, p):
    """Pull form: what arrives in step tau computed from the spike bits of the
    last L steps.  LDS atomics add in arbitrary order, so the comparison is with
    the fp64 oracle at 1e-5 of max(|want|, 1e-2 * sum of |w| into the cell)."""
    rng = np.random.default_rng(40 + batch)
    n_src, n_tgt, L = 211, 190, 6
    src, tgt, w, d, r = _edges(rng, n_src, n_tgt, 15000)
    by_src = net.coo_to_csr(src, tgt, w, d, r, n_rows=n_src, major="source")
    by_tgt = net.coo_to_csr(src, tgt, w, d, r, n_rows=n_tgt, major="target")
    table = ops.SynapseTable.from_numpy(by_tgt)
    words = ops.n_words(n_src * batch)
    hist = torch.zeros(L, words + 1, dtype=torch.int64, device="cuda")
    abs_src = (by_src[0], by_src[1], np.abs(by_src[2]), by_src[3], by_src[4])
    z_of = {}
    syn = torch.full((4, n_tgt * batch), 7.0, device="cuda")      # must be overwritten, not accumulated
    for tau in range(1, 14):
        k = tau - 1                                                  # the newest emitting step
        z_of[k] = (rng.random(n_src * batch) < p).astype(np.uint8)
        hist[k % L] = to_dev(bits_of(z_of[k]))
        ring = np.zeros((L, 4, n_tgt * batch))
        mag = np.zeros((L, 4, n_tgt * batch))
        for kk in range(max(0, tau - (L - 1)), tau):
            orc.deliver_events(np.flatnonzero(z_of[kk]), batch, by_src, ring, n_tgt, kk)
            orc.deliver_events(np.flatnonzero(z_of[kk]), batch, abs_src, mag, n_tgt, kk)
        ops.csr_propagate_pull(hist, n_src, table, syn, n_tgt, batch, tau)
        got = syn.cpu().numpy()
        want, m = ring[tau % L], mag[tau % L]
        assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-2 * m + 1e-30)) < 1e-5
        assert np.all(got[m == 0] == 0)
    assert np.abs(want).max() > 0


@pytest.mark.parametrize("n,batch,L,k", [(1, 1, 6, 400), (255, 1, 6, 300), (257, 3, 6, 250), (5000, 1, 6, 120), (1023, 8, 2, 150), (70, 1, 63, 200), (30011, 2, 6, 100)])
def test_delivery_by_target_ranges_equals_the_walk(n, batch, L, k, monkeypatch):
    """Fewer, as many and more targets than ranges, ranges without targets, several trials, two slots and many: what an atomic per event
    gives, bit for bit (quarter-pA weights: exact sums in any order), from no active element to all."""
    rng = np.random.default_rng(n + batch)
    src, tgt, w, d, r = _edges(rng, n, n, n * k, max_delay=L - 1)
    w = (np.round(w * 4) / 4).astype(np.float32)
    table = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
    if table.nnz < 100 * n or table.range_rows_min(n, batch, L) == 0:
        pytest.skip("not a table for ranges")
    seg = table.ranges(n)
    assert seg is not None and table.ranges(n) is seg
    from bmtk_amd import _lib
    start = torch.as_tensor(np.round(rng.normal(0, 10, (L, 4, n * batch)) * 4) / 4, device="cuda", dtype=torch.float32)
    for share in (0.0, 0.01, 0.2, 1.0):
        on = np.flatnonzero(rng.random(n * batch) < share).astype(np.int32)
        ids, count = to_dev(np.concatenate([on, np.full(1, -7, np.int32)])), to_dev(np.array([on.size], np.int32))
        want, got = start.clone(), start.clone()
        monkeypatch.setattr(ops.SynapseTable, "range_rows_min", lambda *a: 0)
        ops.csr_propagate_scatter(ids, count, table, want, n, batch, 13, max_active=n * batch)
        monkeypatch.undo()
        for rows_min in (0, 1 << 30):
            got.copy_(start)
            _lib.check(_lib.load().bmtk_csr_propagate_scatter_ranges(ids.data_ptr(), count.data_ptr(), batch, *table.pointers(), seg.data_ptr(),
                                                                     -(-n // 256), 256, rows_min, got.data_ptr(), L, n, 13, ops._stream()))
            assert torch.equal(want, got), (share, rows_min)
        got.copy_(start)
        ops.csr_propagate_scatter(ids, count, table, got, n, batch, 13, max_active=n * batch)
        assert torch.equal(want, got)


def test_delivery_by_target_ranges_follows_a_table_that_is_written_to():
    """Weights, delays, receptors and targets changed in place behind the offsets; rows whose order is lost; other row bounds; a table
    that was never sorted: always what an atomic per event gives."""
    rng = np.random.default_rng(3)
    n, L, nnz = 600, 6, 600 * 150
    src, tgt, w, d, r = _edges(rng, n, n, nnz)
    w = (np.round(w * 4) / 4).astype(np.float32)
    table = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
    ids, count = torch.arange(n, device="cuda", dtype=torch.int32), torch.tensor([n], device="cuda", dtype=torch.int32)

    def check(t):
        want, got = torch.zeros(L, 4, n, device="cuda"), torch.zeros(L, 4, n, device="cuda")
        from bmtk_amd import _lib
        _lib.check(_lib.load().bmtk_csr_propagate_scatter(ids.data_ptr(), count.data_ptr(), n, 1, *t.pointers(), want.data_ptr(), L, n, 4, ops._stream()))
        ops.csr_propagate_scatter(ids, count, t, got, n, 1, 4)
        assert torch.equal(want, got) and float(want.abs().max()) > 0

    assert 0 < table.range_rows_min(n, 1, L) <= n
    check(table)
    seg = table.ranges(n)
    table.weights.mul_(-2)
    table.delays.copy_(torch.randint(1, L, (nnz,), device="cuda"))
    table.receptors.copy_(torch.randint(0, 4, (nnz,), device="cuda"))
    check(table)
    table.indices.copy_(torch.randint(0, n, (nnz,), device="cuda"))      # targets leave their ranges, rows are no longer in order
    check(table)
    assert table.ranges(n) is seg
    table.indptr[1:-1] = torch.arange(1, n, device="cuda") * (nnz // n)  # other rows
    check(table)
    assert table.ranges(n) is None
    for order in (torch.arange(nnz - 1, -1, -1, device="cuda"), torch.arange(nnz, device="cuda")):
        t = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
        rows = torch.repeat_interleave(torch.arange(n, device="cuda"), (t.indptr[1:] - t.indptr[:-1]).long())
        by = torch.sort(rows[order], stable=True).indices
        t.indices, t.weights = t.indices[order][by].contiguous(), t.weights[order][by].contiguous()
        check(t)
        assert (t.ranges(n) is None) == (order[0].item() != 0)


def test_a_captured_delivery_follows_row_bounds_written_later():
    """A captured call keeps no offsets: its replays read the row bounds of their own time."""
    rng = np.random.default_rng(5)
    n, L, nnz = 600, 6, 600 * 150
    src, tgt, w, d, r = _edges(rng, n, n, nnz)
    w = (np.round(w * 4) / 4).astype(np.float32)
    table = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
    ids, count = torch.arange(n, device="cuda", dtype=torch.int32), torch.tensor([n], device="cuda", dtype=torch.int32)
    got, want = torch.zeros(L, 4, n, device="cuda"), torch.zeros(L, 4, n, device="cuda")
    ops.csr_propagate_scatter(ids, count, table, got, n, 1, 4)
    assert table.ranges(n) is not None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got.zero_()
        ops.csr_propagate_scatter(ids, count, table, got, n, 1, 4)
    for bounds in (None, torch.arange(1, n, device="cuda") * (nnz // n), torch.arange(1, n, device="cuda") * 3):
        if bounds is not None:
            table.indptr[1:-1] = bounds
        ops.csr_propagate_scatter(ids, count, table, want.zero_(), n, 1, 4)
        graph.replay()
        assert torch.equal(want, got)
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        ops.csr_propagate_scatter(ids, count, table, got.zero_(), n, 1, 4)
    torch.cuda.current_stream().wait_stream(other)
    assert torch.equal(want, got)
    with pytest.raises(RuntimeError):
        ops.csr_propagate_scatter(ids, count, table, torch.zeros(1, 4, n, device="cuda"), n, 1, 4)


def test_delivery_by_target_ranges_of_row_bounds_written_unseen():
    """Row bounds rewritten behind the version counter (a captured write replayed, ``.data``, a DLPack view): shifted and shortened rows,
    all synapses in one row, rows outside their old bounds.  Always what an atomic per event gives, with the offsets of before."""
    rng = np.random.default_rng(7)
    n, L, nnz = 600, 6, 600 * 150
    src, tgt, w, d, r = _edges(rng, n, n, nnz)
    w = (np.round(w * 4) / 4).astype(np.float32)
    table = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
    on = np.union1d(rng.choice(n, n // 2, replace=False), [0, 299, n - 1]).astype(np.int32)
    ids, count = to_dev(on), to_dev(np.array([on.size], np.int32))
    from bmtk_amd import _lib

    def walked():
        want = torch.zeros(L, 4, n, device="cuda")
        _lib.check(_lib.load().bmtk_csr_propagate_scatter(ids.data_ptr(), count.data_ptr(), n, 1, *table.pointers(), want.data_ptr(), L, n, 4, ops._stream()))
        return want

    def ranged():
        got = torch.zeros(L, 4, n, device="cuda")
        ops.csr_propagate_scatter(ids, count, table, got, n, 1, 4)
        return got

    assert 0 < table.range_rows_min(n, 1, L) <= on.size and torch.equal(ranged(), walked())
    before = walked()
    i = torch.arange(1, n, device="cuda", dtype=torch.int32)
    bounds = [i * (nnz // n), i * 3, (i >= 300).to(torch.int32) * nnz, torch.full_like(i, nnz), torch.full_like(i, 0), nnz - (n - i) * 140]
    fresh = torch.zeros_like(i)
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        torch.add(fresh, 0, out=table.indptr[1:-1])
    table.ranges(n)          # (the capture itself was counted, its replays are not)
    seg = table.ranges(n)
    for b in bounds:
        fresh.copy_(b)
        graph.replay()
        want, got = walked(), ranged()
        assert torch.equal(want, got) and not torch.equal(want, before)
        assert table.ranges(n) is seg
    view = torch.from_dlpack(table.indptr.detach())
    for how in (table.indptr.data, view):
        for b in bounds:
            how[1:-1] = b
            assert torch.equal(walked(), ranged())


@pytest.mark.parametrize("sort", [True, False])
def test_delivery_by_target_ranges_of_a_table_made_under_inference_mode(sort):
    """Such tensors have no version counter: delivered in the mode and after it, also where row bounds were rewritten in the mode."""
    rng = np.random.default_rng(8)
    n, L, nnz = 600, 6, 600 * 150
    src, tgt, w, d, r = _edges(rng, n, n, nnz)
    w = (np.round(w * 4) / 4).astype(np.float32)
    from bmtk_amd import _lib
    with torch.inference_mode():
        table = ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n)
        if not sort:
            table.indices = table.indices.flip(0).contiguous()
    assert table.indptr.is_inference()
    on = np.union1d(rng.choice(n, n // 2, replace=False), [0, n - 1]).astype(np.int32)
    ids, count = to_dev(on), to_dev(np.array([on.size], np.int32))

    def check():
        want, got = torch.zeros(L, 4, n, device="cuda"), torch.zeros(L, 4, n, device="cuda")
        _lib.check(_lib.load().bmtk_csr_propagate_scatter(ids.data_ptr(), count.data_ptr(), n, 1, *table.pointers(), want.data_ptr(), L, n, 4, ops._stream()))
        ops.csr_propagate_scatter(ids, count, table, got, n, 1, 4)
        assert torch.equal(want, got) and float(want.abs().max()) > 0

    assert 0 < table.range_rows_min(n, 1, L) <= on.size
    check()
    with torch.inference_mode():
        check()
        table.indptr[1:-1] = torch.arange(1, n, device="cuda") * 3
        check()
    check()
    assert (table.ranges(n) is not None) == sort


def test_delivery_where_the_offsets_find_no_room(monkeypatch):
    """The walk takes the call, and does not ask for the memory again."""
    rng = np.random.default_rng(9)
    n, L, nnz = 600, 6, 600 * 150
    src, tgt, w, d, r = _edges(rng, n, n, nnz)
    w = (np.round(w * 4) / 4).astype(np.float32)
    table, other = (ops.SynapseTable.from_edges(src, tgt, w, d, r, n, n) for _ in range(2))
    ids, count = torch.arange(n, device="cuda", dtype=torch.int32), torch.tensor([n], device="cuda", dtype=torch.int32)
    want, got = torch.zeros(L, 4, n, device="cuda"), torch.zeros(L, 4, n, device="cuda")
    ops.csr_propagate_scatter(ids, count, other, want, n, 1, 4)
    asked = []

    def no_room(self, *a):
        asked.append(a)
        raise torch.OutOfMemoryError("none left")
    monkeypatch.setattr(ops.SynapseTable, "segment_offsets", no_room)
    for _ in range(2):
        ops.csr_propagate_scatter(ids, count, table, got.zero_(), n, 1, 4)
        assert torch.equal(want, got) and len(asked) == 1


@pytest.mark.parametrize("field,dtype", [("indices", torch.int16), ("indices", torch.int64), ("indptr", torch.int64), ("indptr", torch.int16)])
def test_delivery_and_segment_offsets_refuse_other_types_before_reading_them(field, dtype):
    rng = np.random.default_rng(10)
    n, L, nnz = 600, 6, 600 * 150
    table = ops.SynapseTable.from_edges(*_edges(rng, n, n, nnz), n, n)
    setattr(table, field, getattr(table, field).to(dtype))
    ids, count = torch.arange(n, device="cuda", dtype=torch.int32), torch.tensor([n], device="cuda", dtype=torch.int32)
    assert 0 < table.range_rows_min(n, 1, L) <= n
    with pytest.raises(TypeError, match=field):
        ops.csr_propagate_scatter(ids, count, table, torch.zeros(L, 4, n, device="cuda"), n, 1, 4)
    with pytest.raises(TypeError, match=field):
        table.segment_offsets(7, 30)
    assert getattr(table, "_ranges", None) is None


@pytest.mark.parametrize("span,n_groups", [(7, 30), (64, 4), (1, 211), (300, 1), (100, 2)])
def test_segment_offsets_are_what_a_search_finds(span, n_groups):
    """Empty rows, rows of one synapse and of several chunks, repeated targets, targets beyond the last group, first and last groups empty."""
    rng = np.random.default_rng(span)
    lens = rng.integers(0, 200, 50)
    lens[[0, 3, 49]] = 0
    lens[[1, 4]] = 1, 64
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    idx = np.concatenate([np.sort(rng.integers(0, 211, m)) for m in lens]).astype(np.int32)
    one = np.ones(idx.size, np.uint8)
    t = ops.SynapseTable(to_dev(indptr), to_dev(idx), to_dev(one.astype(np.float32)), to_dev(one), to_dev(one), n_rows=50, max_row=200)
    want = np.stack([indptr[j] + np.searchsorted(idx[indptr[j]:indptr[j + 1]], np.arange(n_groups + 1) * span) for j in range(50)])
    np.testing.assert_array_equal(t.segment_offsets(span, n_groups).cpu().numpy(), want)
    t.indices[indptr[-1] - 1] = 0
    with pytest.raises(ValueError):
        t.segment_offsets(span, n_groups)


@pytest.mark.parametrize("batch,p,n_src,L", [(1, 0.3, 211, 6), (5, 0.2, 211, 6), (32, 0.05, 1500, 6), (64, 0.01, 211, 6),
                                              (64, 0.3, 211, 6), (100, 0.1, 97, 6), (130, 0.05, 211, 6),
                                              (64, 0.05, 211, 2), (32, 0.05, 400, 8), (64, 0.05, 211, 9), (5, 0.2, 300, 14)])
def test_two_step_pull_equals_two_pulls(batch, p, n_src, L):
    """``csr_propagate_pull2`` (the arrivals of steps tau-1 and tau in one pass over the table) == two calls of
    ``csr_propagate_pull`` over the same spike history, bit for bit: both add the same Q31.32 weights, whose sum
    does not depend on the order.  (The one-step form is pinned against the oracle above.)  Histories of up to 8
    rows take the form with one byte of activity per source, longer ones the form with one bit per row and
    source; delays run up to L - 1 steps, the longest a history of L rows serves."""
    rng = np.random.default_rng(70 + batch + L)
    n_tgt = 190
    src, tgt, w, d, r = _edges(rng, n_src, n_tgt, 15000, max_delay=L - 1)
    table = ops.SynapseTable.from_numpy(net.coo_to_csr(src, tgt, w, d, r, n_rows=n_tgt, major="target"))
    words = ops.n_words(n_src * batch)
    hist = torch.zeros(L, words + 1, dtype=torch.int64, device="cuda")
    one = torch.full((2, 4, n_tgt * batch), 7.0, device="cuda")
    two = torch.full((2, 4, n_tgt * batch), -3.0, device="cuda")      # must be overwritten, not accumulated
    for tau in range(1, 2 * L + 4):
        hist[(tau - 1) % L] = to_dev(bits_of((rng.random(n_src * batch) < p).astype(np.uint8)))
        if tau <= L:                                                   # both steps need their L-1 steps of history
            continue
        # the row of step tau-1 is never read by the pull of step tau-1: delays are at least one step
        ops.csr_propagate_pull(hist, n_src, table, one[0], n_tgt, batch, tau - 1)
        ops.csr_propagate_pull(hist, n_src, table, one[1], n_tgt, batch, tau)
        ops.csr_propagate_pull2(hist, n_src, table, two, n_tgt, batch, tau)
        assert torch.equal(one, two), tau
        assert float(one[0].abs().max()) > 0 and not torch.equal(one[0], one[1])


@pytest.mark.parametrize("batch,L,two", [(64, 6, True), (12, 6, True), (64, 9, True), (100, 6, True), (64, 6, False)])
def test_pulls_of_one_table_on_two_streams_and_in_a_graph(batch, L, two):
    """Two streams at work at once with histories of their own, and a captured call replayed beside them:
    none reads what another call has laid out."""
    rng = np.random.default_rng(batch + L)
    n_src, n_tgt, reps = 20000, 3000, 30
    src, tgt, w, d, r = _edges(rng, n_src, n_tgt, 400000, max_delay=L - 1)
    table = ops.SynapseTable.from_numpy(net.coo_to_csr(src, tgt, w, d, r, n_rows=n_tgt, major="target"))
    words = ops.n_words(n_src * batch)
    hist = [torch.zeros(L, words + 1, dtype=torch.int64, device="cuda") for _ in range(3)]
    for h in hist:
        h[:, :-1] = torch.as_tensor(rng.integers(0, 2**62, (L, words)) & rng.integers(0, 2**62, (L, words)) & rng.integers(0, 2**62, (L, words)), device="cuda")
    out = lambda: torch.zeros(2 if two else 1, 4, n_tgt * batch, device="cuda")  # noqa: E731

    def pull(h, to):
        if two:
            ops.csr_propagate_pull2(h, n_src, table, to, n_tgt, batch, L)
        else:
            ops.csr_propagate_pull(h, n_src, table, to, n_tgt, batch, L)

    want = [out() for _ in hist]
    for h, x in zip(hist, want):
        pull(h, x)
        torch.cuda.synchronize()
    assert not torch.equal(want[0], want[1])
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [[out() for _ in range(reps)] for _ in streams]
    graph, replayed = torch.cuda.CUDAGraph(), out()
    with torch.cuda.graph(graph):
        pull(hist[2], replayed)
    torch.cuda.synchronize()
    for k in range(reps):
        for s, h, g in zip(streams, hist, got):
            with torch.cuda.stream(s):
                pull(h, g[k])
        replayed.zero_()
        graph.replay()
        if k % 10 == 9:
            torch.cuda.current_stream().synchronize()
            assert torch.equal(replayed, want[2])
    torch.cuda.synchronize()
    for g, x in zip(got, want):
        assert all(torch.equal(y, x) for y in g)


@pytest.mark.parametrize("two", [True, False])
def test_pulls_of_one_table_from_two_threads_share_no_scratch_memory(monkeypatch, two):
    """A call that begins while another thread's is under way, on the same stream, works in memory of its own: the launches of the two
    may come in any order."""
    import threading
    from bmtk_amd import _lib
    rng = np.random.default_rng(3)
    n, L, batch = 500, 6, 64
    src, tgt, w, d, r = _edges(rng, n, n, 20000)
    table = ops.SynapseTable.from_numpy(net.coo_to_csr(src, tgt, w, d, r, n_rows=n, major="target"))
    hist = torch.zeros(L, ops.n_words(n * batch) + 1, dtype=torch.int64, device="cuda")
    hist[:, :-1] = 0x0101010101010101
    name, f = ("bmtk_csr_propagate_pull2", ops.csr_propagate_pull2) if two else ("bmtk_csr_propagate_pull", ops.csr_propagate_pull)
    real, scratch = _lib.load(), []
    out = [torch.zeros(2 if two else 1, 4, n * batch, device="cuda") for _ in range(2)]

    class Lib:
        def __getattr__(self, what):
            return getattr(real, what) if what != name else self.pull

        def pull(self, *args):
            scratch.append(args[-2])
            if len(scratch) == 1:
                other = threading.Thread(target=f, args=(hist, n, table, out[1], n, batch, L))
                other.start()
                other.join()
            return getattr(real, name)(*args)

    monkeypatch.setattr(_lib, "load", lambda *a, **k: lib)
    lib = Lib()
    f(hist, n, table, out[0], n, batch, L)
    assert len(scratch) == 2 and scratch[0] != scratch[1]
    assert torch.equal(*out) and float(out[0].abs().max()) > 0


@pytest.mark.parametrize("n_tgt,nnz,batch,power", [(3, 4000, 64, 1.0), (5000, 70000, 33, 6.0), (9001, 8500000, 32, 3.0), (40000, 8400000, 8, 8.0)])
def test_two_step_pull_of_rows_of_very_unequal_length(n_tgt, nnz, batch, power):
    """Targets drawn as n * x**power: rows from several tenths of the table down to none, empty ones first and last, on either side
    of the size from which workgroups begin at their share of the synapses.  Equal to two calls of the one-step form, bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(n_tgt)
    n_src, L = 700, 6
    tgt = (torch.rand(nnz, device="cuda", generator=g, dtype=torch.float64) ** power * (n_tgt - 2)).long() + (1 if n_tgt > 3 else 0)
    src = torch.randint(0, n_src, (nnz,), device="cuda", generator=g)
    table = ops.SynapseTable.from_edges(tgt, src, torch.randn(nnz, device="cuda", generator=g),
                                        torch.randint(1, L, (nnz,), device="cuda", generator=g, dtype=torch.uint8),
                                        torch.randint(0, 4, (nnz,), device="cuda", generator=g, dtype=torch.uint8), n_tgt, n_src)
    hist = torch.zeros(L, ops.n_words(n_src * batch) + 1, dtype=torch.int64, device="cuda")
    for row in hist:
        row[:-1] = to_dev(bits_of((torch.rand(n_src * batch, device="cuda", generator=g) < 0.01).to(torch.uint8).cpu().numpy()))[:row.numel() - 1]
    one = torch.full((2, 4, n_tgt * batch), 7.0, device="cuda")
    two = torch.full((2, 4, n_tgt * batch), -3.0, device="cuda")
    ops.csr_propagate_pull(hist, n_src, table, one[0], n_tgt, batch, 2 * L - 1)
    ops.csr_propagate_pull(hist, n_src, table, one[1], n_tgt, batch, 2 * L)
    ops.csr_propagate_pull2(hist, n_src, table, two, n_tgt, batch, 2 * L)
    # (the one-step pull of step t - 1 reads the row of step t - 1 as that of step t - 1 - L: no delay is that long)
    assert torch.equal(one, two) and float(two.abs().max()) > 0


@pytest.mark.parametrize("batch,L", [(64, 6), (5, 6), (32, 8), (64, 2), (1, 3)])
def test_two_step_auto_delivery_equals_the_oracle(batch, L):
    """``ops.AutoPropagator2`` (bmtk_csr_propagate_auto2): called every second step, each of the two new steps goes
    out as events or is left to a pull that sums two arrival steps in one pass.  The same run as for the one-step
    switch -- activity from nothing to 20 % and back, so that pushed and pulled steps mix within and across calls
    and arrival slots hold pushed weights when the pull adds its sums -- with quarter-pA weights: after every call
    both arrival slots must equal the fp32 oracle's bit for bit, also with thresholds that force one form."""
    rng = np.random.default_rng(34 + batch + L)
    n, T = 500, 40
    src, tgt, w, d, r = _edges(rng, n, n, 30000, max_delay=L - 1)
    w = (np.round(w * 4) / 4 + np.sign(w) * 0.25).astype(np.float32)
    by_src = net.coo_to_csr(src, tgt, w, d, r, n_rows=n, major="source")
    by_tgt = net.csr_transpose(by_src, n)
    t_src, t_tgt = ops.SynapseTable.from_numpy(by_src), ops.SynapseTable.from_numpy(by_tgt)
    ne = n * batch
    comp_a, comp_b = ops.SpikeCompactor(ne), ops.SpikeCompactor(ne)
    rates = [0.0, 0.0, 0.002, 0.2, 0.002, 0.0, 0.2, 0.2, 0.01, 0.002, 0.2, 0.0, 0.002] * 4
    zs = [(rng.random(ne) < rates[k]).astype(np.uint8) for k in range(T)]
    counts = sorted(int(z.sum()) for z in zs)
    mid = counts[len(counts) // 2]
    for thr in (mid, 0, ne, counts[-1] - 1):
        want = np.zeros((L, 4, ne), np.float32)
        hist = torch.zeros(L, ops.n_words(ne) + 1, dtype=torch.int64, device="cuda")
        ring = torch.zeros(L, 4, ne, device="cuda")
        auto = ops.AutoPropagator2(t_src, t_tgt, hist, ring, n, n, batch, scatter_max_active=thr)
        seen = set()
        for k in range(1, T, 2):
            lists = []
            for step, comp in ((k - 1, comp_a), (k, comp_b)):
                orc.gather_rows(zs[step], batch, by_tgt, want, n, step)
                hist[step % L] = to_dev(bits_of(zs[step]))
                lists += list(comp(to_dev(zs[step])))
            auto.step2(k, *lists)
            pulled = auto.pulled_steps()
            seen |= {bool(pulled[(k - 1) % L]), bool(pulled[k % L])}
            for slot in (k % L, (k + 1) % L):
                np.testing.assert_array_equal(ring[slot].cpu().numpy(), want[slot],
                                              err_msg="call %d slot %d threshold %d" % (k, slot, thr))
                ring[slot].zero_()    # the consumer's part: both slots are read and cleared before the next call
                want[slot] = 0.0
        if thr == mid:
            assert seen == {True, False}      # both forms ran
        elif thr == ne:
            assert seen == {False}


def test_table_from_edges_on_the_device_equals_the_host_build():
    from bmtk_amd import network as net
    rng = np.random.default_rng(5)
    n_rows, n_cols, nnz = 300, 450, 20000
    src, tgt = rng.integers(0, n_rows, nnz), rng.integers(0, n_cols, nnz)
    w = rng.normal(size=nnz).astype(np.float32)
    r = rng.integers(0, 4, nnz).astype(np.uint8)
    for d in (rng.integers(1, 6, nnz), rng.integers(100, 1000, nnz)):
        want = net.coo_to_csr(src, tgt, w, d, r, n_rows, "source")
        got = ops.SynapseTable.from_edges(src, tgt, w, d, r, n_rows, n_cols)
        for a, b in zip(want, (got.indptr, got.indices, got.weights, got.delays, got.receptors)):
            np.testing.assert_array_equal(a, b.cpu().numpy())
            assert a.dtype == b.cpu().numpy().dtype
    with pytest.raises(ValueError):
        ops.SynapseTable.from_edges(src, tgt + n_cols, w, d, r, n_rows, n_cols)


@pytest.mark.parametrize("batch", [1, 24, 64])
def test_auto_delivery_picks_a_form_on_the_device_and_the_ring_is_the_oracles(batch):
    """``ops.AutoPropagator`` (bmtk_csr_propagate_auto): step by step the active count decides on the device whether
    a step's spikes are pushed into the ring as events or left to the pull over the spike history.  A run whose
    activity goes from nothing to 20 % and back mixes the two forms in every way -- pushed steps between pulled
    ones, arrival slots that hold pushed weights when the pull adds its sums, stretches with nothing to pull.
    Quarter-pA weights: after every call the arrival slot must equal the fp32 oracle's bit for bit, whatever the
    mix, also with thresholds that force one form throughout."""
    rng = np.random.default_rng(33)
    n, L, T = 500, 6, 40
    src, tgt, w, d, r = _edges(rng, n, n, 30000)
    w = (np.round(w * 4) / 4 + np.sign(w) * 0.25).astype(np.float32)
    by_src = net.coo_to_csr(src, tgt, w, d, r, n_rows=n, major="source")
    by_tgt = net.csr_transpose(by_src, n)
    t_src, t_tgt = ops.SynapseTable.from_numpy(by_src), ops.SynapseTable.from_numpy(by_tgt)
    ne = n * batch
    comp = ops.SpikeCompactor(ne)
    rates = [0.0, 0.0, 0.002, 0.2, 0.002, 0.0, 0.2, 0.2, 0.01, 0.002] * 4
    zs = [(rng.random(ne) < rates[k]).astype(np.uint8) for k in range(T)]
    counts = sorted(int(z.sum()) for z in zs)
    mid = counts[len(counts) // 2]
    for thr in (mid, 0, ne, counts[-1] - 1):
        want = np.zeros((L, 4, ne), np.float32)
        hist = torch.zeros(L, ops.n_words(ne) + 1, dtype=torch.int64, device="cuda")
        ring = torch.zeros(L, 4, ne, device="cuda")
        auto = ops.AutoPropagator(t_src, t_tgt, hist, ring, n, n, batch, scatter_max_active=thr)
        seen = set()
        for k in range(T):
            orc.gather_rows(zs[k], batch, by_tgt, want, n, k)
            hist[k % L] = to_dev(bits_of(zs[k]))
            ids, cnt = comp(to_dev(zs[k]))
            auto.step(k, ids, cnt)
            seen.add(bool(auto.pulled_steps()[k % L]))
            slot = (k + 1) % L
            np.testing.assert_array_equal(ring[slot].cpu().numpy(), want[slot], err_msg="step %d threshold %d" % (k, thr))
            ring[slot].zero_()        # the consumer's part: the slot is read and cleared before the next call
            want[slot] = 0.0
        assert np.abs(want).max() > 0 or thr == mid
        if thr == mid:
            assert seen == {True, False}      # both forms ran
        elif thr == 0:
            assert seen == {True} or 0 in counts
        elif thr == ne:
            assert seen == {False}


def test_native_pointer_checks_are_the_general_ones():
    """What passes gives the tensor's pointer, what does not the general way's exception, word for word."""
    from bmtk_amd import _ptr
    general = next(f for f in gc_functions() if f.__name__ == "_p")
    x = torch.zeros(4, 6, device="cuda")
    calls = [(None,), (x,), (x, torch.float32), (x, torch.float32, 24), (x, None, 3, "x"), (x[1:],), (x[:0],), (torch.nn.Parameter(x),), (x.requires_grad_(),),
             (x.detach().to(torch.complex64).conj(),), (x, torch.int32, 24, "ring"), (x, torch.float32, 25, "ring"), (x.t(), None, None, "t"), (x[:, :2],), (x.cpu(),),
             (x, torch.float32, 24.0), (x, torch.float32, 1 << 70), (x, "float"), (x.to_sparse(),), (5,), ()]
    for args in calls:
        outs = []
        for f in (_ptr.ptr, general):
            try:
                outs.append(f(*args))
            except Exception as exc:
                outs.append((type(exc), str(exc)))
        assert outs[0] == outs[1], args
    assert _ptr.ptr(x, name="y") == x.data_ptr() and ops._p is _ptr.ptr
    with pytest.raises(ValueError, match="y holds 24"):
        _ptr.ptr(x, numel=25, name="y")


def gc_functions():
    import gc
    import types
    return [f for f in gc.get_objects() if isinstance(f, types.FunctionType) and f.__module__ == "bmtk_amd.ops"]
