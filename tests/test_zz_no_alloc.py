"""e3x_csr_build_static (sort buffers in a static device array, no allocation) against e3x_csr_build.

Integer work: the row pointers and the permutation must be bit-identical.  Two calls in a row share the static
buffers, the second on a smaller edge list, so stale contents of the first call must not leak into it.
"""
import numpy as np
import pytest
import torch

from e3nn_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _build(dst, N, static):
    L = _lib.lib()
    E = dst.numel()
    rowptr = torch.full((N + 1,), -7, dtype=torch.int32, device=DEV)
    perm = torch.full((max(E, 1),), -7, dtype=torch.int32, device=DEV)
    st = _lib.stream_ptr(DEV)
    bits = dst.element_size() * 8
    if static:
        rc = L.e3x_csr_build_static(_lib.ptr(dst), bits, E, N, _lib.ptr(rowptr), _lib.ptr(perm), st)
    else:
        nbytes = L.e3x_csr_workspace_bytes(E, N)
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=DEV)
        rc = L.e3x_csr_build(_lib.ptr(dst), bits, E, N, _lib.ptr(rowptr), _lib.ptr(perm), _lib.ptr(ws), nbytes, st)
    _lib.check(rc)
    torch.cuda.synchronize()
    return rowptr.cpu().numpy(), perm[:E].cpu().numpy()


def _reference(dst, N):
    d = dst.cpu().numpy().astype(np.int64)
    perm = np.argsort(d, kind="stable").astype(np.int32)
    rowptr = np.searchsorted(d[perm], np.arange(N + 1), side="left").astype(np.int32)
    return rowptr, perm


def test_static_scratch_matches_workspace_entry_point_twice_in_a_row():
    g = torch.Generator().manual_seed(5)
    cases = [(200_000, 30_000, torch.int64), (4_321, 97, torch.int32), (0, 11, torch.int64)]
    with torch.cuda.device(DEV):
        for E, N, dt in cases:  # big, then smaller, then empty: all on the same static buffers
            dst = torch.randint(0, N, (E,), generator=g).to(dt).to(DEV)
            rp_s, pm_s = _build(dst, N, static=True)
            rp_w, pm_w = _build(dst, N, static=False)
            rp_r, pm_r = _reference(dst, N)
            assert np.array_equal(rp_s, rp_w) and np.array_equal(pm_s, pm_w), (E, N)
            assert np.array_equal(rp_s, rp_r) and np.array_equal(pm_s, pm_r), (E, N)


def _graph(kind, E, N, n_src, g):
    src, dst = torch.randint(0, n_src, (E,), generator=g), torch.randint(0, N, (E,), generator=g)
    if kind == "grouped":
        dst = torch.sort(dst)[0]
    if kind == "star":  # one row longer than a wavefront puts in order: the general sort
        dst[: E // 2] = N // 2
    if kind == "long":  # the longest that it does
        dst = dst % (N - 1) + 1
        dst[torch.randperm(E, generator=g)[:1024]] = 0
    if kind == "band":  # rows that share sources
        src = (dst + torch.randint(-3, 4, (E,), generator=g)) % n_src
    if kind == "negative":
        src = src - n_src * torch.randint(0, 2, (E,), generator=g)
    return src, dst


@pytest.mark.parametrize("kind,E,N,n_src", [
    ("random", 1, 1, 1), ("random", 2, 5, 3), ("random", 5000, 63, 70), ("random", 4097, 4096, 4096), ("random", 9000, 4097, 4097),
    ("grouped", 6001, 300, 300), ("band", 20000, 2500, 2500), ("star", 6000, 50, 50), ("long", 9000, 400, 400), ("negative", 3000, 200, 150),
    ("random", 300, 1, 40), ("random", 30000, 16384, 16384), ("random", 30000, 16385, 16385), ("random", 3000, 100, 70000), ("band", 60, 8200, 8200),
    # lists that are looked at before they are sorted, and the largest that are not
    ("random", 2_000_001, 20_000, 20_000), ("grouped", 2_000_001, 20_000, 20_000), ("random", 2_000_000, 20_000, 20_000),
    ("random", 2_000_001, 16_000, 16_000), ("star", 2_000_001, 20_000, 20_000),
])  # fmt: skip
@pytest.mark.parametrize("src_t,dst_t", [(torch.int64, torch.int64), (torch.int32, torch.int64)])
def test_edge_list_in_one_call_matches_the_separate_entry_points(kind, E, N, n_src, src_t, dst_t):
    import ctypes

    L = _lib.lib()
    src, dst = (t.to(DEV) for t in _graph(kind, E, N, n_src, torch.Generator().manual_seed(E + N)))
    src, dst = src.to(src_t), dst.to(dst_t)
    st, bits = _lib.stream_ptr(DEV), (src.element_size() * 8, dst.element_size() * 8)
    want_ptr, want_perm = (torch.from_numpy(a).to(DEV) for a in _build(dst, N, static=False))
    want_order, want_pairs = torch.empty(N, dtype=torch.int32, device=DEV), ctypes.c_int32(-1)
    n = L.e3x_row_order_workspace_bytes(N)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    _lib.check(L.e3x_row_order_build(_lib.ptr(src), bits[0], _lib.ptr(want_ptr), _lib.ptr(want_perm), E, N, n_src, _lib.ptr(want_order),
                                     ctypes.byref(want_pairs), _lib.ptr(ws), n, st))  # fmt: skip
    for with_order in (True, False):
        rowptr, perm, order = (torch.full((k,), -7, dtype=torch.int32, device=DEV) for k in (N + 1, E, N))
        grouped, pairs = ctypes.c_int32(-1), ctypes.c_int32(-1)
        n = L.e3x_edges_workspace_bytes(E, N)
        ws = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
        _lib.check(L.e3x_edges_build(_lib.ptr(src), bits[0], _lib.ptr(dst), bits[1], E, N, n_src, _lib.ptr(rowptr), _lib.ptr(perm),
                                     _lib.ptr(order) if with_order else None, ctypes.byref(grouped), ctypes.byref(pairs), _lib.ptr(ws), n, st))  # fmt: skip
        assert torch.equal(rowptr, want_ptr) and torch.equal(perm, want_perm)
        assert grouped.value == int(bool((dst[1:] >= dst[:-1]).all()))
        if with_order:
            assert torch.equal(order, want_order) and pairs.value == want_pairs.value
    for bad_src, bad_dst in ((n_src, 0), (-n_src - 1, 0), (0, N), (0, -1)):
        s, d = src.clone(), dst.clone()
        s[E // 2], d[E // 2] = bad_src, bad_dst
        rc = L.e3x_edges_build(_lib.ptr(s), bits[0], _lib.ptr(d), bits[1], E, N, n_src, _lib.ptr(rowptr), _lib.ptr(perm), _lib.ptr(order),
                               ctypes.byref(grouped), ctypes.byref(pairs), _lib.ptr(ws), n, st)  # fmt: skip
        with pytest.raises(IndexError, match="gather source" if bad_dst == 0 else "scatter destination"):
            _lib.check(rc)


def test_static_scratch_reports_bad_indices_and_clears_the_flag():
    with torch.cuda.device(DEV):
        bad = torch.tensor([0, 3, 9, 1], dtype=torch.int64, device=DEV)
        with pytest.raises(IndexError):
            _build(bad, 5, static=True)
        good = torch.tensor([0, 3, 4, 1], dtype=torch.int64, device=DEV)  # the flag of the failed call is gone
        rp, pm = _build(good, 5, static=True)
        assert rp.tolist() == [0, 1, 2, 2, 3, 4] and pm.tolist() == [0, 3, 1, 2]


def test_static_scratch_rejects_edge_lists_beyond_its_buffers():
    L = _lib.lib()
    cap = L.e3x_csr_static_scratch_bytes()
    E = 1 << 21
    assert L.e3x_csr_workspace_bytes(E, 1 << 20) <= cap  # the documented size always fits
    too_many = cap // 4  # three 4-byte arrays per edge alone exceed the buffer
    one = torch.zeros(1, dtype=torch.int32, device=DEV)
    rc = L.e3x_csr_build_static(_lib.ptr(one), 32, too_many, 8, _lib.ptr(one), _lib.ptr(one), _lib.stream_ptr(DEV))
    assert rc == _lib.ERR_INVALID
    assert b"static buffer" in L.e3x_last_error()


def test_static_scratch_host_threads_take_turns():
    # two host threads on streams of their own share the device's one array; the library serialises them (a per-device
    # lock from the first launch to the final synchronisation), so both get the right answer
    import threading

    g = torch.Generator().manual_seed(9)
    jobs = [(150_000, 20_000), (90_000, 7_000)]
    dsts = [torch.randint(0, N, (E,), generator=g).to(DEV) for E, N in jobs]
    results = [None, None]

    def work(i):
        L = _lib.lib()
        E, N = jobs[i]
        with torch.cuda.device(DEV):
            stream = torch.cuda.Stream(device=DEV)
            rowptr = torch.empty(N + 1, dtype=torch.int32, device=DEV)
            perm = torch.empty(E, dtype=torch.int32, device=DEV)
            torch.cuda.synchronize()
            for _ in range(5):
                rc = L.e3x_csr_build_static(_lib.ptr(dsts[i]), 64, E, N, _lib.ptr(rowptr), _lib.ptr(perm), _lib.c_void_p(stream.cuda_stream))
                if rc != 0:
                    results[i] = rc
                    return
            stream.synchronize()
            results[i] = (rowptr.cpu().numpy(), perm.cpu().numpy())

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, (E, N) in enumerate(jobs):
        assert isinstance(results[i], tuple), results[i]
        rp, pm = _reference(dsts[i], N)
        assert np.array_equal(results[i][0], rp) and np.array_equal(results[i][1], pm)
