"""Save / load (reference tests/test_exact.py:219-239, test_updates.cu:459-498) and searches that
run while another thread adds vectors (test_exact.py:367-405): every search must equal the exact
answer over one of the published prefixes."""

import os
import threading
import time

import numpy as np
import pytest
import torch

import libcertex_amd as certex
import oracle
from tests import data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.uint8, np.float32, np.float16])
def test_save_load(gpu, tmp_path, dtype):
    if dtype == np.uint8:
        X, Q = data.mixture_u8(20_000, seed=1), data.mixture_u8(100, seed=2)
    else:
        X, Q = data.gaussian(20_000, 64, 1, dtype), data.gaussian(100, 64, 2, dtype)
    idx = certex.Index(X.shape[1], metric="l2")
    idx.add(X)
    idx.remove(torch.arange(0, 20_000, 7))
    labels = None
    D0, I0 = idx.search(Q, k=10)
    path = tmp_path / "index.cx"
    idx.save(path)
    back = certex.Index.load(path)
    assert back.ntotal == idx.ntotal and back.dtype == idx.dtype and back.metric == "l2"
    D1, I1 = back.search(Q, k=10)
    np.testing.assert_array_equal(I0, I1)
    np.testing.assert_array_equal(D0, D1)
    back.add(X[:1000])  # a loaded index keeps growing
    assert back.ntotal == idx.ntotal + 1000


@pytest.mark.parametrize("dtype", [np.uint8, np.float32])
def test_save_load_in_chunks(gpu, tmp_path, dtype):
    """Arrays larger than the 64 MiB staging buffers move in several chunks each (an odd count for
    the rows), with labels and lists; the loaded index answers exactly as the saved one."""
    if dtype == np.uint8:
        X = data.mixture_u8(1_300_000, seed=7)  # 166 MB of rows: 3 chunks
        Q = data.mixture_u8(300, seed=8)
    else:
        X = data.gaussian(330_000, 128, 7, np.float32)  # 169 MB of vectors: 3 chunks
        Q = data.gaussian(300, 128, 8, np.float32)
    labels = torch.from_numpy(np.random.default_rng(9).integers(0, 5, len(X)).astype(np.int32))
    idx = certex.Index(128, metric="l2", n_lists=32)
    idx.add(X, labels=labels)
    idx.remove(torch.arange(3, len(X), 101))
    D0, I0 = idx.search(Q, k=10)
    ql = torch.from_numpy(np.random.default_rng(10).integers(0, 5, len(Q)).astype(np.int32))
    Dl0, Il0 = idx.search(Q, k=10, labels=ql)
    path = tmp_path / "big.cx"
    idx.save(path)
    back = certex.Index.load(path)
    assert back.ntotal == idx.ntotal and back.core.lists == idx.core.lists
    assert torch.equal(back.list_order(), idx.list_order())
    D1, I1 = back.search(Q, k=10)
    np.testing.assert_array_equal(I0, I1)
    np.testing.assert_array_equal(D0, D1)
    Dl1, Il1 = back.search(Q, k=10, labels=ql)
    np.testing.assert_array_equal(Il0, Il1)
    np.testing.assert_array_equal(Dl0, Dl1)


def test_load_rejects_foreign_files(gpu, tmp_path):
    bad = tmp_path / "bad.cx"
    bad.write_bytes(b"<f4\x00" + (0x43455258).to_bytes(4, "little") + (1).to_bytes(4, "little") + b"\x00" * 64)
    with pytest.raises(ValueError, match="another version"):
        certex.Index.load(bad)
    with pytest.raises(ValueError):
        (tmp_path / "junk").write_bytes(b"hello world")
        certex.Index.load(tmp_path / "junk")


def search_while_adding(search, add):
    """search(nq) in a thread of its own and add() while it runs: what the search returned (or the
    exception that ended it). A search that did not go on for 20 ms (hundreds of batches) after the rows
    were added runs again with more queries."""
    for nq in (10_000, 40_000, 80_000):
        out = []

        def body():
            try:
                with torch.cuda.stream(torch.cuda.Stream()):
                    out.append(search(nq))
                    out.append(time.perf_counter())
                    torch.cuda.current_stream().synchronize()
            except BaseException as e:  # noqa: B036
                out[:] = [e]

        t = threading.Thread(target=body)
        t.start()
        time.sleep(0.05)
        add()
        torch.cuda.synchronize()
        added = time.perf_counter()
        t.join()
        if isinstance(out[0], BaseException) or out[1] - added > 0.02:
            return out[0]
    pytest.fail("no search went on after the rows were added")


def test_rows_added_past_an_id_map(gpu):
    """A mapped label search of many batches: rows that another thread adds past its map between two
    of them end it. The map is the start of a longer tensor, whose other entries no result may hold."""
    X = data.mixture_u8(3_000, seed=41)
    Xg = torch.from_numpy(X).cuda()
    idx = certex.Index(128)
    idx.add(Xg[:2_000], labels=torch.zeros(2_000, dtype=torch.int32))
    whole = torch.arange(40_000, device="cuda")

    def search(nq):
        n = idx.core.size
        return idx._search(Xg[2_000:].repeat(nq // 1_000, 1), 5, 1, torch.zeros(nq, dtype=torch.int32), None,
                           id_map=whole[:n])

    got = search_while_adding(search, lambda: idx.add(Xg[2_000:], labels=torch.zeros(1_000, dtype=torch.int32)))
    assert isinstance(got, ValueError) and "id map" in str(got), got


@pytest.mark.parametrize("entry", ["cuvsCertexSearch", "cuvsCertexSearchNoAlloc"])
@pytest.mark.parametrize("per_query", [False, True])
def test_rows_added_past_a_filter(gpu, per_query, entry):
    """A filtered search of many batches (row terms, or the filtered kernels of a search without
    allocation and of a mask per query): rows that another thread adds between two of them, whose ids
    the filter does not cover, are in no result. The filter words are the start of a longer tensor
    with every later bit set."""
    import ctypes

    from libcertex_amd import _capi as C

    X = data.mixture_u8(3_008, seed=43)
    Xg = torch.from_numpy(X).cuda()
    idx = certex.Index(128)
    idx.add(Xg[:2_048])
    words = torch.full((6_000_000,), -1, dtype=torch.int32, device="cuda")

    def search(nq):
        nq //= 2 if per_query else 1
        n = idx.core.size
        Q = Xg[2_048:].repeat(nq // 960 + 1, 1)[:nq].contiguous()
        I = torch.empty((nq, 5), dtype=torch.int64, device="cuda")
        D = torch.empty((nq, 5), dtype=torch.float32, device="cuda")
        sp = C.SearchParams(128, 1, 2)
        w = words[: (n * (nq if per_query else 1) + 31) // 32]
        qb, ib, db, wb = C.Borrowed(Q), C.Borrowed(I), C.Borrowed(D), C.Borrowed(w, dtype_override=(C.kDLUInt, 32))
        C.check(getattr(C.lib(), entry)(C.resources(), ctypes.byref(sp), idx.core.h, qb.ptr, ib.ptr, db.ptr,
                                        C.Filter(ctypes.addressof(wb.m), C.BITMAP if per_query else C.BITSET)))
        torch.cuda.current_stream().synchronize()
        return n, I

    n, I = search_while_adding(search, lambda: idx.add(Xg[2_048:]))
    assert bool((I >= 0).all()) and int(I.max()) < n
    assert bool((idx.search(Xg[2_048:], k=1)[1][:, 0] >= 2_048).all())


@pytest.mark.parametrize("host_labels", [True, False])
def test_row_labels_moved_during_a_label_search(gpu, host_labels):
    """A label search of many batches while rows added past the index's capacity move its row labels:
    the last queries, searched after that, see the new rows."""
    X = data.mixture_u8(3_008, seed=45)
    Xg = torch.from_numpy(X).cuda()
    labels = lambda n: torch.zeros(n, dtype=torch.int32)  # noqa: E731
    idx = certex.Index(128, partition_labels=False)
    idx.add(Xg[:2_048], labels=labels(2_048))
    new = len(X) - 2_048

    def search(nq):
        n, lq = idx.core.size, labels(nq)
        Q = Xg[2_048:].repeat(nq // new + 1, 1)[:nq]
        return n, nq, idx.search(Q, k=1, batch=1, labels=lq if host_labels else lq.cuda())[1]

    n, nq, I = search_while_adding(search, lambda: idx.add(Xg[2_048:], labels=labels(new)))
    last = int(I[-1, 0])
    assert last >= 2_048 and np.array_equal(X[2_048 + (last - 2_048) % new], X[2_048 + (nq - 1) % new])
    assert int(I.max()) < idx.core.size


@pytest.mark.parametrize("host_labels", [True, False])
def test_partition_dropped_during_a_label_search(gpu, host_labels):
    """A routed label search of many batches while another thread gives partitioned rows new labels,
    which drops the partition: the last query is answered by the new labels, every id once."""
    import ctypes

    from libcertex_amd import _capi as C

    X = data.mixture_u8(4_000, seed=47)
    Q = data.mixture_u8(1_000, seed=48)
    idx = certex.Index(128)
    idx.add(X, labels=torch.zeros(4_000, dtype=torch.int32))
    Qg = torch.from_numpy(Q).cuda()

    def search(nq):
        lq = torch.zeros(nq, dtype=torch.int32)
        return idx.search(Qg.repeat(nq // 1_000, 1), k=20, batch=1, labels=lq if host_labels else lq.cuda())[1]

    def relabel():
        lb = C.Borrowed(torch.ones(1_500, dtype=torch.int32, device="cuda"))
        C.check(C.lib().cuvsCertexSetLabels(C.resources(), lb.ptr, 0, idx.core.h))

    I = search_while_adding(search, relabel)
    assert idx.core.n_partitioned == 0
    want = oracle.knn(X[1_500:], Q[-1:], 20, "l2")[1] + 1_500
    np.testing.assert_array_equal(I[-1:].cpu().numpy(), want)


@pytest.mark.parametrize("dtype", [np.uint8, np.float32])
def test_concurrent_search_and_add(gpu, dtype):
    """Searches on three streams while a fourth adds rows: every search equals the oracle on one
    published snapshot. Float rows of 256 coordinates take the tiled screen, and additions raise
    the index's fp16 maxima (the certificate's operand bounds) while searches read them."""
    if dtype == np.uint8:
        X = data.mixture_u8(40_000, seed=5)
        Q = data.mixture_u8(200, seed=6)
    else:
        X = data.powerlaw_unit(40_000, 256, seed=5) * np.linspace(1, 3, 40_000, dtype=np.float32)[:, None]
        Q = data.powerlaw_unit(200, 256, seed=6)
    idx = certex.Index(X.shape[1])
    idx.add(X[:20_000])
    sizes = list(range(20_000, 40_001, 2_000))
    refs = [oracle.knn(X[:n], Q, 10, "l2")[1] for n in sizes]
    errors = []

    def writer():
        with torch.cuda.stream(torch.cuda.Stream()):
            for i in range(20_000, 40_000, 2_000):
                idx.add(X[i : i + 2_000])
            torch.cuda.current_stream().synchronize()

    def reader():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                Qg = torch.from_numpy(Q).cuda()
                for _ in range(10):
                    _, I = idx.search(Qg, k=10)
                    torch.cuda.current_stream().synchronize()
                    I = I.cpu().numpy()
                    ok = np.zeros(len(Q), bool)
                    for r in refs:
                        ok |= (I == r).all(1)
                    assert ok.all(), f"{int((~ok).sum())} queries match no snapshot"
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=writer)] + [threading.Thread(target=reader) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]
    assert idx.ntotal == 40_000
    _, I = idx.search(Q, k=10)
    np.testing.assert_array_equal(I, refs[-1])
