"""The status bits of malformed input are the same on every kernel path.

Each case of tests/status_cases.py runs through the C ABI with the workspace
that selects each kernel path, and through the host twins; every one must
report the hand-derived bits.  node2vec validates the whole CSR on every
call, so its bits depend neither on the path nor on the seed; the uniform
walk reports what its walks read.
"""
import ctypes
import time

import numpy as np
import pytest
import torch

import mlx_cluster_amd as mc
from mlx_cluster_amd import _lib, synth
from tests import status_cases as sc

pytestmark = pytest.mark.gpu

N2V_MODES = ("lds", "records", "csr", "few", "few_tables", "direct")
ROWS = (_lib.MLXC_ROWS_UNSORTED, _lib.MLXC_ROWS_SORTED, _lib.MLXC_ROWS_DETECT)


def _t(a, cuda):
    return torch.as_tensor(np.asarray(a, dtype=np.int64)).to(cuda)


def _n2v_status(rowptr, col, start, L, seed, rows, mode, cuda):
    lib = _lib.load()
    rowptr, col, start = _t(rowptr, cuda), _t(col, cuda), _t(start, cuda)
    V, E, N = rowptr.numel() - 1, col.numel(), start.numel()
    p, q, rule = 0.5, 2.0, _lib.MLXC_RULE_REF_CHAIN
    query = lambda n_, l_: lib.mlxc_rejection_sampling_workspace_bytes(V, E, n_, l_, p, q, rule)
    layout = {"direct": _lib.MLXC_N2V_LAYOUT_DIRECT, "csr": _lib.MLXC_N2V_LAYOUT_CSR,
              "records": _lib.MLXC_N2V_LAYOUT_RECORDS_FULL, "lds": _lib.MLXC_N2V_LAYOUT_LDS}
    if mode in layout:
        nbytes = max(lib.mlxc_rejection_sampling_layout_bytes(V, E, N, L, layout[mode]), 32)
    else:
        nbytes = {"few": 64, "few_tables": 64 + (E + 1) // 2 * 16 + 8192}[mode]
    if mode == "lds":
        assert query(N, L) == 256  # the query itself selects the LDS walk here
    ws = torch.full(((nbytes + 7) // 8,), -1, dtype=torch.int64, device=cuda)
    n = torch.empty((N, L + 1), dtype=torch.int64, device=cuda)
    e = torch.empty((N, L), dtype=torch.int64, device=cuda)
    rc = lib.mlxc_rejection_sampling(rowptr.data_ptr(), V, col.data_ptr(), E, start.data_ptr(),
                                     N, L, p, q, seed, 0, rule, rows, n.data_ptr(), e.data_ptr(),
                                     _lib.MLXC_OUT_INT64, ws.data_ptr(), nbytes,
                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    return int(ws[0].item())


@pytest.mark.parametrize("case", sc.N2V_CASES, ids=[c[0] for c in sc.N2V_CASES])
def test_node2vec_status_same_on_every_path(case, cuda):
    name, rowptr, col, start, want = case
    lib = _lib.load()
    L = 3
    for seed in (0, 1):
        for rows in ROWS:
            got = {mode: _n2v_status(rowptr, col, start, L, seed, rows, mode, cuda)
                   for mode in N2V_MODES}
            got["host"] = sc.host_node2vec_status(lib, rowptr, col, start, L, 0.5, 2.0, seed,
                                                  _lib.MLXC_RULE_REF_CHAIN, rows)
            assert all(v == want for v in got.values()), (name, seed, rows, got)
        if want:
            with pytest.raises(ValueError):
                mc.rejection_sampling(_t(rowptr, cuda), _t(col, cuda), _t(start, cuda), L,
                                      0.5, 2.0, seed=seed)
        else:
            mc.rejection_sampling(_t(rowptr, cuda), _t(col, cuda), _t(start, cuda), L, 0.5, 2.0,
                                  seed=seed)


def _uniform_status(rowptr, col, start, L, mode, seeded, cuda):
    lib = _lib.load()
    rowptr, col, start = _t(rowptr, cuda), _t(col, cuda), _t(start, cuda)
    V, E, N = rowptr.numel() - 1, col.numel(), start.numel()
    nbytes = {"lds": 256, "records": 256 + 16 * (E + N), "csr": 256 + 16 * N, "plain": 32}[mode]
    ws = torch.full(((nbytes + 7) // 8,), -1, dtype=torch.int64, device=cuda)
    n = torch.empty((N, L + 1), dtype=torch.int64, device=cuda)
    e = torch.empty((N, max(L, 1)), dtype=torch.int64, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    graph = (rowptr.data_ptr(), V, col.data_ptr(), E, start.data_ptr(), N)
    outs = (n.data_ptr(), e.data_ptr(), _lib.MLXC_OUT_INT64, ws.data_ptr(), nbytes, stream)
    if seeded:
        rc = lib.mlxc_random_walk_seeded(*graph, L, 5, 0, *outs)
    else:
        rand = torch.full((max(N * L, 1),), 0.5, dtype=torch.float32, device=cuda)
        rc = lib.mlxc_random_walk(*graph, rand.data_ptr(), L, *outs)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    return int(ws[0].item())


@pytest.mark.parametrize("case", sc.UNI_CASES, ids=[c[0] for c in sc.UNI_CASES])
def test_uniform_status_same_on_every_path(case, cuda):
    """16 walks (the case's starts repeated), so that N * L is a multiple of
    4 and at least 16: the rand tensor then allows the windowed kernels, and
    the record and CSR workspaces select those walks, the others the flat walk."""
    name, rowptr, col, start, L, want = case
    lib = _lib.load()
    start = np.resize(np.asarray(start, np.int64), 16)
    for seeded in (False, True):
        got = {mode: _uniform_status(rowptr, col, start, L, mode, seeded, cuda)
               for mode in ("lds", "records", "csr", "plain")}
        got["host"] = sc.host_uniform_status(lib, rowptr, col, start, L,
                                             seed=5 if seeded else None)
        assert all(v == want for v in got.values()), (name, seeded, got)


@pytest.mark.parametrize("case", sc.UNI_CASES, ids=[c[0] for c in sc.UNI_CASES])
def test_published_status_is_the_workspace_word(case, cuda):
    """mlxc_publish_status stores the call's status word into host memory and
    then its flag: the word equals workspace word 0 read back by a copy, and
    the compiled binding's check (which waits on those host words) raises
    exactly when it is non-zero."""
    name, rowptr, col, start, L, want = case
    lib = _lib.load()
    hip = ctypes.CDLL("libamdhip64.so")  # the HIP runtime torch has loaded
    words = ctypes.c_void_p()
    flags = 0x40000000 | 0x2 | 0x1  # hipHostMallocCoherent | Mapped | Portable
    assert hip.hipHostMalloc(ctypes.byref(words), ctypes.c_size_t(16), ctypes.c_uint(flags)) == 0
    try:
        h = (ctypes.c_int64 * 2).from_address(words.value)
        start = np.resize(np.asarray(start, np.int64), 16)
        r, c, s = _t(rowptr, cuda), _t(col, cuda), _t(start, cuda)
        V, E, N = r.numel() - 1, c.numel(), s.numel()
        nbytes = 256 + 16 * (E + N)
        ws = torch.full(((nbytes + 7) // 8,), -1, dtype=torch.int64, device=cuda)
        n = torch.empty((N, L + 1), dtype=torch.int64, device=cuda)
        stream = torch.cuda.current_stream().cuda_stream
        for _ in range(2):  # the second time over the first call's host words
            h[0], h[1] = 0, -1
            rc = lib.mlxc_random_walk_seeded(r.data_ptr(), V, c.data_ptr(), E, s.data_ptr(), N, L,
                                             5, 0, n.data_ptr(), None, _lib.MLXC_OUT_INT64,
                                             ws.data_ptr(), nbytes, stream)
            assert rc == 0, _lib.last_error()
            assert lib.mlxc_publish_status(ws.data_ptr(), words, stream) == 0, _lib.last_error()
            deadline = time.monotonic() + 30
            while h[0] == 0:
                assert time.monotonic() < deadline, "the status was not published"
            assert h[1] == int(ws[0].item()) == want, (name, h[1], want)
    finally:
        torch.cuda.synchronize()
        hip.hipHostFree(words)
    if want:
        with pytest.raises(ValueError):
            mc.random_walk(r, c, s, None, L, seed=5)
    else:
        mc.random_walk(r, c, s, None, L, seed=5)


@pytest.fixture
def status_words():
    """Three host words the device can write, with mlxc_set_status_target
    undone afterwards."""
    hip = ctypes.CDLL("libamdhip64.so")
    words = ctypes.c_void_p()
    flags = 0x40000000 | 0x2 | 0x1  # hipHostMallocCoherent | Mapped | Portable
    assert hip.hipHostMalloc(ctypes.byref(words), ctypes.c_size_t(24), ctypes.c_uint(flags)) == 0
    yield words.value, (ctypes.c_int64 * 3).from_address(words.value)
    _lib.load().mlxc_set_status_target(None)
    torch.cuda.synchronize()
    hip.hipHostFree(words)


def test_status_target_of_every_kind_of_call(status_words, cuda):
    """With a thread's status target set, every walk call and CSR build on the
    thread leaves its status bits in word 1 (a build its entry count in word
    2) and 1 in word 0, whichever of its launches publishes them: flat,
    record, LDS and few-walks walks (with and without row tables), calls
    without walks, noalloc, small, large and empty builds.  Validated calls of
    the Python layer keep the target; after NULL nothing is written."""
    lib = _lib.load()
    address, h = status_words
    stream = torch.cuda.current_stream().cuda_stream
    rowptr, col = (t.to(cuda) for t in synth.rmat_csr(12, 40_000, seed=5, symmetrize=True))
    V, E = rowptr.numel() - 1, col.numel()
    N, L = 300, 9
    out = torch.empty((N, L + 1), dtype=torch.int64, device=cuda)
    ws = torch.zeros(1 << 20, dtype=torch.int64, device=cuda)
    good = torch.arange(N, device=cuda) % V
    bad = good.clone()
    bad[7] = V

    def uniform(start, nbytes, n=N):
        return lib.mlxc_random_walk_seeded(rowptr.data_ptr(), V, col.data_ptr(), E,
                                           start.data_ptr(), n, L, 3, 0, out.data_ptr(), None, 0,
                                           ws.data_ptr(), nbytes, stream)

    def n2v(start, nbytes, n=N):
        return lib.mlxc_rejection_sampling(rowptr.data_ptr(), V, col.data_ptr(), E,
                                           start.data_ptr(), n, L, 0.5, 2.0, 3, 0, 0,
                                           _lib.MLXC_ROWS_DETECT, out.data_ptr(), None, 0,
                                           ws.data_ptr(), nbytes, stream)

    rand = torch.zeros(N * L, device=cuda)
    noalloc = lambda start: lib.mlxc_random_walk_noalloc(
        rowptr.data_ptr(), V, col.data_ptr(), E, start.data_ptr(), N, rand.data_ptr(), L,
        out.data_ptr(), None, 0, None, stream)
    tables = 64 + (E + 1) // 2 * 16 + 8192
    walks = {"flat, zeroed word": lambda s: uniform(s, 32), "flat": lambda s: uniform(s, 32 + 4 * N),
             "csr": lambda s: uniform(s, 256 + 16 * N),
             "records": lambda s: uniform(s, 256 + 16 * (E + N)), "few": lambda s: n2v(s, 64),
             "few, tables": lambda s: n2v(s, tables), "direct": lambda s: n2v(s, 32),
             "n2v records": lambda s: n2v(s, lib.mlxc_rejection_sampling_layout_bytes(
                 V, E, N, L, _lib.MLXC_N2V_LAYOUT_RECORDS_FULL)), "noalloc": noalloc}
    small_rp, small_cl = (t.to(cuda) for t in synth.rmat_csr(8, 1000, seed=5))

    def lds(start, nbytes):
        return lib.mlxc_rejection_sampling(small_rp.data_ptr(), 256, small_cl.data_ptr(),
                                           small_cl.numel(), start.data_ptr(), N, L, 0.5, 2.0, 3, 0,
                                           0, _lib.MLXC_ROWS_DETECT, out.data_ptr(), None, 0,
                                           ws.data_ptr(), nbytes, stream)

    walks["lds, words of its blocks"] = lambda s: lds(s.clamp(max=255) + (s == V), 1280)
    walks["lds"] = lambda s: lds(s.clamp(max=255) + (s == V), 256)

    def run(call, *args):
        h[0], h[1], h[2] = 0, -1, -1
        assert call(*args) == 0, _lib.last_error()
        torch.cuda.synchronize()
        return list(h)

    assert lib.mlxc_set_status_target(address) == 0, _lib.last_error()
    assert lib.mlxc_status_target() == address
    for name, call in walks.items():
        assert run(call, good) == [1, 0, -1], name
        assert run(call, bad) == [1, _lib.MLXC_STATUS_BAD_NODE, -1], name
    assert run(uniform, good, 32, 0) == [1, 0, -1]
    assert run(n2v, good, 64, 0) == [1, 0, -1]
    ids = torch.randint(0, 4096, (2, 300_000), device=cuda)
    rp2, cl2 = torch.empty(4097, dtype=torch.int64, device=cuda), torch.empty_like(ids[0])

    def build(n, nodes=4096):
        nbytes = lib.mlxc_csr_build_workspace_bytes(nodes, n, 0)
        assert nbytes <= ws.numel() * 8
        return lib.mlxc_csr_build(ids[0].data_ptr(), ids[1].data_ptr(), n, nodes, 0,
                                  rp2.data_ptr(), cl2.data_ptr(), ws.data_ptr(), nbytes, stream)

    for n in (0, 5_000, 300_000):
        assert run(build, n) == [1, 0, n]
    assert run(build, 5_000, 100)[:2] == [1, _lib.MLXC_STATUS_BAD_NODE]
    assert run(build, 300_000, 100)[:2] == [1, _lib.MLXC_STATUS_BAD_NODE]
    # validated calls of the Python layer wait on words of their own
    mc.random_walk(rowptr, col, good, None, L, seed=3)
    mc.rejection_sampling(rowptr, col, good, L, 0.5, 2.0, seed=3)
    mc.to_csr(ids, 4096)
    with pytest.raises(ValueError):
        mc.random_walk(rowptr, col, bad, None, L, seed=3)
    assert lib.mlxc_status_target() == address
    assert run(walks["flat"], good) == [1, 0, -1]
    assert lib.mlxc_set_status_target(None) == 0 and lib.mlxc_status_target() is None
    assert run(walks["flat"], good) == [0, -1, -1]
    assert run(build, 5_000) == [0, -1, -1]
    mc.random_walk(rowptr, col, good, None, L, seed=3)
    assert lib.mlxc_status_target() is None
