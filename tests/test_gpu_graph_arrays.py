"""The graph arrays the library keeps in HBM, read back through medusa_graph_device_arrays:
CSR as given, CSC offsets and sources, and the CSR-to-CSC slot map (the reference's
msgDstID, built by EdgeArray::buildAA), each equal to the oracle's CSC build on RMAT-20 and
on a small graph with duplicate edges, self-loops and vertices without edges."""
import ctypes

import numpy as np
import pytest

import medusa_amd as md
from medusa_amd import workloads as wl
from conftest import csr_from_edges

pytestmark = pytest.mark.gpu
HIP_MEMCPY_DEVICE_TO_HOST = 2


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[case] {request.node.nodeid}", flush=True)


def _d2h(ptr, count):
    """Copies `count` uint32 from device address `ptr` with the HIP runtime the library uses."""
    memcpy = md.lib().hipMemcpy
    memcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    memcpy.restype = ctypes.c_int
    out = np.empty(count, np.uint32)
    if count:
        assert memcpy(out.ctypes.data, ptr, out.nbytes, HIP_MEMCPY_DEVICE_TO_HOST) == 0
    return out


def _check(oracle, rp, col):
    n, m = len(rp) - 1, len(col)
    cptr, csrc, slot = oracle.csc(rp, col)
    with md.Graph(rp, col) as G:
        a = G.device_arrays()
        assert np.array_equal(_d2h(a["row_ptr"], n + 1), rp)
        assert np.array_equal(_d2h(a["col"], m), col)
        assert np.array_equal(_d2h(a["csc_ptr"], n + 1), cptr)
        assert np.array_equal(_d2h(a["csc_src"], m), csrc)
        assert np.array_equal(_d2h(a["msg_slot"], m), slot)
    # the slot map sends CSR edge e (u -> v) to a CSC position of v whose source is u
    src_of_e = np.repeat(np.arange(n, dtype=np.uint32), np.diff(rp.astype(np.int64)))
    assert np.array_equal(csrc[slot], src_of_e)
    assert np.all((slot >= cptr[col]) & (slot < cptr[col + 1]))
    assert np.array_equal(np.sort(slot), np.arange(m, dtype=np.uint32))  # every CSC position once


def test_device_arrays_match_oracle_csc_small(oracle):
    edges = [(0, 1), (0, 1), (2, 2), (1, 0), (4, 1), (4, 3), (1, 4), (4, 1)]
    rp, col, _ = csr_from_edges(6, edges)
    _check(oracle, rp, col)


def test_device_arrays_match_oracle_csc_rmat20(oracle):
    rp, col = wl.rmat_graph()
    _check(oracle, rp, col)


class _DeviceArray:
    """An allocation of `nbytes` of device memory, every byte 7."""

    def __init__(self, nbytes):
        L = md.lib()
        L.hipMalloc.argtypes, L.hipMalloc.restype = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t], ctypes.c_int
        L.hipFree.argtypes, L.hipFree.restype = [ctypes.c_void_p], ctypes.c_int
        L.hipMemset.argtypes, L.hipMemset.restype = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t], ctypes.c_int
        p = ctypes.c_void_p()
        assert L.hipMalloc(ctypes.byref(p), nbytes) == 0
        self.base, self.nbytes = p.value, nbytes
        self.clear()

    def clear(self):
        assert md.lib().hipMemset(self.base, 7, self.nbytes) == 0
        assert md.lib().hipDeviceSynchronize() == 0

    def at(self, offset):
        class Out:
            data_ptr = lambda _: self.base + offset  # noqa: E731
        return Out()

    def bytes(self):
        return _d2h(self.base, self.nbytes // 4).view(np.uint8)

    def free(self):
        assert md.lib().hipFree(self.base) == 0


@pytest.mark.parametrize("short", [4, 4096])
def test_device_output_past_its_allocation_is_refused(oracle, short):
    """A device output whose allocation ends before the result does is an error of every entry point,
    host- and device-driven, and nothing is written; one that ends where the result does is filled."""
    n, k = 40_000, 9
    rng = np.random.default_rng(short)
    rp, col, _ = csr_from_edges(n, rng.integers(0, n, (4 * n, 2)))
    w = rng.integers(1, 1001, len(col)).astype(np.uint32)
    srcs = rng.integers(0, n, k).astype(np.uint32)
    calls = [(4 * n, lambda G, o: G.bfs(0, out=o), lambda: oracle.bfs_queue(rp, col, 0)),
             (4 * n, lambda G, o: G.bfs(0, out=o, timing=1), lambda: oracle.bfs_queue(rp, col, 0)),
             (4 * n, lambda G, o: G.sssp(0, out=o), lambda: oracle.sssp_dijkstra(rp, col, w, 0)),
             (4 * n, lambda G, o: G.sssp(0, out=o, timing=1), lambda: oracle.sssp_dijkstra(rp, col, w, 0)),
             (4 * n, lambda G, o: G.pagerank(0.85, 3, out=o), lambda: oracle.pagerank_f32(rp, col, 0.85, 3)),
             (k * n, lambda G, o: G.mbfs(srcs, out=o), lambda: oracle.mbfs(rp, col, srcs)),
             (k * n, lambda G, o: G.mbfs(srcs, out=o, timing=1), lambda: oracle.mbfs(rp, col, srcs))]
    with md.Graph(rp, col, w) as G:
        for i, (need, call, want) in enumerate(calls):
            print(f"[case] call {i}", flush=True)
            A = _DeviceArray(need + 256)
            call(G, A.at(256))
            got = A.bytes()
            assert (got[:256] == 7).all() and np.array_equal(got[256:], np.ascontiguousarray(want()).view(np.uint8).ravel())
            A.clear()
            with pytest.raises(md.MedusaError) as e:
                call(G, A.at(256 + short))
            assert e.value.code == -2  # MEDUSA_ERR_HIP
            assert (A.bytes() == 7).all(), i
            A.free()


class _MappedArray:
    """`nbytes` of device memory behind one address range of two mappings (hipMemMap)."""

    class _Location(ctypes.Structure):
        _fields_ = [("type", ctypes.c_int), ("id", ctypes.c_int)]

    class _Prop(ctypes.Structure):
        pass

    class _Access(ctypes.Structure):
        pass

    _Prop._fields_ = [("type", ctypes.c_int), ("handle_types", ctypes.c_int), ("location", _Location),
                      ("win32", ctypes.c_void_p), ("flags", ctypes.c_uint32)]
    _Access._fields_ = [("location", _Location), ("flags", ctypes.c_int)]

    def __init__(self, nbytes):
        L, size, ull = md.lib(), ctypes.c_size_t, ctypes.c_ulonglong
        here = self._Location(1, 0)  # hipMemLocationTypeDevice
        prop = self._Prop(1, 0, here, None, 0)  # hipMemAllocationTypePinned
        gran = size()
        assert L.hipMemGetAllocationGranularity(ctypes.byref(gran), ctypes.byref(prop), ctypes.c_int(1)) == 0
        half = -(-(nbytes // 2) // gran.value) * gran.value
        assert half < nbytes <= 2 * half
        va = ctypes.c_void_p()
        assert L.hipMemAddressReserve(ctypes.byref(va), size(2 * half), size(0), ctypes.c_void_p(), ull(0)) == 0
        self.base, self.half, self.handles = va.value, half, []
        for i in range(2):
            h = ctypes.c_void_p()
            assert L.hipMemCreate(ctypes.byref(h), size(half), ctypes.byref(prop), ull(0)) == 0
            assert L.hipMemMap(ctypes.c_void_p(self.base + i * half), size(half), size(0), h, ull(0)) == 0
            self.handles.append(h)
        access = self._Access(here, 3)  # hipMemAccessFlagsProtReadWrite
        assert L.hipMemSetAccess(va, size(2 * half), ctypes.byref(access), size(1)) == 0

    def data_ptr(self):
        return self.base

    def free(self):
        L = md.lib()
        for i, h in enumerate(self.handles):
            assert L.hipMemUnmap(ctypes.c_void_p(self.base + i * self.half), ctypes.c_size_t(self.half)) == 0
            assert L.hipMemRelease(h) == 0
        assert L.hipMemAddressFree(ctypes.c_void_p(self.base), ctypes.c_size_t(2 * self.half)) == 0


def test_device_output_over_two_mappings(oracle):
    """An output over both mappings of an address range, of which HIP names one at a time, is filled."""
    n, k = 1_048_576, 8
    rng = np.random.default_rng(5)
    rp, col, _ = csr_from_edges(n, rng.integers(0, n, (4 * n, 2)))
    w = rng.integers(1, 1001, len(col)).astype(np.uint32)
    srcs = rng.integers(0, n, k).astype(np.uint32)
    calls = [(4 * n, lambda G, o: G.bfs(0, out=o), lambda: oracle.bfs_queue(rp, col, 0)),
             (4 * n, lambda G, o: G.sssp(0, out=o), lambda: oracle.sssp_dijkstra(rp, col, w, 0)),
             (4 * n, lambda G, o: G.pagerank(0.85, 3, out=o), lambda: oracle.pagerank_f32(rp, col, 0.85, 3)),
             (k * n, lambda G, o: G.mbfs(srcs, out=o), lambda: oracle.mbfs(rp, col, srcs))]
    with md.Graph(rp, col, w) as G:
        for i, (need, call, want) in enumerate(calls):
            print(f"[case] call {i}", flush=True)
            A = _MappedArray(need)
            call(G, A)
            got = _d2h(A.data_ptr(), need // 4)
            assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want()).view(np.uint8).ravel()), i
            A.free()
