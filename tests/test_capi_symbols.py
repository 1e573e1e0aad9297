"""CPU-side checks of the C ABI: the library loads, exports every symbol that
include/hgcalml_amd.h declares, and rejects bad arguments on the host before
anything is launched (no GPU needed for any of this)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "hgcalml_amd.h")
LIB = os.path.join(ROOT, "hgcalml_amd", "libhgcalml_amd.so")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(hgc_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def capi():
    if not os.path.exists(LIB):
        from hgcalml_amd import build
        build.build(verbose=False)
    return ctypes.CDLL(LIB)


def test_header_declares_the_expected_entry_points():
    names = declared_symbols()
    for must in ("hgc_bin_by_coordinates", "hgc_binned_select_knn", "hgc_index_replacer", "hgc_accumulate_knn",
                 "hgc_accumulate_knn_grad", "hgc_binned_assign_to_condensates"):
        assert must in names


def test_library_exports_every_declared_symbol(capi):
    for name in declared_symbols():
        assert hasattr(capi, name), "missing export: " + name


def test_python_binding_covers_every_declared_symbol(capi):
    from hgcalml_amd import _lib
    assert sorted(_lib.EXPORTED_SYMBOLS) == declared_symbols()


def test_host_side_argument_checks(capi):
    capi.hgc_last_error.restype = ctypes.c_char_p
    assert capi.hgc_version() >= 100
    # total bins: host arithmetic
    nb = (ctypes.c_int * 3)(30, 29, 31)
    out = ctypes.c_int(0)
    assert capi.hgc_bin_by_coordinates_total_bins(nb, 3, 17, ctypes.byref(out)) == 0
    assert out.value == 30 * 29 * 31 * 16
    nb[1] = 0
    assert capi.hgc_bin_by_coordinates_total_bins(nb, 3, 17, ctypes.byref(out)) == -1
    assert b"positive" in capi.hgc_last_error()
    # kNN shape rules of the reference op: 2 <= binning dims <= 5, >= 2 coordinates
    null = ctypes.c_void_p(None)
    args_tail = [null] * 9
    f = capi.hgc_binned_select_knn
    f.argtypes = [ctypes.c_void_p] * 9 + [ctypes.c_int] * 7 + [ctypes.c_void_p]
    assert f(*args_tail, 10, 4, 3, 1, 5, 0, 0, null) == -1
    assert b"at least 2 binning dimensions" in capi.hgc_last_error()
    assert f(*args_tail, 10, 4, 3, 6, 5, 0, 0, null) == -1
    assert b"maximum 5 binning dimensions" in capi.hgc_last_error()
    assert f(*args_tail, 10, 4, 1, 2, 5, 0, 0, null) == -1
    assert f(*args_tail, 10, 4, 3, 3, 5, 0, 0, null) == -1 and b"null pointer" in capi.hgc_last_error()
    assert f(*args_tail, 0, 4, 3, 3, 5, 0, 0, null) == 0  # empty input is fine
    assert f(*args_tail, 150_000_000, 1, 8, 3, 5, 0, 0, null) == -1 and b"4 GiB" in capi.hgc_last_error()
    # accumulate: output width must match mean_and_max
    g = capi.hgc_accumulate_knn
    g.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int] * 6 + [ctypes.c_void_p]
    assert g(*([null] * 5), 10, 4, 8, 8, 0, 1, null) == -1
    assert g(*([null] * 5), 0, 4, 8, 16, 0, 1, null) == 0
    # workspace queries are pure host functions
    capi.hgc_sort_by_bin_workspace_bytes.restype = ctypes.c_size_t
    capi.hgc_inverse_neighbour_index_workspace_bytes.restype = ctypes.c_size_t
    assert capi.hgc_sort_by_bin_workspace_bytes(150000, 27000) >= 2 * 150000 * 4
    # the sorted keys, plus whatever rocPRIM asks for itself
    assert capi.hgc_inverse_neighbour_index_workspace_bytes(1000, 64) >= 64000 * 4
    # the one-call condensate wrapper: sizes checked on the host, the empty input needs no workspace
    capi.hgc_build_and_assign_condensates_workspace_bytes.restype = ctypes.c_size_t
    assert capi.hgc_build_and_assign_condensates_workspace_bytes(1000, 4, 2, 6, 3) > 1000 * 4 * 4
    assert capi.hgc_build_and_assign_condensates_workspace_bytes(1000, 17, 2, 6, 3) == 0
    c = capi.hgc_build_and_assign_condensates
    c.argtypes = ([ctypes.c_void_p] * 5 + [ctypes.c_int] * 3 + [ctypes.c_float] * 2 + [ctypes.c_int] * 3 +
                  [ctypes.c_void_p] * 6 + [ctypes.c_size_t, ctypes.c_void_p])
    one = ctypes.c_void_p(256)
    assert c(one, one, one, null, one, 10, 17, 1, 0.1, 1.0, 1, 3, 5, one, one, one, one, one, null, 0, null) == -1
    assert b"coordinate dimensions" in capi.hgc_last_error()
    assert c(one, one, one, null, one, 10, 4, 1, 0.1, 1.0, 1, 0, 5, one, one, one, one, one, null, 0, null) == -1
    assert c(one, one, one, null, one, 10, 4, 1, 0.1, 0.0, 1, 3, 5, one, one, one, one, one, null, 0, null) == -1
    assert b"distance_threshold" in capi.hgc_last_error()
    assert c(one, one, one, null, one, 10, 4, 1, 0.1, 1.0, 1, 3, 5, one, one, one, one, one, null, 0, null) == -2
    # missing workspace is reported, not dereferenced
    h = capi.hgc_sort_by_bin
    h.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                  ctypes.c_size_t, ctypes.c_void_p]
    assert h(one, 10, 10, one, one, null, 0, null) == -2


def test_limits_of_the_gravnet_passes(capi):
    """tables of up to 2^31 - 1 slots, as everywhere else, and rows of any width a tensor has: what is missing here is only the
    pointers"""
    capi.hgc_last_error.restype = ctypes.c_char_p
    p, i = ctypes.c_void_p, ctypes.c_int
    null = p(None)
    for f, before, after in ((capi.hgc_gravnet_drop_self, 2, 3), (capi.hgc_gravnet_drop_self_grad, 2, 2),
                             (capi.hgc_sumw_distance_grad, 3, 2)):
        f.argtypes = [p] * before + [i, i] + [p] * after
        for n, k, text in ((32537631, 66, b"null pointer"), (1 << 25, 64, b"2^31")):   # 2^31 - 2 and 2^31 slots
            assert f(*[null] * before, n, k, *[null] * after) == -1 and text in capi.hgc_last_error()
    capi.hgc_gravnet_join.argtypes = [p] * 3 + [i] * 3 + [p] * 2
    capi.hgc_gravnet_join_grad.argtypes = [p] + [i] * 3 + [p] * 4
    for f, x in ((4, 3 << 20), (3 << 20, 4)):
        assert capi.hgc_gravnet_join(*[null] * 3, 5, f, x, *[null] * 2) == -1 and b"null pointer" in capi.hgc_last_error()
        assert capi.hgc_gravnet_join_grad(null, 5, f, x, *[null] * 4) == -1 and b"null pointer" in capi.hgc_last_error()


def test_scratch_of_the_accumulation_gradient(capi):
    """the quotients: one float per vertex and feature, and none where the kernel that reads it is not taken (small tables; large ones
    in the next test)"""
    f = capi.hgc_accumulate_knn_grad_scratch_bytes
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int] * 4
    for mean_and_max in (0, 1):
        assert f(1000, 40, 64, mean_and_max) == 1000 * 64 * 4
        assert f(1000, 64, 64, mean_and_max) == 0                       # a power of two: no quotients needed
        assert f(1000, 40, 15, mean_and_max) == 0 and f(1000, 40, 129, mean_and_max) == 0
        assert f(0, 40, 64, mean_and_max) == 0
    assert f(1000, 255, 64, 1) == 0 and f(1000, 255, 64, 0) == 1000 * 64 * 4    # arg-max slots are bytes
    assert f(5000000, 40, 128, 1) == 0 and f(5000000, 40, 128, 0) == 5000000 * 128 * 4   # rows beyond 32-bit offsets


def test_scratch_of_the_weight_gradients_in_list_order(capi):
    """from 16 million slots, 24 neighbours and 64 features on, with the maximum, one float per slot and an int behind the
    quotients; a buffer that holds the quotients alone is taken, less is not (what is missing after that are only pointers)"""
    f, call = capi.hgc_accumulate_knn_grad_scratch_bytes, capi.hgc_accumulate_knn_grad_scratch
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int] * 4
    call.argtypes = [ctypes.c_void_p] * 11 + [ctypes.c_int] * 6 + [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]

    def up(n):
        return (n + 255) // 256 * 256
    at = ctypes.c_void_p(256)  # (an address that nothing looks at: each call ends before)
    for n, k, feat, listed in ((250000, 64, 64, True), (249999, 64, 64, False), (400013, 40, 100, True), (700000, 23, 64, False),
                               (300000, 60, 63, False), (666667, 24, 64, True)):
        quotients = 0 if k & (k - 1) == 0 else up(n * feat * 4)
        assert f(n, k, feat, 0) == quotients
        assert f(n, k, feat, 1) == quotients + (up(n * k * 4) + 256 if listed else 0)
        for size, code in ((quotients, -1), (quotients - 1, -2)):
            if size >= 0:
                rc = call(*[None] * 9, at, at, n, k, feat, 2 * feat, 1, 0, at, size, None)
                assert rc == code, (n, k, feat, size, rc)


def test_settings_are_per_thread(capi):
    """the status word, the choice of the kNN grid and the last error text belong to the thread that set
    them: another thread sees the initial state, and what it sets does not leak back"""
    import threading
    capi.hgc_get_status_word.restype = ctypes.c_void_p
    capi.hgc_set_status_word.argtypes = [ctypes.c_void_p]
    capi.hgc_last_error.restype = ctypes.c_char_p
    assert capi.hgc_set_knn_grid(1) == 0 and capi.hgc_get_knn_grid() == 1
    assert capi.hgc_set_status_word(ctypes.c_void_p(4096)) == 0 and capi.hgc_get_status_word() == 4096
    nb = (ctypes.c_int * 1)(0)
    out = ctypes.c_int(0)
    assert capi.hgc_bin_by_coordinates_total_bins(nb, 1, 2, ctypes.byref(out)) == -1
    mine = capi.hgc_last_error()
    assert mine
    seen = {}

    def other():
        seen["grid"] = capi.hgc_get_knn_grid()
        seen["word"] = capi.hgc_get_status_word()
        seen["error"] = capi.hgc_last_error()
        capi.hgc_set_knn_grid(0)
        capi.hgc_set_status_word(ctypes.c_void_p(8192))

    th = threading.Thread(target=other)
    th.start()
    th.join()
    assert seen == {"grid": 0, "word": None, "error": b""}
    assert capi.hgc_get_knn_grid() == 1 and capi.hgc_get_status_word() == 4096 and capi.hgc_last_error() == mine
    capi.hgc_set_knn_grid(0)
    capi.hgc_set_status_word(None)


def test_package_refuses_cpu_tensors(capi):
    import torch
    from hgcalml_amd import AccumulateLinKnn
    with pytest.raises(RuntimeError, match="GPU"):
        AccumulateLinKnn(torch.ones(4, 2), torch.ones(4, 3), torch.zeros(4, 2, dtype=torch.int32))


def test_knn_workspace_query_covers_every_number_of_neighbours(capi):
    """the size is checked before anything is launched; without a GPU the launch that follows is an error of its own.
    (A call with 2-D points, one event of 30,000 and K = 43 was refused with the workspace that the query asks for.)"""
    torch = pytest.importorskip("torch")
    if torch.cuda.is_available():
        pytest.skip("the pointers of this test lead nowhere")
    query, call = capi.hgc_binned_select_knn_pipeline_workspace_bytes, capi.hgc_binned_select_knn_pipeline
    query.restype = ctypes.c_size_t
    somewhere, null = ctypes.c_void_p(1 << 20), ctypes.c_void_p(None)
    for c in (2, 3, 4, 5, 6):
        for events in (1, 2, 7, 64):
            for n in (1, 100, 1000, 5000, 20000, 30000, 100000, 150000, 500000, 1000000):
                need = query(n, c, events + 1, 30, 3, 0)
                for k in list(range(2, 70)) + [100, 300]:
                    rc = call(somewhere, somewhere, null, n, c, events + 1, k, 30, 3, 0, ctypes.c_float(-1.0), somewhere,
                              somewhere, null, somewhere, ctypes.c_size_t(need), null)
                    assert rc not in (0, -2), (c, events, n, k)
