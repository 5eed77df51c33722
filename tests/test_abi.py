"""The C-ABI library loads without a GPU, exports every symbol include/gnnhip.h
declares, validates arguments on the host and reports errors through status codes."""
import ctypes
import os
import re

import numpy as np
import pytest

from graphnn_amd import _lib as binding

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gnnhip.h")


def _declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gnnhip_[a-z0-9_]+)\s*\(", text)))


def test_library_is_built_in_tree():
    assert os.path.exists(binding.library_path()), "run `python -m graphnn_amd.build`"


def test_every_declared_symbol_is_exported_and_bound():
    lib = ctypes.CDLL(binding.library_path())
    declared = _declared_symbols()
    assert len(declared) >= 30
    for name in declared:
        assert hasattr(lib, name), "declared in gnnhip.h but not exported: " + name
    # the Python binding declares a prototype for each of them, and nothing else
    assert sorted(binding.SIGNATURES) == declared


def test_header_cites_the_reference_for_every_entry():
    text = open(HEADER).read()
    # each block comment introducing entry points names a reference file
    blocks = re.findall(r"/\* ----(.*?)\*/", text, flags=re.S)
    assert len(blocks) >= 20
    for b in blocks:
        if "No counterpart in the reference" in b:      # the entry for callers that cannot allocate
            continue
        assert re.search(r"(src|include|examples)/[\w/]+\.(cpp|cu|h)", b), b[:80]


def test_argument_validation_needs_no_gpu():
    lib = binding.load_library()
    f = ctypes.c_float
    # negative sizes, bad op codes, null pointers: rejected before any device work
    assert lib.gnnhip_spmm_csr_f32(-1, 1, 1, 0, f(1), None, None, None, None, 1, f(0), None, 1, None) == -1
    assert b"negative" in lib.gnnhip_last_error()
    assert lib.gnnhip_spmm_csr_f32(4, 4, 8, 0, f(1), None, None, None, None, 8, f(0), None, 8, None) == -1
    assert lib.gnnhip_gemm_f32(2, 0, 1, 1, 1, f(1), None, 1, None, 1, f(0), None, 1, None) == -1
    assert lib.gnnhip_unary_f32(99, None, 10, f(0), f(0), None) == -1
    assert lib.gnnhip_reduce_f32(9, None, 10, None, None) == -1
    assert lib.gnnhip_row_argmax_f32(None, 3, 0, None, None) == -1
    assert lib.gnnhip_s2v_forward_f32(0, 1, 1, 1, 1, 1, 1, 0, *([None] * 19), None, None) == -1
    x = np.zeros(8, np.float32)
    p = x.ctypes.data_as(ctypes.c_void_p)
    assert lib.gnnhip_s2v_level_f32(2, 4, 0, p, p, p, p, p, None, None, p, None) == -1      # in place is refused
    assert b"in place" in lib.gnnhip_last_error()
    # empty work is a successful no-op
    assert lib.gnnhip_unary_f32(6, None, 0, f(0), f(0), None) == 0
    assert lib.gnnhip_spmm_csr_f32(0, 0, 0, 0, f(1), None, None, None, None, 0, f(0), None, 0, None) == 0
    assert lib.gnnhip_memset0(None, 0, None) == 0


def test_bindings_take_no_integer_for_a_device_tensor():
    """every float* / int* parameter of the compiled bindings refuses an address (sizes are zero: nothing could be launched);
    the host pointers, marked @ in the argument lists, are the only ones that take one"""
    b = binding.load_bindings()
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    tried = 0
    for name, params in re.findall(r"\bint gnnhip_([a-z0-9_]+)\s*\(([^)]*)\)", text):
        fn = getattr(b, name, None)
        if fn is None or not fn.__doc__:
            continue
        kinds = [p.strip() for p in params.split(",")][:-1]        # the stream is not passed
        names = [a.strip() for a in fn.__doc__.split(",")]
        assert len(kinds) == len(names), name
        args = [None if "*" in k else 0.0 if k.startswith("float") else 0 for k in kinds]
        for i, (kind, arg) in enumerate(zip(kinds, names)):
            if not re.match(r"(const )?(float|int)\*", kind) or arg.startswith("@"):
                continue
            with pytest.raises(ValueError, match="^%s must be" % arg):
                fn(*args[:i], 4096, *args[i + 1:])
            tried += 1
    assert tried > 200


@pytest.mark.parametrize("rows,n,fits", [(1, 1, 1), (7_450, 16_380, 1), (9_000, 60_000, 1), (100_000, 60_000, 1), (156_000, 65_536, 1),
                                         (157_500, 65_536, 0), (300_000, 65_536, 0), (2_000_000, 1_000, 1), (2_700_000, 1_000, 0), (100, 65_537, 0),
                                         (0, 5, 0), (5, 0, 0)])
def test_grouping_in_one_launch_is_a_rule_of_its_own(rows, n, fits):
    """which (rows, pairs) one launch groups: 2.35 bytes per pair and 4 per row of a 64th of the rows in 160 KB, at most 65,536 pairs.
    The host layer asks this to choose between the device and its own loop"""
    assert binding.load_library().gnnhip_csr_group_one_launch(rows, n) == fits


def test_plan_entries_reject_what_is_not_a_plan():
    lib = binding.load_library()
    x = np.zeros(8, np.float32)
    p = x.ctypes.data_as(ctypes.c_void_p)
    f = ctypes.c_float
    assert lib.gnnhip_spmm_csr_planned_f32(p, 4, f(1), p, 4, f(0), p, 4, None) == -1
    assert b"not a live CSR plan" in lib.gnnhip_last_error()
    assert lib.gnnhip_s2v_level_planned_f32(None, 64, p, p, None, None, p, None) == -1
    assert lib.gnnhip_csr_plan_destroy(None) == 0
    assert lib.gnnhip_csr_plan_destroy(p) == -1
    n = ctypes.c_size_t()
    assert lib.gnnhip_csr_plan_bytes(p, ctypes.byref(n)) == -1
    h = ctypes.c_void_p()
    assert lib.gnnhip_csr_plan_create(-1, 1, p, p, p, None, ctypes.byref(h)) == -1
    assert lib.gnnhip_csr_plan_create(1, 1, None, p, p, None, ctypes.byref(h)) == -1
    assert lib.gnnhip_csr_plan_create(1, 1, p, p, p, None, None) == -1


def test_compute_before_init_is_refused():
    import torch
    if torch.cuda.is_available():
        pytest.skip("on a GPU box another test may already have initialised the library")
    lib = binding.load_library()
    x = np.zeros(8, np.float32)
    p = x.ctypes.data_as(ctypes.c_void_p)
    assert lib.gnnhip_unary_f32(6, p, 8, ctypes.c_float(0), ctypes.c_float(0), None) == -4
    assert b"gnnhip_init" in lib.gnnhip_last_error()
    out = ctypes.c_void_p()
    assert lib.gnnhip_malloc(ctypes.byref(out), 1024) == -4
    # no device here: init reports it instead of crashing
    assert lib.gnnhip_init(0) in (-3, -1)
    assert lib.gnnhip_shutdown() == 0


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(binding, "_lib", None)
    monkeypatch.setattr(binding, "_LIB_PATH", str(tmp_path / "libgnnhip.so"))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        binding.load_library()


def test_bindings_make_empty_tensors_of_every_kind():
    """one letter: a tensor of the sizes given; several: a tuple, each taking its sizes in turn; too few or too many are refused"""
    import torch
    from graphnn_amd import _lib
    empty = _lib.load_bindings().empty
    cpu = torch.device("cpu")
    one = empty(cpu, "f", 2, 3, 4)
    assert one.shape == (2, 3, 4) and one.dtype == torch.float32 and one.is_contiguous()
    a, b, c = empty(one, "iFf", 3, 4, 5, 0)
    assert (a.shape, b.shape, c.shape) == ((3,), (4, 5), (0,)) and (a.dtype, b.dtype, c.dtype) == (torch.int32, torch.float32, torch.float32)
    for bad in (("ff", 3), ("f", 1, 2, 3, 4), ("F" "f", 3, 4)):
        with pytest.raises(TypeError):
            empty(cpu, *bad)
    with pytest.raises(RuntimeError):
        empty(cpu, "f", -2)


@pytest.mark.parametrize("args", [("", 3), ("ff", 3, 4, 5), ("iF", 3, 4, 5, 6), ("F", 3), ("F", 3, 4, 5), ("x", 3), ("fx", 3, 4), ("d", 3), ("I", 3),
                                  ("\u00e9", 3), ("f\0", 3, 4), ("f",), ("i", 1, 2, 3, 4)])
def test_bindings_make_no_tensors_of_a_list_that_does_not_add_up(args):
    """no letters, letters that name no type, sizes left over or missing"""
    import torch
    from graphnn_amd import _lib
    with pytest.raises(TypeError):
        _lib.load_bindings().empty(torch.device("cpu"), *args)


@pytest.mark.parametrize("offsets", [
    np.array([0, 2, 5], np.int64), np.array([0, 2, 5], np.float32), np.array([0, 2, 5], np.uint32), np.array([0, 2, 5], ">i4"), b"\0" * 12,
    np.array([0, 2], np.int32), np.array([], np.int32), np.zeros((3, 1), np.int32), np.int32(5), np.int64(1 << 40),
    np.array([0, 9, 2, 9, 5, 9], np.int32)[::2]])
def test_bindings_refuse_host_arrays_of_another_kind(offsets):
    """row offsets on the host are an int32 array with an element more than there are rows: other elements, a shorter array, another
    number of dimensions, gaps, and a number in numpy's dress are refused before anything reads them"""
    from graphnn_amd import _lib
    with pytest.raises((ValueError, BufferError)):
        _lib.load_bindings().csr_consecutive_rows_host_f32(2, offsets, 0, None, None, None)


@pytest.mark.parametrize("offsets", [np.array([0, 2, 5], np.int32), np.array([0, 2, 5, 7], "<i4"), (ctypes.c_int * 3)(0, 2, 5),
                                     memoryview(np.array([0, 2, 5], np.int32)).toreadonly(), 1 << 40])
def test_bindings_take_host_arrays_of_int32_and_addresses(offsets):
    """past the arguments: what refuses the call is the entry behind them (no row pointers to write), or no device to run it on.  The
    address is never read: the null row pointers are found first"""
    from graphnn_amd import _lib
    with pytest.raises((RuntimeError, _lib.GnnHipError)):
        _lib.load_bindings().csr_consecutive_rows_host_f32(2, offsets, 0, None, None, None)


@pytest.mark.parametrize("which", [np.zeros(1, np.float32), np.zeros(1, np.int64), np.zeros(0, np.int32), b"\0\0\0\0",
                                   memoryview(np.zeros(1, np.int32)).toreadonly(), np.int32(0)])
def test_bindings_refuse_host_results_of_another_kind(which):
    """the entry writes which buffer holds the last level: into one writable int32"""
    from graphnn_amd import _lib
    args = [0] * 8 + [None] * 19
    with pytest.raises((ValueError, BufferError)):
        _lib.load_bindings().s2v_forward_f32(*args, which)
