"""The C-ABI library loads without a GPU and exports every symbol that
include/managan_hip.h declares (no compute calls here)."""
import ctypes
import importlib
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "managan_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mg_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported():
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib = L.load()
    names = _declared()
    assert len(names) >= 25
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in the header but not exported"
    # and the Python binding table covers exactly the declared entry points
    assert sorted(L.exported_symbols()) == names


def test_host_only_entry_points():
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib = L.load()
    assert lib.mg_abi_version() == 1
    nd = (ctypes.c_int * 3)()
    assert lib.mg_neighbour_ndiv(5.0, 55.0, 55.0, 55.0, ctypes.byref(nd)) == 0
    assert list(nd) == [11, 11, 11]
    assert lib.mg_neighbour_ndiv(6.0, 70.0, 70.0, 70.0, ctypes.byref(nd)) == 0
    assert list(nd) == [12, 12, 12]
    nbytes = ctypes.c_size_t(0)
    assert lib.mg_neighbour_workspace_bytes(8, 16384, 5.0, 55.0, 55.0, 55.0, ctypes.byref(nbytes)) == 0
    # preferred size: 256 neighbour entries of 2 bytes per atom (boxes of at most 65536 atoms: 67 MB for 131072 atoms)
    # plus the sorted records and cell tables; 4-byte entries for larger boxes
    assert 8 * 16384 * 256 * 2 < nbytes.value < 8 * 16384 * 256 * 2 + 8_000_000
    assert lib.mg_neighbour_workspace_bytes(1, 70000, 5.0, 90.0, 90.0, 90.0, ctypes.byref(nbytes)) == 0
    assert 70000 * 256 * 4 < nbytes.value < 70000 * 256 * 4 + 5_000_000
    # box smaller than 3 cells: the reference's error, as a status code
    assert lib.mg_neighbour_workspace_bytes(1, 10, 5.5, 10.0, 10.0, 10.0, ctypes.byref(nbytes)) == L.MG_ERR_BOX_TOO_SMALL
    assert b"3*cutoff" in lib.mg_status_string(L.MG_ERR_BOX_TOO_SMALL)
    assert lib.mg_status_string(0) == b"ok"


def test_a_sort_workspace_serves_every_smaller_count():
    """Chunks grow with the count, so that one more element may need fewer of them: what is asked for never falls, and covers a count's
    own chunks (512 counts each, one row of totals, spare keys and values and the positions between passes)."""
    lib = importlib.import_module("learned-dynamics_amd._lib").load()
    size, before = ctypes.c_size_t(0), 0
    edges = [512 * 2 ** k + d for k in range(13) for d in (-1, 0, 1)] + [4096 * 300 + d for d in (-1, 0, 1)]
    for count in sorted({0, 1, 2, 511, *edges, *range(1000, 1400000, 7919)}):
        assert lib.mg_sort_by_key_workspace_bytes(count, ctypes.byref(size)) == 0
        per = next(p for p in (2, 4, 8, 16) if p == 16 or count <= 65536 * p)
        chunks = -(-count // (256 * per))
        assert size.value >= max(before, 4 * ((chunks + 1) * 512 + 3 * count)), count
        before = size.value


def test_shims_expose_reference_symbols():
    pkg = importlib.import_module("learned-dynamics_amd")
    pkg.install_shims()
    import codegen_tensops_cuda
    import neighbour_grid_cuda
    import tensor_ops_cuda
    import torch_scatter
    for name in ("get_neighbours", "edges_read", "edges_reduce", "get_edges"):      # neighbour_grid.cpp:198-203
        assert callable(getattr(neighbour_grid_cuda, name))
    assert callable(tensor_ops_cuda.tensor_linear)                                  # tensor_ops.cpp:180-182
    assert callable(torch_scatter.segment_coo)
    expected = ["set_kern_attributes", "bee_fwd_cuda", "bee_bwl_cuda", "bee_bwr_cuda", "cow_o0_fwd_cuda",
                "cow_o0_bwl_cuda", "cow_o0_bwr_cuda", "cow_o1_fwd_cuda", "cow_o1_bwl_cuda", "cow_o1_bwr_cuda"]
    for o in ("o0", "o1", "o2", "oc"):
        for suffix in ("", "_backward", "_backleft", "_wtsback"):
            expected.append(f"ant16_{o}{suffix}_cuda")
    for name in expected:                                                            # codegen_tensops.cpp:1980-2011
        assert callable(getattr(codegen_tensops_cuda, name)), name


def test_torch_binding_loads_and_exports_the_reference_names():
    """managan_torch_ext.so (csrc/torch_binding.cpp) imports without a GPU and carries the functions the reference's
    compiled extensions export (neighbour_grid.cpp:198-203, tensor_ops.cpp:180-182, codegen_tensops.cpp:2001-2010)."""
    L = importlib.import_module("learned-dynamics_amd._lib")
    ext = L.load_torch_ext()
    for name in ("get_neighbours", "edges_read", "edges_reduce", "get_edges", "tensor_linear", "tensor_prods",
                 "tensor_prods_supported", "bee_fwd_cuda", "bee_bwl_cuda", "bee_bwr_cuda", "cow_o0_fwd_cuda", "cow_o0_bwl_cuda",
                 "cow_o0_bwr_cuda", "cow_o1_fwd_cuda", "cow_o1_bwl_cuda", "cow_o1_bwr_cuda"):
        assert callable(getattr(ext, name)), name
    import torch
    try:
        ext.tensor_linear(0, torch.zeros(4, 4), torch.zeros(2, 4))
    except RuntimeError as e:                       # host tensors are refused before anything touches a device
        assert "must be a CUDA tensor" in str(e)
    else:
        raise AssertionError("a host tensor was accepted")


def test_message_gradient_takes_the_struct_with_a_pointer_per_product():
    """mg_bee_message_grad (include/managan_hip.h): 13 gradients by product and then the graph, as callers in C lay it out.  With one
    gradient missing the call names it and launches nothing (the other pointers are never followed)."""
    import ctypes
    L = importlib.import_module("learned-dynamics_amd._lib")
    lib = L.load()

    class Args(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in ("l_0", "l_1", "l_2", "enc", "rh")] + [("dy", ctypes.c_void_p * 13)] + \
                   [(n, ctypes.c_void_p) for n in ("row_ptr", "dst", "dst_row_ptr", "perm")] + [("E", ctypes.c_long)] + \
                   [(n, ctypes.c_int) for n in ("n_src", "n_rows", "chan")] + \
                   [(n, ctypes.c_void_p) for n in ("workspace", "d_0", "d_1", "d_2", "d_enc", "d_rh")]

    for missing in (0, 7, 12):
        a = Args(E=10, n_src=3, n_rows=4, chan=64)
        for name, kind in Args._fields_:
            if kind is ctypes.c_void_p:
                setattr(a, name, 16)
        for k in range(13):
            a.dy[k] = None if k == missing else 16
        assert lib.mg_bee_message_grad_run(ctypes.byref(a), None) != 0
        assert f"gradient {missing} is null" in lib.mg_last_error().decode()
