"""The shared libraries load and export every entry point their headers declare (no
compute calls, so no GPU is needed), and the Python-visible operator module exposes
the reference's operator names."""
import ctypes
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "compressgnn_amd")
sys.path.insert(0, PKG)


def declared(header):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(cgnn_[a-z0-9_]+)\s*\(", text)))


def test_device_library_exports_every_declared_symbol():
    names = declared("compressgnn_abi.h")
    assert len(names) >= 18
    lib = ctypes.CDLL(os.path.join(PKG, "lib", "libcgnn_hip.so"))
    for n in names:
        assert hasattr(lib, n), n
    lib.cgnn_version.restype = ctypes.c_char_p
    assert b"gfx950" in lib.cgnn_version()
    from compressgnn_amd import abi
    assert sorted(abi.EXPORTS) == names


def test_prep_library_exports_every_declared_symbol():
    names = declared("compressgnn_prep.h")
    lib = ctypes.CDLL(os.path.join(PKG, "lib", "libcgnn_prep.so"))
    for n in names:
        assert hasattr(lib, n), n
    import compressgnn_offline as off
    assert sorted(off.EXPORTS) == names


def test_argument_checks_without_a_gpu():
    """Entry points validate their arguments before touching the device."""
    from compressgnn_amd import abi
    lib = abi.lib()
    s = abi.CsrStruct()
    s.rows, s.cols, s.nnz = 4, 4, 1 << 40
    rc = lib.cgnn_spmm(ctypes.byref(s), 0, None, None, ctypes.c_int64(8), 0, 0, None, ctypes.c_size_t(0), None)
    assert rc == 1 and b"2^31" in lib.cgnn_last_error()
    assert lib.cgnn_spmm(None, 0, None, None, ctypes.c_int64(8), 0, 0, None, ctypes.c_size_t(0), None) == 1
    rc = lib.cgnn_lsh_hash(ctypes.c_int64(4), ctypes.c_int64(4), 31, 0, None, None, None, None, None)
    assert rc == 1 and b"[0,30]" in lib.cgnn_last_error()
    assert lib.cgnn_copy_bytes(None, None, ctypes.c_size_t(7), None) == 1
    assert lib.cgnn_lsh_scan_workspace_bytes(16) >= 64


@pytest.mark.parametrize("F,nnz,double,parts,groups,run", [
    (257, 49784, False, 3, 4, 24), (513, 985767, False, 5, 4, 64), (602, 49784, False, 3, 4, 24), (4096, 49784, False, 8, 4, 16),
    (2048, 131071, False, 4, 4, 20), (2048, 131072, False, 8, 4, 20), (602, 985767, False, 3, 4, 32), (602, 1000, False, 3, 4, 8),
    (256, 49784, False, 1, 4, 8), (512, 49784, False, 1, 4, 8), (768, 985767, False, 3, 4, 32), (256, 49784, True, 4, 4, 8),
    (64, 985767, False, 1, 16, 36)])
def test_entries_per_workgroup_of_products_of_int64_arrays(F, nnz, double, parts, groups, run):
    """Every part of a wide product looks for the rows of its entries: runs are counted for the parts together, where a search
    costs much beside what it is for."""
    from compressgnn_amd import abi
    arrivals = ctypes.c_int64(-1)
    total = abi.lib().cgnn_spmm_once_workspace_bytes(abi.i64(1000), abi.i64(nnz), abi.i64(F), int(double), ctypes.byref(arrivals))
    workgroups = -(-nnz // (groups * run))
    assert arrivals.value == workgroups * parts
    assert total == 2 * workgroups * F * (8 if double else 4)


def test_kernels_spill_no_registers(tmp_path):
    """What the compiler says of the kernels of the device library: none puts registers aside in memory."""
    from compressgnn_amd import abi
    tools = "/opt/rocm/llvm/bin"
    if not os.path.exists(os.path.join(tools, "llvm-readelf")):
        pytest.skip("no llvm-readelf")
    shutil.copy(abi.LIB_PATH, tmp_path / "lib.so")  # the code objects are written beside it
    subprocess.run([os.path.join(tools, "llvm-objdump"), "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    kernels, spilled = 0, []
    for part in sorted(tmp_path.glob("*gfx950")):
        notes = subprocess.run([os.path.join(tools, "llvm-readelf"), "--notes", str(part)], check=True, stdout=subprocess.PIPE, text=True).stdout
        for kernel in re.split(r"\n  - ", notes):
            name, count = re.findall(r"\.symbol:\s+(\S+)", kernel), re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)
            if count:
                kernels += 1
                spilled += [name[-1]] if int(count[1]) else []
    assert kernels > 400 and not spilled


def test_runtime_module_has_the_reference_operator_names():
    import compressgnn_runtime as rt
    for name in ["spmm_func", "cluster_forward", "cluster_workspace", "cluster_assign", "cluster_mean",
                 "cluster_mean_backward", "cluster_reconstruct", "cluster_reconstruct_backward"]:
        assert hasattr(rt, name), name
    import torch
    with pytest.raises(RuntimeError, match="GPU"):
        rt.spmm_func(torch.zeros(2, dtype=torch.long), torch.zeros(0, dtype=torch.long), torch.zeros(0),
                     torch.zeros(1, 3), "rowbalance", None)
    with pytest.raises(RuntimeError):
        rt.cluster_assign(torch.zeros(3, 4), torch.zeros(4, 2), 2, [])


def test_sampler_module_has_the_reference_names():
    """compressgnn_sample, the module name the reference builds from src/sample
    (function.cpp:7-9): both functions, GPU tensors only."""
    import torch
    import compressgnn_sample as sampler
    for name in ["neighbor_sample_cg_sim", "neighbor_sample_ori_impl"]:
        assert callable(getattr(sampler, name)), name
    ptr = torch.zeros(3, dtype=torch.long)
    with pytest.raises(RuntimeError, match="GPU"):
        sampler.neighbor_sample_ori_impl(ptr, torch.zeros(0, dtype=torch.long), torch.zeros(1, dtype=torch.long), [2])
