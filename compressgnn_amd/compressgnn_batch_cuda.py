"""GPU batch compressor behind the reference's optional module name
(src/offline/bindings/batch_cuda.cpp:3-9: `is_available()` and
`compress_csr_batch(vlist, elist, rounds=12, min_pair_frequency=16)`), which
loader/compression_backend.py:6-40 picks when `compression_backend` is 'auto' or 'cuda'.

The rounds run as HIP kernels (csrc/merger.hip) on the current GPU and return the same
arrays as the host compressor compressgnn_offline.compress_csr_batch: (vlist int32,
elist int32, vertex_cnt, rule_cnt).  Input checks and errors follow the reference's bridge
(src/offline/bindings/batch_bridge.hpp:8-26): ValueError for non-integer, negative or
too large values and for min_pair_frequency < 3."""
import os
import sys

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))


def is_available():
    if not os.path.exists(os.path.join(_HERE, "lib", "libcgnn_hip.so")):
        return False
    import torch
    return torch.cuda.is_available()


def compress_csr_batch(vlist, elist, rounds=12, min_pair_frequency=16, release_cache=False):
    """release_cache=True hands the workspace (60 to 85 bytes per edge) back to the device
    afterwards with torch.cuda.empty_cache(), which also flushes whatever else the caller's
    allocator holds cached: for a preparation script that goes on to build a large model."""
    import torch
    if _HERE not in sys.path:
        sys.path.append(_HERE)
    import compressgnn_runtime
    arrays = []
    for arr in (vlist, elist):
        a = np.asarray(arr)
        if a.ndim != 1 or a.dtype.kind not in "iu":
            raise ValueError("CSR arrays must be one-dimensional integer arrays")
        if a.dtype not in (np.int64, np.int32):  # which the operator checks on their way to the device
            if a.size and (int(a.max()) > np.iinfo(np.int32).max or int(a.min()) < 0):
                raise ValueError("CSR value exceeds int32 range")
            a = a.astype(np.int64)
        arrays.append(torch.from_numpy(np.ascontiguousarray(a)))
    usable = min_pair_frequency >= 3 and rounds >= 1 and len(arrays[0]) > 0 and torch.cuda.is_available()
    if not usable:  # what follows raises or returns, after a value out of range does
        for a in arrays:
            if len(a) and (int(a.max()) > np.iinfo(np.int32).max or int(a.min()) < 0):
                raise ValueError("CSR value exceeds int32 range")
    if min_pair_frequency < 3:
        raise ValueError("Batch compression needs min_pair_frequency >= 3")
    if rounds < 1:
        raise ValueError("rounds must be positive")
    if len(arrays[0]) == 0:
        return np.zeros(1, np.int32), np.zeros(0, np.int32), 0, 0
    if not usable:
        raise RuntimeError("GPU compression requested but no usable device is available")
    ptr, col, rules = compressgnn_runtime.compress_csr_batch(*arrays, rounds, min_pair_frequency)
    if release_cache:
        torch.cuda.empty_cache()
    return ptr.numpy(), col.numpy(), len(arrays[0]) - 1, rules
