"""Downloads into page-locked buffers (one kernel for all arrays) equal those into ordinary ones (a copy each): several
subsets of arrays, unaligned destinations, ordinary ones beside page-locked ones in one call, the reference's order,
and boxes on both sides of the size where the copies take over."""
import ctypes

import numpy as np
import pytest

import tigerpm_amd as T

pytestmark = pytest.mark.gpu
FIELDS = ["x", "y", "z", "vx", "vy", "vz", "rung", "gx", "gy", "gz", "pot"]


@pytest.fixture
def pinned():
    """Page-locked buffers from the HIP runtime that the library is linked to (a second runtime in the process, as
    another package may bring, would not know them as such)."""
    T.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    held = []

    def make(n, dtype, shift):
        size = n * np.dtype(dtype).itemsize + 64
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), 0) == 0
        held.append(p)
        whole = np.frombuffer((ctypes.c_uint8 * size).from_address(p.value), np.uint8)
        whole.fill(0xA5)
        return whole, whole[shift : shift + size - 64].view(dtype)

    yield make
    for p in held:
        assert hip.hipHostFree(p) == 0


@pytest.mark.parametrize("n", [1, 63, 257, 30011, 1800000])
@pytest.mark.parametrize("order", [T.TPM_ORDER_DEVICE, T.TPM_ORDER_REFERENCE])
def test_pinned_equals_pageable(gpu_ctx, pinned, n, order):
    rng = np.random.default_rng(n)
    xyz = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    v = [rng.standard_normal(n).astype(np.float32) for _ in range(3)]
    gpu_ctx.set_params(T.baseline_params(32, 32, 3, n_total=n))
    gpu_ctx.set_host_order(order)
    gpu_ctx.upload(*xyz, *v, rng.integers(0, 9, n).astype(np.int8))
    gpu_ctx.chainmesh_create()
    want = gpu_ctx.download()
    for names, shift in ((FIELDS, 0), (["rung"], 1), (["x", "rung", "pot"], 4), (["vz", "gx"], 8)):
        kept = {k: pinned(n, want[k].dtype, shift) for k in names}
        ptr = [ctypes.c_void_p(kept[k][1].ctypes.data) if k in kept else None for k in FIELDS]
        assert T.lib().tpm_particles_download(gpu_ctx._h, *ptr) == 0
        for k in names:
            whole, view = kept[k]
            assert np.array_equal(view, want[k]), k
            assert (whole[:shift] == 0xA5).all() and (whole[shift + view.nbytes :] == 0xA5).all(), k
        # one pageable destination among page-locked ones
        if len(names) > 1:
            mixed = np.empty(n, want[names[0]].dtype)
            ptr[FIELDS.index(names[0])] = ctypes.c_void_p(mixed.ctypes.data)
            assert T.lib().tpm_particles_download(gpu_ctx._h, *ptr) == 0
            assert np.array_equal(mixed, want[names[0]])
            for k in names[1:]:
                assert np.array_equal(kept[k][1], want[k]), k
