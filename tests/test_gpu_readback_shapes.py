"""GPU: downloads into page-locked buffers that one kernel may not write as they are: 4-byte arrays at addresses that
are no multiple of four, and one buffer given for several arrays, where the last array's entries stay, as with copies
made one after the other."""
import ctypes

import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_readback import FIELDS, pinned  # noqa: F401  (a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 30011])
@pytest.mark.parametrize("order", [T.TPM_ORDER_DEVICE, T.TPM_ORDER_REFERENCE])
def test_unaligned_and_shared_buffers(gpu_ctx, pinned, n, order):  # noqa: F811
    rng = np.random.default_rng(n)
    xyz = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    v = [rng.standard_normal(n).astype(np.float32) for _ in range(3)]
    gpu_ctx.set_params(T.baseline_params(32, 32, 3, n_total=n))
    gpu_ctx.set_host_order(order)
    gpu_ctx.upload(*xyz, *v, rng.integers(0, 9, n).astype(np.int8))
    gpu_ctx.chainmesh_create()
    want = gpu_ctx.download()
    for shift in (1, 2, 3):
        whole, _ = pinned(4 * n, np.uint8, 0)
        ptr = [ctypes.c_void_p(whole.ctypes.data + shift) if k == "vy" else None for k in FIELDS]
        assert T.lib().tpm_particles_download(gpu_ctx._h, *ptr) == 0
        assert np.array_equal(whole[shift : shift + 4 * n], want["vy"].view(np.uint8))
        assert (whole[:shift] == 0xA5).all() and (whole[shift + 4 * n :] == 0xA5).all()
    whole, _ = pinned(4 * n, np.uint8, 0)
    ptr = [ctypes.c_void_p(whole.ctypes.data) if k in ("x", "vz", "pot") else None for k in FIELDS]
    assert T.lib().tpm_particles_download(gpu_ctx._h, *ptr) == 0
    assert np.array_equal(whole[: 4 * n], want["pot"].view(np.uint8))
