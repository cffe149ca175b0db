"""GPU test of the radix sort at the edges of its tile sizes, against numpy's
stable argsort (bit-exact: keys and permutation)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 511, 512, 513, 32768, 32769, 131072, 131073, 262144, 262145]


@pytest.mark.parametrize("kind", ["random", "few", "equal"])
@pytest.mark.parametrize("n", SIZES)
def test_sort_at_tile_edges(n, kind):
    import torch
    from paratreet_amd import _lib
    fn = _lib.load().pt_sort_noalloc
    fn.argtypes = [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
    fn.restype = C.c_int
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 2**64, n, dtype=np.uint64)
    if kind == "few":
        keys = keys[rng.integers(0, min(n, 7), n)]
    elif kind == "equal":
        keys[:] = keys[0]
    k = torch.from_numpy(keys.view(np.int64)).cuda()
    out = torch.zeros_like(k)
    perm = torch.zeros(n, dtype=torch.int32, device="cuda")
    assert fn(k.data_ptr(), n, out.data_ptr(), perm.data_ptr(),
              torch.cuda.current_stream().cuda_stream) == 0
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(perm.cpu().numpy(), want)
    assert np.array_equal(out.cpu().numpy().view(np.uint64), keys[want])
