"""GPU: the stable radix sort at the edges of its tiles (2,048 pairs) and of a
digit row's scan round (256 tiles), against numpy's stable argsort (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 2047, 2048, 2049, 4097, 255 * 2048, 256 * 2048 + 1,
                               257 * 2048 + 77])
@pytest.mark.parametrize("distinct", [3, 1 << 32])
def test_sort_pairs_stable_at_tile_edges(n, distinct):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from jaxabm_amd._lib import check, lib, ptr, stream_handle

    rng = np.random.default_rng(n)
    keys = rng.integers(0, distinct, n, dtype=np.uint64).astype(np.uint32)
    if distinct == 3:
        keys *= np.uint32(0x01010101)   # ties in every digit
    dk = torch.from_numpy(keys.view(np.int32).copy()).cuda()
    dv = torch.arange(n, dtype=torch.int32, device="cuda")
    nbytes = int(lib().abm_permutation_workspace(n))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    check(lib().abm_sort_pairs_u32(ptr(dk), ptr(dv), n, ptr(ws), nbytes, stream_handle()), "sort")
    order = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(dv.cpu().numpy(), order)
    np.testing.assert_array_equal(dk.cpu().numpy().view(np.uint32), keys[order])
