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


# the tiles (of 2,048) where the scan of a segment's counts changes its form
@pytest.mark.parametrize("tiles", [1, 2, 4, 5, 16, 17, 32, 33])
@pytest.mark.parametrize("segments", [1, 15, 16])
@pytest.mark.parametrize("ragged", [0, 1])
def test_segments_equal_single_permutations(tiles, segments, ragged):
    import torch

    import oracle as O
    from jaxabm_amd import random as jr

    n = tiles * 2048 - ragged * 77
    keys = np.random.default_rng(tiles).integers(0, 1 << 32, (segments, 2), dtype=np.uint64)
    keys = keys.astype(np.uint32)
    got = jr.permutation_each(torch.from_numpy(keys.view(np.int32)).cuda(), n, 1).cpu().numpy()
    for k in {0, segments // 2, segments - 1}:
        np.testing.assert_array_equal(got[k], O.permutation(keys[k], n, 1))
    assert (np.sort(got, axis=1) == np.arange(n)).all()
