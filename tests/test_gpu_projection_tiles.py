"""The stacked projection of a prompt (queries, keys and values in one GEMM with three outputs) in the wider tiles and with K
cut, where every output is a multiple of 128 columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# whole tiles, K ranges, hybrid and stream-K cuts; the last three are no forms of this launch: the closed rule
@pytest.mark.parametrize("tile", [-1, 13, 14, 16, 18, 215, 415, 213, 10313, 20013, 20015, 216, 30013])
def test_tiles_and_cuts_of_the_stacked_projection(fdx, modelgen, tile):
    """One row block to tiles that cross sequences, three outputs in the first layer and two in the last, against a session of
    17 sequences, which takes a launch for each (fp32 sums of 256 products in another order: 1e-5)."""
    stacked_projection(fdx, modelgen, tile, 0)


@pytest.mark.parametrize("cap", [8, 10])
@pytest.mark.parametrize("tile", [13, 14, 16, 18, 415, 213, 10213, 10313, 20013])
def test_stacked_projection_several_tiles_a_workgroup(fdx, modelgen, tile, cap):
    """A grid of `cap` workgroups: each walks tiles of several outputs, and of 12 or 48 tiles of 128 x 128 the hybrid cuts leave
    whole ones beside a cut remainder."""
    stacked_projection(fdx, modelgen, tile, cap)


def stacked_projection(fdx, modelgen, tile, cap):
    js = modelgen.dumps(modelgen.gpt2(seed=231, layers=2, d_model=256, heads=4, vocab=33000, max_pos=128, bias_std=0.1,
                                      random_affine=True, std=0.1))
    model = fdx.Model(js, verify=False)
    ids = np.random.default_rng(232).integers(0, 33000, (17, 90))
    wide = fdx.Session(model, 17, 96)
    some = {B: fdx.Session(model, B, 96) for B in (1, 5, 16)}
    lo = 0
    for n in (2, 3, 16, 63):
        want, _ = wide.prefill(ids[:, lo:lo + n])
        fdx.lib.fdx_debug_force_tile(tile)
        fdx.lib.fdx_debug_persist_cap(cap)
        try:
            got = {B: s.prefill(ids[:B, lo:lo + n])[0] for B, s in some.items()}
        finally:
            fdx.lib.fdx_debug_force_tile(-1)
            fdx.lib.fdx_debug_persist_cap(0)
        for B in some:
            err = np.abs(got[B] - want[:B]).max() / np.abs(want[:B]).max()
            assert err <= 1e-5, (B, n, err)
        lo += n
