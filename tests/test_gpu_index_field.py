"""Bit-exact addressing of the one-kernel fields (KK_FIELD): the index-map test
build with VKFX_FIELD=1 against one Stockham permutation per axis. The cases hold
every radix, several fields a block with a ragged last one, the copied-in first
stage, axes of one stage and of many, and every rank-2 and rank-3 shape of the
N-D list of the axis passes that is small enough (the list itself runs on the
axis passes in test_gpu_index.py)."""
import numpy as np
import pytest

from oracle import index_maps as im
from test_gpu_index import F32, F64, FWD, INV, ND, idx_ctx, run, tagged  # noqa: F401

pytestmark = pytest.mark.gpu

FIELDS = [([2, 2], 1), ([2, 2], 3001), ([3, 5], 2000), ([13, 11], 1500), ([9, 7], 1), ([12, 10], 30), ([64, 48], 2),
          ([32, 32], 1030), ([2, 1000], 2), ([1000, 2], 2), ([16, 8, 8], 700), ([10, 12, 15], 3), ([3, 2, 26], 4),
          ([49, 81], 2), ([72, 44], 3), ([16, 16, 16], 2), ([4, 512], 2), ([13, 13, 13], 2), ([11, 22, 6], 5)]
SMALL = [(d, b) for d, b, _ in ND if len(d) in (2, 3) and int(np.prod(d)) <= 4096 and max(d) < 4099]


def field_maps(dims, p):
    """One line map per axis: the radices run last axis first."""
    maps, at = [None] * len(dims), 0
    for i, stages in enumerate(p["axis_stages"][:len(dims)]):
        ax = len(dims) - 1 - i
        radices = p["radices"][at:at + stages]
        assert int(np.prod(radices)) == dims[ax], p
        maps[ax] = im.stockham_perm(dims[ax], radices)
        at += stages
    assert at == len(p["radices"]), p
    return maps


@pytest.mark.parametrize("prec", [F32, F64])
@pytest.mark.parametrize("dims,batch", FIELDS + SMALL)
def test_field(idx_ctx, dims, batch, prec):  # noqa: F811
    x = tagged(int(np.prod(dims)) * batch, prec)
    for direction in (FWD, INV):
        out, desc = run(idx_ctx, dims, batch, prec, direction, x, env={"VKFX_FIELD": "1"})
        assert [p["kernel"] for p in desc["passes"]] == ["field"], desc["passes"]
        v = x.reshape((batch,) + tuple(dims))
        for ax, src in enumerate(field_maps(dims, desc["passes"][0])):
            v = np.take(v, src, axis=ax + 1)
        assert np.array_equal(out, v.reshape(-1)), (dims, batch)
