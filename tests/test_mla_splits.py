"""The default number of key splits of the sparse MLA (no GPU: 256 CUs assumed)."""
import pytest

from xtier_amd import ops


@pytest.mark.parametrize('rows', [1, 4, 32, 33, 64, 96, 128, 255, 256, 2048])
def test_short_latent_lists_are_not_split(rows):
    """Below 512 keys a split would round the FP32 accumulators to FP16 partials."""
    assert {ops.default_mla_splits(rows, topk) for topk in range(512)} == {1}


@pytest.mark.parametrize('rows,topk,splits', [(1, 383, 1), (32, 384, 3), (33, 384, 1), (32, 511, 3), (33, 511, 1),
                                              (64, 320, 1), (61, 512, 4), (61, 640, 4), (128, 512, 2), (200, 640, 1)])
def test_page_lists(rows, topk, splits):
    """The pages' partials are FP32; short lists split only where the merge costs less than the split gains."""
    assert ops.default_mla_splits(rows, topk, True) == splits


@pytest.mark.parametrize('rows', [1, 7, 64, 96, 255])
@pytest.mark.parametrize('v4', [False, True])
def test_one_round_of_workgroups(rows, v4):
    for topk in (512, 640, 1024, 2048, 8192):
        s = ops.default_mla_splits(rows, topk, v4)
        assert s >= 1 and (rows * s <= 256 or s == ops.default_mla_splits(1 << 20, topk, v4))
