"""What the block-sparse prefill (kv_fp4.py:369-404) refuses on the host, before any launch: no GPU needed, and the
library's entries are replaced so that none can be reached."""
import pytest
import torch

from xtier_amd import ops

PAGES, KH, BLOCK, D = 4, 2, 128, 128


class Reached(Exception):
    """A library entry was about to be called."""


@pytest.fixture(autouse=True)
def no_launch(monkeypatch):
    class Library:
        def __getattr__(self, name):
            raise Reached(name)
    monkeypatch.setattr(ops._lib, 'lib', Library)


def _args(cu, n, blocks=None):
    """Queries of the ragged batch cu over arrays of n requests."""
    pay = torch.zeros(PAGES, KH, BLOCK, D // 2, dtype=torch.uint8)
    sc = torch.zeros(PAGES, KH, BLOCK, D // 16, dtype=torch.uint8)
    total = max(cu)
    kw = dict(q=torch.zeros(total, 2 * KH, D, dtype=torch.bfloat16), k_cache=pay, v_cache=pay.clone(), sink=None,
              req_to_token=torch.zeros(8, 512, dtype=torch.int32), slot_ids=torch.zeros(n, dtype=torch.int64),
              topk_idx=torch.zeros(KH, max(1, total), 2, dtype=torch.int32), block_size_q=1, block_size_k=BLOCK,
              cu_seqlens=torch.tensor(cu, dtype=torch.int32), seq_lens=torch.ones(n, dtype=torch.int32),
              prefix_lens=torch.zeros(n, dtype=torch.int32), max_seqlen_q=total, k_sc=sc, v_sc=sc.clone())
    if blocks is not None:
        kw['cu_seqblocks_q'] = torch.tensor(blocks, dtype=torch.int32)
    return kw


@pytest.mark.parametrize('name', ['cu_seqblocks_q', 'k_sc', 'v_sc', 'slot_ids', 'cu_seqlens', 'topk_idx'])
def test_each_tensor_must_be_on_the_gpu(monkeypatch, name):
    """One tensor on the host, every other one taken for a GPU tensor."""
    kw = _args([0, 3, 5], 2, [0, 3, 5])
    host = kw[name].untyped_storage().data_ptr()

    def need_cuda(*tensors):
        if any(t is not None and t.untyped_storage().data_ptr() == host for t in tensors):
            raise ValueError('on the host')
    monkeypatch.setattr(ops, '_need_cuda', need_cuda)
    with pytest.raises(ValueError, match='on the host'):
        ops.fp4_prefill_gqa_share_sparse(**kw)


@pytest.mark.parametrize('cu,n,blocks', [([0, 3, 5], 1, None), ([0, 3, 5], 0, None), ([0, 0, 5], 1, [0, 0, 5]),
                                         ([0, 3, 5], 2, [0]), ([0, 2, 4, 5], 2, [0, 2, 4, 5])])
def test_arrays_short_of_the_requests_with_rows_are_refused(monkeypatch, cu, n, blocks):
    """They were indexed out of bounds once; taken as they are, another request's keys would answer."""
    monkeypatch.setattr(ops, '_need_cuda', lambda *tensors: None)
    with pytest.raises(ValueError, match='requests'):
        ops.fp4_prefill_gqa_share_sparse(**_args(cu, n, blocks))


@pytest.mark.parametrize('cu,n,blocks', [([0, 3, 5], 2, None), ([0, 3, 5, 5, 5], 2, None), ([0, 3, 5, 5], 2, [0, 3, 5]),
                                         ([0, 3, 5], 4, None), ([0], 1, None)])
def test_arrays_that_cover_every_row_are_taken(monkeypatch, cu, n, blocks):
    """Requests without rows at the end need no entries, and longer arrays do no harm."""
    monkeypatch.setattr(ops, '_need_cuda', lambda *tensors: None)
    kw = _args(cu, n, blocks)
    if not kw['q'].shape[0]:
        kw['q'] = torch.zeros(2, 2 * KH, D, dtype=torch.bfloat16)
    with pytest.raises(Reached, match='xt_block_prefill_rows'):
        ops.fp4_prefill_gqa_share_sparse(**kw)
