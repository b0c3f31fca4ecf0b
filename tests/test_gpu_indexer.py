"""The top-k producers on the GPU against the oracle (oracle/topk.py): the selection bit for bit on the same FP32
logits; the QSA indexer logits (qsa_prefill.py:77-102) and the DSA FP8 logits (indexer_torch.py:28-72) within the
rounding of FP32 sums of exact products, the masked columns exactly; the hooks that carry them."""
import math

import numpy as np
import pytest
import torch

from oracle import topk as ref
from xtier_amd import glm, ops, qsa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('cols,k', [(1, 1), (100, 64), (5000, 2048), (4999, 1000), (100000, 2048), (70000, 4096)])
def test_topk_rows_bit_for_bit(cols, k):
    g = torch.Generator().manual_seed(cols + k)
    x = torch.randn(7, cols, generator=g)
    x[0] = torch.round(x[0] * 4) / 4                      # heavy ties
    x[1, : cols // 2] = -math.inf                        # masked half
    x[2] = -math.inf                                     # nothing finite
    if cols > 3:
        x[3, 1], x[3, 2] = math.nan, math.inf            # not finite: never taken
    x[4] = 1.0                                           # all equal: the lowest positions
    zero = torch.where(torch.rand(cols, generator=g) < 0.5, -0.0, 0.0)
    x[6] = torch.where(torch.arange(cols) % 7 == 3, x[6].abs() + 0.5, zero)   # -0 and +0 tie below the positives
    xg = x.cuda()
    got = ops.topk_rows(xg, k).cpu().numpy()
    want = ref.topk_rows(x.numpy(), k)
    assert np.array_equal(got, want)


@pytest.mark.parametrize('cols,k', [(96256, 2048), (70000, 512)])
def test_topk_rows_values_placed_by_position(cols, k):
    """Rows whose largest values sit at positions picked by the row's layout (one element of every other
    2048-position block, its complement, one lane of every 64, one position in 97): the selection must not depend
    on where in the row the large values are."""
    g = torch.Generator().manual_seed(cols)
    pos = torch.arange(cols)
    chunk, lane, elem = pos // 2048, (pos // 4) % 512, pos % 4
    picked = (chunk % 2 == 0) & (elem == (chunk // 2) % 4)
    x = torch.randn(4, cols, generator=g)
    x[0] = torch.where(picked, x[0], x[0] + 10)           # large values everywhere but the picked positions
    x[1] = torch.where(picked, x[1] + 10, x[1])           # large values only at the picked positions
    x[2] = torch.where(lane % 64 == 5, x[2] + 10, x[2])   # the large values all in one lane of every wavefront
    x[3] = torch.where(pos % 97 == 0, x[3], -math.inf)    # about cols / 97 finite values, fewer than k
    got = ops.topk_rows(x.cuda(), k).cpu().numpy()
    assert np.array_equal(got, ref.topk_rows(x.numpy(), k))


@pytest.mark.parametrize('cols', [1024, 2048, 2049, 4095, 4096, 4097, 8192, 8196, 16384, 16385, 32768, 32772, 49152, 49153, 65536, 65540,
                                  98304, 98305])
def test_topk_rows_edges_of_the_register_forms(cols):
    """Rows that just fill a form and that are just past it; random, with ties at the threshold, and masked."""
    g = torch.Generator().manual_seed(cols)
    x = torch.randn(4, -(-cols // 4) * 4, generator=g)[:, :cols]
    x[1] = torch.round(x[1] * 8) / 8
    x[2, 100:cols - 700] = -math.inf
    x[3] = 0.0
    x[3, -5:] = 1.0
    for k in (1, 2048):
        got = ops.topk_rows(x.cuda(), k).cpu().numpy()
        assert np.array_equal(got, ref.topk_rows(x.numpy(), k))


@pytest.mark.parametrize('rows,cols', [(300, 65540), (300, 20000), (270, 32768), (270, 49152), (300, 65533), (260, 98304), (257, 70001), (3, 98308), (2, 196608), (2, 196609),
                                       (2, 150003)])
def test_topk_rows_packed_forms(rows, cols):
    """More rows than CUs and rows past 98304 columns keep 16 bits per key: values that differ below those bits, ties
    that overflow the candidate lists, masked and non-finite columns."""
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows, -(-cols // 4) * 4, generator=g)[:, :cols]
    n = min(rows, 5)
    x[0] = 1.0 + torch.randint(0, 1 << 15, (cols,), generator=g) * 2.0 ** -23   # one bucket, differing low bits
    x[1] = torch.round(x[1] * 2) / 2
    if rows > 2:
        x[2, 5:cols - 900] = -math.inf
        x[-1, ::3] = math.nan
    for k in (1, 2048):
        got = ops.topk_rows(x.cuda(), k).cpu().numpy()
        for r in {0, 1, *range(n), rows - 1}:
            assert np.array_equal(got[r:r + 1], ref.topk_rows(x[r:r + 1].numpy(), k)), r


@pytest.mark.parametrize('rows,cols,skip', [(3, 4093, 0), (5, 5000, 1), (3, 32767, 3), (2, 65537, 2), (300, 30001, 0),
                                            (2, 131075, 1)])
def test_topk_rows_off_16_byte_alignment(rows, cols, skip):
    """Rows whose stride or base is not a multiple of 16 bytes."""
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows * cols + skip, generator=g)
    x[skip + 1::97] = -math.inf
    got = ops.topk_rows(x.cuda()[skip:].view(rows, cols), 2048).cpu().numpy()
    n = min(rows, 5)
    assert np.array_equal(got[:n], ref.topk_rows(x[skip:].view(rows, cols)[:n].numpy(), 2048))
    assert np.array_equal(got[-1:], ref.topk_rows(x[skip:].view(rows, cols)[-1:].numpy(), 2048))


@pytest.mark.parametrize('cols', [1, 3, 4, 255, 1000])
def test_topk_rows_short_rows_of_many(cols):
    """More than two rows per CU: rows of any length take the register forms."""
    g = torch.Generator().manual_seed(cols)
    x = torch.round(torch.randn(520, cols, generator=g) * 64) / 64
    x[1], x[2, ::2], x[3] = -math.inf, math.nan, 0.0
    for k in (1, 300):
        assert np.array_equal(ops.topk_rows(x.cuda(), k).cpu().numpy(), ref.topk_rows(x.numpy(), k))


def test_topk_rows_empty_rows():
    x = torch.randn(3, 8, device='cuda')[:, :0]          # rows of no column: nothing is read, every entry is -1
    assert np.array_equal(ops.topk_rows(x, 5).cpu().numpy(), np.full((3, 5), -1, np.int32))


def test_topk_rows_strided_rows_and_out():
    x = torch.randn(5, 3000, device='cuda')
    out = torch.full((5, 100), 7, dtype=torch.int32, device='cuda')
    ops.topk_rows(x[:, :2500], 100, out=out)
    assert np.array_equal(out.cpu().numpy(), ref.topk_rows(x[:, :2500].cpu().numpy(), 100))


def _bound_qsa(q, k, scale):
    """FP32 summation bound of the head sum of ReLU(q . k) / scale: exact products summed over dim, then over heads."""
    a = np.einsum('rhd,nd->rn', np.abs(q), np.abs(k))
    dim, heads = q.shape[2], q.shape[1]
    return (dim + heads + 2) * 2.0 ** -24 * a / scale


@pytest.mark.parametrize('rows,heads,dim,keys,dtype', [
    (37, 4, 128, 1000, torch.bfloat16), (352, 4, 128, 4096, torch.bfloat16), (5, 1, 64, 333, torch.bfloat16),
    (9, 8, 256, 700, torch.float16), (3, 32, 128, 257, torch.bfloat16), (20, 16, 64, 2100, torch.float16)])
def test_qsa_indexer_logits(rows, heads, dim, keys, dtype):
    g = torch.Generator().manual_seed(rows * keys)
    q = torch.randn(rows, heads, dim, generator=g).to(dtype)
    k = torch.randn(keys, 1, dim, generator=g).to(dtype)
    # causal ranges as the reference's check builds them (tests/qsa_prefill_check.py:25-33), plus empty and clipped
    pos = torch.arange(rows) * (keys // max(1, rows)) + keys // 3
    starts = torch.zeros(rows, dtype=torch.int32)
    ends = torch.clamp((pos + 1), max=keys + 50).to(torch.int32)
    starts[0], ends[0] = 5, 5
    if rows > 2:
        starts[2] = keys // 2
    got = ops.qsa_indexer_logits(q.cuda(), k.cuda(), starts.cuda(), ends.cuda()).cpu().numpy()
    qn, kn = q.float().numpy().astype(np.float64), k[:, 0].float().numpy().astype(np.float64)
    want = ref.qsa_indexer_logits(qn, kn, starts.numpy(), ends.numpy())
    assert np.array_equal(np.isinf(got), np.isinf(want)) and not np.isnan(got).any()
    fin = np.isfinite(want)
    err = np.abs(got.astype(np.float64)[fin] - want[fin])
    # the kernel multiplies by 1 / score_scale: one rounding of the reciprocal and one of the product
    bound = (_bound_qsa(qn, kn, math.sqrt(dim)) + np.abs(want) * 2.0 ** -23)[fin]
    assert (err <= bound).all(), float((err / bound).max())


@pytest.mark.parametrize('rows,heads,dim,keys,dtype', [
    (32, 4, 128, 63, torch.bfloat16), (33, 4, 128, 65, torch.float16), (129, 4, 128, 33000, torch.bfloat16),
    (1, 1, 128, 1, torch.bfloat16), (300, 1, 64, 70000, torch.bfloat16), (70, 2, 256, 129, torch.float16),
    (33, 8, 128, 64, torch.bfloat16), (40, 16, 128, 20000, torch.bfloat16), (17, 32, 256, 127, torch.float16),
    (9, 32, 128, 31, torch.bfloat16), (2, 1, 64, (1 << 20) + 5, torch.bfloat16)])
def test_qsa_indexer_logits_edges_of_the_tiles(rows, heads, dim, keys, dtype):
    """Rows at and past one workgroup's for one, two and four column groups, keys at stage edges, and rows too long for
    the 31-bit store offsets."""
    test_qsa_indexer_logits(rows, heads, dim, keys, dtype)


def _check_qsa(logits, q, k, starts, ends, scale):
    """Every logit against FP64 on the GPU, within the FP32 summation bound (_bound_qsa)."""
    heads, dim, keys = q.shape[1], q.shape[2], k.shape[0]
    kd, at = k.double(), torch.arange(keys, device='cuda')
    for r in range(q.shape[0]):
        qd = q[r].double()
        want = torch.clamp(qd @ kd.T, min=0).sum(0) / scale
        bound = (qd.abs().sum(0) @ kd.abs().T) * ((dim + heads + 2) * 2.0 ** -24 / scale) + want * 2.0 ** -23
        ok = (at >= int(starts[r])) & (at < int(ends[r]))
        assert (logits[r].double()[ok] - want[ok]).abs().le(bound[ok]).all(), r
        assert (logits[r][~ok] == -math.inf).all(), r


def _qsa_case(rows, heads, dim, keys, dtype):
    g = torch.Generator().manual_seed(rows * keys + heads)
    q = torch.randn(rows, heads, dim, generator=g).to(dtype).cuda()
    k = torch.randn(keys, dim, generator=g).to(dtype).cuda()
    ends = (torch.arange(rows) * (keys // rows) + keys // 3).clamp(max=keys).int()
    starts = torch.zeros(rows, dtype=torch.int32)
    starts[rows // 2], ends[0] = keys // 5, keys + 9
    return q, k, starts, ends


@pytest.mark.parametrize('rows,heads,dim,keys,dtype', [
    (300, 2, 128, 33000, torch.bfloat16), (70, 8, 128, 33001, torch.bfloat16), (70, 8, 64, 40000, torch.float16),
    (70, 16, 128, 40003, torch.bfloat16), (40, 16, 64, 33000, torch.float16), (30, 32, 64, 50001, torch.bfloat16),
    (30, 32, 128, 33000, torch.float16), (70, 32, 256, 20001, torch.bfloat16), (130, 8, 256, 20000, torch.bfloat16)])
def test_qsa_indexer_logits_most_column_groups(rows, heads, dim, keys, dtype):
    """Enough rows and keys for four column groups per wavefront (256 dims: two) at every number of heads."""
    q, k, starts, ends = _qsa_case(rows, heads, dim, keys, dtype)
    _check_qsa(ops.qsa_indexer_logits(q, k, starts.cuda(), ends.cuda()), q, k, starts, ends, math.sqrt(dim))


@pytest.mark.parametrize('heads', [1, 2, 4, 8, 16, 32])
@pytest.mark.parametrize('dim,dtype,odd', [(64, torch.bfloat16, 0), (64, torch.float16, 1), (128, torch.bfloat16, 1),
                                           (128, torch.float16, 0), (256, torch.bfloat16, 0), (256, torch.float16, 1)])
def test_qsa_indexer_logits_rows_far_apart(heads, dim, dtype, odd):
    """Logit rows so far apart that a workgroup's rows pass 2^31 bytes; the columns past the keys stay as they are."""
    rows, keys = 7, 1000 + 37 * odd
    ld = (heads << 20) + 4 + odd
    q, k, starts, ends = _qsa_case(rows, heads, dim, keys, dtype)
    buf = torch.empty(rows, ld, device='cuda')
    buf[:, keys:keys + 64] = 7.0
    s, e = starts.cuda(), ends.cuda()
    lib = ops._lib
    lib.check(lib.lib().xt_qsa_indexer_logits(
        q.data_ptr(), q.stride(0), q.stride(1), rows, heads, dim, k.data_ptr(), k.stride(0), keys, s.data_ptr(),
        e.data_ptr(), 1.5, lib.XT_DTYPE_BF16 if dtype == torch.bfloat16 else lib.XT_DTYPE_F16, buf.data_ptr(), ld,
        torch.cuda.current_stream().cuda_stream), 'qsa_indexer_logits')
    _check_qsa(buf[:, :keys], q, k, starts, ends, 1.5)
    assert (buf[:, keys:keys + 64] == 7.0).all()


@pytest.mark.parametrize('rows,prefix', [(352, 380000), (1000, 100000), (64, 8192), (4096, 30000), (37, 500000)])
def test_qsa_indexer_logits_reference_cases(rows, prefix):
    """The cases of tests/qsa_prefill_check.py:25-53: 4 heads x 128, compressed keys (ratio 4) up to the last row, each
    row's range [0, (pos + 1) / 4)."""
    g = torch.Generator().manual_seed(20261023 + rows)
    keys = (prefix + rows) // 4
    q = torch.randn(rows, 4, 128, generator=g).bfloat16()
    k = torch.randn(keys, 1, 128, generator=g).bfloat16()
    starts = torch.zeros(rows, dtype=torch.int32)
    ends = ((torch.arange(prefix, prefix + rows) + 1) // 4).to(torch.int32)
    got = ops.qsa_indexer_logits(q.cuda(), k.cuda(), starts.cuda(), ends.cuda()).cpu().numpy()
    qn, kn = q.float().numpy().astype(np.float64), k[:, 0].float().numpy().astype(np.float64)
    want = ref.qsa_indexer_logits(qn, kn, starts.numpy(), ends.numpy())
    fin = np.isfinite(want)
    assert np.array_equal(np.isinf(got), ~fin) and not np.isnan(got).any()
    a = np.zeros(want.shape)
    for h in range(4):
        a += np.abs(qn[:, h]) @ np.abs(kn).T
    bound = (130 + 4 + 2) * 2.0 ** -24 * a / math.sqrt(128) + np.abs(want) * 2.0 ** -23
    assert (np.abs(got.astype(np.float64)[fin] - want[fin]) <= bound[fin]).all()


def test_qsa_prefill_hook():
    calls = []
    original = lambda *a: calls.append(a) or 'original'
    q = torch.randn(4, 4, 128).bfloat16()
    k = torch.randn(9, 1, 128).bfloat16()
    s, e = torch.zeros(4, dtype=torch.int32), torch.full((4,), 9, dtype=torch.int32)
    assert qsa.qsa_mqa_prefill(original, q, k, s, e) == 'original'            # CPU tensors
    assert qsa.qsa_mqa_prefill(original, q.cuda()[:, :3], k.cuda(), s, e) == 'original'   # 3 heads
    got = qsa.qsa_mqa_prefill(original, q.cuda(), k.cuda(), s.cuda(), e.cuda(), 2.0)
    assert len(calls) == 2 and got.shape == (4, 9)
    want = ref.qsa_indexer_logits(q.float().numpy(), k[:, 0].float().numpy(), s.numpy(), e.numpy(), 2.0)
    assert np.allclose(got.cpu().numpy(), want, rtol=1e-5, atol=1e-5)


def _fp8(shape, g, scale=2.0):
    return (torch.randn(*shape, generator=g) * scale).to(torch.float8_e4m3fn)


@pytest.mark.parametrize('num_q,heads,num_kv,clean', [(300, 32, 1000, False), (64, 64, 5000, True),
                                                      (7, 96, 33, False)])
def test_dsa_mqa_logits(num_q, heads, num_kv, clean):
    """The shapes of tests/glm_indexer_torch_check.py:27-43 (300 queries x 1000 keys, 32 heads x 128) and wider."""
    g = torch.Generator().manual_seed(num_q + heads)
    q, k = _fp8((num_q, heads, 128), g), _fp8((num_kv, 128), g)
    k_scale = torch.rand(num_kv, generator=g) + 0.5
    w = torch.randn(num_q, heads, generator=g)
    ks = torch.randint(0, max(1, num_kv // 2), (num_q,), generator=g, dtype=torch.int32)
    ke = ks + torch.randint(1, num_kv, (num_q,), generator=g, dtype=torch.int32)
    got = glm.fp8_mqa_logits(None, q.cuda(), (k.cuda(), k_scale.cuda()), w.cuda(), ks.cuda(), ke.cuda(), clean)
    assert got.shape == (num_q, num_kv) and got.stride(0) == (num_kv + 3) // 4 * 4
    got = got.cpu().numpy().astype(np.float64)
    want = ref.dsa_mqa_logits(q.float().numpy(), k.float().numpy(), k_scale.numpy(), w.numpy(), ks.numpy(),
                              ke.numpy(), clean)
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fin = np.isfinite(want)
    rel = np.linalg.norm(got[fin] - want[fin]) / np.linalg.norm(want[fin])
    assert rel < 1e-5, rel                                 # the reference's own bound (glm_indexer_torch_check.py:42)
    a = (np.einsum('qhd,nd->qhn', np.abs(q.float().numpy()), np.abs(k.float().numpy())) *
         np.abs(w.numpy())[:, :, None]).sum(1) * k_scale.numpy()[None, :]
    assert (np.abs(got[fin] - want[fin]) <= ((128 + heads + 4) * 2.0 ** -24 * a)[fin] + 1e-30).all()


@pytest.mark.parametrize('scale', [0.05, 2.0, 20.0])
def test_dsa_logits_one_head_within_the_fp32_sum_bound(scale):
    """With one-hot head weights and unit key scales each logit is ReLU of one 128-term FP8 dot product: held to the
    bound of an FP32 sum of exact products (an FP8 matrix instruction that rounds inside its 16-product sums misses it
    by hundreds of units in the last place)."""
    g = torch.Generator().manual_seed(7)
    num_q, heads, num_kv, dim = 256, 32, 1024, 128
    q, k = _fp8((num_q, heads, dim), g, scale), _fp8((num_kv, dim), g, scale)
    w = torch.zeros(num_q, heads)
    w[torch.arange(num_q), torch.arange(num_q) % heads] = 1.0
    ks = torch.zeros(num_q, dtype=torch.int32)
    ke = torch.full((num_q,), num_kv, dtype=torch.int32)
    got = ops.dsa_mqa_logits(q.cuda(), (k.cuda(), torch.ones(num_kv, device='cuda')), w.cuda(), ks.cuda(),
                             ke.cuda()).cpu().numpy().astype(np.float64)
    qs = q.float().numpy().astype(np.float64)[np.arange(num_q), np.arange(num_q) % heads]
    kd = k.float().numpy().astype(np.float64)
    exact = np.maximum(qs @ kd.T, 0.0)
    assert (np.abs(got - exact) <= (dim + 2) * 2.0 ** -24 * (np.abs(qs) @ np.abs(kd).T)).all()


def test_dsa_paged_mqa_logits():
    """The decode case of tests/glm_indexer_torch_check.py:44-65: 3 rows over 8 pages of 64 in a pool of 40."""
    g = torch.Generator().manual_seed(20261029)
    H, D, BLOCK, pages = 32, 128, 64, 40
    kv = torch.empty(pages, BLOCK * (D + 4), dtype=torch.uint8)
    vals = _fp8((pages, BLOCK, D), g)
    scl = torch.rand(pages, BLOCK, generator=g) + 0.5
    kv[:, :BLOCK * D] = vals.view(torch.uint8).reshape(pages, -1)
    kv[:, BLOCK * D:] = scl.view(torch.uint8).reshape(pages, -1)
    kv4 = kv.view(pages, BLOCK, 1, D + 4)
    table = torch.randperm(pages, generator=g)[:24].view(3, 8).to(torch.int32)
    lens = torch.tensor([512, 300, 77], dtype=torch.int32)
    q = _fp8((3, 1, H, D), g)
    w = torch.randn(3, H, generator=g)
    for clean in (False, True):
        for msl in (8 * BLOCK, 8 * BLOCK + 100):
            got = glm.fp8_paged_mqa_logits(None, q.cuda(), kv4.cuda(), w.cuda(), lens.view(3, 1).cuda(),
                                           table.cuda(), None, msl, clean).cpu().numpy().astype(np.float64)
            want = ref.dsa_paged_mqa_logits(q[:, 0].float().numpy(), kv.numpy(), w.numpy(), lens.numpy(),
                                            table.numpy(), msl, clean)
            assert np.array_equal(np.isinf(got), np.isinf(want)) and got.shape == want.shape
            fin = np.isfinite(want) & (want != 0)
            assert np.linalg.norm(got[fin] - want[fin]) / np.linalg.norm(want[fin]) < 1e-5
            assert np.array_equal(got[~fin & ~np.isinf(want)], want[~fin & ~np.isinf(want)])


@pytest.mark.parametrize('heads,dim,block,msl', [
    (32, 128, 64, 640), (64, 128, 32, 2083), (64, 64, 128, 1), (128, 64, 96, 31), (32, 256, 64, 33), (96, 64, 256, 4096),
    (32, 128, 48, 500), (64, 256, 64, 300), (128, 128, 64, 300)])
def test_dsa_paged_logits_edges(heads, dim, block, msl):
    """Lengths at the edges of 32-key blocks, pages and the table, negative and out-of-range table entries (the first
    reads page 0, the others no key), page sizes off the 32-key grid and head counts past the register budget; every
    logit within the FP32 summation bound."""
    g = torch.Generator().manual_seed(heads + dim + block + msl)
    lens = torch.tensor([0, 1, 31, 32, 33, block - 1, block, block + 1, msl - 1, msl, msl + 500], dtype=torch.int32)
    rows, width, pages = len(lens), max(1, -(-msl // block)), 37
    vals = _fp8((pages, block, dim), g)
    scl = torch.rand(pages, block, generator=g) + 0.5
    kv = torch.empty(pages, block * (dim + 4), dtype=torch.uint8)
    kv[:, :block * dim] = vals.view(torch.uint8).reshape(pages, -1)
    kv[:, block * dim:] = scl.view(torch.uint8).reshape(pages, -1)
    table = torch.randint(0, pages, (rows, width), generator=g, dtype=torch.int32)
    table[2, 0], table[9, width // 2], table[10, width - 1] = -1, pages, 2 ** 31 - 1
    q, w = _fp8((rows, 1, heads, dim), g), torch.randn(rows, heads, generator=g)
    for clean in (False, True):
        got = ops.dsa_paged_mqa_logits(q.cuda(), kv.view(pages, block, 1, dim + 4).cuda(), w.cuda(), lens.cuda(),
                                       table.cuda(), None, msl, clean).cpu().numpy().astype(np.float64)
        fill = -np.inf if clean else 0.0
        for r in range(rows):
            n = min(int(lens[r]), msl, width * block)
            page = table[r].clamp(min=0).long().repeat_interleave(block)[:n]
            live = (page < pages).numpy()
            page = page.clamp(max=pages - 1)
            at = torch.arange(n) % block
            k, ks = vals[page, at].float().numpy().astype(np.float64), scl[page, at].numpy().astype(np.float64)
            qd, wd = q[r, 0].float().numpy().astype(np.float64), w[r].numpy().astype(np.float64)
            want = np.where(live, (np.maximum(qd @ k.T, 0) * wd[:, None]).sum(0) * ks, fill)
            bound = (dim + heads + 4) * 2.0 ** -24 * ((np.abs(qd) @ np.abs(k).T) * np.abs(wd)[:, None]).sum(0) * ks
            same = got[r, :n] == want
            assert (same | (np.abs(got[r, :n] - np.where(np.isinf(want), 0, want)) <= bound + 1e-30)).all(), r
            assert (got[r, n:] == fill).all(), r


@pytest.mark.parametrize('rows,heads,dim,block,msl,run', [
    (32, 32, 128, 64, 4096, 2), (48, 64, 128, 32, 4096, 3), (41, 32, 256, 96, 5000, 4), (24, 128, 64, 64, 6001, 3),
    (80, 96, 64, 128, 4095, 5), (64, 32, 128, 64, 65536, 64), (65, 64, 64, 256, 65536 + 33, 64)])
def test_dsa_paged_logits_runs_of_blocks(rows, heads, dim, block, msl, run):
    """Runs of several 32-key blocks per wavefront, up to the 64 table entries it holds: lengths that end at every block
    of a run and inside it, pages crossed within a run, bad table entries in its middle. Every key against FP64."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert min(64, -(-(-(-msl // 32) * rows) // (8 * cus))) == run or cus != 256   # as the launch sizes it
    g = torch.Generator().manual_seed(rows + heads + msl)
    width, pages = -(-msl // block), 37
    vals, scl = _fp8((pages, block, dim), g), torch.rand(pages, block, generator=g) + 0.5
    kv = torch.empty(pages, block * (dim + 4), dtype=torch.uint8)
    kv[:, :block * dim] = vals.view(torch.uint8).reshape(pages, -1)
    kv[:, block * dim:] = scl.view(torch.uint8).reshape(pages, -1)
    table = torch.randint(0, pages, (rows, width), generator=g, dtype=torch.int32)
    bad = torch.rand(rows, width, generator=g)
    table[bad < 0.03], table[bad > 0.97] = -1, pages
    table[-1, width // 2] = 2 ** 31 - 1
    r = torch.arange(rows)
    lens = (msl // 2 // (32 * run) * run + r % (run + 1)) * 32 + torch.tensor([0, 1, 17, 31])[r // (run + 1) % 4]
    lens[::5] = msl
    lens[1], lens[2], lens[3] = 0, 32 * run + 1, msl + 500
    q, w = _fp8((rows, 1, heads, dim), g), torch.randn(rows, heads, generator=g)
    qd, kd = q[:, 0].cuda().double(), vals.view(-1, dim).cuda().double()
    wd, sd = w.cuda().double(), scl.view(-1).cuda().double()
    n = lens.clamp(max=min(msl, width * block)).cuda().view(-1, 1)
    at = torch.arange(msl, device='cuda')
    page = table.cuda().long().clamp(min=0)[:, (at // block).clamp(max=width - 1)]
    live = (at < n) & (page < pages)
    slot = page.clamp(max=pages - 1) * block + at % block
    for clean in (False, True):
        got = ops.dsa_paged_mqa_logits(q.cuda(), kv.view(pages, block, 1, dim + 4).cuda(), w.cuda(), lens.int().cuda(),
                                       table.cuda(), None, msl, clean).double()
        for i in range(rows):
            score = (torch.clamp(qd[i] @ kd.T, min=0) * wd[i].view(-1, 1)).sum(0) * sd
            bound = ((qd[i].abs() @ kd.abs().T) * wd[i].abs().view(-1, 1)).sum(0) * sd * ((dim + heads + 4) * 2.0 ** -24)
            ok = live[i]
            assert (got[i][ok] - score[slot[i][ok]]).abs().le(bound[slot[i][ok]] + 1e-30).all(), i
            assert (got[i][~ok] == (-math.inf if clean else 0.0)).all(), i


def test_glm_schedule_and_sm_count():
    assert glm.get_paged_mqa_logits_metadata(None, 1, 2, x=3) is None
    assert glm.get_num_sms(None) == torch.cuda.get_device_properties(0).multi_processor_count
    assert {t for t, _ in glm.HOOKS} == {'deep_gemm.fp8_mqa_logits', 'deep_gemm.fp8_paged_mqa_logits',
                                         'deep_gemm.get_paged_mqa_logits_metadata', 'deep_gemm.get_num_sms'}
