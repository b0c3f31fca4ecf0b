"""The calls a serving program makes of this package, as timed cases: sparse decode and prefill attention over NVFP4
pools (GQA, head-major pages, latent caches), the FP8 latent pages, the index scores that pick their keys, the
selection, and the quantized append of new keys and values. Sizes are those of the package's workloads
(xtier_amd/workloads.py, bench.py), with smaller, ragged and odd ones among the drawn cases.

prepare() builds what the program holds before a call: the quantized pools, tables, lists and activations; run() is one
pass through the public entry points; exact() is the same result in 64 bits from plain torch.
"""
import math

import torch

from xtier_amd import ops
from xtier_amd.pool import KVPool, LatentPool

DEV = 'cuda'


def listed():
    return [
        # one chat request, two wide KV heads, SGLang's pool and token table: every layer of every token pays its latency
        {'name': 'decode_one', 'path': 'decode', 'rows': 1, 'q_heads': 16, 'kv_heads': 2, 'dim': 256, 'ctx': 4099,
         'topk': 512, 'page': 1, 'layout': 'split', 'ragged': False},
        # a full decode batch at 32K context, the package's own pool layout
        {'name': 'decode_batch', 'path': 'decode', 'rows': 32, 'q_heads': 32, 'kv_heads': 4, 'dim': 128, 'ctx': 32768,
         'topk': 2048, 'page': 64, 'layout': 'interleaved', 'ragged': False},
        # a chunk of a long prompt: its keys and values quantized into the pool, then each query over its own keys
        {'name': 'prefill_chunk', 'path': 'prefill', 'rows': 4096, 'q_heads': 32, 'kv_heads': 4, 'dim': 128,
         'ctx': 65536, 'topk': 2048, 'page': 64},
        # a decode batch over head-major pages: the layer's index block scores and its attention over picked blocks
        {'name': 'block_decode', 'path': 'block_decode', 'rows': 32, 'q_heads': 64, 'kv_heads': 4, 'dim': 128,
         'ctx': 32768, 'blocks': 16, 'ragged': False},
        # the same layer on a chunk of a long prompt
        {'name': 'block_prefill', 'path': 'block_prefill', 'rows': 4096, 'q_heads': 64, 'kv_heads': 4, 'dim': 128,
         'ctx': 61440, 'blocks': 16},
        # latent attention: a decode batch with 128 heads
        {'name': 'mla_decode', 'path': 'mla', 'rows': 64, 'heads': 128, 'ctx': 16384, 'topk': 2048, 'causal': False},
        # latent attention: a prompt chunk, the largest call
        {'name': 'mla_prefill', 'path': 'mla', 'rows': 2048, 'heads': 128, 'ctx': 65536, 'topk': 2048, 'causal': True},
        # FP8 latent pages: a window list and a list of compressed keys, lists of differing lengths, a sink
        {'name': 'mla_pages', 'path': 'mla_pages', 'rows': 61, 'heads': 64, 'window': 128, 'extra': 512},
        # the index logits of a prompt chunk against a long context
        {'name': 'index_prefill', 'path': 'index_prefill', 'rows': 352, 'heads': 4, 'dim': 128, 'keys': 95088},
        # the index logits of a decode batch over its paged FP8 index cache
        {'name': 'index_decode', 'path': 'index_decode', 'rows': 32, 'heads': 32, 'dim': 128, 'ctx': 32768},
        # the selection of a decode batch and of a prompt chunk
        {'name': 'select_decode', 'path': 'select', 'rows': 32, 'cols': 32768, 'topk': 2048, 'ragged': True},
        {'name': 'select_prefill', 'path': 'select', 'rows': 352, 'cols': 95088, 'topk': 2048, 'ragged': True},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(['decode', 'decode', 'prefill', 'block_decode', 'block_prefill', 'mla', 'mla', 'mla_pages',
                       'index_prefill', 'index_decode', 'select', 'select'])
    if path == 'decode':
        q_heads, kv_heads, dim = rng.choice([(32, 4, 128), (8, 1, 128), (16, 2, 256), (32, 2, 256), (16, 4, 64),
                                             (40, 8, 128)])
        rows = _spread(rng, 1, 64)
        return {'path': path, 'rows': rows, 'q_heads': q_heads, 'kv_heads': kv_heads, 'dim': dim,
                'ctx': _spread(rng, 600, min(131072, (1 << 20) // rows)), 'topk': rng.choice([512, 1024, 2048]),
                'page': rng.choice([1, 16, 64]), 'layout': rng.choice(['interleaved', 'split']),
                'ragged': rng.random() < 0.7}
    if path == 'prefill':
        return {'path': path, 'rows': _spread(rng, 65, 4096), 'q_heads': 32, 'kv_heads': rng.choice([2, 4, 8]),
                'dim': 128, 'ctx': _spread(rng, 2500, 65536), 'topk': rng.choice([512, 1024, 2048]), 'page': 64}
    if path == 'block_decode':
        rows = _spread(rng, 1, 48)
        return {'path': path, 'rows': rows, 'q_heads': rng.choice([32, 64]), 'kv_heads': rng.choice([2, 4]),
                'dim': 128, 'ctx': _spread(rng, 2500, (1 << 20) // rows // 2), 'blocks': rng.choice([8, 16]),
                'ragged': rng.random() < 0.7}
    if path == 'block_prefill':
        return {'path': path, 'rows': _spread(rng, 65, 4096), 'q_heads': rng.choice([32, 64]), 'kv_heads': 4,
                'dim': 128, 'ctx': _spread(rng, 128, 480) * 128, 'blocks': rng.choice([8, 16])}
    if path == 'mla':
        causal = rng.random() < 0.4
        return {'path': path, 'rows': _spread(rng, 129, 2048) if causal else _spread(rng, 1, 96),
                'heads': rng.choice([64, 128, 128]), 'ctx': _spread(rng, 3000, 65536 if causal else 10000),
                'topk': rng.choice([512, 1024, 2048]), 'causal': causal}
    if path == 'mla_pages':
        return {'path': path, 'rows': _spread(rng, 1, 512), 'heads': rng.choice([64, 128]), 'window': 128,
                'extra': rng.choice([0, 128, 512, 1024])}
    if path == 'index_prefill':
        return {'path': path, 'rows': _spread(rng, 1, 512), 'heads': rng.choice([1, 2, 4, 8, 16]),
                'dim': rng.choice([64, 128]), 'keys': _spread(rng, 600, 65536)}
    if path == 'index_decode':
        rows = _spread(rng, 1, 64)
        return {'path': path, 'rows': rows, 'heads': rng.choice([32, 64]), 'dim': 128,
                'ctx': _spread(rng, 600, (1 << 20) // rows)}
    rows = _spread(rng, 1, 512)
    return {'path': path, 'rows': rows, 'cols': _spread(rng, 600, min(262144, (1 << 25) // rows)),
            'topk': rng.choice([512, 1024, 2048]), 'ragged': rng.random() < 0.7}


# --- inputs ---------------------------------------------------------------------------------------------------------

_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(shape, g, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def _activations(n, heads, dim, g):
    """Keys or values: normal, with one channel in a hundred eight times as large."""
    x = torch.randn(n, heads, dim, generator=g, device=DEV)
    pick = torch.randperm(heads * dim, generator=g, device=DEV)[:max(1, heads * dim // 100)]
    scale = torch.ones(heads * dim, device=DEV)
    scale[pick] = 8.0
    return x.mul_(scale.view(1, heads, dim)).to(torch.bfloat16)


def _global_scale(x):
    return (x.abs().amax().float() / 2688).clamp(min=1e-12).reshape(1)


def _nvfp4(x, g):
    """Plain NVFP4 quantization: (payload, scale bytes) of BF16 rows [n, heads, dim] with the global scale g [1]."""
    n, heads, dim = x.shape
    pay = torch.empty(n, heads, dim // 2, dtype=torch.uint8, device=x.device)
    sc = torch.empty(n, heads, dim // 16, dtype=torch.uint8, device=x.device)
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=x.device)
    step = max(1, (1 << 27) // (heads * dim))
    for i in range(0, n, step):
        b = x[i:i + step].float().reshape(-1, heads, dim // 16, 16)
        s = (b.abs().amax(-1) / (6.0 * g)).clamp(max=448.0).to(torch.float8_e4m3fn)
        y = b / (s.float() * g).clamp(min=1e-30).unsqueeze(-1)
        code = torch.bucketize(y.abs(), mid, out_int32=True).to(torch.uint8)   # ties to the lower code
        code |= (y < 0).to(torch.uint8) << 3
        code = code.reshape(-1, heads, dim // 2, 2)
        pay[i:i + step] = code[..., 0] | (code[..., 1] << 4)
        sc[i:i + step] = s.view(torch.uint8)
    return pay, sc


def _table64(device):
    t = torch.tensor(_E2M1, dtype=torch.float64, device=device)
    return torch.cat([t, -t])


def _decode64(pay, sc):
    """NVFP4 rows [..., width / 2], scale bytes [..., width / 16] -> FP64 [..., width], without the global scale."""
    t = _table64(pay.device)
    v = torch.stack([t[(pay & 15).long()], t[(pay >> 4).long()]], -1).flatten(-2)
    s = sc.contiguous().view(torch.float8_e4m3fn).double()
    return (v.unflatten(-1, (-1, 16)) * s.unsqueeze(-1)).flatten(-2)


def _lists(limits, n, g):
    """Per row n distinct sorted positions below limits[row], one in each n-th of the range; shorter ranges give every
    position, then -1."""
    lim = limits.to(torch.int64).view(-1, 1)
    i = torch.arange(n, device=DEV).view(1, -1)
    lo, hi = lim * i // n, lim * (i + 1) // n
    u = torch.rand(lim.shape[0], n, generator=g, device=DEV, dtype=torch.float64)
    pos = lo + torch.minimum((u * (hi - lo)).long(), (hi - lo - 1).clamp(min=0))
    return torch.where(lim >= n, pos, torch.where(i < lim, i, -1))


def _pages(rows, ctx, page, g):
    n = -(-ctx // page)
    return torch.randperm(rows * n, generator=g, device=DEV).view(rows, n)


def _lengths(case, lo, g):
    if not case['ragged']:
        return torch.full((case['rows'],), case['ctx'], dtype=torch.int32, device=DEV)
    return torch.randint(min(lo, case['ctx']), case['ctx'] + 1, (case['rows'],), generator=g, device=DEV,
                         dtype=torch.int32)


def _kv_pool(slots, heads, dim, layout, g):
    pool = KVPool(slots, heads, dim, DEV, layout=layout)
    for pay, sc, gs in ((pool.k_pay, pool.k_sf, pool.gk), (pool.v_pay, pool.v_sf, pool.gv)):
        x = _activations(slots, heads, dim, g)
        gs.copy_(_global_scale(x))
        p, s = _nvfp4(x, gs)
        pay.copy_(p)
        sc.copy_(s)
    return pool


def _recent_lists(pos, topk, g):
    """Causal lists: the 128 most recent positions and the others spread below them."""
    near = min(128, topk // 2)
    lo = pos - near + 1
    far = _lists(lo, topk - near, g)
    return torch.cat([far, lo.view(-1, 1) + torch.arange(near, device=DEV)], 1)


def _prepare_decode(c, g):
    rows, page = c['rows'], c['page']
    table = _pages(rows, c['ctx'], page, g)
    pool = _kv_pool(table.numel() * page, c['kv_heads'], c['dim'], c['layout'], g)
    seq = _lengths(c, 300, g)
    return {'q': _randn((rows, c['q_heads'], c['dim']), g), 'pool': pool, 'table': table.int(), 'seq': seq,
            'req': torch.arange(rows, device=DEV), 'idx': _lists(seq, c['topk'], g).int(), 'scale': c['dim'] ** -0.5}


def _prepare_prefill(c, g):
    ctx, n, page = c['ctx'], c['rows'], c['page']
    total = ctx + n
    table = _pages(1, total, page, g)
    pool = _kv_pool(table.numel() * page, c['kv_heads'], c['dim'], 'interleaved', g)
    pos = torch.arange(ctx, total, device=DEV)
    slots = table[0, pos // page] * page + pos % page
    # the chunk's rows are new: cleared here, appended by the pass
    pool.buffer[slots] = 0
    return {'q': _randn((n, c['q_heads'], c['dim']), g), 'pool': pool, 'table': table.int(), 'slots': slots,
            'k': _activations(n, c['kv_heads'], c['dim'], g),
            'v': _activations(n, c['kv_heads'], c['dim'], g),
            'idx': _recent_lists(pos, c['topk'], g).int(), 'pos': pos.int(), 'seq': (pos + 1).int(),
            'req': torch.zeros(n, dtype=torch.int64, device=DEV), 'scale': c['dim'] ** -0.5}


def _block_pools(pages, kv_heads, dim, g):
    """Head-major pages of K and V and the one-head index pages, unit global scale."""
    one = torch.ones(1, device=DEV)
    out = []
    for heads in (kv_heads, kv_heads, 1):
        p, s = _nvfp4(_activations(pages * 128, heads, dim, g), one)
        out += [t.view(pages, 128, heads, -1).permute(0, 2, 1, 3).contiguous() for t in (p, s)]
    return out[:4] + [out[4].squeeze(1), out[5].squeeze(1)]


def _prepare_blocks(c, g):
    prefill = c['path'] == 'block_prefill'
    rows, kh, dim = c['rows'], c['kv_heads'], c['dim']
    reqs, total = (1, c['ctx'] + rows) if prefill else (rows, c['ctx'])
    width = -(-total // 128) * 128
    table = _pages(reqs, total, 128, g)
    kp, ks, vp, vs, ip, isc = _block_pools(table.numel(), kh, dim, g)
    r2t = (table[:, :, None] * 128 + torch.arange(128, device=DEV)).reshape(reqs, width).int()
    s = {'k': kp, 'ks': ks, 'v': vp, 'vs': vs, 'ip': ip, 'is': isc, 'r2t': r2t,
         'q': _randn((rows, c['q_heads'], dim), g), 'iq': _randn((rows, 4, dim), g), 'scale': dim ** -0.5,
         'sid': torch.arange(reqs, device=DEV),
         'score': torch.full((4, rows, width // 128), -math.inf, device=DEV)}
    if prefill:
        pos = torch.arange(c['ctx'], total, device=DEV)
        own = (pos // 128).view(1, -1).expand(kh, -1)
        far = _lists(own.reshape(-1), c['blocks'] - 1, g).view(kh, rows, -1)
        i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
        s |= {'idx': torch.cat([own.unsqueeze(2), far], 2).int(), 'cu': i32(0, rows), 'seq': i32(total),
              'pre': i32(c['ctx'])}
    else:
        s['seq'] = _lengths(c, 300, g)
        nb = ((s['seq'] + 127) // 128).repeat(kh)
        s['idx'] = _lists(nb, c['blocks'], g).view(kh, rows, -1).int()
    return s


def _prepare_mla(c, g):
    rows, ctx, causal = c['rows'], c['ctx'], c['causal']
    reqs, total = (1, ctx + rows) if causal else (rows, ctx)
    table = _pages(reqs, total, 64, g)
    slots = table.numel() * 64
    pool = LatentPool(slots, device=DEV)
    lat = _activations(slots, 1, 512, g)
    pool.g = _global_scale(lat)
    p, s = _nvfp4(lat, pool.g)
    pool.pay.copy_(p.view(slots, -1))
    pool.scales.copy_(s.view(slots, -1))
    pool.rope.copy_(_randn((slots, 64), g))
    if causal:
        pos = _recent_lists(torch.arange(ctx, total, device=DEV), c['topk'], g)
    else:
        pos = _lists(torch.full((rows,), ctx, device=DEV), c['topk'], g)
    req = torch.zeros(rows, dtype=torch.int64, device=DEV) if causal else torch.arange(rows, device=DEV)
    at = pos.clamp(min=0)
    idx = torch.where(pos >= 0, table[req[:, None], at // 64] * 64 + at % 64, -1).int()
    return {'q': _randn((rows, 1, c['heads'], 576), g, scale=0.5), 'pool': pool, 'idx': idx.unsqueeze(1),
            'scale': 576 ** -0.5}


def _fp8_pages(tokens, page, g):
    """FP8 latent pages [pages, page, 1, 584]: E4M3 values, exponents around 1, BF16 rope values."""
    n = tokens // page
    buf = torch.zeros(n, page * 584, dtype=torch.uint8, device=DEV)
    data = buf[:, :page * 576].view(n, page, 576)
    data[..., :448] = _randn((n, page, 448), g, torch.float8_e4m3fn, 32.0).view(torch.uint8)
    data[..., 448:] = _randn((n, page, 64), g).view(torch.uint8)
    sc = buf[:, page * 576:].view(n, page, 8)
    sc[..., :7] = torch.randint(120, 125, (n, page, 7), generator=g, device=DEV, dtype=torch.uint8)
    return buf.as_strided((n, page, 1, 584), (page * 584, 584, 584, 1))


def _prepare_mla_pages(c, g):
    rows, extra = c['rows'], c['extra']
    s = {'q': _randn((rows, 1, c['heads'], 512), g), 'cache': _fp8_pages(rows * 256, 256, g), 'scale': 512 ** -0.5,
         'sink': _randn((c['heads'],), g, torch.float32), 'cache2': None, 'idx2': None, 'len2': None}
    base = torch.arange(rows, device=DEV).view(rows, 1, 1)
    s['idx'] = (base * 256 + torch.arange(c['window'], device=DEV) + 64).int()
    s['len'] = torch.randint(c['window'] // 2, c['window'] + 1, (rows,), generator=g, device=DEV, dtype=torch.int32)
    if extra:
        s['cache2'] = _fp8_pages(rows * 4096, 128, g)
        pick = _lists(torch.full((rows,), 4096, device=DEV), extra, g).unsqueeze(1)
        s['idx2'] = (base * 4096 + pick).int()
        s['len2'] = torch.randint(extra // 2, extra + 1, (rows,), generator=g, device=DEV, dtype=torch.int32)
    return s


def _prepare_index_prefill(c, g):
    rows, keys = c['rows'], c['keys']
    # the chunk's queries are the last positions of the context: each sees the keys up to its own
    end = torch.arange(keys - rows, keys, device=DEV).clamp(min=0) + 1
    return {'q': _randn((rows, c['heads'], c['dim']), g), 'k': _randn((keys, 1, c['dim']), g),
            'start': torch.zeros(rows, dtype=torch.int32, device=DEV), 'end': end.int()}


def _prepare_index_decode(c, g):
    rows, dim = c['rows'], c['dim']
    table = _pages(rows, c['ctx'], 64, g)
    n = table.numel()
    cache = torch.empty(n, 64, 1, dim + 4, dtype=torch.uint8, device=DEV)
    flat = cache.view(n, -1)
    flat[:, :64 * dim] = _randn((n, 64 * dim), g, torch.float32, 100.0).clamp(-448, 448).to(torch.float8_e4m3fn).view(
        torch.uint8)
    flat[:, 64 * dim:] = (torch.rand(n, 64, generator=g, device=DEV) * 0.01 + 0.01).view(torch.uint8)
    return {'q': _randn((rows, 1, c['heads'], dim), g, torch.float8_e4m3fn), 'cache': cache, 'table': table.int(),
            'w': torch.rand(rows, c['heads'], generator=g, device=DEV) / c['heads'],
            'lens': torch.randint(min(300, c['ctx']), c['ctx'] + 1, (rows,), generator=g, device=DEV,
                                  dtype=torch.int32), 'ctx': c['ctx']}


def _prepare_select(c, g):
    rows, cols = c['rows'], c['cols']
    x = torch.randn(rows, cols, generator=g, device=DEV)
    if c['ragged']:   # a row's scores end at its length, with -inf behind
        n = torch.randint(cols // 2, cols + 1, (rows, 1), generator=g, device=DEV)
        x.masked_fill_(torch.arange(cols, device=DEV) >= n, -math.inf)
    return {'x': x, 'topk': c['topk']}


_PREPARE = {'decode': _prepare_decode, 'prefill': _prepare_prefill, 'block_decode': _prepare_blocks,
            'block_prefill': _prepare_blocks, 'mla': _prepare_mla, 'mla_pages': _prepare_mla_pages,
            'index_prefill': _prepare_index_prefill, 'index_decode': _prepare_index_decode, 'select': _prepare_select}


def prepare(case, seed):
    return {'path': case['path'], 'page': case.get('page', 1), **_PREPARE[case['path']](case, _gen(seed))}


# --- one pass -------------------------------------------------------------------------------------------------------

def run(s):
    path = s['path']
    if path == 'decode':
        return ops.sparse_decode(s['q'], s['pool'].raw, s['table'], s['idx'], s['seq'], s['scale'],
                                 page_size=s['page'], row_req=s['req'])
    if path == 'prefill':
        s['pool'].append(s['k'], s['v'], s['slots'])
        out = ops.sparse_decode(s['q'], s['pool'].raw, s['table'], s['idx'], s['seq'], s['scale'],
                                page_size=s['page'], row_req=s['req'], query_pos=s['pos'])
        return out, s['pool'].buffer
    if path == 'block_decode':
        # no forced blocks: their 1e29 would hide the other scores in a comparison
        ops.minimax_decode_scores(s['iq'], s['ip'], s['is'], s['r2t'], s['score'], s['seq'], s['sid'], 128, s['scale'],
                                  1.0, 0, 0)
        return s['score'], ops.fp4_sparse_decode(s['q'], s['k'], s['ks'], s['v'], s['vs'], s['r2t'], s['sid'],
                                                 s['idx'], s['seq'], 128, s['scale'])
    if path == 'block_prefill':
        n = s['q'].shape[0]
        ops.minimax_prefill_scores(s['iq'], s['ip'], s['is'], s['r2t'], s['score'], s['cu'], s['seq'], s['pre'],
                                   s['sid'], 128, s['scale'], 1.0, n)
        return s['score'], ops.fp4_prefill_gqa_share_sparse(s['q'], s['k'], s['v'], None, s['r2t'], s['sid'], s['idx'],
                                                            1, 128, s['cu'], s['seq'], s['pre'], n, s['scale'],
                                                            k_sc=s['ks'], v_sc=s['vs'])
    if path == 'mla':
        return ops.sparse_mla(s['q'], s['pool'], s['idx'], None, None, s['scale'])
    if path == 'mla_pages':
        return ops.sparse_mla(s['q'], s['cache'], s['idx'], s['len'], s['sink'], s['scale'], s['cache2'], s['idx2'],
                              s['len2'])
    if path == 'index_prefill':
        return ops.qsa_indexer_logits(s['q'], s['k'], s['start'], s['end'])
    if path == 'index_decode':
        return ops.dsa_paged_mqa_logits(s['q'], s['cache'], s['w'], s['lens'], s['table'], None, s['ctx'])
    return ops.topk_rows(s['x'], s['topk'])


def work(case):
    """What a pass cannot do without: each key it attends to read once per list that names it (in prefill, where lists
    share keys, each context key once), its queries, lists and outputs."""
    c = case
    rows, path = c['rows'], c['path']
    if path in ('decode', 'prefill'):
        keys = rows * min(c['topk'], c['ctx'])
        row = c['kv_heads'] * 2 * (c['dim'] // 2 + c['dim'] // 16)
        io = rows * c['q_heads'] * c['dim'] * 4 + rows * c['topk'] * 4
        if path == 'prefill':
            return {'bytes': (c['ctx'] + rows) * row + io + rows * c['kv_heads'] * 4 * c['dim'],
                    'flops': keys * c['q_heads'] * 4 * c['dim']}
        return {'bytes': keys * row + io, 'flops': keys * c['q_heads'] * 4 * c['dim']}
    if path in ('block_decode', 'block_prefill'):
        keys = rows * min(c['blocks'] * 128, c['ctx'])
        row = c['kv_heads'] * 2 * (c['dim'] // 2 + c['dim'] // 16)
        io = rows * (c['q_heads'] * 4 + 4 * 2) * c['dim'] + rows * c['kv_heads'] * c['blocks'] * 4
        mean = c['ctx'] * (0.5 if c.get('ragged') else 1) + (rows / 2 if path == 'block_prefill' else 0)
        total = c['ctx'] + rows if path == 'block_prefill' else rows * mean
        read = (total if path == 'block_prefill' else keys) * row + total * (c['dim'] // 2 + c['dim'] // 16 + 4)
        return {'bytes': read + io + rows * mean / 128 * 16,
                'flops': keys * c['q_heads'] * 4 * c['dim'] + rows * mean * 4 * 2 * c['dim']}
    if path == 'mla':
        keys = rows * min(c['topk'], c['ctx'])
        read = c['ctx'] + rows if c['causal'] else keys
        return {'bytes': read * 416 + rows * c['heads'] * (576 + 512) * 2 + keys * 4,
                'flops': keys * c['heads'] * 2 * (576 + 512)}
    if path == 'mla_pages':
        keys = rows * (c['window'] + c['extra']) * 0.75
        return {'bytes': keys * 587 + rows * c['heads'] * 2048, 'flops': keys * c['heads'] * 2048}
    if path == 'index_prefill':
        return {'bytes': (rows * c['heads'] + c['keys']) * c['dim'] * 2 + rows * c['keys'] * 4,
                'flops': rows * c['keys'] * c['heads'] * 2 * c['dim']}
    if path == 'index_decode':
        keys = rows * c['ctx'] / 2
        return {'bytes': keys * (c['dim'] + 4) + rows * c['ctx'] * 4, 'flops': keys * c['heads'] * 2 * c['dim']}
    return {'bytes': rows * c['cols'] * 4 + rows * c['topk'] * 4, 'flops': 0}


def tolerance(case):
    path = case['path']
    if path == 'select':
        return 'exact'
    if path in ('index_prefill', 'index_decode'):
        return {'rel': 1e-6}     # FP32 sums of exact products: 6e-8 from 64 bits
    # BF16 outputs (1.7e-3 from 64 bits; the pages' probabilities are BF16 too: 2.2e-3); sums and scores are far inside
    return {'rel': 9e-3 if path == 'mla_pages' else 7e-3}


# --- the same in 64 bits --------------------------------------------------------------------------------------------

def _attend(q, k, v, live, scale):
    """q [n, kv, group, d], k / v [n, kv, keys, d], live [n, kv or 1, keys] -> (out, natural-log sum)."""
    x = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    x = x.masked_fill(~live.unsqueeze(2), -math.inf)
    lse = torch.logsumexp(x, 3)
    p = torch.exp(x - lse.masked_fill(lse == -math.inf, 0.0).unsqueeze(3))
    return torch.matmul(p, v), lse


def _gqa64(q, kd, vd, slots, live, scale, step):
    """Attention of rows q [n, heads, d] over pool slots [n, kv or 1, keys]; kd / vd(slots [m, kv, keys], n0) -> FP64."""
    n, heads, d = q.shape
    out = torch.empty(n, heads, d, dtype=torch.float64, device=q.device)
    for i in range(0, n, step):
        s, ok = slots[i:i + step], live[i:i + step]
        k, v = kd(s), vd(s)
        kv = k.shape[1]
        o, _ = _attend(q[i:i + step].double().view(-1, kv, heads // kv, d), k, v, ok, scale)
        out[i:i + step] = o.reshape(-1, heads, d)
    return out


def _exact_gqa(c, s):
    pool, page, idx = s['pool'], s['page'], s['idx'].long()
    if c['path'] == 'prefill':
        for x, gs, pay, sc in ((s['k'], pool.gk, pool.k_pay, pool.k_sf), (s['v'], pool.gv, pool.v_pay, pool.v_sf)):
            p, b = _nvfp4(x, gs)
            pay[s['slots']] = p
            sc[s['slots']] = b
    live = (idx >= 0) & (idx < s['seq'].long()[:, None])
    at = idx.clamp(min=0)
    slots = s['table'].long()[s['req'][:, None], at // page] * page + at % page
    # [n, keys, kv, d] -> [n, kv, keys, d]
    kd = lambda t: (_decode64(pool.k_pay[t], pool.k_sf[t]) * pool.gk.double()).transpose(1, 2)  # noqa: E731
    vd = lambda t: (_decode64(pool.v_pay[t], pool.v_sf[t]) * pool.gv.double()).transpose(1, 2)  # noqa: E731
    out = _gqa64(s['q'], kd, vd, slots, live.unsqueeze(1), s['scale'], 64)
    return (out, None) if c['path'] == 'prefill' else out


def _exact_blocks(c, s):
    prefill = c['path'] == 'block_prefill'
    rows, kh, dim = c['rows'], c['kv_heads'], c['dim']
    idx = s['idx'].long().permute(1, 0, 2)                                     # [rows, kv, blocks]
    pos = (idx.clamp(min=0).unsqueeze(3) * 128 + torch.arange(128, device=DEV)).flatten(2)
    limit = (s['pre'].long() + torch.arange(1, rows + 1, device=DEV)) if prefill else s['seq'].long()
    live = (idx >= 0).repeat_interleave(128, 2) & (pos < limit.view(-1, 1, 1))
    req = torch.zeros(rows, dtype=torch.int64, device=DEV) if prefill else torch.arange(rows, device=DEV)
    r2t = s['r2t'].long()
    slots = r2t[req.view(-1, 1, 1), pos.clamp(max=r2t.shape[1] - 1)]
    head = torch.arange(kh, device=DEV).view(1, kh, 1)
    kd = lambda t: _decode64(s['k'][t // 128, head, t % 128], s['ks'][t // 128, head, t % 128])  # noqa: E731
    vd = lambda t: _decode64(s['v'][t // 128, head, t % 128], s['vs'][t // 128, head, t % 128])  # noqa: E731
    out = _gqa64(s['q'], kd, vd, slots, live, s['scale'], 64)
    score = torch.full(s['score'].shape, -math.inf, dtype=torch.float64, device=DEV)
    width = r2t.shape[1]
    step = 1 if not prefill else 64
    for i in range(0, rows, step):
        if not prefill or i == 0:
            t = r2t[req[i]]
            keys = _decode64(s['ip'][t // 128, t % 128], s['is'][t // 128, t % 128])   # [width, dim]
        x = torch.matmul(s['iq'][i:i + step].double(), keys.t()) * (s['scale'] * math.log2(math.e))
        ok = torch.arange(width, device=DEV).view(1, -1) < limit[i:i + step].view(-1, 1)
        x = x.masked_fill(~ok.unsqueeze(1), -math.inf)
        score[:, i:i + step] = x.unflatten(2, (-1, 128)).amax(3).permute(1, 0, 2)
    return score, out


def _mla64(q, keys, value, live, sink, scale):
    x = torch.matmul(q, keys.transpose(1, 2).contiguous()) * scale
    x = x.masked_fill(~live.unsqueeze(1), -math.inf)
    lse = torch.logsumexp(x, 2)
    total = lse if sink is None else torch.logaddexp(lse, sink.double().view(1, -1))
    return torch.matmul(torch.exp(x - total.unsqueeze(2)), value), lse


def _exact_mla(c, s):
    pool, n = s['pool'], c['rows']
    out = torch.empty(n, 1, c['heads'], 512, dtype=torch.float64, device=DEV)
    lse = torch.empty(n, c['heads'], 1, dtype=torch.float64, device=DEV)
    for i in range(0, n, 64):
        idx = s['idx'][i:i + 64, 0].long()
        at = idx.clamp(min=0)
        lat = _decode64(pool.pay[at], pool.scales[at]) * pool.g.double()
        keys = torch.cat([lat, pool.rope[at].double()], 2)
        o, e = _mla64(s['q'][i:i + 64, 0].double(), keys, lat, idx >= 0, None, s['scale'])
        out[i:i + 64, 0], lse[i:i + 64, :, 0] = o, e
    return out, lse


def _pages64(cache, idx):
    """FP64 rows [n, keys, 512] of FP8 latent pages at token slots idx."""
    n, page = cache.shape[:2]
    flat = torch.as_strided(cache, (n, page * 584), (cache.stride(0), 1))
    data = flat[:, :page * 576].view(n, page, 576)[idx // page, idx % page]
    ex = flat[:, page * 576:].view(n, page, 8)[idx // page, idx % page][..., :7].double()
    nope = data[..., :448].contiguous().view(torch.float8_e4m3fn).double().unflatten(-1, (7, 64))
    rope = data[..., 448:].contiguous().view(torch.bfloat16).double()
    return torch.cat([(nope * torch.exp2(ex - 127).unsqueeze(-1)).flatten(-2), rope], -1)


def _exact_mla_pages(c, s):
    n = c['rows']
    out = torch.empty(n, 1, c['heads'], 512, dtype=torch.float64, device=DEV)
    lse = torch.empty(n, c['heads'], 1, dtype=torch.float64, device=DEV)
    for i in range(0, n, 64):
        keys, live = [], []
        for cache, idx, ln in ((s['cache'], s['idx'], s['len']), (s['cache2'], s['idx2'], s['len2'])):
            if cache is not None:
                keys.append(_pages64(cache, idx[i:i + 64, 0].long()))
                live.append(torch.arange(idx.shape[2], device=DEV).view(1, -1) < ln[i:i + 64].view(-1, 1))
        k = torch.cat(keys, 1)
        o, e = _mla64(s['q'][i:i + 64, 0].double(), k, k, torch.cat(live, 1), s['sink'], s['scale'])
        out[i:i + 64, 0], lse[i:i + 64, :, 0] = o, e
    return out, lse


def _exact_index_prefill(c, s):
    k = s['k'][:, 0].double().t().contiguous()
    out = torch.empty(c['rows'], c['keys'], dtype=torch.float64, device=DEV)
    at = torch.arange(c['keys'], device=DEV).view(1, -1)
    for i in range(0, c['rows'], 64):
        x = torch.matmul(s['q'][i:i + 64].double(), k).clamp(min=0).sum(1) / math.sqrt(c['dim'])
        out[i:i + 64] = x.masked_fill(at >= s['end'][i:i + 64].long().view(-1, 1), -math.inf)
    return out


def _exact_index_decode(c, s):
    rows, dim, ctx = c['rows'], c['dim'], c['ctx']
    out = torch.zeros(rows, ctx, dtype=torch.float64, device=DEV)
    n = s['cache'].shape[0]
    flat = s['cache'].view(n, -1)
    for r in range(rows):
        p = flat[s['table'][r].long()]
        k = p[:, :64 * dim].contiguous().view(torch.float8_e4m3fn).double().view(-1, dim)[:ctx]
        ks = p[:, 64 * dim:].contiguous().view(torch.float32).double().reshape(-1)[:ctx]
        x = torch.matmul(s['q'][r, 0].double(), k.t().contiguous()).clamp(min=0)
        x = (x * s['w'][r].double().view(-1, 1)).sum(0) * ks
        out[r] = torch.where(torch.arange(ctx, device=DEV) < s['lens'][r], x, 0.0)
    return out


_EXACT = {'decode': _exact_gqa, 'prefill': _exact_gqa, 'block_decode': _exact_blocks, 'block_prefill': _exact_blocks,
          'mla': _exact_mla, 'mla_pages': _exact_mla_pages, 'index_prefill': _exact_index_prefill,
          'index_decode': _exact_index_decode}


def exact(case, seed):
    if case['path'] not in _EXACT:
        return None
    return _EXACT[case['path']](case, prepare(case, seed))
