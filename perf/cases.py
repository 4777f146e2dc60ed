"""The work a program has this framework do, as timed cases.

Six kinds of call, each through a public entry point, over the sizes that the
framework's configurations, tests and benchmark use:

* ``decode``: one decode step of one layer over a paged KV pool, every request
  at its own context length (``paged_ops.paged_decode_batch``: append + attention).
* ``attend``: append and causal attention of n tokens per request on split
  heads, what ``PagedKVCache.attention`` runs per layer for a prefill and for a
  ``decode_step`` (``paged_ops.paged_append`` + ``paged_ops.paged_attention``).
* ``prefill``: append and causal attention of n tokens per request from one
  fused QKV projection (``paged_ops.paged_prefill``).
* ``ragged``: the same for prompts of different lengths in one call
  (``paged_ops.paged_prefill_ragged``).
* ``mlp``: the MLP of a decode step (``mt_decode_projection``: fc with tanh
  GELU, then the down projection as split sums).
* ``generate``: a whole model call: prompts prefilled into paged caches, then
  decode steps, logits of every step (``DecoderLM.prefill_batch`` and
  ``decode_batch``).

Context and prompt lengths are the quantiles of the stated distribution, dealt
to the requests in an order drawn from the seed, so that every seed asks for
the same amount of work.
"""
import functools
import math

import numpy as np
import torch

from minitorch_amd import paged_ops
from minitorch_amd.amp import autocast
from minitorch_amd.dtypes import dtype_code
from minitorch_amd.model import DecoderLM, fragment_tiled, model_library
from minitorch_amd.paged_kv_cache import KVPagePool
from minitorch_amd.runtime import DeviceTensor, F, I, P, call

TORCH_DTYPE = {'float32': torch.float32, 'float16': torch.float16, 'bfloat16': torch.bfloat16}
SIZE = {'float32': 4, 'float16': 2, 'bfloat16': 2}
PAGES_PER_SLAB = 64


# ------------------------------------------------------------------ cases ---
def listed():
    return [
        # the smallest call: four short requests in the default precision
        dict(name='decode 4 fp32', op='decode', batch=4, heads=12, dim=64, page=16, dtype='float32',
             lengths='uniform', low=7, high=120),
        # the benchmark's headline: GPT-2-small heads, 64 requests
        dict(name='decode 64 fp16', op='decode', batch=64, heads=12, dim=64, page=16, dtype='float16',
             lengths='uniform', low=128, high=1024),
        # one layer of GPT-2-medium serving 128 requests at steady state
        dict(name='decode 128 bf16', op='decode', batch=128, heads=16, dim=64, page=16, dtype='bfloat16',
             lengths='lognormal', low=16, high=1024),
        # the ragged tail: GPT-2-XL heads, 512 requests, the longest at 8192 tokens
        dict(name='decode 512 bf16 ragged', op='decode', batch=512, heads=25, dim=64, page=32, dtype='bfloat16',
             lengths='lognormal', low=1, high=8192),
        # a few users with long conversations: latency, not throughput
        dict(name='decode 3 fp16 long', op='decode', batch=3, heads=12, dim=64, page=16, dtype='float16',
             lengths='uniform', low=3000, high=8000),
        # PagedKVCache: one more token for each row of a cache (decode_step), default precision
        dict(name='attend 1 token fp32', op='attend', batch=2, heads=12, dim=64, page=16, dtype='float32',
             tokens=1, offset=700),
        # PagedKVCache: a prefill of four prompts of odd length, default precision
        dict(name='attend 333 tokens fp32', op='attend', batch=4, heads=12, dim=64, page=16, dtype='float32',
             tokens=333, offset=0),
        # one long prompt, GPT-2-medium heads
        dict(name='prefill 1000 bf16', op='prefill', batch=1, heads=16, dim=64, page=16, dtype='bfloat16',
             tokens=1000, offset=0),
        # a chunk of a long document behind the part that is already cached
        dict(name='prefill 2048 bf16 chunk', op='prefill', batch=1, heads=16, dim=64, page=16, dtype='bfloat16',
             tokens=2048, offset=2048),
        # sixteen prompts admitted together, DistilGPT-2 heads
        dict(name='ragged 16 fp16', op='ragged', prompts=16, heads=12, dim=64, page=16, dtype='float16',
             low=32, high=512, offset=0),
        # the MLP of a GPT-2-medium decode step
        dict(name='mlp 40 bf16', op='mlp', rows=40, width=1024, dtype='bfloat16'),
        # DistilGPT-2: eight prompts, then six decode steps
        dict(name='generate 8 fp16', op='generate', requests=8, low=32, high=160, steps=6, page=16, dtype='float16'),
    ]


def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    op = rng.choices(['decode', 'attend', 'prefill', 'ragged', 'mlp', 'generate'], [9, 4, 3, 3, 2, 1])[0]
    heads, page = rng.choice([12, 16, 25]), rng.choice([8, 16, 16, 32])
    dtype = rng.choice(['float32', 'float16', 'bfloat16'])
    if op == 'decode':
        high = _log(rng, 40, 8192)
        case = dict(op=op, batch=_log(rng, 1, 512), heads=heads, dim=rng.choice([64, 64, 64, 64, 128, 80, 32]),
                    page=page, dtype=dtype, lengths=rng.choice(['uniform', 'lognormal']),
                    low=max(1, high // rng.choice([2, 8, 32])), high=high)
        while case['batch'] > 1 and work(case)['bytes'] > 1.5e9:
            case['batch'] = case['batch'] * 2 // 3
        return case
    if op == 'attend':
        case = dict(op=op, batch=_log(rng, 1, 8), heads=heads, dim=rng.choice([64, 64, 64, 128, 80, 32]), page=page,
                    dtype=dtype, tokens=_log(rng, 1, 1024), offset=rng.choice([0, _log(rng, 1, 4000)]))
        if case['tokens'] == 1 and case['offset'] == 0:
            case['offset'] = _log(rng, 16, 4000)
        return _fewer(case, 8e6)
    if op == 'prefill':
        case = dict(op=op, batch=_log(rng, 1, 8), heads=heads, dim=rng.choice([64, 64, 128]), page=page,
                    dtype=dtype, tokens=_log(rng, 16, 2048), offset=rng.choice([0, 0, _log(rng, 16, 4000)]))
        return _fewer(case, 8e6 if dtype == 'float32' else 60e6)
    if op == 'ragged':
        high = _log(rng, 32, 1024)
        case = dict(op=op, prompts=_log(rng, 2, 32), heads=heads, dim=rng.choice([64, 64, 128]), page=page,
                    dtype=rng.choice(['float16', 'bfloat16']), low=max(1, high // rng.choice([2, 16])), high=high,
                    offset=rng.choice([0, 0, _log(rng, 16, 1000)]))
        return _fewer(case, 60e6)
    if op == 'mlp':
        return dict(op=op, rows=_log(rng, 1, 128), width=rng.choice([768, 1024]),
                    dtype=rng.choice(['float16', 'bfloat16']))
    high = _log(rng, 16, 160)
    return dict(op=op, requests=_log(rng, 1, 8), low=max(1, high // 4), high=high, steps=rng.randint(1, 6),
                page=page, dtype=dtype)


def _fewer(case, most):
    """The case with as many fewer requests, then tokens, as keep its
    (head, query, key) triples within ``most``."""
    count = 'prompts' if case['op'] == 'ragged' else 'batch'
    while case[count] > 1 and _pairs(case) * case['heads'] > most:
        case[count] = case[count] * 2 // 3
    while case['op'] != 'ragged' and case['tokens'] > 1 and _pairs(case) * case['heads'] > most:
        case['tokens'] = case['tokens'] * 2 // 3
    return case


# ------------------------------------------------------------------- work ---
def _quantiles(n, low, high, kind='uniform'):
    """n lengths in [low, high]: evenly spread, or lognormal about a quarter
    of ``high`` (sigma 1.2 from 4096 tokens on, else 0.8), clipped."""
    u = (np.arange(n) + 0.5) / n
    if kind == 'uniform':
        x = low + u * (high - low)
    else:
        sigma = 1.2 if high >= 4096 else 0.8
        median = 256 if high >= 1024 else max(low, high / 4)
        # the normal quantile function by bisection on erf
        z = np.zeros(n)
        a, b = np.full(n, -6.0), np.full(n, 6.0)
        for _ in range(50):
            z = (a + b) / 2
            below = np.array([0.5 * (1 + math.erf(t / math.sqrt(2))) for t in z]) < u
            a, b = np.where(below, z, a), np.where(below, b, z)
        x = np.exp(math.log(median) + sigma * z)
        x[-1] = high
    return np.clip(np.round(x), low, high).astype(np.int64)


def _lengths(case):
    if case['op'] == 'decode':
        return _quantiles(case['batch'], case['low'], case['high'], case['lengths'])
    return _quantiles(case['prompts'] if case['op'] == 'ragged' else case['requests'], case['low'], case['high'])


def _pairs(case):
    """(query, key) pairs of one head, over every request of the call."""
    tokens = _lengths(case) if case['op'] == 'ragged' else np.full(case['batch'], case['tokens'])
    return int(np.sum(tokens * case['offset'] + tokens * (tokens + 1) // 2))


def work(case):
    s = SIZE[case['dtype']]
    if case['op'] == 'decode':
        L, hd = _lengths(case), case['heads'] * case['dim']
        b = case['batch']
        # cached K and V, q/k/v in, out and the new rows written, table entries and offsets
        return dict(bytes=int(2 * (L.sum() - b) * hd * s + 6 * b * hd * s + 4 * np.sum(-(-L // case['page'])) + 4 * b),
                    flops=int(4 * L.sum() * hd))
    if case['op'] in ('attend', 'prefill', 'ragged'):
        hd = case['heads'] * case['dim']
        tokens = _lengths(case) if case['op'] == 'ragged' else np.full(case['batch'], case['tokens'])
        new, old = int(tokens.sum()), len(tokens) * case['offset']
        return dict(bytes=(6 * new + 2 * old) * hd * s + 4 * int(np.sum(-(-(tokens + case['offset']) // case['page']))),
                    flops=4 * _pairs(case) * hd)
    if case['op'] == 'mlp':
        m, d = case['rows'], case['width']
        return dict(bytes=8 * d * d * s + 4 * d * s + m * d * s + m * 4 * d * s + MLP_SPLITS * m * d * 4,
                    flops=2 * 8 * d * d * m)
    L, d, layers, vocab = _lengths(case), 768, 6, 50257
    rows = int(L.sum())
    weights = (12 * d * d * layers + vocab * d) * s
    r, steps = case['requests'], case['steps']
    logits = r * vocab * s
    kv = 2 * layers * d * s * (rows + sum(rows + r * t for t in range(1, steps + 1)))
    per_row = 2 * 12 * d * d * layers
    return dict(bytes=(steps + 1) * (weights + logits) + kv,
                flops=per_row * (rows + r * steps) + 2 * (steps + 1) * r * vocab * d
                + 4 * d * layers * int(np.sum(L * (L + 1) // 2)))


# Four times the largest difference seen between a path and its 64-bit result
# or another order of its sums (relative 2-norm), per type of the result.
def tolerance(case):
    if case['op'] == 'generate':
        return dict(rel={'float32': 1e-5, 'float16': 3e-3, 'bfloat16': 3e-2}[case['dtype']])
    return dict(rel={'float32': 2e-6, 'float16': 1e-3, 'bfloat16': 8e-3}[case['dtype']])


# ------------------------------------------------------------------ paged ---
def _deal(lengths, seed):
    return lengths[np.random.default_rng([seed, 1]).permutation(len(lengths))]


class _Pool:
    """A page pool [slabs, 1 layer, K and V, pages, heads, page, dim] whose
    requests' pages lie at random places, with its device tables; cached
    values are N(0, 1)."""

    def __init__(self, case, totals, seed):
        h, d, page, t = case['heads'], case['dim'], case['page'], TORCH_DTYPE[case['dtype']]
        gen = torch.Generator('cuda').manual_seed(seed)
        need = -(-totals // page)
        self.slabs = -(-(int(need.sum()) + 8) // PAGES_PER_SLAB)
        self.columns = int(need.max())
        self.pages = torch.randn((self.slabs, 1, 2, PAGES_PER_SLAB, h, page, d), device='cuda', dtype=t, generator=gen)
        order = torch.randperm(self.slabs * PAGES_PER_SLAB, device='cuda', generator=gen).to(torch.int32)
        table = torch.full((len(totals), self.columns), -1, device='cuda', dtype=torch.int32)
        owned = torch.arange(self.columns, device='cuda')[None, :] < torch.from_numpy(need).cuda()[:, None]
        table[owned] = order[:int(need.sum())]
        self.table, self.totals, self.need = table, totals, need
        slab_bytes = self.pages[0].numel() * self.pages.element_size()
        self.slab_table = (self.pages.data_ptr() + slab_bytes * torch.arange(self.slabs, dtype=torch.int64)).cuda()
        self.gen, self.t = gen, t

    def randn(self, *shape):
        return torch.randn(shape, device='cuda', dtype=self.t, generator=self.gen)

    def common(self, case):
        return dict(h=case['heads'], d=case['dim'], page_size=case['page'], pages_per_slab=PAGES_PER_SLAB,
                    num_slabs=self.slabs, columns=self.columns, layer=0, layers=1, dtype=case['dtype'])

    def places(self, r, first, count):
        """Slab, slot and row in the page of tokens [first, first + count) of request r."""
        pos = torch.arange(first, first + count, device='cuda')
        page = self.table[r, pos // self.pages.shape[5]].long()
        return page // PAGES_PER_SLAB, page % PAGES_PER_SLAB, pos % self.pages.shape[5]

    def written(self, writes):
        """The pages with K/V rows [count, heads, dim] written at (request, first token)."""
        out = self.pages.clone()
        for r, first, k, v in writes:
            slab, slot, row = self.places(r, first, k.shape[0])
            out[slab, 0, 0, slot, :, row] = k
            out[slab, 0, 1, slot, :, row] = v
        return out

    def cached(self, pages, r, count):
        """K and V [heads, count, dim] of request r's first tokens, in 64 bits."""
        slab, slot, row = self.places(r, 0, count)
        return tuple(pages[slab, 0, kv, slot, :, row].double().permute(1, 0, 2).contiguous() for kv in (0, 1))


def _causal(q, k, v, offset):
    """softmax(q k^T / sqrt(d)) v for q [heads, n, dim] at ``offset``, in 64 bits."""
    n, keys = q.shape[1], k.shape[1]
    hidden = torch.arange(keys, device='cuda')[None, :] > offset + torch.arange(n, device='cuda')[:, None]
    out = torch.empty_like(q)
    for head in range(q.shape[0]):
        scores = (q[head] @ k[head].t().contiguous()) / math.sqrt(q.shape[2])
        out[head] = torch.softmax(scores.masked_fill_(hidden, -math.inf), 1) @ v[head]
    return out


def _prepare_decode(case, seed):
    lengths = _deal(_lengths(case), seed)
    pool = _Pool(case, lengths, seed)
    shape = (case['batch'], case['heads'], 1, case['dim'])
    q, k, v = (pool.randn(*shape) for _ in range(3))
    offsets = torch.from_numpy((lengths - 1).astype(np.int32)).cuda()
    return dict(op='decode', pool=pool, q=q, k=k, v=v, offsets=offsets, out=torch.empty_like(q),
                args=dict(b=case['batch'], **pool.common(case)))


def _run_decode(s):
    pool = s['pool']
    paged_ops.paged_decode_batch(s['out'].data_ptr(), s['q'].data_ptr(), s['k'].data_ptr(), s['v'].data_ptr(),
                                 pool.slab_table.data_ptr(), pool.table.data_ptr(), s['offsets'].data_ptr(),
                                 **s['args'])
    return dict(out=s['out'], pages=pool.pages)


def _exact_decode(case, s):
    pool = s['pool']
    pages = pool.written([(r, int(n) - 1, s['k'][r].transpose(0, 1), s['v'][r].transpose(0, 1))
                          for r, n in enumerate(pool.totals)])
    out = torch.empty(s['q'].shape, device='cuda', dtype=torch.float64)
    for r, n in enumerate(pool.totals):
        k, v = pool.cached(pages, r, int(n))
        w = torch.softmax((k * s['q'][r].double()).sum(2) / math.sqrt(case['dim']), 1)
        out[r, :, 0] = (w[:, :, None] * v).sum(1)
    return dict(out=out, pages=pages)


def _prepare_attend(case, seed):
    n, offset, b = case['tokens'], case['offset'], case['batch']
    pool = _Pool(case, np.full(b, offset + n), seed)
    q, k, v = (pool.randn(b, case['heads'], n, case['dim']) for _ in range(3))
    return dict(op='attend', pool=pool, q=q, k=k, v=v, out=torch.empty_like(q), n=n, offset=offset,
                args=dict(b=b, offset=offset, **pool.common(case)))


def _run_attend(s):
    pool = s['pool']
    paged_ops.paged_append(s['k'].data_ptr(), s['v'].data_ptr(), pool.slab_table.data_ptr(), pool.table.data_ptr(),
                           n=s['n'], **s['args'])
    paged_ops.paged_attention(s['out'].data_ptr(), s['q'].data_ptr(), pool.slab_table.data_ptr(),
                              pool.table.data_ptr(), nq=s['n'], nk=s['offset'] + s['n'], **s['args'])
    return dict(out=s['out'], pages=pool.pages)


def _exact_attend(case, s):
    pool, n, offset = s['pool'], s['n'], s['offset']
    pages = pool.written([(r, offset, s['k'][r].transpose(0, 1), s['v'][r].transpose(0, 1))
                          for r in range(case['batch'])])
    out = torch.empty(s['q'].shape, device='cuda', dtype=torch.float64)
    for r in range(case['batch']):
        out[r] = _causal(s['q'][r].double(), *pool.cached(pages, r, offset + n), offset)
    return dict(out=out, pages=pages)


def _prepare_prefill(case, seed):
    n, b, hd = case['tokens'], case['batch'], case['heads'] * case['dim']
    pool = _Pool(case, np.full(b, case['offset'] + n), seed)
    qkv = pool.randn(b * n, 3 * hd)
    return dict(op='prefill', pool=pool, qkv=qkv, hd=hd, tokens=[n] * b,
                out=torch.empty((b * n, hd), device='cuda', dtype=pool.t),
                args=dict(b=b, n=n, offset=case['offset'], qkv_stride=3 * hd, **pool.common(case)))


def _run_prefill(s):
    pool, q, step = s['pool'], s['qkv'].data_ptr(), s['hd'] * s['qkv'].element_size()
    paged_ops.paged_prefill(s['out'].data_ptr(), q, q + step, q + 2 * step, pool.slab_table.data_ptr(),
                            pool.table.data_ptr(), **s['args'])
    return dict(out=s['out'], pages=pool.pages)


def _prepare_ragged(case, seed):
    tokens, hd = _deal(_lengths(case), seed), case['heads'] * case['dim']
    pool = _Pool(case, tokens + case['offset'], seed)
    rows = int(tokens.sum())
    row_bytes = 4 * pool.columns
    return dict(op='ragged', pool=pool, qkv=pool.randn(rows, 3 * hd), hd=hd, tokens=[int(n) for n in tokens],
                out=torch.empty((rows, hd), device='cuda', dtype=pool.t),
                tables=[pool.table.data_ptr() + row_bytes * r for r in range(len(tokens))],
                offsets=[case['offset']] * len(tokens), args=dict(qkv_stride=3 * hd, **pool.common(case)))


def _run_ragged(s):
    pool, q, step = s['pool'], s['qkv'].data_ptr(), s['hd'] * s['qkv'].element_size()
    paged_ops.paged_prefill_ragged(s['out'].data_ptr(), q, q + step, q + 2 * step, pool.slab_table.data_ptr(),
                                   s['tables'], s['tokens'], s['offsets'], **s['args'])
    return dict(out=s['out'], pages=pool.pages)


def _exact_rows(case, s):
    """``prefill`` and ``ragged``: token-major rows, prompt after prompt."""
    pool, h, d, offset = s['pool'], case['heads'], case['dim'], case['offset']
    q, k, v = (t.reshape(-1, h, d) for t in s['qkv'].split(s['hd'], 1))
    first = np.concatenate([[0], np.cumsum(s['tokens'])])
    part = [slice(int(a), int(b)) for a, b in zip(first[:-1], first[1:])]
    pages = pool.written([(r, offset, k[p], v[p]) for r, p in enumerate(part)])
    out = torch.empty((q.shape[0], h, d), device='cuda', dtype=torch.float64)
    for r, p in enumerate(part):
        out[p] = _causal(q[p].double().transpose(0, 1).contiguous(),
                         *pool.cached(pages, r, offset + s['tokens'][r]), offset).transpose(0, 1)
    return dict(out=out.reshape(-1, s['hd']), pages=pages)


# -------------------------------------------------------------------- MLP ---
MLP_SPLITS = 4  # ranges of the down projection's k, as a decode step of these widths takes
TILED_WEIGHTS = 4  # mt_decode_projection's layout bit for fragment-tiled weights
GELU, PARTIALS = 1, 2


def _tiled(w):
    """``fragment_tiled`` of a device matrix (made once per model by a program)."""
    n, k = w.shape
    return w.reshape(n // 16, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous().reshape(-1)


def _prepare_mlp(case, seed):
    m, d, t = case['rows'], case['width'], TORCH_DTYPE[case['dtype']]
    gen = torch.Generator('cuda').manual_seed(seed)

    def randn(*shape, std=1.0):
        return (std * torch.randn(shape, device='cuda', generator=gen)).to(t)

    w_fc, w_proj = randn(4 * d, d, std=0.02), randn(d, 4 * d, std=0.02)
    return dict(op='mlp', m=m, d=d, code=dtype_code(case['dtype']), x=randn(m, d), w_fc=w_fc, b_fc=randn(4 * d, std=0.1),
                w_proj=w_proj, fc_tiled=_tiled(w_fc), proj_tiled=_tiled(w_proj),
                hidden=torch.empty((m, 4 * d), device='cuda', dtype=t),
                sums=torch.empty((MLP_SPLITS, m, d), device='cuda', dtype=torch.float32))


def _run_mlp(s):
    m, d, lib, types = s['m'], s['d'], model_library(), [P, P, P, P, I, I, I, I, I, I, I]
    call(lib, 'mt_decode_projection', types, s['hidden'].data_ptr(), s['x'].data_ptr(), s['fc_tiled'].data_ptr(),
         s['b_fc'].data_ptr(), m, 4 * d, d, 1, GELU, s['code'], TILED_WEIGHTS)
    call(lib, 'mt_decode_projection', types, s['sums'].data_ptr(), s['hidden'].data_ptr(), s['proj_tiled'].data_ptr(),
         None, m, d, 4 * d, MLP_SPLITS, PARTIALS, s['code'], TILED_WEIGHTS)
    return dict(hidden=s['hidden'], sums=s['sums'])


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_mlp(case, s):
    hidden = _gelu(s['x'].double() @ s['w_fc'].double().t() + s['b_fc'].double())
    step = 4 * s['d'] // MLP_SPLITS
    w = s['w_proj'].double()
    sums = [hidden[:, i * step:(i + 1) * step] @ w[:, i * step:(i + 1) * step].t() for i in range(MLP_SPLITS)]
    return dict(hidden=hidden, sums=torch.stack(sums))


# ------------------------------------------------------------------ model ---
@functools.lru_cache(maxsize=1)
def _model():
    """DistilGPT-2's architecture with seeded weights, loaded once by a program
    (its prompts come from each case's seed)."""
    return DecoderLM(n_vocab=50257, n_embd=768, n_head=12, n_layer=6, n_positions=1024, seed=0).eval()


class _Precision:
    """The autocast scope of a compute type; float32 runs outside any."""

    def __init__(self, dtype):
        self.scope = None if dtype == 'float32' else autocast(dtype)

    def __enter__(self):
        return self.scope and self.scope.__enter__()

    def __exit__(self, *exc):
        return self.scope and self.scope.__exit__(*exc)


class _Shared:
    """A framework tensor's memory as torch sees it; keeps the tensor alive."""

    def __init__(self, tensor):
        self.tensor = tensor
        kind = '<f4' if tensor.dtype == 'float32' else '<f2' if tensor.dtype == 'float16' else '<i2'
        self.__cuda_array_interface__ = dict(shape=tensor.shape, typestr=kind, data=(tensor.ptr, False), version=2)


def _as_torch(tensor):
    shared = torch.as_tensor(_Shared(tensor), device='cuda')
    return shared.view(torch.bfloat16) if tensor.dtype == 'bfloat16' else shared


def _prepare_generate(case, seed):
    model, lengths = _model(), _deal(_lengths(case), seed)
    rng = np.random.default_rng([seed, 2])
    prompts = [rng.integers(0, model.n_vocab, size=int(n)) for n in lengths]
    later = rng.integers(0, model.n_vocab, size=(case['steps'], len(prompts), 1))
    with _Precision(case['dtype']):
        pool = KVPagePool(model, page_size=case['page'], max_bytes=64 << 20, pages_per_slab=4)
        model._weights(case['dtype'])
    return dict(op='generate', model=model, pool=pool, prompts=prompts, later=later, dtype=case['dtype'],
                page=case['page'], steps=[DeviceTensor.from_numpy(ids.astype(np.float32)) for ids in later],
                capacity=[int(n) + case['steps'] for n in lengths])


def _run_generate(s):
    model = s['model']
    with _Precision(s['dtype']):
        caches = [model.create_kv_cache(1, c, page_size=s['page'], page_pool=s['pool']) for c in s['capacity']]
        logits = [model.prefill_batch(s['prompts'], caches)]
        for ids in s['steps']:
            logits.append(model.decode_batch(ids, caches))
        for cache in caches:
            cache.close()
    return [_as_torch(t) for t in logits]


def _exact_generate(case, s):
    model, t = s['model'], TORCH_DTYPE[case['dtype']]
    weights = {}

    def get(name, rounded=True):
        if name not in weights:
            w = torch.from_numpy(model.state[name]).cuda()
            weights[name] = (w.to(t) if rounded else w).double()
        return weights[name]

    def norm(x, name):
        y = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + model.ln_eps)
        return y * get(name + '.weight', False) + get(name + '.bias', False)

    def linear(x, name):
        return x @ get(name + '.weight') + get(name + '.bias')

    steps, h = case['steps'], model.n_head
    out = [torch.empty((len(s['prompts']), 1, model.n_vocab), device='cuda', dtype=torch.float64)
           for _ in range(steps + 1)]
    for r, prompt in enumerate(s['prompts']):
        ids = torch.from_numpy(np.concatenate([prompt, s['later'][:, r, 0]])).cuda()
        n = len(ids)
        x = get('transformer.wte.weight', False)[ids] + get('transformer.wpe.weight', False)[:n]
        for i in range(model.n_layer):
            p = f'transformer.h.{i}.'
            q, k, v = (y.reshape(n, h, -1).transpose(0, 1).contiguous()
                       for y in linear(norm(x, p + 'ln_1'), p + 'attn.c_attn').split(model.n_embd, 1))
            y = _causal(q, k, v, 0).transpose(0, 1).reshape(n, -1)
            x = x + linear(y, p + 'attn.c_proj')
            x = x + linear(_gelu(linear(norm(x, p + 'ln_2'), p + 'mlp.c_fc')), p + 'mlp.c_proj')
        head = torch.from_numpy(model.state['transformer.wte.weight']).cuda().to(t).double()
        logits = norm(x, 'transformer.ln_f')[len(prompt) - 1:] @ head.t()
        for step in range(steps + 1):
            out[step][r, 0] = logits[step]
    return out


# -------------------------------------------------------------- interface ---
_PREPARE = dict(decode=_prepare_decode, attend=_prepare_attend, prefill=_prepare_prefill, ragged=_prepare_ragged,
                mlp=_prepare_mlp, generate=_prepare_generate)
_RUN = dict(decode=_run_decode, attend=_run_attend, prefill=_run_prefill, ragged=_run_ragged, mlp=_run_mlp,
            generate=_run_generate)
_EXACT = dict(decode=_exact_decode, attend=_exact_attend, prefill=_exact_rows, ragged=_exact_rows, mlp=_exact_mlp,
              generate=_exact_generate)


def prepare(case, seed):
    state = _PREPARE[case['op']](case, seed)
    # the framework launches on the calling thread's own stream, torch on its
    # default one: the inputs are there before the first call
    torch.cuda.synchronize()
    return state


def run(state):
    return _RUN[state['op']](state)


def exact(case, seed):
    return _EXACT[case['op']](case, prepare(case, seed))
