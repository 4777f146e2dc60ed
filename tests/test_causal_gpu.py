"""GPU parity of the matrix-core causal attention at the edges of its tiles and
of its dispatch, against the float64 oracle: head dims that do not fill the
kernel's 64 or 128 columns, fp32, query counts around the 32-, 64- and
128-query tiles, every workgroup shape and keys split over workgroups; fp32's
precision, small weights, and both sides of the lines to the per-query kernel
(which the small fp32 grids of the tile edges run on at head dims 64 and 128;
test_few_queries has the large ones).
Tolerances are in tests/tolerances.py."""
import numpy as np
import pytest

from oracle import paged_oracle as po
from test_prefill_gpu import (CODES, key_split_launches, prefill_case, run_prefill, run_fused_single,
                              run_ragged)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,dim', [('float32', 64), ('float32', 128), ('float32', 20), ('float16', 32),
                                       ('bfloat16', 80), ('float16', 128), ('bfloat16', 8)])
@pytest.mark.parametrize('nq,offset', [(2, 0), (31, 33), (33, 0), (65, 31), (129, 250)])
def test_causal_tile_edges(dtype, dim, nq, offset):
    case = prefill_case(200 + dim + nq, batch=2, heads=2, dim=dim, page_size=16, nk=offset + nq, dtype=dtype,
                        layers=2, layer=1)
    run_prefill(case, nq, offset + nq, offset, seed=nq)
    one = prefill_case(300 + dim + nq, batch=1, heads=2, dim=dim, page_size=8, nk=offset + nq, dtype=dtype)
    run_fused_single(one, nq, offset, seed=nq)


# (batch, heads, queries): 64-query tiles in one round of the compute units,
# two 64-query workgroups per compute unit, 128-query tiles
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('batch,heads,nq,offset', [(3, 20, 200, 5), (3, 40, 200, 5), (5, 60, 140, 5)])
def test_causal_workgroup_shapes(dtype, batch, heads, nq, offset):
    case = prefill_case(400 + nq, batch=batch, heads=heads, dim=64, page_size=16, nk=offset + nq, dtype=dtype)
    run_prefill(case, nq, offset + nq, offset, seed=heads)


# (batch, heads, queries, offset, head dim) about the lines between the causal
# and the per-query kernel, and of prompts of at most 32 queries over one round
# of the compute units, whose tiles are narrow: fp32 in grids that the causal
# kernel takes at few queries or keys, then few queries on the per-query kernel
@pytest.mark.parametrize('dtype,shape', [
    ('float32', (8, 70, 2, 10, 64)), ('float32', (4, 20, 31, 33, 64)), ('float32', (4, 20, 33, 0, 64)),
    ('float32', (3, 30, 65, 31, 64)), ('float32', (5, 52, 20, 300, 64)), ('float32', (6, 50, 20, 300, 64)),
    ('float32', (6, 50, 20, 300, 128)), ('float32', (4, 140, 7, 150, 128)), ('bfloat16', (6, 50, 20, 300, 80)),
    ('float32', (30, 10, 4, 508, 64)), ('float32', (30, 10, 4, 1021, 64)), ('float32', (30, 10, 3, 1022, 128)),
    ('float32', (4, 80, 7, 150, 128)), ('float32', (1, 12, 20, 380, 128)), ('float16', (30, 20, 3, 200, 64)),
    ('bfloat16', (30, 20, 4, 508, 64)), ('float16', (30, 10, 3, 317, 128)), ('float16', (30, 10, 3, 318, 128))])
def test_few_queries(dtype, shape):
    batch, heads, nq, offset, dim = shape
    case = prefill_case(450 + nq + heads, batch=batch, heads=heads, dim=dim, page_size=16, nk=offset + nq, dtype=dtype)
    run_prefill(case, nq, offset + nq, offset, seed=heads)


@pytest.mark.parametrize('dtype,dim', [('float32', 64), ('bfloat16', 64), ('float16', 80)])
@pytest.mark.parametrize('nq,offset', [(3, 4090), (40, 2500)])
def test_causal_keys_split_over_workgroups(dtype, dim, nq, offset):
    # few tiles, many rounds of keys; a hole is NaN for every query through the merge
    case = prefill_case(500 + nq, batch=1, heads=2, dim=dim, page_size=8, nk=offset + nq, dtype=dtype,
                        pages_per_slab=16)
    before = key_split_launches()
    run_prefill(case, nq, offset + nq, offset, seed=nq)
    assert key_split_launches() == before + 1
    run_fused_single(case, nq, offset, seed=nq)
    assert key_split_launches() == before + 2
    case.table[0, 100] = -1
    run_prefill(case, nq, offset + nq, offset, seed=nq)
    assert key_split_launches() == before + 3


@pytest.mark.parametrize('dtype,dim', [('float32', 64), ('bfloat16', 80)])
def test_causal_ragged_splits_over_workgroups(dtype, dim):
    before = key_split_launches()
    run_ragged(dtype, dim, [1, 33, 20], [2600, 17, 2100], h=2, seed=dim)
    assert key_split_launches() == before + 1


# Largest relative 2-norm error against 64 bits: 3 % over what the per-query
# kernel measured on such inputs (1.031e-7, 1.253e-7, 1.436e-7), whose sums are
# short chains over 16 groups of lanes. One chain over a block's 32 keys gave
# 1.137e-7, 1.382e-7 and 1.541e-7.
@pytest.mark.parametrize('dim,n,bound', [(64, 60, 1.06e-7), (64, 333, 1.29e-7), (128, 333, 1.48e-7)])
def test_fp32_sums_keep_the_per_query_kernels_precision(dim, n, bound):
    case = prefill_case(700 + n, batch=4, heads=12, dim=dim, page_size=16, nk=n, dtype='float32')
    got, ref = run_prefill(case, n, n, 0, seed=n)
    error = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f'head dim {dim}, {n} tokens: relative error {error:.4e}')
    assert error < bound


@pytest.mark.parametrize('dtype', ['float16', 'bfloat16'])
@pytest.mark.parametrize('n', [2, 5, 40])
def test_many_small_weights_beside_large_ones(dtype, n):
    # In every block of 32 keys one scores 0, with zero values, and 31 score
    # about -12.75: weights of 2.9e-6, 48.7 of fp16's smallest steps, times
    # values of 30000 make the whole output, 2.7. Rounded down to whole steps
    # the weights lost 1 % of it, ten times the tolerance.
    nk = 1500
    case = prefill_case(800 + n, batch=1, heads=1, dim=64, page_size=16, nk=nk, dtype=dtype)
    q = np.random.default_rng(n).standard_normal((1, 1, n, 64), dtype=np.float32)  # as run_prefill draws it
    q = po.decode(po.encode(q, CODES[dtype]), CODES[dtype])[0, 0].astype(np.float64)
    k = np.zeros((1, 1, nk, 64), np.float32)
    k[0, 0] = np.linalg.pinv(q) @ np.full(n, -12.75 * 8)
    v = np.full_like(k, 30000)
    k[0, 0, ::32] = v[0, 0, ::32] = 0
    po.image_append(case.image, case.table, case.columns, po.encode(k, CODES[dtype]), po.encode(v, CODES[dtype]), 0)
    got, ref = run_prefill(case, n, nk, nk - n, seed=n)
    assert 2 < ref[0, 0, 0, 0] < 4
