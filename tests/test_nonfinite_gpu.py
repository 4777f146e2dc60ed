"""GPU parity of causal attention over values that are not finite: a query's
output holds Inf or NaN in a dim only where a key that it attends does. Against
the float64 oracle, which sums the attended keys alone; the finite outputs by
tests/tolerances.py, the others exactly."""
import numpy as np
import pytest

from minitorch_amd import paged_ops
from minitorch_amd.runtime import DeviceTensor, runtime
from minitorch_amd.workloads import DevicePagedCase
from oracle import paged_oracle as po
from test_prefill_gpu import CODES, prefill_case
from tolerances import assert_attention_close

pytestmark = pytest.mark.gpu


def assert_same_values(got, ref, dtype, context):
    assert np.array_equal(np.isnan(got), np.isnan(ref)), f'{context}: NaN pattern differs'
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf]) and not np.isinf(got[~inf]).any(), f'{context}: Inf pattern differs'
    assert_attention_close(np.where(inf, 0, got), np.where(inf, 0, ref), dtype, context=context)


# Workgroup shapes of the causal kernel: one and two key blocks, few and many
# tiles, keys split over workgroups.
SHAPES = [(2, 3, 5, 40, 64), (2, 30, 20, 30, 64), (30, 10, 33, 0, 64), (1, 2, 70, 300, 64), (1, 2, 40, 2500, 80),
          (3, 20, 200, 5, 64), (3, 40, 100, 200, 64), (5, 60, 140, 5, 64), (2, 40, 70, 60, 128), (4, 40, 30, 30, 128)]


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('batch,heads,n,offset,dim', SHAPES)
def test_non_finite_values_reach_only_queries_that_attend_them(dtype, batch, heads, n, offset, dim):
    case = prefill_case(500 + n + heads, batch=batch, heads=heads, dim=dim, page_size=16, nk=offset + n, dtype=dtype)
    hd = heads * dim
    qkv = np.random.default_rng(n).standard_normal((batch, n, 3 * hd), dtype=np.float32)
    v = qkv[:, :, 2 * hd:].reshape(batch, n, heads, dim)
    # dims of one head of the first request and of all heads of the last
    v[0, n // 2, 1, 3] = np.inf
    v[0, n // 2, 1, dim - 1] = np.nan
    v[0, n - 1, 0, 7] = -np.inf
    v[-1, n // 3, :, 5] = -np.inf
    v[-1, n - 1, :, 5] = np.inf
    v[-1, n - 2, :, 11] = np.nan
    v[-1, 0, heads - 1, 2] = np.inf
    qkv = po.encode(qkv, CODES[dtype])
    parts = [np.ascontiguousarray(qkv[:, :, i * hd:(i + 1) * hd].reshape(batch, n, heads, dim).transpose(0, 2, 1, 3))
             for i in range(3)]
    image = case.image.copy()
    po.image_append(image, case.table, case.columns, parts[1], parts[2], 0, offset=offset)
    checked = sorted({0, batch - 1})  # the requests with such values
    ref = po.image_paged_attention(image, CODES[dtype], case.table[checked], case.columns, parts[0][checked], 0,
                                   offset, offset + n)
    assert np.isinf(ref).any() and np.isnan(ref).any() and np.isfinite(ref).any()
    item = 4 if dtype == 'float32' else 2
    common = dict(h=heads, d=dim, page_size=16, pages_per_slab=case.pages_per_slab, num_slabs=case.num_slabs,
                  columns=case.columns, layer=0, layers=1, dtype=dtype)

    def upload(x):
        t = DeviceTensor(x.shape, dtype)
        runtime().h2d(t.ptr, x)
        return t

    for entry in ('attention', 'prefill', 'ragged'):
        dev = DevicePagedCase(case)
        if entry == 'attention':
            q, k, vv = (upload(x) for x in parts)
            out = DeviceTensor(parts[0].shape, dtype)
            paged_ops.paged_append(k.ptr, vv.ptr, dev.slab_table.ptr, dev.block_table.ptr, b=batch, n=n,
                                   offset=offset, **common)
            paged_ops.paged_attention(out.ptr, q.ptr, dev.slab_table.ptr, dev.block_table.ptr, b=batch, nq=n,
                                      nk=offset + n, offset=offset, **common)
        else:
            rows = upload(qkv)
            out = DeviceTensor((batch * n, hd), dtype)
            q, k, vv = (rows.ptr + i * hd * item for i in range(3))
            if entry == 'prefill':
                paged_ops.paged_prefill(out.ptr, q, k, vv, dev.slab_table.ptr, dev.block_table.ptr, b=batch, n=n,
                                        offset=offset, qkv_stride=3 * hd, **common)
            else:
                tables = [dev.block_table.ptr + 4 * r * case.columns for r in range(batch)]
                paged_ops.paged_prefill_ragged(out.ptr, q, k, vv, dev.slab_table.ptr, tables, [n] * batch,
                                               [offset] * batch, qkv_stride=3 * hd, out_stride=hd, **common)
        runtime().synchronize()
        got = out.to_numpy()
        if entry != 'attention':
            got = got.reshape(batch, n, heads, dim).transpose(0, 2, 1, 3)
        assert_same_values(got[checked], ref, dtype, f'{entry} n={n} offset={offset}')
        assert np.array_equal(dev.pool_image().view(np.uint8), image.view(np.uint8)), f'{entry}: append differs'
        others = np.delete(got, checked, axis=0)
        assert np.isfinite(others).all()
