"""GPU parity of the paths that read rows element by element: head dims whose
rows are not whole 16-byte chunks, and operands at addresses that are not
16-byte aligned, through every entry point (decode, unsplit and split; append
and causal attention; prefill and ragged prefill). Against the float64 oracle;
pool images bit for bit. Tolerances are in tests/tolerances.py."""
import numpy as np
import pytest

from minitorch_amd import paged_ops
from minitorch_amd.runtime import RawDeviceBuffer, runtime
from minitorch_amd.workloads import make_decode_case, DevicePagedCase
from oracle import paged_oracle as po
from test_paged_gpu import check_case
from test_prefill_gpu import CODES, prefill_case, run_fused_single, run_prefill, run_ragged
from tolerances import assert_attention_close

pytestmark = pytest.mark.gpu
ODD_ROWS = [('float32', 33), ('float16', 20), ('float16', 100), ('bfloat16', 7)]


@pytest.mark.parametrize('dtype,dim', ODD_ROWS)
@pytest.mark.parametrize('lengths', [[1, 7, 33, 500], [1, 1025, 3000]])
def test_decode(dtype, dim, lengths):
    pages = sum(-(-n // 16) for n in lengths)
    check_case(make_decode_case(620 + dim, batch=len(lengths), heads=3, dim=dim, page_size=16, lengths=lengths,
                                pool_pages=-(-pages // 4) * 4, pages_per_slab=4, dtype=dtype))


@pytest.mark.parametrize('dtype,dim', ODD_ROWS)
@pytest.mark.parametrize('n,offset', [(1, 90), (5, 40), (70, 33), (3, 2100)])
def test_attention_and_prefill(dtype, dim, n, offset):
    case = prefill_case(630 + dim + n, batch=2, heads=3, dim=dim, page_size=16, nk=offset + n, dtype=dtype)
    run_prefill(case, n, offset + n, offset, seed=n)
    one = prefill_case(640 + dim + n, batch=1, heads=3, dim=dim, page_size=8, nk=offset + n, dtype=dtype)
    run_fused_single(one, n, offset, seed=n)


@pytest.mark.parametrize('dtype,dim', ODD_ROWS)
def test_ragged(dtype, dim):
    run_ragged(dtype, dim, [17, 1, 40], [0, 12, 5], h=2, seed=dim)


def at_odd_address(x):
    """A device buffer that holds x one element past its start."""
    buffer = RawDeviceBuffer(x.nbytes + 16)
    assert buffer.ptr % 16 == 0
    buffer.upload(x.reshape(-1), x.itemsize)
    return buffer


@pytest.mark.parametrize('dtype', ['float32', 'float16', 'bfloat16'])
@pytest.mark.parametrize('n,offset', [(1, 700), (20, 30)])
def test_unaligned_operands(dtype, n, offset):
    # whole chunks (head dim 64) at addresses one element off
    b, h, d = 2, 3, 64
    case = prefill_case(650 + n, batch=b, heads=h, dim=d, page_size=16, nk=offset + n, dtype=dtype)
    rng = np.random.default_rng(n)
    q, k, v = (po.encode(rng.standard_normal((b, h, n, d), dtype=np.float32), CODES[dtype]) for _ in range(3))
    image = case.image.copy()
    po.image_append(image, case.table, case.columns, k, v, 0, offset=offset)
    ref = po.image_paged_attention(image, CODES[dtype], case.table, case.columns, q, 0, offset, offset + n)
    common = dict(b=b, h=h, d=d, page_size=16, pages_per_slab=case.pages_per_slab, num_slabs=case.num_slabs,
                  columns=case.columns, layer=0, layers=1, dtype=dtype)
    rows = [np.ascontiguousarray(x.transpose(0, 2, 1, 3)) for x in (q, k, v)]  # [b, n, h, d]
    for entry in ('attention', 'prefill', 'decode'):
        if entry == 'decode' and n > 1:
            continue
        dev = DevicePagedCase(case)
        buffers = [at_odd_address(x) for x in (rows if entry == 'prefill' else (q, k, v))]
        out = at_odd_address(np.zeros_like(q))
        qp, kp, vp, op = (t.ptr + q.itemsize for t in (*buffers, out))
        if entry == 'attention':
            paged_ops.paged_append(kp, vp, dev.slab_table.ptr, dev.block_table.ptr, n=n, offset=offset, **common)
            paged_ops.paged_attention(op, qp, dev.slab_table.ptr, dev.block_table.ptr, nq=n, nk=offset + n,
                                      offset=offset, **common)
        elif entry == 'prefill':
            paged_ops.paged_prefill(op, qp, kp, vp, dev.slab_table.ptr, dev.block_table.ptr, n=n, offset=offset,
                                    **common)
        else:
            paged_ops.paged_decode_batch(op, qp, kp, vp, dev.slab_table.ptr, dev.block_table.ptr, dev.offsets.ptr,
                                         **common)
        runtime().synchronize()
        got = po.decode(out.download(q.dtype, q.size, q.itemsize), CODES[dtype]).reshape((b, n, h, d) if entry == 'prefill' else (b, h, n, d))
        if entry == 'prefill':
            got = got.transpose(0, 2, 1, 3)
        assert_attention_close(got, ref, dtype, context=entry)
        assert np.array_equal(dev.pool_image().view(np.uint8), image.view(np.uint8)), f'{entry}: append differs'
