"""GPU parity of one query per request on the decode kernel: through
``mt_paged_attention`` and ``mt_paged_prefill`` at one length for all rows
(unsplit, split at odd lengths, past 2048 keys, a missing page), and through
``mt_paged_decode_batch`` where few rows with long tables are split finer than
1024 tokens. Against the float64 oracle; tolerances are in tests/tolerances.py."""
import numpy as np
import pytest

from minitorch_amd import paged_ops
from minitorch_amd.runtime import DeviceTensor, runtime
from minitorch_amd.workloads import make_decode_case, DevicePagedCase
from oracle import paged_oracle as po
from test_paged_gpu import check_case
from test_prefill_gpu import CODES, prefill_case, run_prefill, run_fused_single
from tolerances import assert_attention_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,dim', [('float32', 64), ('float32', 128), ('float32', 12), ('bfloat16', 64),
                                       ('float16', 80), ('bfloat16', 120)])
@pytest.mark.parametrize('keys', [1, 64, 65, 577, 2049, 4100])
def test_one_token_attention(dtype, dim, keys):
    case = prefill_case(600 + keys + dim, batch=2, heads=3, dim=dim, page_size=16, nk=keys, dtype=dtype, layers=2,
                        layer=1, pages_per_slab=8)
    run_prefill(case, 1, keys, keys - 1, seed=keys)
    one = prefill_case(700 + keys + dim, batch=1, heads=3, dim=dim, page_size=8, nk=keys, dtype=dtype,
                       pages_per_slab=8)
    run_fused_single(one, 1, keys - 1, seed=keys)


@pytest.mark.parametrize('keys,hole', [(100, 2), (100, 6), (3000, 100), (3000, 187)])
def test_one_token_attention_missing_page(keys, hole):
    # a hole anywhere, also at the new token's page, makes the row NaN
    case = prefill_case(800 + keys + hole, batch=2, heads=2, dim=64, page_size=16, nk=keys, dtype='bfloat16',
                        pages_per_slab=8)
    case.table[1, hole] = -1
    got, _ = run_prefill(case, 1, keys, keys - 1, seed=hole)
    assert np.isnan(got[1]).all() and not np.isnan(got[0]).any()


@pytest.mark.parametrize('dtype,dim', [('float32', 64), ('bfloat16', 64), ('float16', 128), ('bfloat16', 40)])
@pytest.mark.parametrize('batch,lengths', [(1, [3333]), (3, [1, 1025, 5000]), (9, [7, 64, 65, 300, 512, 513, 1024, 1500, 2000])])
def test_decode_batch_few_rows_long_tables(dtype, dim, batch, lengths):
    case = make_decode_case(900 + batch + dim, batch=batch, heads=3, dim=dim, page_size=16, lengths=lengths,
                            pool_pages=-(-sum(-(-n // 16) for n in lengths) // 8) * 8, pages_per_slab=8, dtype=dtype)
    check_case(case)
