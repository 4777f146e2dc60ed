"""Captured calls whose split partials lie in the library's workspace: a graph
holds the workspace's address, which later and larger calls of the thread must
leave valid. Each graph is replayed several times, with the thread's own eager
calls (one of them growing the workspace) and synchronizations in between, and
every replay equals the eager result bit for bit. Tolerances of the eager result
are in tests/tolerances.py."""
import ctypes as ct
import threading

import numpy as np
import pytest

from minitorch_amd import paged_ops
from minitorch_amd.runtime import DeviceTensor, runtime
from minitorch_amd.workloads import DevicePagedCase, make_decode_case
from oracle import paged_oracle as po
from test_prefill_gpu import CODES, prefill_case
from tolerances import assert_attention_close

pytestmark = pytest.mark.gpu


class Call:
    """A call with its own buffers: the decode of ragged rows, or causal
    attention of the last nq tokens."""

    def __init__(self, nq, lengths, dtype='float16', heads=3):
        self.nq, self.dtype = nq, dtype
        if nq == 0:
            pages = sum(-(-n // 16) for n in lengths)
            self.case = make_decode_case(40, batch=len(lengths), heads=heads, dim=64, page_size=16, lengths=lengths,
                                         pool_pages=-(-pages // 8) * 8, pages_per_slab=8, dtype=dtype)
            self.dev = DevicePagedCase(self.case)
            self.out = self.dev.out
        else:
            nk = lengths[0]
            self.case = c = prefill_case(41, batch=len(lengths), heads=heads, dim=64, page_size=16, nk=nk, dtype=dtype,
                                         pages_per_slab=8)
            self.dev = DevicePagedCase(c)
            rng = np.random.default_rng(nq)
            self.q = po.encode(rng.standard_normal((c.batch, heads, nq, 64), dtype=np.float32), CODES[dtype])
            self.q_dev = DeviceTensor(self.q.shape, dtype)
            runtime().h2d(self.q_dev.ptr, self.q)
            self.out = DeviceTensor(self.q.shape, dtype)
        self.blank = np.zeros(self.out.shape, self.out.raw_numpy().dtype)

    def __call__(self):
        c, d = self.case, self.dev
        if self.nq == 0:
            paged_ops.paged_decode_batch(d.out.ptr, d.q.ptr, d.k.ptr, d.v.ptr, d.slab_table.ptr, d.block_table.ptr,
                                         d.offsets.ptr, **d.kwargs())
        else:
            nk = int(c.lengths[0])
            paged_ops.paged_attention(self.out.ptr, self.q_dev.ptr, d.slab_table.ptr, d.block_table.ptr, b=c.batch,
                                      h=c.heads, nq=self.nq, nk=nk, d=64, page_size=16,
                                      pages_per_slab=c.pages_per_slab, num_slabs=c.num_slabs, columns=c.columns,
                                      layer=0, layers=1, offset=nk - self.nq, dtype=self.dtype)

    def clear(self):
        runtime().h2d(self.out.ptr, self.blank)

    def result(self):
        runtime().synchronize()
        return self.out.raw_numpy()

    def check(self):
        c = self.case
        if self.nq == 0:
            ref = po.image_decode_batch(c.image.copy(), CODES[c.dtype], c.table, c.columns, c.q, c.k, c.v, c.offsets,
                                        c.layer)
        else:
            nk = int(c.lengths[0])
            ref = po.image_paged_attention(c.image, CODES[c.dtype], c.table, c.columns, self.q, 0, nk - self.nq, nk)
        runtime().synchronize()
        assert_attention_close(self.out.to_numpy(), ref, c.dtype)


def in_new_thread(work):
    """Runs ``work`` in a thread of its own, whose workspace starts empty."""
    errors = []

    def run():
        try:
            work()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize('before', [False, True])
@pytest.mark.parametrize('nq,lengths', [(0, [2500, 100]), (1, [3000]), (40, [4040])])
def test_replays_after_the_workspace_has_grown(nq, lengths, before):
    # `before`: the workspace is there when the capture begins, else it grows
    # within it.
    def work():
        lib = runtime().lib
        lib.mt_graph_end.argtypes = [ct.POINTER(ct.c_void_p)]
        lib.mt_graph_launch.argtypes = [ct.c_void_p]
        lib.mt_graph_destroy.argtypes = [ct.c_void_p]
        call, small, large = Call(nq, lengths), Call(0, [1500, 9]), Call(0, [6000, 5000, 2000, 9], heads=12)
        if before:
            call()
        runtime().synchronize()
        graph = ct.c_void_p()
        assert lib.mt_graph_begin() == 0
        call()
        assert lib.mt_graph_end(ct.byref(graph)) == 0
        call.clear()
        assert lib.mt_graph_launch(graph) == 0
        first = call.result()
        call.check()
        for other in (small, large, small, large):
            other()
            call.clear()
            assert lib.mt_graph_launch(graph) == 0
            other.check()
            assert np.array_equal(call.result(), first)
        call.clear()
        call()
        assert np.array_equal(call.result(), first)
        assert lib.mt_graph_destroy(graph) == 0

    in_new_thread(work)
