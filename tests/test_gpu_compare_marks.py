"""GPU: the first pass of a comparison finds a single differing element wherever it lies.

Lengths around a workgroup's units, a chunk and several chunks; every element width and second
destination; one planted element at the ends and inside, of the destination or of the second one.
Counts are whole numbers: they must be exact.  After each find the plan compares clean again, so no
mark outlives its call.  The allocation-free entry point also runs on a plan that has never run and
so has no chunk table: its first pass is then the persistent one, without workgroups per piece.
"""

import numpy as np
import pytest
import torch

from elasticmegatron_amd import _native
from elasticmegatron_amd._native import SEGMENT_DTYPE

pytestmark = pytest.mark.gpu

CAST, DUP = 1, 4


@pytest.mark.parametrize("no_alloc,table", [(False, True), (True, True), (True, False)],
                         ids=["compare", "compare_static", "compare_static_without_chunk_table"])
@pytest.mark.parametrize("elem,flags", [(4, 0), (4, CAST), (4, DUP), (2, 0), (2, DUP), (1, 0), (8, DUP)])
def test_one_element(gpu_device, elem, flags, no_alloc, table):
    lens = [1, 3, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 4097, 9000]
    segs, off = [], 0
    for k, n in enumerate(lens):   # every other segment on 16 bytes, the rest an element off where they fall
        off = (off + 15) // 16 * 16 if k % 2 == 0 else off
        segs.append((0, 0, elem, flags, n, 1, off, 0, off, 0, 1 if flags else 0, off))
        off += n
    t = np.zeros(len(lens), dtype=SEGMENT_DTYPE)
    for r, (sb, db, eb, fl, n, rows, so, ss, do, ds, ab, ao) in zip(t, segs):
        r["src_buf"], r["dst_buf"], r["elem_bytes"], r["flags"], r["len"], r["rows"] = sb, db, eb, fl, n, rows
        r["src_off"], r["dst_off"], r["aux_buf"], r["aux_off"] = so, do, ab, ao
    nbytes = off * elem
    src = torch.randint(0, 100, (nbytes,), dtype=torch.uint8, device=gpu_device)
    dst, aux = torch.zeros_like(src), torch.zeros_like(src)
    plan = _native.Plan(t, [nbytes], [nbytes, nbytes])
    st = torch.cuda.current_stream(gpu_device).cuda_stream
    sp, dp = [src.data_ptr()], [dst.data_ptr(), aux.data_ptr()]
    plan.execute(sp, dp, st)
    if not table:
        plan = _native.Plan(t, [nbytes], [nbytes, nbytes])
    m = len(lens)
    groups, aux_groups = np.arange(m, dtype=np.uint32), np.arange(m, 2 * m, dtype=np.uint32)

    def mismatches():
        return plan.compare(sp, dp, groups, aux_groups, 2 * m, st, no_alloc=no_alloc)["mismatches"].astype(int)

    print(f"case one element: {elem} bytes, flags {flags}, no_alloc {no_alloc}, chunk table {table}", flush=True)
    assert not mismatches().any()
    for k, n in enumerate(lens):
        for second in ([False, True] if flags else [False]):
            width = 2 if second and flags == CAST else elem
            buf = aux if second else dst
            for i in sorted({0, n // 2, n - 1}):
                at = (segs[k][11 if second else 8] + i) * width
                buf[at] ^= 1
                want = np.zeros(2 * m, dtype=int)
                want[m + k if second else k] = 1
                assert (mismatches() == want).all(), (n, second, i)
                buf[at] ^= 1
    assert not mismatches().any()
