"""Row units: segments whose source, destination or length is no whole number of 16-byte units.

On the CPU, ``tests/native/row_units.cpp`` checks the placement of every unit (csrc/segment.h) over
element sizes, lengths, pitches and base addresses.  On the GPU, the copy must equal numpy slicing
and write nothing beside the rows, under every launch schedule, and a comparison must count every
element once, also those that two units hold.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

from elasticmegatron_amd import _native
from elasticmegatron_amd.resharding.layout import SEGMENT_DTYPE
from tests.helpers import bf16_rne_bits

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TYPES = {2: np.uint16, 4: np.uint32, 8: np.uint64}


def test_units_cover_every_element_once_and_stay_inside_their_rows(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ is needed to build the host check")
    exe = tmp_path / "row_units"
    r = subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "elasticmegatron_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "row_units.cpp"), "-o", str(exe)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout.split()[1]) > 10_000


def _segments(eb):
    """One-run and strided segments around the edges: rows of 15 to 17 bytes' worth of elements, of a
    line and of 512 bytes less and plus one element, and one long odd row; offsets off 16 bytes, off
    a line, and co-aligned.  Destinations are disjoint."""
    per, line = 16 // eb, 128 // eb
    out, src, dst, aux = [], 0, 0, 0
    k = 0
    for n in (per - 1, per, per + 1, line - 1, line + 1, 4 * line - 1, 4 * line + 1, 2 * line * line + 5):
        for rows, gap in ((1, 0), (3, 0), (5, 1), (4, line // 2 + 1)):
            for so, do in ((1, 0), (0, 1), (3, 3), (per // 2 + 1, line - 1)):
                if n < 1 or (n > 100 * line and rows > 1):
                    continue
                flags = (0, 1 if eb == 4 else 4, 4, 2, 3 if eb == 4 else 6)[k % 5]
                k += 1
                ss, ds, asr = (n + 2, n + gap, n + 1) if rows > 1 else (0, 0, 0)
                has_aux = flags & 5
                out.append((0, 0, eb, flags, src + so, dst + do, n, rows, ss, ds, 1 if has_aux else 0, 0,
                            aux // (2 if flags & 1 else eb) + k % 3 if has_aux else 0, asr if has_aux else 0))
                src += (rows * (n + 2) + 2 * line) // line * line
                dst += (rows * (n + gap) + 3 * line) // line * line
                aux += (rows * (n + 1) + 3 * line) // line * 128   # bytes
    t = np.zeros(len(out), dtype=SEGMENT_DTYPE)
    t[:] = out
    return t, (src + line) * eb, (dst + line) * eb, aux + 128


def _expected(t, src, dst, aux):
    eb = int(t[0]["elem_bytes"])
    a, b, d, h = src.view(TYPES[eb]), dst.view(TYPES[eb]), aux.view(TYPES[eb]), aux.view(np.uint16)
    for s in t:
        n, flags = int(s["len"]), int(s["flags"])
        for r in range(int(s["rows"])):
            so, do, ao = (int(s[f]) + r * int(s[g]) for f, g in
                          (("src_off", "src_stride"), ("dst_off", "dst_stride"), ("aux_off", "aux_stride")))
            v = np.zeros(n, dtype=a.dtype) if flags & 2 else a[so:so + n]
            b[do:do + n] = v
            if flags & 1:
                h[ao:ao + n] = bf16_rne_bits(v)
            if flags & 4:
                d[ao:ao + n] = v


@pytest.mark.gpu
@pytest.mark.parametrize("eb", [2, 4, 8])
@pytest.mark.parametrize("tuning", [{}, dict(lanes=256), dict(units=4, xcd_remap=2), dict(chunk_index=False),
                                    dict(buffer_ops=True), dict(persistent=True), dict(nontemporal=False)])
def test_row_units_copy_and_compare(gpu_device, eb, tuning):
    print(f"case row units elem {eb} tuning {tuning}", flush=True)
    t, ns, nd, na = _segments(eb)
    rng = np.random.default_rng(eb)
    src_h = rng.integers(0, 256, ns, dtype=np.uint8)
    want, want_aux = (rng.integers(0, 256, n, dtype=np.uint8) for n in (nd, na))
    # Bases 16 bytes off a line, as a tensor inside another buffer may be.
    src, dst, aux = (torch.zeros(n + 16, dtype=torch.uint8, device=gpu_device) for n in (ns, nd, na))
    src[16:].copy_(torch.from_numpy(src_h))
    dst[16:].copy_(torch.from_numpy(want))
    aux[16:].copy_(torch.from_numpy(want_aux))
    _expected(t, src_h, want, want_aux)
    plan = _native.Plan(t, [ns], [nd, na], check_disjoint=True)
    bases = [src.data_ptr() + 16], [dst.data_ptr() + 16, aux.data_ptr() + 16]
    st = torch.cuda.current_stream().cuda_stream
    try:
        _native.set_tuning(**tuning)
        plan.execute(*bases, st)
    finally:
        _native.set_tuning()
    torch.cuda.synchronize()
    assert np.array_equal(dst[16:].cpu().numpy(), want) and np.array_equal(aux[16:].cpu().numpy(), want_aux)
    assert not dst[:16].any() and not aux[:16].any()

    # Every element counted once; damage to the first, second, middle and last element of rows is found.
    # The allocation-free entry point runs on a second plan too, one that has never run and so has no
    # chunk table: its first pass is then the persistent one.
    n = len(t)
    groups = np.arange(n, dtype=np.uint32)
    fresh = _native.Plan(t, [ns], [nd, na])
    for p, no_alloc in ((fresh, True), (plan, False), (plan, True)):
        got = p.compare(*bases, groups, groups + n, 2 * n, st, no_alloc=no_alloc)
        assert not got["mismatches"].any()
        assert np.array_equal(got["elements"][:n], t["len"] * t["rows"])
    d, hits = dst[16:].view({2: torch.int16, 4: torch.int32, 8: torch.int64}[eb]), np.zeros(n, dtype=np.uint64)
    for i in range(0, n, 3):
        ln, r = int(t[i]["len"]), int(t[i]["rows"]) - 1
        cols = {0, 1 % ln, ln // 2, ln - 1}
        for c in cols:
            d[int(t[i]["dst_off"]) + r * int(t[i]["dst_stride"]) + c] ^= 1
        hits[i] = len(cols)
    aux_hits = np.zeros(n, dtype=np.uint64)   # the last element of the second destination's last row
    for i in range(1, n, 3):
        s, fl = t[i], int(t[i]["flags"])
        if fl & 5:
            at = int(s["aux_off"]) + (int(s["rows"]) - 1) * int(s["aux_stride"]) + int(s["len"]) - 1
            aux[16 + at * (2 if fl & 1 else eb)] ^= 1
            aux_hits[i] = 1
    assert aux_hits.any()
    for p, no_alloc in ((fresh, True), (plan, False), (plan, True)):
        got = p.compare(*bases, groups, groups + n, 2 * n, st, no_alloc=no_alloc)
        assert np.array_equal(got["mismatches"][:n], hits) and np.array_equal(got["mismatches"][n:], aux_hits)
