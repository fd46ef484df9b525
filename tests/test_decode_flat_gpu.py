"""Flat buckets (a column range that is no multiple of the 256, 512 or 1024 substreams):
bit-exact against the input weights through the op's first call, its cached plan, a
DecodePlan of several tensors and the allocation-free batch; the status words stay clear."""
import ctypes

import numpy as np
import pytest
import torch

import MPServe_cuda
import oracle
from mpserve_amd import _native
from mpserve_amd.decode import DecodePlan, sidecar_decode_args
from mpserve_amd.mpserve_cuda import _descriptor, _stream_handle, read_status
from tests.helpers import decode_args, synth, to_torch
from tests.test_decode_gpu import _esc_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(bf, q, sides):
    """Every way to decode ``q`` with each of the sidecars, into buffers of another value."""
    items = [(torch.from_numpy(np.ascontiguousarray(q)).to(DEV), to_torch(s, DEV)) for s in sides]
    blank = lambda: torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=DEV)  # noqa: E731
    same = lambda o, what: np.testing.assert_array_equal(o.view(torch.uint16).cpu().numpy(), bf, err_msg=what)  # noqa: E731
    read_status(torch.device(DEV))
    for q_t, sc_t in items:
        for what in ("first call", "plan"):
            same(MPServe_cuda.huffman_decode_fp8(*decode_args(sc_t, q_t), out=blank()), what)
    outs = [blank() for _ in items]
    plan = DecodePlan([(q_t, sc_t, o) for (q_t, sc_t), o in zip(items, outs)])
    plan.decode()
    assert plan.read_status() == 0
    for o in outs:
        same(o, "DecodePlan")
    outs = [blank() for _ in items]
    descs = [_descriptor(*sidecar_decode_args(q_t, sc_t)[:13], o) for (q_t, sc_t), o in zip(items, outs)]
    arr = (_native.MpsFp8Tensor * len(descs))(*descs)
    _native.check(_native.lib().mps_fp8_decode_batch_noalloc(
        arr, len(descs), 7, ctypes.c_void_p(_stream_handle(torch.device(DEV)))))
    for o in outs:
        same(o, "batch")
    assert read_status(torch.device(DEV)) == 0
    return plan.info()["work_items"]


@pytest.mark.parametrize("n,m", [
    (300, 1000),    # rows shorter than 1024 substreams, 4 | m
    (140, 5000),    # several slabs a row
    (140, 1028), (140, 2044),  # one quad past, one short of a multiple
    (130, 1021), (130, 1022), (130, 1023), (130, 4099),  # odd widths: elements split over two rows
    (129, 257), (600, 36), (600, 35),  # many rows a slab
    (2000, 5),      # rows of about one lane's elements
    (2000, 4), (2000, 3),  # the narrowest; below it (general path)
    (1, 4099), (2, 513),   # one or two rows: fewer elements than some k
])
def test_flat_widths(n, m):
    print(f"[flat] {n}x{m}", flush=True)
    bf, q, sc = synth(n, m, seed=n + m)
    sc[n // 2:] = sc[0]  # buckets of 128 rows beside small ones
    _check(bf, q, [oracle.encode(bf, q, sc, 7, k) for k in (256, 512, 1024)])


@pytest.mark.parametrize("n,m", [(128, 1500), (128, 1501), (40, 3003)])
def test_flat_esc(n, m):
    print(f"[flat] esc {n}x{m}", flush=True)
    bf, q, scales = _esc_inputs(n, m, n + m)
    sides = [oracle.encode(bf, q, scales, 7, k, with_stats=True) for k in (256, 1024)]
    assert all(st["esc_elements"] > 0 for _, st in sides)
    _check(bf, q, [s for s, _ in sides])


@pytest.mark.parametrize("bs0,bs1", [(128, 128), (128, 100), (96, 130), (40, 1500)])
def test_flat_column_ranges(bs0, bs1):
    """Blocks: column ranges that start inside a row."""
    print(f"[flat] blocks {bs0}x{bs1}", flush=True)
    n, m = 2 * bs0, 3 * bs1
    bf, q, _ = synth(n, m, seed=bs1)
    sc = np.random.default_rng(bs0).integers(0x2000, 0x2003, size=(2, 3), dtype=np.uint16)
    _check(bf, q, [oracle.encode(bf, q, sc, 7, k) for k in (256, 1024)])


@pytest.mark.parametrize("m", [12008, 12007])
def test_flat_ranges(m):
    """Buckets of 128 rows that a plan cuts into ranges of slabs, which start inside a row;
    side by side at k = 256 and 512."""
    print(f"[flat] ranges {m}", flush=True)
    bf, q, sc = synth(300, m, seed=m)
    sides = [oracle.encode(bf, q, sc[:1].copy(), 7, k) for k in (256, 512, 1024)]
    for s in sides:
        assert _check(bf, q, [s]) > s["bucket_table_i32"].shape[0]


@pytest.mark.parametrize("k", [256, 1024])
def test_flat_runs_share_tables(k):
    """More blocks of three scales than CUs: a plan decodes several after one table set-up. A row
    index out of range costs its own block only."""
    print(f"[flat] runs k{k}", flush=True)
    bs, g = 64, 30
    bf, q, _ = synth(bs * g, bs * g, seed=k)
    sc = np.random.default_rng(k).integers(0x2000, 0x2003, size=(g, g), dtype=np.uint16)
    side = oracle.encode(bf, q, sc, 7, k)
    assert _check(bf, q, [side]) < g * g
    side["row_indices_i32"] = side["row_indices_i32"].copy()
    hit = 17 * g + 5  # a bucket's index: block row 17, block column 5
    side["row_indices_i32"][hit * bs + 3] = bs * g
    out = torch.zeros(q.shape, dtype=torch.bfloat16, device=DEV)
    plan = DecodePlan([(torch.from_numpy(q).to(DEV), to_torch(side, DEV), out)])
    plan.decode()
    assert plan.read_status() == _native.MPS_STATUS_BAD_ROW
    want = bf.copy()
    want[17 * bs:18 * bs, 5 * bs:6 * bs] = 0
    np.testing.assert_array_equal(out.view(torch.uint16).cpu().numpy(), want)


@pytest.mark.parametrize("n,m,k", [
    (256, 1024, 1024), (300, 3072, 1024), (512, 4096, 1024), (140, 14336, 1024),  # P of 1, 3, 4, 14 blocks a row
    (1000, 3000, 1024), (257, 2001, 512),                                         # flat
    (512, 256, 256), (700, 1536, 512), (512, 4096, 256),                          # ranges side by side
])
def test_small_tensors_in_short_ranges(n, m, k):
    """A tensor of fewer than 64 elements a lane and CU: ranges of down to 16 elements a lane."""
    print(f"[flat] short ranges {n}x{m} k{k}", flush=True)
    bf, q, sc = synth(n, m, seed=n + m)
    sc[:] = sc[0]  # buckets of 128 rows
    side = oracle.encode(bf, q, sc, 7, k)
    items = _check(bf, q, [side])
    assert items > side["bucket_table_i32"].shape[0]
