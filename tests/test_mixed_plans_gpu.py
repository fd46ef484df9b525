"""Plans of weights that take different paths in one launch: each set of paths has a kernel of
its own (awq_decode_plan<kRanges>, fp8_decode_plan), and every weight decodes as in a plan alone."""
import numpy as np
import pytest
import torch

import oracle
from mpserve_amd import awq
from mpserve_amd.decode import DecodePlan
from mpserve_amd.synthetic import make_awq_weight
from tests.helpers import synth, to_torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _awq_item(n, m, group, k, one_scale=True):
    w = make_awq_weight(n, m, group, seed=n + m + k, device=DEV)
    if one_scale:  # buckets of 128 rows, or of 1024 groups
        s = w.scale_u16.view(torch.int16)
        s.copy_(s.reshape(-1)[0].clone().expand_as(s))
    return w.int4_u8, awq.build_awq_sidecar(w.bf16, w.int4_u8, w.scale_u16, 11, k, 1024, group is not None)


ROWS = (512, 4096, None, 1024)     # whole buckets of k = 1024, or row ranges of them
BESIDE = (512, 1024, None, 256)    # ranges side by side
GROUPS = (512, 1024, 128, 1024)    # runs of by-scale buckets
TINY = (40, 2, None, 1024, False)  # buckets of one code a lane


def _check_awq(shapes, monkeypatch):
    items = [_awq_item(*s) for s in shapes]
    blank = lambda q: torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=DEV)  # noqa: E731
    bits = lambda t: t.view(torch.int16)  # noqa: E731
    monkeypatch.setenv("MPSERVE_AWQ_SLAB", "0")
    want = [blank(q) for q, _ in items]
    for (q, sc), o in zip(items, want):
        awq.AwqDecodePlan([(q, sc, o)]).decode()
    torch.cuda.synchronize()
    monkeypatch.delenv("MPSERVE_AWQ_SLAB")
    got = [blank(q) for q, _ in items]
    plan = awq.AwqDecodePlan([(q, sc, o) for (q, sc), o in zip(items, got)])
    for _ in range(2):
        plan.decode()
    for s, a, b in zip(shapes, got, want):
        assert torch.equal(bits(a), bits(b)), s


@pytest.mark.parametrize("shapes", [
    (ROWS, BESIDE), (ROWS, TINY), (ROWS, BESIDE, TINY), (GROUPS, ROWS, BESIDE), (GROUPS, TINY), (BESIDE, TINY),
])
def test_awq_aligned_weights_of_several_kinds(shapes, monkeypatch):
    print(f"[mixed] awq {shapes}", flush=True)
    _check_awq(shapes, monkeypatch)


FLAT = (300, 1000, None, 1024)     # rows that are no multiple of the substreams
FLAT256 = (140, 1021, None, 256)
OTHER = (512, 1024, 64, 1024)      # groups of another size than 128 columns
OTHER256 = (600, 1024, 64, 256)


@pytest.mark.parametrize("shapes", [
    (ROWS, FLAT), (GROUPS, FLAT, TINY), (ROWS, TINY, FLAT256),           # <13>
    (BESIDE, FLAT256), (BESIDE, TINY, FLAT),                             # <14>
    (ROWS, BESIDE, FLAT),                                                # <11>
    (GROUPS, OTHER), (GROUPS, OTHER, FLAT, TINY), (BESIDE, OTHER256), (OTHER, OTHER256, FLAT256),  # <30>
    (ROWS, BESIDE, TINY, FLAT), (ROWS, OTHER, FLAT), (ROWS, BESIDE, OTHER, TINY),                  # <31>
])
def test_awq_aligned_and_flat_weights(shapes, monkeypatch):
    print(f"[mixed] awq {shapes}", flush=True)
    _check_awq(shapes, monkeypatch)


@pytest.mark.parametrize("shapes", [
    ((512, 4096, 1024), (140, 5000, 1024)),                        # a large flat share
    ((512, 4096, 1024), (2, 1000, 1024)), ((512, 4096, 256), (2, 1021, 256)),  # few and short flat buckets
    ((512, 4096, 1024), (1, 10000, 512)),                          # few, but long
    ((512, 4096, 1024), (512, 1024, 256), (300, 1021, 512), (3, 700, 1024)),
])
def test_fp8_aligned_and_flat_weights(shapes):
    print(f"[mixed] fp8 {shapes}", flush=True)
    items = []
    for n, m, k in shapes:
        bf, q, sc = synth(n, m, seed=n + m + k)
        sc[:] = sc[0]
        side = to_torch(oracle.encode(bf, q, sc, 7, k), DEV)
        out = torch.full((n, m), float("nan"), dtype=torch.bfloat16, device=DEV)
        items.append((bf, (torch.from_numpy(q).to(DEV), side, out)))
    plan = DecodePlan([x for _, x in items])
    for _ in range(2):
        plan.decode()
    assert plan.read_status() == 0
    for (bf, (_, _, out)), s in zip(items, shapes):
        np.testing.assert_array_equal(out.view(torch.uint16).cpu().numpy(), bf, err_msg=str(s))


@pytest.mark.parametrize("n,m,group,k", [
    (40, 1500, None, 1024), (300, 4099, None, 256),   # flat: one range; several side by side
    (256, 1024, 64, 1024), (512, 1024, 256, 256), (40, 1500, 1500, 512),
])
@pytest.mark.parametrize("at", [0.0, 0.99])
def test_awq_bad_row_is_dropped_alone(n, m, group, k, at, monkeypatch):
    """A row (group) index out of range in sidecars that left the per-lane path: flagged, and the other
    rows decode as they do there."""
    print(f"[mixed] bad row {n}x{m} group {group} k{k} at {at}", flush=True)
    from mpserve_amd._native import MPS_STATUS_BAD_ROW

    q, sc = _awq_item(n, m, group, k)
    key = "group_rows_i32" if group else "row_indices_i32"
    sc[key] = sc[key].clone()
    sc[key][int(at * sc[key].numel())] = n
    outs = []
    for slab in ("0", "1"):
        monkeypatch.setenv("MPSERVE_AWQ_SLAB", slab)
        out = torch.zeros((n, m), dtype=torch.bfloat16, device=DEV)
        plan = awq.AwqDecodePlan([(q, sc, out)])
        plan.decode()
        assert plan.read_status() & MPS_STATUS_BAD_ROW
        outs.append(out.view(torch.int16))
    assert torch.equal(outs[0], outs[1]) and int((outs[0] != 0).any(dim=1).sum()) >= n - 1
