"""Plans of weights that take different paths in one launch: each set of paths has a kernel of
its own (awq_decode_plan<kRanges>, fp8_decode_plan), and every weight decodes as in a plan alone."""
import pytest
import torch

from mpserve_amd import awq
from mpserve_amd.synthetic import make_awq_weight

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
