"""AWQ sidecars whose buckets are not whole blocks of the 128-column slab path: flat row
buckets of any width, by-scale groups of other sizes. Bit-exact to the per-lane path's
output (MPSERVE_AWQ_SLAB=0) and, where the coding is lossless, to the input weights."""
import pytest
import torch

import MPServe_cuda
from mpserve_amd import awq
from mpserve_amd.mpserve_cuda import read_status
from mpserve_amd.synthetic import make_awq_weight
from tests.test_awq_oracle import esc_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _args(q, sc, by_scale):
    n, m = q.shape
    mid = (("bucket_group_offsets_i32", "group_rows_i32", "group_col_start_i32") if by_scale else
           ("bucket_col_start_i32", "bucket_col_len_i32", "bucket_row_offsets_i32", "row_indices_i32"))
    head = (q, sc["bitstream_u64"], sc["decode_syms_u16"], sc["decode_lens_u8"], sc["bucket_table_i32"])
    tail = (sc["bucket_thread_startbit_u32"], sc["bucket_bit_base_i64"], n, m, 11)
    return head + tuple(sc[x] for x in mid) + tail + ((int(sc["shape_nmkg_i64"][3]),) if by_scale else ())


def _check(bf16, q, scales, k, by_scale, cap, monkeypatch, flat):
    sc, st = awq.build_awq_sidecar(bf16, q, scales, 11, k, cap, by_scale, with_stats=True)
    blank = lambda: torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=DEV)  # noqa: E731
    bits = lambda t: t.view(torch.int16)  # noqa: E731
    read_status(torch.device(DEV))
    monkeypatch.setenv("MPSERVE_AWQ_SLAB", "0")
    want = blank()
    plan = awq.AwqDecodePlan([(q, sc, want)])
    plan.decode()
    lane_items = plan.info()["work_items"]
    monkeypatch.delenv("MPSERVE_AWQ_SLAB")
    outs = [blank(), blank()]
    plan = awq.AwqDecodePlan([(q, sc, o) for o in outs])
    for _ in range(2):
        plan.decode()
    status = plan.read_status()
    if st["esc_collisions"] == 0:
        assert torch.equal(bits(want), bits(bf16)) and status == 0
    for o in outs:
        assert torch.equal(bits(o), bits(want))
    op = (MPServe_cuda.huffman_decode_awq_int4_bucket_by_scale if by_scale else
          MPServe_cuda.huffman_decode_awq_int4_bucket)
    for _ in range(2):
        assert torch.equal(bits(op(*_args(q, sc, by_scale), out=blank())), bits(want))
    if st["esc_collisions"] == 0:
        assert read_status(torch.device(DEV)) == 0
    if flat:
        assert plan.info()["work_items"] >= 2 * min(lane_items, sc["bucket_table_i32"].shape[0])


@pytest.mark.parametrize("k", [256, 512, 1024])
@pytest.mark.parametrize("n,m", [
    (140, 5000), (140, 1028), (130, 1021), (130, 4099),  # quads, odd widths
    (129, 257), (300, 36), (300, 35), (2000, 5), (2000, 4), (2000, 3),  # many rows a slab; too narrow for a range
    (128, 2048), (1, 4099), (1, 300),  # fewer than four blocks a row; single rows
])
def test_rows_of_any_width(n, m, k, monkeypatch):
    print(f"[awq flat] rows {n}x{m} k{k}", flush=True)
    w = make_awq_weight(n, m, None, seed=n + m, device=DEV)
    s = w.scale_u16.view(torch.int16)
    s[n // 2:] = s[0].clone()  # a bucket of up to 128 rows beside small ones
    _check(w.bf16, w.int4_u8, w.scale_u16, k, False, 1024, monkeypatch, False)


@pytest.mark.parametrize("m", [12008, 12007])
def test_ranges_of_slabs(m, monkeypatch):
    print(f"[awq flat] ranges {m}", flush=True)
    w = make_awq_weight(300, m, None, seed=m, device=DEV)
    for k in (256, 512, 1024):
        _check(w.bf16, w.int4_u8, w.scale_u16[:1].clone(), k, False, 1024, monkeypatch, True)


@pytest.mark.parametrize("m", [1500, 1501])
@pytest.mark.parametrize("by_scale", [False, True])
def test_flat_esc(m, by_scale, monkeypatch):
    print(f"[awq flat] esc {m} by_scale {by_scale}", flush=True)
    bits, q, sc = esc_inputs(with_zero=False)
    bits, q = (torch.from_numpy(x.reshape(-1)[:40 * m].reshape(40, m).copy()).to(DEV) for x in (bits.view("int16"), q))
    sc = torch.from_numpy(sc.view("int16")).view(torch.uint16).to(DEV)[:1].reshape(1)
    for k in (256, 1024):
        _check(bits.view(torch.bfloat16), q, sc, k, by_scale, 1024, monkeypatch, False)


@pytest.mark.parametrize("n,m,group,k,cap", [
    (512, 1024, 64, 1024, 1024), (512, 1024, 64, 512, 1024), (512, 1024, 64, 256, 1024), (300, 1024, 64, 1024, 37),
    (512, 1024, 256, 1024, 1024), (512, 1024, 256, 256, 1024), (256, 2048, 512, 1024, 100),
    (512, 1024, 32, 1024, 1024),  # narrower than a wave: the per-lane path
    (300, 1500, None, 1024, 1024), (300, 1501, None, 256, 64), (300, 2048, None, 512, 1024),  # a row a group
    (200, 3000, 1500, 1024, 1024),
])
def test_by_scale_groups(n, m, group, k, cap, monkeypatch):
    print(f"[awq flat] by scale {n}x{m} group {group} k{k} cap {cap}", flush=True)
    w = make_awq_weight(n, m, group, seed=n + m, device=DEV)
    s = w.scale_u16.view(torch.int16)
    s.copy_(torch.where(torch.arange(s.numel(), device=DEV).view(s.shape) % 3 == 0, s, s.reshape(-1)[0]))  # large buckets
    _check(w.bf16, w.int4_u8, w.scale_u16, k, True, cap, monkeypatch, False)


@pytest.mark.parametrize("n,m,group,k", [
    (512, 4096, None, 1024), (140, 14336, None, 1024),                             # 4 and 14 blocks a row
    (512, 1024, None, 256), (300, 2048, None, 512),                                # ranges side by side
    (700, 3000, None, 1024), (257, 2001, None, 512),                               # flat
    (512, 4096, 128, 256), (512, 4096, 128, 1024), (512, 2048, 64, 512),           # slabs of groups
])
def test_small_weights_in_short_ranges(n, m, group, k, monkeypatch):
    """A weight of fewer than 64 elements a lane and CU: ranges of down to 16 elements a lane."""
    print(f"[awq flat] short ranges {n}x{m} group {group} k{k}", flush=True)
    w = make_awq_weight(n, m, group, seed=n + m, device=DEV)
    s = w.scale_u16.view(torch.int16)
    s.copy_(s.reshape(-1)[0].clone().expand_as(s))  # buckets of 128 rows, or of 1024 groups
    _check(w.bf16, w.int4_u8, w.scale_u16, k, group is not None, 1024, monkeypatch, False)
