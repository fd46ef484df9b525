"""The builder ops are complete when they return: the stream they ran on is idle, so their outputs
and inputs may be used, rewritten or freed on another stream without an event between."""
import pytest
import torch

import MPServe_cuda
from mpserve_amd.decode import DecodePlan, sidecar_decode_args
from mpserve_amd.synthetic import make_awq_weight

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _fp8(n, m):
    g = torch.Generator(device=DEV).manual_seed(n)
    w = torch.randn((n, m), generator=g, device=DEV).mul_(0.02).to(torch.bfloat16)
    s = w.float().abs().amax(dim=1) / 448.0
    q = (w.float() / s[:, None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)
    return w, q.contiguous(), s.to(torch.float16).view(torch.uint16)


@pytest.mark.parametrize("max_len", [7, 12])  # the unit passes; the general path
def test_fp8_build_on_a_side_stream_is_complete(max_len):
    print(f"[streams] fp8 max_len {max_len}", flush=True)
    w, q, s = _fp8(4096, 8192)  # the last pass over it runs for tens of microseconds
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for _ in range(3):
        with torch.cuda.stream(side):
            sc = MPServe_cuda.huffman_build_fp8_decode_tables(w, q, s, max_len, 1024)
        assert side.query()
    if max_len != 7:
        return
    src = w.clone()
    out = torch.empty_like(w)
    MPServe_cuda.huffman_decode_fp8(*sidecar_decode_args(q, sc), out=out)  # the first call, on the current stream
    assert torch.equal(out.view(torch.int16), src.view(torch.int16))
    with torch.cuda.stream(side):
        sc = MPServe_cuda.huffman_build_fp8_decode_tables(w, q, s, max_len, 1024)
    w.zero_()  # the input is the caller's again
    plan = DecodePlan([(q, sc, out)])  # its checkpoints walk reads the stream just written
    plan.decode()
    assert torch.equal(out.view(torch.int16), src.view(torch.int16)) and plan.read_status() == 0


@pytest.mark.parametrize("by_scale", [False, True])
def test_awq_build_on_a_side_stream_is_complete(by_scale):
    print(f"[streams] awq by_scale {by_scale}", flush=True)
    w = make_awq_weight(4096, 8192, 128 if by_scale else None, seed=3, device=DEV)
    torch.cuda.synchronize()
    build = (MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables_by_scale if by_scale else
             MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables)
    side = torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(side):
            build(w.bf16, w.int4_u8, w.scale_u16, 11, 1024)
        assert side.query()


@pytest.mark.parametrize("n_sym", [3000, 65536])
def test_general_path_takes_the_unit_passes_block(n_sym, monkeypatch):
    """A build whose pairs overflow the unit passes' tables (random bits) asks for one block of work
    memory beside the scales', as one that stays on them does."""
    from mpserve_amd._common import BuilderOutputs

    print(f"[streams] work memory, {n_sym} symbols", flush=True)
    real, work = BuilderOutputs._alloc, []

    def count(self, ctx, slot, nbytes):
        if slot < 0:
            work.append(nbytes)
        return real(self, ctx, slot, nbytes)

    monkeypatch.setattr(BuilderOutputs, "_alloc", count)
    g = torch.Generator(device=DEV).manual_seed(n_sym)
    w = torch.randint(0, n_sym, (256, 900), generator=g, device=DEV).to(torch.int16).view(torch.bfloat16)
    q = torch.randint(0, 256 if n_sym == 65536 else 2, (256, 900), generator=g, device=DEV, dtype=torch.uint8)
    s = torch.full((1,), 0x1C00, dtype=torch.int16, device=DEV).view(torch.uint16)
    MPServe_cuda.huffman_build_fp8_decode_tables(w, q, s, 7, 1024)
    assert len(work) == 2
