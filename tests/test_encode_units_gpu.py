"""The builder's unit passes at their edges, byte for byte against the CPU oracle:
units a bucket, partial steps, odd widths and offsets, substream counts that do not
divide a workgroup, the two sizes of the code-word table, and calls that leave the
passes for the general path (pairs that overflow a table, few substreams)."""
import numpy as np
import pytest
import torch

import MPServe_cuda
import oracle
from mpserve_amd.synthetic import make_awq_weight
from tests.helpers import synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _fp8(bf, q, sc, L, k, shift=0):
    """Builds on the device from tensors `shift` elements into their storage."""
    def put(a, dt):
        a = np.ascontiguousarray(a)
        base = torch.empty(a.size + shift, dtype=dt, device=DEV)
        base[shift:] = torch.from_numpy(a.reshape(-1)).to(DEV)
        return base[shift:].view(a.shape)
    b = put(bf.view(np.int16), torch.int16).view(torch.bfloat16)
    got = MPServe_cuda.huffman_build_fp8_decode_tables(b, put(q, torch.uint8), torch.from_numpy(sc), L, k)
    return {x: v.cpu().numpy() for x, v in got.items()}


def _same(got, want):
    assert list(got) == list(want)
    for x in want:
        assert got[x].shape == want[x].shape and np.array_equal(got[x], want[x]), x


@pytest.mark.parametrize("n,m,k,shift", [
    (300, 520, 1024, 0),    # several units a bucket, 8-element loads
    (300, 521, 1024, 0),    # odd width: rows start anywhere
    (300, 520, 1024, 1),    # the same loads from tensors at odd offsets
    (260, 1000, 320, 0),    # 1024 / k pieces leave work-items over
    (257, 999, 33, 0), (257, 999, 32, 0),  # many pieces side by side
    (257, 999, 31, 0),      # too few substreams: general path
    (5000, 8, 1024, 0), (5000, 3, 512, 0), (20000, 2, 64, 0),  # units bounded by their rows, not their elements
    (3, 17, 1024, 0),       # fewer elements than substreams
])
def test_units_per_row(n, m, k, shift):
    print(f"[units] {n}x{m} k{k} shift {shift}", flush=True)
    bf, q, sc = synth(n, m, seed=n + m + k)
    sc[n // 3:] = sc[0]  # one scale with many rows, the others few
    _same(_fp8(bf, q, sc, 7, k, shift), oracle.encode(bf, q, sc, 7, k))


@pytest.mark.parametrize("L", [1, 6, 7, 10, 11, 12])
def test_units_code_lengths(L):
    print(f"[units] L {L}", flush=True)
    bf, q, sc = synth(200, 300, seed=L)
    _same(_fp8(bf, q, sc[:1].copy(), L, 256), oracle.encode(bf, q, sc[:1].copy(), L, 256))


@pytest.mark.parametrize("syms,qs", [(2900, 2), (3500, 2), (6000, 2), (65536, 256)])
def test_units_table_sizes(syms, qs):
    """Pairs of one scale: within 3/4 of the smaller table, of the larger, near its end, and beyond any table."""
    print(f"[units] {syms} symbols x {qs}", flush=True)
    rng = np.random.default_rng(syms)
    bf = rng.integers(0, syms, size=(256, 900)).astype(np.uint16)
    q = rng.integers(0, qs, size=bf.shape).astype(np.uint8)
    sc = np.array([0x1C00], dtype=np.uint16)
    _same(_fp8(bf, q, sc, 7, 1024), oracle.encode(bf, q, sc, 7, 1024))


@pytest.mark.parametrize("n_sym", [2, 12, 64])
def test_short_list_with_a_count_that_could_wrap(n_sym):
    """A key of few symbols, one of them 2.3 million times: its merge runs in sequence."""
    print(f"[units] {n_sym} symbols, one very frequent", flush=True)
    rng = np.random.default_rng(n_sym)
    bf = np.full((2304, 1024), 0x3C00, dtype=np.uint16)
    rare = rng.choice(bf.size, 5000, replace=False)
    bf.flat[rare] = 0x3C00 + rng.integers(1, n_sym, size=rare.size) ** 2 if n_sym > 2 else 0x3C01
    q = np.full(bf.shape, 0x40, dtype=np.uint8)
    sc = np.array([0x1C00], dtype=np.uint16)
    _same(_fp8(bf, q, sc, 7, 1024), oracle.encode(bf, q, sc, 7, 1024))


@pytest.mark.parametrize("bs", [(128, 128), (64, 40), (2, 3)])
def test_units_blocks(bs):
    print(f"[units] blocks {bs}", flush=True)
    n, m = bs[0] * 4, bs[1] * 20
    bf, q, _ = synth(n, m, seed=bs[1])
    sc = np.random.default_rng(bs[0]).integers(0x2000, 0x2006, size=(4, 20), dtype=np.uint16)
    _same(_fp8(bf, q, sc, 7, 256), oracle.encode(bf, q, sc, 7, 256))


@pytest.mark.parametrize("n,m,group,k,by_scale,cap", [
    (512, 1024, 128, 1024, True, 1024), (512, 1024, 64, 256, True, 7), (300, 1000, 40, 512, True, 100000),
    (300, 999, None, 1024, True, 64), (300, 999, None, 256, False, 1024), (256, 640, 128, 1024, False, 1024),
])
def test_units_awq(n, m, group, k, by_scale, cap):
    print(f"[units] awq {n}x{m} group {group} k{k} by_scale {by_scale}", flush=True)
    w = make_awq_weight(n, m, group, seed=n + m + k)
    args = (w.bf16.to(DEV), w.int4_u8.to(DEV), w.scale_u16, 11, k)
    if by_scale:
        got = MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables_by_scale(*args, cap)
    else:
        got = MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables(*args)
    want = oracle.awq_encode(w.bf16.view(torch.uint16).numpy(), w.int4_u8.numpy(), w.scale_u16.numpy(), 11, k, cap,
                             by_scale)
    got = {x: v.cpu().numpy() for x, v in got.items()}
    assert list(got) == list(want)
    for x, v in want.items():
        assert got[x].shape == v.shape and np.array_equal(got[x].view(v.dtype), v), x


@pytest.mark.parametrize("L", [7, 12])
def test_handle_calls_give_the_ops_outputs(L):
    """The C ABI's handle (its own allocations, copied out) against the op's tensors; L = 12 takes the general path."""
    import ctypes

    from mpserve_amd import _native
    from mpserve_amd.encode import _OUTPUTS

    print(f"[units] handle L {L}", flush=True)
    bf, q, sc = (torch.from_numpy(x).to(DEV) for x in synth(300, 520, seed=3))
    want = MPServe_cuda.huffman_build_fp8_decode_tables(bf.view(torch.bfloat16), q, sc, L, 256)
    a = _native.MpsFp8EncodeIn()
    a.bf16, a.fp8, a.scales, a.numel, a.ndim, a.scale_ndim = bf.data_ptr(), q.data_ptr(), sc.data_ptr(), bf.numel(), 2, 1
    a.dims[0], a.dims[1], a.scale_dims[0], a.scale_numel, a.max_len, a.threads_per_block = 300, 520, 300, 300, L, 256
    lib, h, sizes, ptrs = _native.lib(), ctypes.c_void_p(), (ctypes.c_int64 * 17)(), (ctypes.c_void_p * 17)()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _native.check(lib.mps_fp8_encode(ctypes.byref(a), stream, ctypes.byref(h)))
    _native.check(lib.mps_fp8_sidecar_sizes(h, sizes))
    got = [torch.empty(sizes[i], dtype=dt) for i, (_, dt) in enumerate(_OUTPUTS)]
    for i, t in enumerate(got):
        ptrs[i] = t.data_ptr()
    _native.check(lib.mps_fp8_sidecar_copy(h, ptrs, stream))
    _native.check(lib.mps_fp8_sidecar_free(h))
    for (key, _), t in zip(_OUTPUTS, got):
        assert np.array_equal(t.numpy(), want[key].cpu().numpy().reshape(-1)), key


def test_builder_reports_no_memory():
    """An allocator without memory ends the build with an error, and the next build works."""
    from mpserve_amd._common import BuilderOutputs

    print("[units] no memory", flush=True)
    bf, q, sc = (torch.from_numpy(x).to(DEV) for x in synth(64, 256, seed=4))
    real, left = BuilderOutputs._alloc, [3]

    def few(self, ctx, slot, nbytes):
        left[0] -= 1
        return real(self, ctx, slot, nbytes) if left[0] >= 0 else None

    BuilderOutputs._alloc = few
    try:
        with pytest.raises(MemoryError, match="no device memory"):
            MPServe_cuda.huffman_build_fp8_decode_tables(bf.view(torch.bfloat16), q, sc, 7, 256)
    finally:
        BuilderOutputs._alloc = real
    out = MPServe_cuda.huffman_build_fp8_decode_tables(bf.view(torch.bfloat16), q, sc, 7, 256)
    want = oracle.encode(bf.cpu().numpy(), q.cpu().numpy(), sc.cpu().numpy(), 7, 256)
    _same({x: v.cpu().numpy() for x, v in out.items()}, want)


@pytest.mark.parametrize("entries", [65, 66, 127, 129, 511, 512, 513, 1025, 2046, 2047, 2048, 2049, 2300, 5000])
def test_long_lists(entries):
    """One key's list at the edges of the codebook kernels' sizes: few ties and many, with ESC past 2^L."""
    print(f"[units] list of {entries}", flush=True)
    rng = np.random.default_rng(entries)
    vals = np.concatenate([np.arange(entries), (entries * rng.random(90000) ** (1.5 + entries % 7)).astype(np.int64)])
    vals = vals[:vals.size // 64 * 64] if entries != 513 else np.repeat(np.arange(entries), 128)  # 513: all counts tie
    bf = rng.permutation(vals).astype(np.uint16).reshape(-1, 64)
    q = np.full(bf.shape, 5, dtype=np.uint8)
    sc = np.array([0x1C00], dtype=np.uint16)
    for L in (7, 11):
        _same(_fp8(bf, q, sc, L, 256), oracle.encode(bf, q, sc, L, 256))
    rows = np.full(bf.shape[0], 0x3C00, dtype=np.uint16)
    args = (torch.from_numpy(bf).to(DEV).view(torch.bfloat16), torch.from_numpy(q).to(DEV), torch.from_numpy(rows), 11, 256)
    for by_scale in (True, False):
        op = ("huffman_build_awq_int4_bucket_decode_tables" + ("_by_scale" if by_scale else ""))
        got = getattr(MPServe_cuda, op)(*args, *((1024,) if by_scale else ()))
        _same({x: v.cpu().numpy() for x, v in got.items()}, oracle.awq_encode(bf, q, rows, 11, 256, 1024, by_scale))


@pytest.mark.parametrize("n,shift,distinct", [
    (1, 0, 8), (7, 0, 8), (8, 0, 8), (9, 0, 8), (8192, 0, 8), (33000, 0, 8), (33000, 1, 1), (33001, 8, 300),
    (8191, 0, 4095), (8192, 0, 1), (8193, 0, 4096),    # from 8192 rows they are dealt to their scales on the GPU
    (9000, 0, 4096), (9000, 0, 4097), (20000, 0, 20000),  # with up to 4096 distinct scales
    (600000, 0, 1000),                                 # tiles of more than 2048 rows
])
def test_scales_ranked_and_dealt(n, shift, distinct):
    """Scales in memory at an offset, in numbers that leave loads, waves and tiles incomplete."""
    print(f"[units] {n} scales of {distinct}, shift {shift}", flush=True)
    rng = np.random.default_rng(n)
    bf, q = rng.integers(0, 50, size=(n, 2)).astype(np.uint16), rng.integers(0, 4, size=(n, 2)).astype(np.uint8)
    sc = rng.choice(65536, size=distinct, replace=False).astype(np.uint16)
    sc = rng.permutation(np.concatenate([sc, rng.choice(sc, size=max(0, n - distinct))])[:n])
    base = torch.zeros(n + shift, dtype=torch.int16, device=DEV)
    base[shift:] = torch.from_numpy(sc.view(np.int16)).to(DEV)
    got = MPServe_cuda.huffman_build_fp8_decode_tables(
        torch.from_numpy(bf.view(np.int16)).to(DEV).view(torch.bfloat16), torch.from_numpy(q).to(DEV),
        base[shift:].view(torch.uint16), 7, 64)
    _same({x: v.cpu().numpy() for x, v in got.items()}, oracle.encode(bf, q, sc, 7, 64))


@pytest.mark.parametrize("n,m,group,distinct", [
    (1100, 512, 64, 150), (1100, 512, 64, 4096),  # 8800 groups dealt to their scales on the GPU
    (1100, 512, 64, 4097), (1100, 512, 64, 8800),  # with too many scales for that: the host's loop into the same outputs
    (2731, 24, 8, 7),                              # 8193 groups, three a row
])
@pytest.mark.parametrize("cap", [1024, 37])
def test_groups_dealt_to_their_scales(n, m, group, distinct, cap):
    """By-scale builds of 8192 groups and more: rows and columns of every bucket's groups, in order."""
    print(f"[units] awq {n}x{m} group {group}, {distinct} scales, cap {cap}", flush=True)
    rng = np.random.default_rng(distinct)
    bf = (0x3C00 + rng.integers(0, 40, size=(n, m))).astype(np.uint16)
    q = rng.integers(0, 16, size=(n, m)).astype(np.uint8)
    sc = rng.choice(65536, size=distinct, replace=False).astype(np.uint16)
    groups = n * (m // group)
    sc = rng.permutation(np.concatenate([sc, rng.choice(sc, size=groups - distinct)])).reshape(n, m // group)
    got = MPServe_cuda.huffman_build_awq_int4_bucket_decode_tables_by_scale(
        torch.from_numpy(bf.view(np.int16)).to(DEV).view(torch.bfloat16), torch.from_numpy(q).to(DEV),
        torch.from_numpy(sc.view(np.int16)).view(torch.uint16), 11, 64, cap)
    want = oracle.awq_encode(bf, q, sc, 11, 64, cap, True)
    got = {x: v.cpu().numpy() for x, v in got.items()}
    assert list(got) == list(want)
    for x, v in want.items():
        assert got[x].shape == v.shape and np.array_equal(got[x].view(v.dtype), v), x


@pytest.mark.parametrize("L,n_sym", [(7, 65), (7, 128), (11, 513), (11, 2048)])
def test_long_list_with_sums_that_could_wrap(L, n_sym):
    """A key of 179.5 million elements (past (2^31 - 1) / 12): its list's merge runs in sequence, in each of the
    workgroup-a-key kernels. Code lengths against the oracle's package-merge of the counts."""
    print(f"[units] {n_sym} symbols, 179.5 million elements", flush=True)
    n, m = 13000, 13808
    rng = np.random.default_rng(n_sym)
    counts = np.maximum(1, (rng.random(n_sym) ** 6 * 1e6).astype(np.int64))
    counts = np.maximum(1, counts * (n * m) // counts.sum())
    counts[counts.argmax()] += n * m - counts.sum()
    assert counts.sum() == n * m and counts.min() >= 1
    syms = 0x3C00 + np.arange(n_sym)
    bf = torch.repeat_interleave(torch.from_numpy(syms.astype(np.int16)).to(DEV), torch.from_numpy(counts).to(DEV))
    q = torch.full((n, m), 0x40, dtype=torch.uint8, device=DEV)
    sc = torch.full((1,), 0x1C00, dtype=torch.int16, device=DEV).view(torch.uint16)
    got = MPServe_cuda.huffman_build_fp8_decode_tables(bf.view(n, m).view(torch.bfloat16), q, sc, L, 1024)
    order = np.lexsort((syms, counts))
    lens = np.empty(n_sym, dtype=np.int64)
    lens[order] = oracle.package_merge([int(c) for c in counts[order]], L)
    table = got["decode_syms_u16"].cpu().numpy()
    packed = got["decode_lens_u8"].cpu().numpy()
    assert table.shape == (1, 1 << L)
    nib = np.stack([packed & 15, packed >> 4], axis=-1).reshape(-1)
    entry = table[0].astype(np.int64) - 0x3C00
    assert np.array_equal(np.bincount(entry, minlength=n_sym), 1 << (L - lens)) and np.array_equal(nib, lens[entry])
    # codes of a length in list order, ascending
    starts = np.concatenate([[True], entry[1:] != entry[:-1]])
    want = order[np.argsort(lens[order], kind="stable")]
    assert np.array_equal(entry[starts], want)
    assert int(got["bucket_bit_base_i64"][-1]) > 0
    total = int((counts * lens).sum())
    bits = got["bucket_thread_startbit_u32"].cpu().numpy().astype(np.int64)[:, -1].sum()
    assert bits == total
