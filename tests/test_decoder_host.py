"""Host-side behaviour of the batched decoder (no kernel launches): argument checks and
their error types (reference src/pagedcore/decoder.py:113-177), weight stacking, the RoPE
table and the allocator's fused-write checks."""

from __future__ import annotations

import pytest
import torch

from oracle import decoder_reference as dref
from pagedcore_amd import _hip
from pagedcore_amd import decoder as dec
from pagedcore_amd.engine_types import KVReservation, RequestId
from pagedcore_amd.kv_cache import KVAllocator
from tests.support import CpuCopyWriter


@pytest.fixture(scope="module")
def small():
    weights = dec.random_weights(device="cpu", seed=1, layers=2, vocab=31, intermediate=32)
    return dec.TinyLlamaWeights(weights.embedding, weights.layers * 11, weights.final_norm, weights.lm_head)


def _allocator(lengths=(5,)):
    pool = torch.zeros((22, 2, 8, 16, 4, 64), dtype=torch.float16)
    allocator = KVAllocator(pool, kv_writer=CpuCopyWriter())
    requests = []
    for index, length in enumerate(lengths):
        request = RequestId(f"r{index}")
        allocator.create(KVReservation(request, 2))
        if length:
            allocator.append(request, *[torch.zeros(22, length, 4, 64, dtype=torch.float16)] * 2)
        requests.append(request)
    return allocator, tuple(requests)


def test_random_weights_shapes_and_stacking(small):
    layer = small.layers[0]
    assert small.embedding.shape == small.lm_head.shape == (31, 2048)
    assert layer.q_proj.shape == (2048, 2048) and layer.k_proj.shape == layer.v_proj.shape == (256, 2048)
    assert layer.gate_proj.shape == layer.up_proj.shape == (32, 2048) and layer.down_proj.shape == (2048, 32)
    assert all(t.dtype == torch.float16 for t in (layer.q_proj, layer.input_norm, small.lm_head))
    assert torch.equal(layer.input_norm, torch.ones(2048, dtype=torch.float16))
    fused = dec._fused(layer)
    # views of the stacked storage: no copy
    assert fused.qkv.data_ptr() == layer.q_proj.data_ptr() and fused.qkv.shape == (2560, 2048)
    assert fused.gate_up.data_ptr() == layer.gate_proj.data_ptr() and fused.gate_up.shape == (64, 2048)
    assert torch.equal(fused.qkv[2048:2304], layer.k_proj) and torch.equal(fused.gate_up[32:], layer.up_proj)
    assert dec._fused(layer) is fused


def test_separate_weights_are_concatenated_and_packed(small):
    layer = small.layers[0]
    separate = dec.LayerWeights(**{name: getattr(layer, name).clone() for name in dref._LAYER_FIELDS})
    fused = dec._fused(separate)
    assert fused.qkv.data_ptr() != separate.q_proj.data_ptr()
    assert torch.equal(fused.qkv, dec._fused(layer).qkv)
    packed = dec.pack_weights(dec.TinyLlamaWeights(small.embedding, (separate,) * 22, small.final_norm, small.lm_head))
    assert dec._fused(packed.layers[0]).qkv.data_ptr() == packed.layers[0].q_proj.data_ptr()


def test_rope_table_is_the_reference_expression():
    table = dec.rope_table(torch.device("cpu"))
    cosine, sine = dref.rope_cos_sin(torch.arange(2048)[None], torch.float16)
    assert torch.equal(table[:, 0], cosine[0, 0, :, :32]) and torch.equal(table[:, 1], sine[0, 0, :, :32])
    assert table.is_contiguous() and dec.rope_table(torch.device("cpu")) is table


def test_decode_paged_argument_checks(small):
    allocator, requests = _allocator((5, 7))
    good = torch.tensor([[1], [2]])
    with pytest.raises(ValueError, match=r"int64 \[batch, 1\]"):
        dec.decode_paged(good.int(), small, allocator, requests)
    with pytest.raises(ValueError, match=r"int64 \[batch, 1\]"):
        dec.decode_paged(good[:1], small, allocator, requests)
    with pytest.raises(ValueError, match="22 decoder layers"):
        dec.decode_paged(good, dec.TinyLlamaWeights(small.embedding, small.layers[:2], small.final_norm, small.lm_head), allocator, requests)
    with pytest.raises(KeyError):
        dec.decode_paged(good, small, allocator, (requests[0], RequestId("unknown")))
    counts = allocator.capacity()
    # no CPU fallback: a CPU pool is refused before anything is staged
    with pytest.raises(RuntimeError, match="runs on the GPU"):
        dec.decode_paged(good, small, allocator, requests)
    assert allocator.capacity() == counts and allocator._decode_appends is None
    assert [allocator.cached_length(r) for r in requests] == [5, 7]


def test_prefill_paged_argument_checks(small):
    allocator, (request, empty) = _allocator((5, 0))
    ids = torch.tensor([[1, 2, 3]])
    with pytest.raises(ValueError, match="empty request cache"):
        dec.prefill_paged(ids, small, allocator, request)
    with pytest.raises(ValueError, match=r"int64 \[1, tokens\]"):
        dec.prefill_paged(ids.repeat(2, 1), small, allocator, empty)
    with pytest.raises(ValueError, match="1 to 2048"):
        dec.prefill_paged(torch.zeros(1, 2049, dtype=torch.int64), small, allocator, empty)
    with pytest.raises(ValueError, match="22 decoder layers"):
        dec.prefill_paged(ids, dec.TinyLlamaWeights(small.embedding, small.layers[:3], small.final_norm, small.lm_head), allocator, empty)
    with pytest.raises(KeyError):
        dec.prefill_paged(ids, small, allocator, RequestId("unknown"))
    with pytest.raises(RuntimeError, match="runs on the GPU"):
        dec.prefill_paged(ids, small, allocator, empty)
    assert allocator.cached_length(empty) == 0


def test_fused_decode_write_checks_before_any_write():
    allocator, requests = _allocator((5, 16))
    table = dec.rope_table(torch.device("cpu"))
    qkv = torch.zeros(2, 2560, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="staged append"):
        allocator.write_decode_layers_rotary(requests, 0, qkv, table)
    counts = allocator.capacity()
    with pytest.raises(RuntimeError, match="every cache layer"), allocator.append_decode(requests):
        with pytest.raises(ValueError, match="written once in order"):
            allocator.write_decode_layers_rotary(requests, 1, qkv, table)
        with pytest.raises(ValueError, match="qkv"):
            allocator.write_decode_layers_rotary(requests, 0, qkv[:, :2552], table)
        with pytest.raises(ValueError, match="qkv"):
            allocator.write_decode_layers_rotary(requests, 0, qkv.float(), table)
        with pytest.raises(ValueError, match="rope_table"):
            allocator.write_decode_layers_rotary(requests, 0, qkv, table[:100])
        with pytest.raises(ValueError, match="distinct"):
            allocator.write_decode_layers_rotary((requests[0], requests[0]), 0, qkv, table)
        with pytest.raises(RuntimeError, match="does not rotate"):
            allocator.write_decode_layers_rotary(requests, 0, qkv, table)
        assert all(append.written_layers == 0 for append in allocator._decode_appends.values())
        slots, positions = allocator._decode_slots(requests, [allocator._decode_appends[r] for r in requests])
        # position = cached length before the step; slot = its block * 16 + offset
        assert positions.tolist() == [5, 16]
        assert slots.tolist() == [allocator.block_table(requests[0])[0] * 16 + 5, allocator._decode_appends[requests[1]].sequence.blocks[1] * 16]
    assert allocator.capacity() == counts


@pytest.mark.parametrize("rows", [1, 129, 1536, 1537])
@pytest.mark.parametrize("form", ["plain", "strided", "misaligned"])
def test_qkv_route_takes_only_what_the_kernel_reads(monkeypatch, rows, form):
    """_qkv_rope gives pc_qkv_rope_append contiguous, aligned weights up to 1536 rows and every
    other call to the projection and a RoPE launch, with the same outputs passed on."""
    n, k = dec.QKV_WIDTH, dec.HIDDEN
    x = torch.zeros((rows, k), dtype=torch.float16)
    if form == "strided":
        weight = torch.zeros((n, 2 * k), dtype=torch.float16)[:, ::2]
    elif form == "misaligned":
        weight = torch.zeros(n * k + 1, dtype=torch.float16)[1:].view(n, k)
    else:
        weight = torch.zeros((n, k), dtype=torch.float16)
    calls = []
    monkeypatch.setattr(_hip, "qkv_rope_append", lambda q, x, w, p, t, **out: calls.append(("fused", out)))
    monkeypatch.setattr(_hip, "rope_kv_append", lambda q, qkv, p, t, **out: calls.append(("rope", out)))
    monkeypatch.setattr(_hip, "rope_kv_append_parts", lambda q, qkv, p, t, **out: calls.append(("parts", out)))
    monkeypatch.setattr(_hip, "gemm_m128", lambda out, x, w, **options: None)
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: torch.zeros((x.shape[0], w.shape[0]), dtype=torch.float16))
    outputs = {"pool": x, "layer": 2, "slot_mapping": x}
    dec._qkv_rope(x, x, weight, None, None, **outputs)
    expected = "fused" if form == "plain" and rows <= 1536 else "rope"
    assert [name for name, _ in calls] == [expected] and calls[0][1] == outputs


@pytest.mark.parametrize("rows,route", [(1, "m128"), (128, "m128"), (129, "rows"), (1536, "rows"), (1537, "library")])
@pytest.mark.parametrize("form", ["plain", "strided", "misaligned"])
def test_eager_qkv_route_adds_as_the_fused_launch(monkeypatch, rows, route, form):
    """_qkv_projection takes the kernels that add in pc_qkv_rope_append's order, unsplit, wherever
    _qkv_rope takes that launch, and F.linear wherever it does not."""
    n, k = dec.QKV_WIDTH, dec.HIDDEN
    x = torch.zeros((rows, k), dtype=torch.float16)
    if form == "strided":
        weight = torch.zeros((n, 2 * k), dtype=torch.float16)[:, ::2]
    elif form == "misaligned":
        weight = torch.zeros(n * k + 1, dtype=torch.float16)[1:].view(n, k)
    else:
        weight = torch.zeros((n, k), dtype=torch.float16)
    calls = []

    def product(name):
        return lambda out, x, w, *, splits=1, epilogue=_hip.GEMM_PARTIALS: calls.append((name, splits, out.shape[-2:]))

    monkeypatch.setattr(_hip, "gemm_m128", product("m128"))
    monkeypatch.setattr(_hip, "gemm_rows", product("rows"))
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: torch.zeros((x.shape[0], w.shape[0]), dtype=torch.float16))
    qkv = dec._qkv_projection(x, weight)
    assert qkv.shape[-2:] == (rows, n) and qkv.ndim == (3 if calls and route == "m128" else 2)
    assert calls == ([(route, 1, (rows, n))] if form == "plain" and route != "library" else [])


@pytest.mark.parametrize("rows", [1, 64, 128, 129, 384, 640, 1024, 2048])
@pytest.mark.parametrize("form", ["plain", "strided", "misaligned", "odd_k", "odd_n"])
def test_projection_route_takes_only_what_the_kernels_read(monkeypatch, rows, form):
    """_linear_parts and _swiglu hand the GEMM kernels contiguous, aligned operands whose K
    divides into 64-column splits, and give every other form to the library product, bit for
    bit. The kernels are stood in for by fp32 products of the same arguments."""
    n, k = (96 if form == "odd_n" else 128), (72 if form == "odd_k" else 256)
    n += 1 if form == "odd_n" else 0
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, k), generator=gen).half()
    if form == "strided":
        weight = torch.randn((n, 2 * k), generator=gen).half()[:, ::2]
    elif form == "misaligned":
        weight = torch.randn(n * k + 1, generator=gen).half()[1:].view(n, k)
    else:
        weight = torch.randn((n, k), generator=gen).half()
    calls = []

    def stand_in(out, x, w, *, splits=1, epilogue=_hip.GEMM_PARTIALS):
        calls.append(epilogue)
        assert x.is_contiguous() and w.is_contiguous() and w.data_ptr() % 16 == 0
        assert w.shape[0] % 32 == 0 and w.shape[1] % (64 * splits) == 0
        if epilogue == _hip.GEMM_SWIGLU:
            assert w.shape[0] % 64 == 0
            y = (x.float() @ w.float().t()).half().float()
            half = w.shape[0] // 2
            out.copy_((torch.nn.functional.silu(y[:, :half]).half().float() * y[:, half:]).half())
            return
        span = w.shape[1] // splits
        products = [x[:, s * span : (s + 1) * span].float() @ w[:, s * span : (s + 1) * span].float().t() for s in range(splits)]
        out.copy_(torch.stack(products) if epilogue == _hip.GEMM_PARTIALS else products[0].half())

    def silu_mul(out, gate_up):
        half = gate_up.shape[1] // 2
        out.copy_((torch.nn.functional.silu(gate_up[:, :half].float()).half().float() * gate_up[:, half:].float()).half())

    monkeypatch.setattr(_hip, "gemm_m128", stand_in)
    monkeypatch.setattr(_hip, "gemm_rows", stand_in)
    monkeypatch.setattr(_hip, "silu_mul", silu_mul)
    library = torch.nn.functional.linear(x, weight)
    got = dec._linear_parts(x, weight, 4)
    got = got.sum(0).half() if got.ndim == 3 else got
    if form == "plain":
        assert calls == [_hip.GEMM_PARTIALS]
        # one fp16 rounding of sums taken in another order
        torch.testing.assert_close(got, library, atol=2e-3 * library.abs().max().item(), rtol=0)
    else:
        assert calls == [] and torch.equal(got, library)
    if form != "odd_n":
        calls.clear()
        fused = dec._swiglu(x, weight)
        expected = torch.empty_like(fused)
        silu_mul(expected, library)
        assert calls == ([_hip.GEMM_SWIGLU] if form == "plain" else [])
        torch.testing.assert_close(fused, expected, atol=4e-3 * expected.abs().max().item(), rtol=0)


@pytest.mark.parametrize("rows,width,k,taken", [(65536, 5632, 64, True), (65537, 5632, 64, False), (40000, 28672, 64, False)])
def test_swiglu_beyond_the_kernels_sizes_is_the_librarys(monkeypatch, rows, width, k, taken):
    """More rows, or more output elements, than pc_gemm_rows takes go to F.linear and pc_silu_mul, as
    every row count above 128 did before that kernel."""
    calls = []
    monkeypatch.setattr(_hip, "gemm_rows", lambda out, x, w, **options: calls.append("rows"))
    monkeypatch.setattr(_hip, "silu_mul", lambda out, gate_up: calls.append("library"))
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: None)
    monkeypatch.setattr(dec, "_rows_swiglu", lambda rows, width: True)
    dec._swiglu(torch.empty((rows, k), dtype=torch.float16), torch.empty((2 * width, k), dtype=torch.float16))
    assert calls == (["rows"] if taken else ["library"])


@pytest.mark.parametrize("n,k", [(2560, 2048), (2048, 2048), (2048, 5632), (32000, 2048)])
def test_rows_splits_always_divide_into_the_decoders_shapes(n, k):
    for rows in range(129, 2049):
        splits = dec._rows_splits(rows, n, k)
        assert splits in (0, 1, 2, 4)
        if splits:
            assert k % (64 * splits) == 0
        if splits > 1:
            # the partials stay a fraction of the weight they save reading late
            assert splits * rows * n * 4 <= 32 << 20


def test_rows_whose_k_does_not_divide_are_the_librarys(monkeypatch):
    """65 units of K cannot be split in four, the count the rule names at this size."""
    assert dec._rows_splits(129, 128, 4160) == 4
    monkeypatch.setattr(_hip, "gemm_rows", lambda *args, **options: pytest.fail("not divisible"))
    x, weight = torch.ones((129, 4160), dtype=torch.float16), torch.ones((128, 4160), dtype=torch.float16)
    assert torch.equal(dec._linear_parts(x, weight, 4), torch.nn.functional.linear(x, weight))
