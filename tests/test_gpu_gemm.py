"""pc_gemm_m128 (the decode step's projections at up to 128 rows) and the split-K consumers.

The GEMM is compared with an fp32 torch product of the same fp16 inputs (fp32 accumulation
in both; only the summation order differs), split by split so that a wrong K range cannot
hide in the total. The fp16 and SwiGLU epilogues are checked against the fp16 rounding of
that product and against pc_silu_mul applied to the library's own fp16 projections. The
split-K consumers are checked bit for bit against the fp16 path fed fp16(sum of the parts),
summed in the same split order.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from pagedcore_amd import _hip
from pagedcore_amd import decoder as dec

pytestmark = pytest.mark.gpu

# (m, n, k, splits): the decode step's q|k|v, o_proj and down projections at batch 128 and
# 64 (the serving graph), and ragged row counts.
PARTIAL_SHAPES = [
    (128, 2560, 2048, 4),
    (128, 2048, 2048, 4),
    (128, 2048, 5632, 8),
    (64, 2560, 2048, 4),
    (37, 2048, 2048, 4),
    (1, 2048, 5632, 8),
    (128, 11264, 2048, 1),
]


def _inputs(device, m, n, k, seed):
    gen = torch.Generator(device=device).manual_seed(seed)
    x = (torch.randn((m, k), device=device, generator=gen) * 0.5).half()
    w = (torch.randn((n, k), device=device, generator=gen) * 0.02).half()
    return x, w


def _bits(t: torch.Tensor) -> np.ndarray:
    return t.detach().cpu().contiguous().view(torch.int16).numpy()


@pytest.mark.parametrize("m,n,k,splits", PARTIAL_SHAPES)
def test_gemm_partials_match_fp32_split_by_split(device, m, n, k, splits):
    x, w = _inputs(device, m, n, k, seed=m + n + k + splits)
    out = torch.full((splits, m, n), float("nan"), dtype=torch.float32, device=device)
    _hip.gemm_m128(out, x, w, splits=splits, epilogue=_hip.GEMM_PARTIALS)
    torch.cuda.synchronize()
    span = k // splits
    worst = 0.0
    for s in range(splits):
        part = x[:, s * span : (s + 1) * span].float() @ w[:, s * span : (s + 1) * span].float().t()
        err = (out[s] - part).abs().max().item()
        scale = part.abs().max().item()
        worst = max(worst, err / scale)
        # fp32 accumulation of the same products in another order: a few ulp of the sums.
        assert err <= 2e-6 * scale + 1e-7, (s, err, scale)
    print(f"m {m} n {n} k {k} splits {splits}: max error / max |part| {worst:.2e}")


@pytest.mark.parametrize("m,n,k", [(128, 11264, 2048), (128, 2048, 2048), (5, 2048, 2048)])
def test_gemm_half_rounds_the_fp32_product(device, m, n, k):
    x, w = _inputs(device, m, n, k, seed=7 + m)
    out = torch.empty((m, n), dtype=torch.float16, device=device)
    _hip.gemm_m128(out, x, w, splits=1, epilogue=_hip.GEMM_HALF)
    exact = x.float() @ w.float().t()
    torch.cuda.synchronize()
    # fp16(Y), Y the fp32 partial-sum path of the same kernel, bit for bit; and Y differs
    # from the exact product by the summation order only: within a half fp16 ulp plus the
    # fp32 accumulation error (absolute, a few 1e-7 of the largest sums: it dominates where
    # the sum cancels to a tiny value).
    parts = torch.empty((1, m, n), dtype=torch.float32, device=device)
    _hip.gemm_m128(parts, x, w, splits=1, epilogue=_hip.GEMM_PARTIALS)
    torch.cuda.synchronize()
    assert np.array_equal(_bits(out), _bits(parts[0].half()))
    ulp = torch.finfo(torch.float16).eps * exact.abs().clamp_min(2.0**-14)
    slack = 2e-6 * exact.abs().max().item()
    assert ((out.float() - exact).abs() <= ulp + slack).all()
    assert (out == exact.half()).float().mean().item() > 0.99


@pytest.mark.parametrize("m", [128, 64, 3])
def test_gemm_swiglu_equals_silu_mul_of_the_fp16_projections(device, m):
    """The SwiGLU epilogue on the stacked [gate | up] weight equals pc_silu_mul applied to
    the fp16 projections of the same kernel configuration, bit for bit (the projections
    themselves are checked against fp32 in test_gemm_half_rounds_the_fp32_product)."""
    width = 5632
    x, w = _inputs(device, m, 2 * width, 2048, seed=11 + m)
    fused = torch.empty((m, width), dtype=torch.float16, device=device)
    _hip.gemm_m128(fused, x, w, splits=1, epilogue=_hip.GEMM_SWIGLU)
    projected = torch.empty((m, 2 * width), dtype=torch.float16, device=device)
    _hip.gemm_m128(projected, x, w, splits=1, epilogue=_hip.GEMM_HALF)
    separate = torch.empty_like(fused)
    _hip.silu_mul(separate, projected)
    torch.cuda.synchronize()
    assert np.array_equal(_bits(fused), _bits(separate))
    # and the reference expression (dense.py:102-104, torch's silu) on those projections
    # within two ulp of the product (silu's own last bit may differ from x / (1 + e^-x)).
    gate, up = projected[:, :width].float(), projected[:, width:].float()
    expected = (torch.nn.functional.silu(gate).half().float() * up).half().float()
    ulp = torch.finfo(torch.float16).eps * expected.abs().clamp_min(2.0**-14)
    assert ((fused.float() - expected).abs() <= 2 * ulp + 2.0**-24).all()


@pytest.mark.parametrize("m", [80, 81, 127, 128])
@pytest.mark.parametrize("n,k", [(64, 64), (192, 192), (320, 2048), (11264, 256), (12352, 128)])
def test_gemm_swiglu_short_tiles(device, m, n, k):
    """Either side of the rows and columns that take 64 x 96 tiles, columns that end inside a tile,
    fewer K stages than the ring has: bit equal to pc_silu_mul of the fp16 projections, and
    nothing written past the output."""
    x, w = _inputs(device, m, n, k, seed=3 * m + n + k)
    guard = torch.full((m * (n // 2) + 64,), -77.0, dtype=torch.float16, device=device)
    fused = guard[: m * (n // 2)].view(m, n // 2).fill_(float("nan"))
    _hip.gemm_m128(fused, x, w, epilogue=_hip.GEMM_SWIGLU)
    projected = torch.empty((m, n), dtype=torch.float16, device=device)
    _hip.gemm_m128(projected, x, w, epilogue=_hip.GEMM_HALF)
    separate = torch.empty((m, n // 2), dtype=torch.float16, device=device)
    _hip.silu_mul(separate, projected)
    torch.cuda.synchronize()
    assert (guard[m * (n // 2) :] == -77.0).all()
    assert np.array_equal(_bits(fused), _bits(separate))


def _sum_in_split_order(parts: torch.Tensor) -> torch.Tensor:
    total = parts[0].clone()
    for s in range(1, parts.shape[0]):
        total = total + parts[s]
    return total.half()


@pytest.mark.parametrize("rows,splits", [(128, 4), (64, 8), (3, 1), (128, 16), (7, 64)])
def test_add_rms_norm_parts_equals_the_fp16_path(device, rows, splits):
    gen = torch.Generator(device=device).manual_seed(rows * splits)
    width = 2048
    parts = torch.randn((splits, rows, width), device=device, generator=gen) * 0.3
    hidden = torch.randn((rows, width), device=device, generator=gen).half()
    weight = (1 + 0.1 * torch.randn(width, device=device, generator=gen)).half()
    h1, h2 = hidden.clone(), hidden.clone()
    out1 = torch.empty_like(hidden)
    out2 = torch.empty_like(hidden)
    _hip.add_rms_norm(out1, h1, _sum_in_split_order(parts), weight, dec.RMS_EPS)
    _hip.add_rms_norm_parts(out2, h2, parts, weight, dec.RMS_EPS)
    torch.cuda.synchronize()
    assert np.array_equal(_bits(h1), _bits(h2))
    assert np.array_equal(_bits(out1), _bits(out2))


@pytest.mark.parametrize("tokens,splits", [(128, 4), (5, 8), (128, 16), (3, 64)])
def test_rope_kv_append_parts_equals_the_fp16_path(device, tokens, splits):
    gen = torch.Generator(device=device).manual_seed(tokens + splits)
    parts = torch.randn((splits, tokens, 2560), device=device, generator=gen) * 0.5
    positions = torch.randint(0, 2048, (tokens,), device=device, generator=gen)
    blocks = 20
    slots = torch.randperm(blocks * 16, device=device, generator=gen)[:tokens]
    table = dec.rope_table(device)
    results = []
    for use_parts in (False, True):
        pool = torch.full((22, 2, blocks, 16, 4, 64), float("nan"), dtype=torch.float16, device=device)
        query = torch.empty(tokens, 32, 64, dtype=torch.float16, device=device)
        keys = torch.empty(tokens, 4, 64, dtype=torch.float16, device=device)
        values = torch.empty_like(keys)
        common = dict(key_out=keys, value_out=values, pool=pool, layer=3, slot_mapping=slots)
        if use_parts:
            _hip.rope_kv_append_parts(query, parts, positions, table, **common)
        else:
            _hip.rope_kv_append(query, _sum_in_split_order(parts), positions, table, **common)
        torch.cuda.synchronize()
        results.append((query, keys, values, pool))
    for a, b in zip(*results):
        assert np.array_equal(_bits(a), _bits(b))


# --- exact properties at the decode step's shapes ------------------------------------------


@pytest.mark.parametrize("m,n,k,splits", [s for s in PARTIAL_SHAPES if s[0] == 128])
def test_gemm_partials_permute_and_scale_exactly(device, m, n, k, splits):
    """Permuting the activation rows permutes the partials' rows, permuting the weight rows
    permutes their columns, and doubling the weight doubles them, all bit for bit: every
    output element is the same sequence of MFMA sums wherever its row and column sit in
    the tiles, and a power-of-two scale rounds nothing."""
    x, w = _inputs(device, m, n, k, seed=7 * n + k)
    gen = torch.Generator(device="cpu").manual_seed(n + splits)
    rows, cols = torch.randperm(m, generator=gen).to(device), torch.randperm(n, generator=gen).to(device)

    def run(xx, ww):
        out = torch.full((splits, m, n), float("nan"), dtype=torch.float32, device=device)
        _hip.gemm_m128(out, xx.contiguous(), ww.contiguous(), splits=splits, epilogue=_hip.GEMM_PARTIALS)
        torch.cuda.synchronize()
        return out

    base = run(x, w)
    assert not torch.isnan(base).any()
    assert torch.equal(run(x[rows], w), base[:, rows])
    assert torch.equal(run(x, w[cols]), base[:, :, cols])
    assert torch.equal(run(x, w * 2), base * 2)


def test_gemm_swiglu_permutes_exactly(device):
    """The SwiGLU epilogue (output column c from gate row c and up row half + c): the same
    permutation of the gate rows and of the up rows permutes the output columns, and
    permuting the activation rows permutes the output rows, bit for bit."""
    m, n, k = 128, 11264, 2048
    half = n // 2
    x, w = _inputs(device, m, n, k, seed=91)
    gen = torch.Generator(device="cpu").manual_seed(92)
    rows, cols = torch.randperm(m, generator=gen).to(device), torch.randperm(half, generator=gen).to(device)

    def run(xx, ww):
        out = torch.full((m, half), float("nan"), dtype=torch.float16, device=device)
        _hip.gemm_m128(out, xx.contiguous(), ww.contiguous(), epilogue=_hip.GEMM_SWIGLU)
        torch.cuda.synchronize()
        return out

    base = run(x, w)
    assert not torch.isnan(base).any()
    assert torch.equal(run(x[rows], w), base[rows])
    permuted = torch.cat((w[:half][cols], w[half:][cols]))
    assert torch.equal(run(x, permuted), base[:, cols])


# --- the streaming form: edges of its row tiles, column tiles and K units --------------------

# (n, k, splits): one unit and one tile; odd units per wave, a last 24-column SwiGLU tile that
# is partly outside (160 / 24), tiles not a multiple of 8; the decode step's shapes.
STREAM_SHAPES = [(64, 64, 1), (320, 704, 1), (96, 1408, 2), (2560, 2048, 2), (2048, 5632, 4), (2048, 2048, 4)]


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 97, 128])
@pytest.mark.parametrize("n,k,splits", STREAM_SHAPES)
def test_gemm_row_and_tile_edges(device, m, n, k, splits):
    """Every row count at the edges of the row tiles: partials against fp32 split by split,
    nothing written past the output, and with one split the fp16 and SwiGLU epilogues bit
    equal to the rounded partials (the same sums under every epilogue)."""
    x, w = _inputs(device, m, n, k, seed=3 * m + n + k)
    guard = torch.full((splits * m * n + 64,), -77.0, dtype=torch.float32, device=device)
    out = guard[: splits * m * n].view(splits, m, n).fill_(float("nan"))
    _hip.gemm_m128(out, x, w, splits=splits, epilogue=_hip.GEMM_PARTIALS)
    torch.cuda.synchronize()
    assert (guard[splits * m * n :] == -77.0).all()
    span = k // splits
    for s in range(splits):
        part = x[:, s * span : (s + 1) * span].float() @ w[:, s * span : (s + 1) * span].float().t()
        scale = part.abs().max().item()
        # fp32 accumulation of the same products in another order
        assert (out[s] - part).abs().max().item() <= 2e-6 * scale + 1e-7
    if splits == 1:
        half = torch.empty((m, n), dtype=torch.float16, device=device)
        _hip.gemm_m128(half, x, w, epilogue=_hip.GEMM_HALF)
        fused = torch.empty((m, n // 2), dtype=torch.float16, device=device)
        _hip.gemm_m128(fused, x, w, epilogue=_hip.GEMM_SWIGLU)
        separate = torch.empty_like(fused)
        _hip.silu_mul(separate, half)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(half), _bits(out[0].half()))
        assert np.array_equal(_bits(fused), _bits(separate))


# (n, k, splits): K ranges of one to three units (fewer than waves); short splits in several rounds; 48-row W
# tiles of every epilogue that end inside a tile, at one and at two rounds; columns where
# 64-row tiles of all rows take one round and 48-row tiles do not.
FORM_SHAPES = [(64, 64, 1), (96, 192, 1), (1024, 1024, 8), (512, 512, 8), (4096, 512, 8), (11296, 256, 1), (20480, 320, 1), (14336, 256, 1), (3104, 1536, 4)]


@pytest.mark.parametrize("m", [16, 17, 32, 33, 40, 48, 49, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("n,k,splits", FORM_SHAPES)
def test_gemm_forms(device, m, n, k, splits):
    """Shapes on either side of the choice between the kernel's forms: partials against float64 split
    by split, nothing written past the output, and with one split the same sums under every
    epilogue."""
    x, w = _inputs(device, m, n, k, seed=7 * m + n + k)
    guard = torch.full((splits * m * n + 64,), -77.0, dtype=torch.float32, device=device)
    out = guard[: splits * m * n].view(splits, m, n).fill_(float("nan"))
    _hip.gemm_m128(out, x, w, splits=splits, epilogue=_hip.GEMM_PARTIALS)
    torch.cuda.synchronize()
    assert (guard[splits * m * n :] == -77.0).all()
    span = k // splits
    for s in range(splits):
        xs, ws = x[:, s * span : (s + 1) * span].double(), w[:, s * span : (s + 1) * span].double()
        bound = span * 2.0**-24 * (xs.abs() @ ws.abs().t())  # `span` exact products added in fp32, in any order
        assert ((out[s].double() - xs @ ws.t()).abs() <= bound).all()
    if splits == 1:
        half = torch.empty((m, n), dtype=torch.float16, device=device)
        _hip.gemm_m128(half, x, w, epilogue=_hip.GEMM_HALF)
        assert np.array_equal(_bits(half), _bits(out[0].half()))
        if n % 64 == 0:
            fused = torch.full((m * (n // 2) + 64,), -77.0, dtype=torch.float16, device=device)
            _hip.gemm_m128(fused[: m * (n // 2)].view(m, n // 2), x, w, epilogue=_hip.GEMM_SWIGLU)
            separate = torch.empty((m, n // 2), dtype=torch.float16, device=device)
            _hip.silu_mul(separate, half)
            torch.cuda.synchronize()
            assert (fused[m * (n // 2) :] == -77.0).all()
            assert np.array_equal(_bits(fused[: m * (n // 2)]), _bits(separate.view(-1)))


@pytest.mark.parametrize("epilogue", [_hip.GEMM_PARTIALS, _hip.GEMM_HALF])
def test_gemm_of_the_longest_k(device, epilogue):
    """K past the streams' 32-bit row offsets (2^24), few columns: small integers in a few columns of K
    at both ends and across the limit, so that every sum is exact."""
    m, n, k = 17, 32, (1 << 24) + 64
    columns = torch.tensor([0, 63, 64, (1 << 23) + 5, (1 << 24) - 1, 1 << 24, (1 << 24) + 1, k - 1], device=device)
    gen = torch.Generator(device=device).manual_seed(1)
    few_x = torch.randint(-4, 5, (m, len(columns)), device=device, generator=gen).half()
    few_w = torch.randint(-4, 5, (n, len(columns)), device=device, generator=gen).half()
    x, w = (torch.zeros((rows, k), dtype=torch.float16, device=device) for rows in (m, n))
    x[:, columns], w[:, columns] = few_x, few_w
    expected = few_x.double() @ few_w.double().T
    out = torch.full((1, m, n) if epilogue == _hip.GEMM_PARTIALS else (m, n), float("nan"), device=device,
                     dtype=torch.float32 if epilogue == _hip.GEMM_PARTIALS else torch.float16)
    _hip.gemm_m128(out, x, w, epilogue=epilogue)
    torch.cuda.synchronize()
    assert torch.equal(out.view(m, n).double(), expected)


@pytest.mark.parametrize("rows,full", [(1, 64), (16, 64), (17, 64), (33, 64), (48, 64), (49, 64), (65, 128), (80, 128), (81, 128), (97, 128)])
def test_decoder_projections_do_not_depend_on_the_batch(device, rows, full):
    """The projections a decode step issues, at its split counts: a row has the same bits in every batch
    of 1 to 64 rows, and in every batch of 65 to 128 (between the two the sums are in another order)."""
    gen = torch.Generator(device=device).manual_seed(rows)

    def weight(n, k):
        return (torch.randn((n, k), device=device, generator=gen) * 0.02).half()

    fewer = 2 if rows <= dec.GEMM_FEW_ROWS else 1
    x = torch.randn((full, 2048), device=device, generator=gen).half()
    wide = torch.randn((full, 5632), device=device, generator=gen).half()
    products = [
        (x, weight(2560, 2048), lambda t, w: dec._qkv_projection(t, w)),
        (x, weight(2048, 2048), lambda t, w: dec._linear_parts(t, w, dec.O_PROJ_SPLITS // fewer)),
        (wide, weight(2048, 5632), lambda t, w: dec._linear_parts(t, w, dec.DOWN_SPLITS // fewer)),
        (x, weight(11264, 2048), lambda t, w: dec._swiglu(t, w)),
    ]
    for inputs, w, product in products:
        some, all_rows = product(inputs[:rows].contiguous(), w), product(inputs, w)
        assert some.shape[:-2] == all_rows.shape[:-2]
        assert np.array_equal(_bits(some), _bits(all_rows[..., :rows, :]))


# --- pc_gemm_rows (a prompt's rows) -----------------------------------------------------------

# (n, k, splits, rows): every tile shape of the dispatch under every epilogue that reaches it (64 x 64,
# 128 x 64, 128 x 128, 128 x 192; SwiGLU 48, 96 and 128 output columns, and 96 on two stages; the
# streams of an unsplit product of few columns), rows one short of, at and one past a tile, column
# counts that end inside a tile, fewer K stages than the ring has, and the decoder's own shapes.
ROWS_SHAPES = [
    (64, 64, 1, (1, 63, 64, 65, 200)),
    (352, 128, 1, (129, 255)),
    (2560, 2048, 2, (129, 192, 256, 333)),
    (2048, 5632, 4, (129, 300, 513)),
    (2080, 1408, 2, (641, 1025)),
    (11264, 256, 1, (129, 300, 600, 700)),
    (2048, 2048, 1, (257, 288, 289, 385, 512, 513, 897, 1023, 1024, 1025)),
    (2560, 2048, 1, (145, 289, 769, 1536, 1537)),
    (2048, 5632, 2, (769, 1024)),
    (11264, 2048, 1, (256, 257, 513, 640, 641, 1409)),
]


@pytest.mark.parametrize("n,k,splits,m", [(n, k, s, m) for n, k, s, rows in ROWS_SHAPES for m in rows])
def test_gemm_rows_tiles(device, m, n, k, splits):
    """Partials against float64 split by split, nothing written past the output; with one split the
    fp16 epilogue bit equal to the rounded partials, and SwiGLU bit equal to pc_silu_mul of its
    two projections (its tiles may differ, the K order does not)."""
    x, w = _inputs(device, m, n, k, seed=5 * m + n + k)
    guard = torch.full((splits * m * n + 64,), -77.0, dtype=torch.float32, device=device)
    out = guard[: splits * m * n].view(splits, m, n).fill_(float("nan"))
    _hip.gemm_rows(out, x, w, splits=splits, epilogue=_hip.GEMM_PARTIALS)
    torch.cuda.synchronize()
    assert (guard[splits * m * n :] == -77.0).all()
    span = k // splits
    for s in range(splits):
        xs, ws = x[:, s * span : (s + 1) * span].double(), w[:, s * span : (s + 1) * span].double()
        # `span` exact products added in fp32, whatever the order: each of at most `span`
        # additions rounds by 2^-24 of a partial sum no larger than the sum of magnitudes.
        bound = span * 2.0**-24 * (xs.abs() @ ws.abs().t())
        assert ((out[s].double() - xs @ ws.t()).abs() <= bound).all()
    if splits == 1:
        half = torch.empty((m, n), dtype=torch.float16, device=device)
        _hip.gemm_rows(half, x, w, epilogue=_hip.GEMM_HALF)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(half), _bits(out[0].half()))
        if n % 64 == 0:
            fused = torch.full((m * (n // 2) + 64,), -77.0, dtype=torch.float16, device=device)
            _hip.gemm_rows(fused[: m * (n // 2)].view(m, n // 2), x, w, epilogue=_hip.GEMM_SWIGLU)
            separate = torch.empty((m, n // 2), dtype=torch.float16, device=device)
            _hip.silu_mul(separate, half)
            torch.cuda.synchronize()
            assert (fused[m * (n // 2) :] == -77.0).all()
            assert np.array_equal(_bits(fused[: m * (n // 2)]), _bits(separate.view(-1)))


# --- the split-K consumers' instances (1, 2, 4, 8 and any other split count; row lengths) ------


@pytest.mark.parametrize("splits", [1, 2, 3, 4, 6, 8, 9])
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 504), (5, 2048), (2, 2056), (2, 4096), (3, 4104), (2, 5632), (2, 6152), (3, 8192)])
def test_add_rms_norm_instances(device, rows, width, splits):
    """Parts bit equal to the fp16 path fed their rounded sum, and that path against float64:
    the residual exact, the output within its two fp16 roundings."""
    gen = torch.Generator(device=device).manual_seed(rows * width + splits)
    parts = torch.randn((splits, rows, width), device=device, generator=gen) * 0.3
    hidden = torch.randn((rows, width), device=device, generator=gen).half()
    weight = (1 + 0.1 * torch.randn(width, device=device, generator=gen)).half()
    delta = _sum_in_split_order(parts)
    results = []
    for given in (parts, delta, None):
        guard = torch.full((2, rows * width + 32), 7.0, dtype=torch.float16, device=device)
        h, out = guard[0, : rows * width].view(rows, width), guard[1, : rows * width].view(rows, width)
        h.copy_(hidden)
        (_hip.add_rms_norm_parts if given is parts else _hip.add_rms_norm)(out, h, given, weight, dec.RMS_EPS)
        torch.cuda.synchronize()
        assert (guard[:, rows * width :] == 7.0).all()
        results.append((h, out))
        summed = hidden if given is None else (hidden.float() + delta.float()).half()
        assert torch.equal(h, summed)
        exact = summed.double() * torch.rsqrt(summed.double().square().mean(-1, keepdim=True) + dec.RMS_EPS) * weight.double()
        # two roundings to fp16 (the second may be of a value rounded first), fp32 elsewhere
        assert ((out.double() - exact).abs() <= exact.abs() * (2.0**-10 + 2.0**-18) + 2.0**-23).all()
    assert np.array_equal(_bits(results[0][0]), _bits(results[1][0]))
    assert np.array_equal(_bits(results[0][1]), _bits(results[1][1]))


@pytest.mark.parametrize("splits", [1, 2, 3, 4, 8, 9])
@pytest.mark.parametrize("outputs", ["pool", "contiguous", "both"])
def test_rope_kv_append_instances(device, splits, outputs):
    """Parts bit equal to the fp16 path (checked against the oracle elsewhere) with each set of
    outputs; slots of -1 and past the pool, and their neighbours' rows, stay untouched."""
    tokens, blocks = 9, 4
    gen = torch.Generator(device=device).manual_seed(splits)
    parts = torch.randn((splits, tokens, 2560), device=device, generator=gen) * 0.5
    positions = torch.randint(0, 2048, (tokens,), device=device, generator=gen)
    slots = torch.randperm(blocks * 16, device=device, generator=gen)[:tokens]
    slots[2], slots[5] = -1, blocks * 16
    table = dec.rope_table(device)
    results = []
    for use_parts in (False, True):
        pool = torch.full((22, 2, blocks, 16, 4, 64), 7.0, dtype=torch.float16, device=device)
        query = torch.empty(tokens, 32, 64, dtype=torch.float16, device=device)
        keys = torch.full((tokens, 4, 64), 7.0, dtype=torch.float16, device=device)
        values = torch.full_like(keys, 7.0)
        given = {} if outputs == "pool" else {"key_out": keys, "value_out": values}
        if outputs != "contiguous":
            given.update(pool=pool, layer=21, slot_mapping=slots)
        if use_parts:
            _hip.rope_kv_append_parts(query, parts, positions, table, **given)
        else:
            _hip.rope_kv_append(query, _sum_in_split_order(parts), positions, table, **given)
        torch.cuda.synchronize()
        results.append((query, keys, values, pool))
        written = torch.zeros(blocks * 16, dtype=torch.bool, device=device)
        if outputs != "contiguous":
            written[slots[(slots >= 0) & (slots < blocks * 16)]] = True
        assert (pool[:21] == 7.0).all() and (pool[21].view(2, -1, 4, 64)[:, ~written] == 7.0).all()
        if outputs == "both":
            kept = (slots >= 0) & (slots < blocks * 16)
            assert torch.equal(pool[21, 0].view(-1, 4, 64)[slots[kept]], keys[kept])
            assert torch.equal(pool[21, 1].view(-1, 4, 64)[slots[kept]], values[kept])
    for a, b in zip(*results):
        assert np.array_equal(_bits(a), _bits(b))


# --- pc_qkv_rope_append (the q|k|v projection with RoPE and the KV write as its epilogue) ------


def _qkv_inputs(device, m, k, seed):
    gen = torch.Generator(device=device).manual_seed(seed)
    x = torch.randn((m, k), device=device, generator=gen).half()
    w = (0.05 * torch.randn((2560, k), device=device, generator=gen)).half()
    positions = torch.randint(0, 2048, (m,), device=device, generator=gen)
    blocks = m // 16 + 2
    slots = torch.randperm(blocks * 16, device=device, generator=gen)[:m].contiguous()
    return x, w, positions, slots, blocks


# The edges of the forms' rows: 16 rows; then 48 per X tile of 16, up to 192; 288; and one workgroup
# per CU of 64 x 64, 128 x 64 and 128 x 128 tiles.
@pytest.mark.parametrize("m", [1, 7, 16, 17, 48, 49, 96, 97, 144, 145, 192, 193, 288, 289, 384, 385, 768, 769, 1536, 1537])
@pytest.mark.parametrize("k", [64, 320, 2048])
def test_qkv_rope_append_forms(device, m, k):
    """Every output against float64: the projection within its fp32 accumulation (k 2^-24 of the
    sum of magnitudes) and one rounding, the rotation within its three; pool rows equal to the
    contiguous ones; rows of tokens without a slot, and memory past the outputs, untouched."""
    x, w, positions, slots, blocks = _qkv_inputs(device, m, k, 7 * m + k)
    dropped = torch.arange(m, device=device) % 5 == 3
    slots[dropped] = torch.where(torch.arange(m, device=device)[dropped] % 2 == 0, -1, blocks * 16)
    table = dec.rope_table(device)
    pool = torch.full((22, 2, blocks, 16, 4, 64), 7.0, dtype=torch.float16, device=device)
    guard = torch.full((3, m * 2048 + 64), 7.0, dtype=torch.float16, device=device)
    query = guard[0, : m * 2048].view(m, 32, 64)
    key, value = (guard[i, : m * 256].view(m, 4, 64) for i in (1, 2))
    _hip.qkv_rope_append(query, x, w, positions, table, key_out=key, value_out=value, pool=pool, layer=3, slot_mapping=slots)
    torch.cuda.synchronize()
    assert (guard[0, m * 2048 :] == 7.0).all() and (guard[1:, m * 256 :] == 7.0).all()
    flat = pool[3].view(2, -1, 4, 64)
    kept = slots[~dropped]
    assert torch.equal(flat[0][kept], key[~dropped]) and torch.equal(flat[1][kept], value[~dropped])
    untouched = torch.ones(blocks * 16, dtype=torch.bool, device=device)
    untouched[kept] = False
    assert (flat[:, untouched] == 7.0).all() and (pool[:3] == 7.0).all() and (pool[4:] == 7.0).all()

    y = x.double() @ w.double().T
    delta = k * 2.0**-24 * (x.double().abs() @ w.double().abs().T)
    delta = delta + 2.0**-11 * (y.abs() + delta) + 2.0**-25  # one rounding to fp16
    heads, errors = y.view(m, 40, 64), delta.view(m, 40, 64)
    c, s = (table[positions, i].double()[:, None] for i in (0, 1))
    lo, hi = heads[:, :36, :32], heads[:, :36, 32:]
    elo, ehi = errors[:, :36, :32], errors[:, :36, 32:]
    got = torch.cat((query, key), 1).double()
    for part, a, b, ea, eb, sign in ((got[..., :32], lo, hi, elo, ehi, -1), (got[..., 32:], hi, lo, ehi, elo, 1)):
        exact = a * c + sign * b * s
        moved = ea * c.abs() + eb * s.abs()
        magnitudes = (a * c).abs() + (b * s).abs() + moved
        bound = moved + 2.0**-11 * 2 * magnitudes * (1 + 2.0**-10) + 3 * 2.0**-25
        assert ((part - exact).abs() <= bound).all()
    assert ((value.double() - heads[:, 36:]).abs() <= errors[:, 36:]).all()


@pytest.mark.parametrize("m", [1, 16, 17, 48, 49, 64])
def test_qkv_rope_append_adds_as_the_projection_with_one_split(device, m):
    """The same bits as pc_gemm_m128 with one split and pc_rope_kv_append_parts, which eager decode
    runs; each output left out in turn; a position past the table gives NaN rows (v kept) and
    no pool write."""
    x, w, positions, slots, blocks = _qkv_inputs(device, m, 2048, m)
    positions[m // 2] = 2048
    table = dec.rope_table(device)
    parts = torch.empty((1, m, 2560), dtype=torch.float32, device=device)
    _hip.gemm_m128(parts, x, w)
    for outputs in ("pool", "contiguous", "both"):
        results = []
        for fused in (False, True):
            pool = torch.full((22, 2, blocks, 16, 4, 64), 7.0, dtype=torch.float16, device=device)
            query = torch.empty(m, 32, 64, dtype=torch.float16, device=device)
            key = torch.full((m, 4, 64), 7.0, dtype=torch.float16, device=device)
            value = torch.full_like(key, 7.0)
            given = {} if outputs == "pool" else {"key_out": key, "value_out": value}
            if outputs != "contiguous":
                given.update(pool=pool, layer=0, slot_mapping=slots)
            if fused:
                _hip.qkv_rope_append(query, x, w, positions, table, **given)
            else:
                _hip.rope_kv_append_parts(query, parts, positions, table, **given)
            torch.cuda.synchronize()
            assert query[m // 2].isnan().all()
            results.append((query, key, value, pool))
        for a, b in zip(*results):
            assert np.array_equal(_bits(a), _bits(b))


# Either side of the row tiles of the stream form up to 288 rows, then of the tile forms, then the library.
@pytest.mark.parametrize("m", [65, 97, 128, 129, 144, 145, 192, 193, 256, 257, 288, 289, 384, 385, 600, 768, 769, 1536, 1537])
def test_eager_projection_has_the_bits_of_the_fused_launch(device, m):
    """The q|k|v projection of eager decode, rotated and written by the RoPE launch, against
    pc_qkv_rope_append (what a DecodeGraph issues): the same bits at every row count."""
    x, w, positions, slots, blocks = _qkv_inputs(device, m, 2048, m)
    table = dec.rope_table(device)
    results = []
    for fused in (False, True):
        pool = torch.full((22, 2, blocks, 16, 4, 64), 7.0, dtype=torch.float16, device=device)
        query = torch.empty(m, 32, 64, dtype=torch.float16, device=device)
        outputs = {"pool": pool, "layer": 1, "slot_mapping": slots}
        if fused:
            dec._qkv_rope(query, x, w, positions, table, **outputs)
        else:
            qkv = dec._qkv_projection(x, w)
            (_hip.rope_kv_append_parts if qkv.ndim == 3 else _hip.rope_kv_append)(query, qkv, positions, table, **outputs)
        torch.cuda.synchronize()
        results.append((query, pool))
    for a, b in zip(*results):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
