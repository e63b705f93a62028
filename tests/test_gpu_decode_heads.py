"""GPU parity of decode on head_dim 64 and on GQA ratios that are no power of
two: MFMA instances whose probabilities, weights and V enter PV in fp32.

Tolerance: the kernel's own error is that of fp32 sums (2e-5 of the result's
norm), so the distance from the oracle is that of rounding the oracle's result
to the type, and no more."""
import pytest
import torch

from oracle.attention import paged_decode_ref
from oracle.fog import fog_bias
from tests.exact64 import attend64, close_to_rounding, paged
from tests.inputs import decode_case, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def mfma_only(monkeypatch):
    """A call that would run on the generic kernel is an error in this file."""
    monkeypatch.setenv("KESSIE_REQUIRE_MFMA", "1")

DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _check(out, q, pool, table, lens, vs, bias, window, dtype):
    for i, n in enumerate(lens):
        if n == 0:
            assert not out[i].any()
            continue
        row = table[i].long()[: -(-n // pool.shape[1])].cpu()
        ref = paged_decode_ref(q[i:i + 1].cpu(), pool[row.to(pool.device)].cpu(), torch.arange(len(row)).int()[None],
                               torch.tensor([n]), None if vs is None else vs.view(-1, vs.shape[-1])[i % vs.shape[0]].cpu(),
                               None if bias is None else bias[i:i + 1].cpu(), window)
        err = (out[i:i + 1].double().cpu() - ref.double()).norm()
        rounding = (ref.to(dtype).double() - ref.double()).norm()
        assert err <= 1.05 * rounding + 2e-5 * ref.double().norm(), f"sequence {i} ({n} tokens): {err:.3e} {rounding:.3e}"


@pytest.mark.parametrize("hq,hkv,d,ctx,lens,page,window,fog,dt", [
    (32, 8, 64, 300, [300, 1, 15, 16, 17, 0, 64], 16, 0, "vscale", "bf16"),
    (3, 3, 64, 700, [700, 31], 32, 0, "none", "fp16"),             # an odd number of kv heads, larger pages
    (16, 1, 64, 5000, [5000], 16, 100, "bias", "bf16"),            # GQA 16, window, one sequence
    (14, 2, 64, 400, [400, 399], 64, 33, "both", "fp16"),          # GQA 7
    (24, 8, 128, 900, [900, 77, 16], 16, 0, "both", "bf16"),       # GQA 3
    (12, 1, 128, 2000, [2000, 5], 32, 500, "vscale", "fp16"),      # GQA 12
    (32, 8, 64, 9000, [9000] + [40 + 9 * i for i in range(30)], 16, 0, "bias", "bf16"),   # balanced splits
    (24, 8, 128, 9000, [9000] + [40 + 9 * i for i in range(15)], 16, 0, "vscale", "fp16"),
])
def test_decode_exact_p_shapes(dev, hq, hkv, d, ctx, lens, page, window, fog, dt):
    from kessie_amd import ops

    b, dtype = len(lens), DT[dt]
    q, pool, table, lens_d = decode_case(b, hq, hkv, d, ctx, page, dtype, dev, seed=51, ctx_lens=lens)
    vs = torch.rand(b, ctx, generator=gen(dev, 52), device=dev) if fog in ("vscale", "both") else None
    bias = fog_bias(ctx, 0.5, 0.5, {3, 17}, 0.1).to(dev).repeat(b, 1) if fog in ("bias", "both") else None
    out = torch.full_like(q, float("nan"))
    ops.fog_decode(q, pool, table, lens_d, ctx, fog_vscale=vs, fog_bias=bias, window=window, out=out)
    torch.cuda.synchronize()
    _check(out, q, pool, table, lens, vs, bias, window, dtype)


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (6, 2, 128)])
@pytest.mark.parametrize("lo,hi,vmul", [(1e4, 1e4, 1.0), (1e-6, 1e-6, 1e3), (1e-6, 1e4, 1.0), (-900.0, 900.0, 1.0)])
def test_decode_fp16_weights_of_any_magnitude(dev, hq, hkv, d, lo, hi, vmul):
    """V weights far from 1 (constant, or rising or changing sign along the context): p * w leaves fp16's range."""
    from kessie_amd import ops

    lens = [500, 33]
    q, pool, table, lens_d = decode_case(2, hq, hkv, d, 500, 16, torch.float16, dev, seed=53, ctx_lens=lens)
    pool, q = pool * vmul, q / vmul
    ramp = torch.linspace(0, 1, 500, device=dev)
    w = (lo + (hi - lo) * ramp if lo * hi < 0 else lo * (hi / lo) ** ramp).float().view(1, -1)
    out = ops.fog_decode(q, pool, table, lens_d, 500, fog_vscale=w.view(-1))
    _check(out, q, pool, table, lens, w, None, 0, torch.float16)


def test_decode_exact_p_invalid_page(dev):
    from kessie_amd import ops

    q, pool, table, lens = decode_case(2, 12, 4, 64, 200, 16, torch.bfloat16, dev, seed=54, ctx_lens=[200, 100])
    bad = table.clone()
    bad[0, 3], bad[1, 0] = -1, pool.shape[0]
    out = ops.fog_decode(q, pool, bad, lens, 200)
    hide = torch.zeros(2, 200, device=dev)  # their tokens contribute nothing
    hide[0, 48:64], hide[1, :16] = -float("inf"), -float("inf")
    _check(out, q, pool, table, [200, 100], None, hide, 0, torch.bfloat16)


SHAPES = pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (6, 2, 128)])


@SHAPES
@pytest.mark.parametrize("dt", ["fp16", "bf16"])
def test_decode_small_probabilities(dev, monkeypatch, hq, hkv, d, dt):
    """One key 12 above all others, with a small V (an attention sink): the result rests on probabilities of e^-12,
    which 16-bit operands of fp16's range hold to a part in 1,000 only.  (One split: the sink is every key's.)"""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_DECODE_WGS", "1")
    dtype, n = DT[dt], 4096
    k = torch.zeros(n, hkv, d, device=dev, dtype=dtype)
    k[5] = 12 / d ** 0.5
    v = (1 + 0.1 * torch.randn(n, hkv, d, generator=gen(dev, 61), device=dev)).to(dtype)
    v[5] = 2.0 ** -10
    q = torch.ones(1, hq, d, device=dev, dtype=dtype)
    pool, table, lens = paged(k, v)
    close_to_rounding(ops.fog_decode(q, pool, table, lens, n), attend64(q, k, v, n - 1), dtype)


@SHAPES
@pytest.mark.parametrize("where", ["faint", "window"])
def test_decode_fp16_one_large_weight(dev, hq, hkv, d, where):
    """A weight of 2^16 on a key whose probability is negligible, or that the window hides, costs the others nothing."""
    from kessie_amd import ops

    n, window = 700, 500 if where == "window" else 0
    k, v = (torch.randn(n, hkv, d, generator=gen(dev, 62 + i), device=dev).half() for i in (0, 1))
    q = torch.randn(1, hq, d, generator=gen(dev, 64), device=dev).half()
    w, bias = torch.ones(n, device=dev), torch.zeros(n, device=dev)
    w[190] = 2.0 ** 16
    if where == "faint":
        bias[190] = -60.0
    pool, table, lens = paged(k, v)
    out = ops.fog_decode(q, pool, table, lens, n, fog_vscale=w, fog_bias=bias, window=window)
    close_to_rounding(out, attend64(q, k, v, n - 1, w, bias, window), torch.float16)


@SHAPES
def test_decode_fp16_weights_under_a_mask(dev, hq, hkv, d):
    """Every key under a mask of -1e9: the splits, whose weights differ, still count alike."""
    from kessie_amd import ops

    n = 1000
    k = torch.zeros(n, hkv, d, device=dev, dtype=torch.float16)
    v = torch.randn(n, hkv, d, generator=gen(dev, 65), device=dev).half()
    q = torch.randn(1, hq, d, generator=gen(dev, 66), device=dev).half()
    w = torch.logspace(0, -4, n, device=dev)
    bias = torch.full((n,), -1e9, device=dev)
    pool, table, lens = paged(k, v)
    out = ops.fog_decode(q, pool, table, lens, n, fog_vscale=w, fog_bias=bias)
    close_to_rounding(out, attend64(q, k, v, n - 1, w, bias), torch.float16)


@SHAPES
@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("what", ["v", "-v", "weight", "hidden weight"])
def test_decode_infinities(dev, hq, hkv, d, dt, what):
    """An infinity in V or in a weight shows as an infinity where its key takes part, and not at all where its
    probability is zero."""
    from kessie_amd import ops

    dtype, n = DT[dt], 300
    k, v = (torch.randn(n, hkv, d, generator=gen(dev, 67 + i), device=dev).to(dtype) for i in (0, 1))
    q = torch.randn(1, hq, d, generator=gen(dev, 69), device=dev).to(dtype)
    w, bias = torch.ones(n, device=dev), torch.zeros(n, device=dev)
    if what.endswith("v"):
        v[130, :, 3] = float("-inf" if what == "-v" else "inf")
    else:
        w[130] = float("inf")
        if what == "hidden weight":
            bias[130] = -float("inf")
    pool, table, lens = paged(k, v)
    out = ops.fog_decode(q, pool, table, lens, n, fog_vscale=w, fog_bias=bias).double().cpu()
    ref = attend64(q, k, v, n - 1, w, bias)
    finite = ref.isfinite()
    assert finite.all() == (what == "hidden weight") and not ref.isnan().any()
    assert torch.equal(out[~finite], ref[~finite])
    close_to_rounding(torch.where(finite, out, 0.0), torch.where(finite, ref, 0.0), dtype)
