"""GPU parity of chunked prefill on head_dim 64 and on GQA ratios that are no
power of two: MFMA instances whose probabilities enter PV as two bf16 operands.

Tolerance: the kernel's own error is that of fp32 sums and of probabilities to
2^-16 (2e-5 of the result's norm), so the distance from the oracle is that of
rounding the oracle's result to the type, and no more."""
import pytest
import torch

from oracle.attention import paged_prefill_ref
from oracle.fog import fog_bias
from tests.exact64 import attend64, close_to_rounding, paged
from tests.inputs import decode_case, gen, randn

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def mfma_only(monkeypatch):
    """A call that would run on the generic kernel is an error in this file."""
    monkeypatch.setenv("KESSIE_REQUIRE_MFMA", "1")

DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _close(out, ref, dtype):
    err = (out.double().cpu() - ref.double()).norm()
    rounding = (ref.to(dtype).double() - ref.double()).norm()
    assert err <= 1.02 * rounding + 2e-5 * ref.double().norm(), f"error {err:.3e}, rounding alone {rounding:.3e}"


def _fog(kind, b, ctx, dev):
    vs = torch.rand(b, ctx, generator=gen(dev, 5), device=dev) if kind in ("vscale", "both") else None
    bias = fog_bias(ctx, 0.5, 0.5, {3, 17}, 0.1).to(dev).repeat(b, 1) if kind in ("bias", "both") else None
    return vs, bias


@pytest.mark.parametrize("hq,hkv,d,c,ctxs,page,window,fog,dt,splits", [
    (32, 8, 64, 70, [200, 70], 16, 0, "vscale", "bf16", 0),    # a query tile and six rows
    (8, 8, 64, 256, [256], 16, 0, "none", "fp16", 0),          # one query tile, fresh prompt
    (32, 8, 64, 1, [1, 64, 65], 16, 0, "both", "bf16", 0),     # one query, edges of a key tile
    (32, 4, 64, 33, [1500], 32, 100, "bias", "fp16", 3),       # larger pages, window, key splits
    (32, 8, 64, 1100, [1100], 16, 0, "bias", "bf16", 1),       # several rounds, longest tiles first
    (24, 8, 128, 86, [300, 86], 16, 0, "vscale", "fp16", 0),   # GQA 3: 85 positions a workgroup
    (40, 8, 128, 52, [900, 31], 16, 64, "both", "bf16", 2),    # GQA 5, splits, a chunk longer than its context
    (28, 4, 64, 37, [400], 32, 0, "vscale", "fp16", 0),        # GQA 7, head_dim 64
    (12, 1, 128, 22, [1000], 64, 0, "none", "bf16", 0),        # GQA 12: 21 positions a workgroup
])
def test_prefill_exact_p_shapes(dev, monkeypatch, hq, hkv, d, c, ctxs, page, window, fog, dt, splits):
    from kessie_amd import ops

    if splits:
        monkeypatch.setenv("KESSIE_PREFILL_SPLITS", str(splits))
    b, mx, dtype = len(ctxs), max(ctxs), DT[dt]
    _, pool, table, lens = decode_case(b, hq, hkv, d, mx, page, dtype, dev, seed=7, ctx_lens=ctxs)
    q = randn((b, c, hq, d), dtype, dev, 8)
    vs, bias = _fog(fog, b, mx, dev)
    out = torch.full_like(q, float("nan"))
    ops.fog_prefill(q, pool, table, lens, mx, fog_vscale=vs, fog_bias=bias, window=window, out=out)
    torch.cuda.synchronize()
    for i, n in enumerate(ctxs):
        live = max(0, c - n)  # queries before position 0 see no key: zeros
        assert not out[i, :live].any()
        ref = paged_prefill_ref(q[i:i + 1, live:].cpu(), pool.cpu(), table[i:i + 1].cpu(), lens[i:i + 1].cpu(),
                                None if vs is None else vs[i:i + 1].cpu(),
                                None if bias is None else bias[i:i + 1].cpu(), window)
        _close(out[i:i + 1, live:], ref, dtype)


@pytest.mark.parametrize("hq,hkv,d,page", [(32, 8, 64, 16), (24, 8, 128, 32), (32, 8, 128, 16)])
def test_prefill_batch_matches_per_sequence(dev, monkeypatch, hq, hkv, d, page):
    """One launch over ragged chunks equals the per-sequence launches bit for bit (one key split)."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", "1")
    chunks, ctxs = [90, 1, 33, 260], [200, 64, 33, 700]
    _, pool, table, lens = decode_case(4, hq, hkv, d, max(ctxs), page, torch.bfloat16, dev, seed=17, ctx_lens=ctxs)
    starts = [0, 90, 91, 124, 384]
    qsl = torch.tensor(starts, dtype=torch.int32, device=dev)
    q = randn((384, hq, d), torch.bfloat16, dev, 18)
    bias = fog_bias(max(ctxs), 0.5, 0.5, {3}, 0.1).to(dev).repeat(4, 1)
    out = torch.full_like(q, float("nan"))
    listed = d == 128 and (hq // hkv) & (hq // hkv - 1) == 0
    assert ops.fog_prefill_varlen(q, qsl, 260, pool, table, lens, max(ctxs), fog_bias=bias, out=out) == listed
    assert ops.fog_prefill_batch(q, qsl, 260, pool, table, lens, max(ctxs), fog_bias=bias, out=out)
    for i in range(4):
        s, e = starts[i], starts[i + 1]
        one = ops.fog_prefill(q[s:e][None], pool, table[i:i + 1], lens[i:i + 1], max(ctxs), fog_bias=bias[i:i + 1])
        assert torch.equal(out[s:e], one[0]), i


@pytest.mark.parametrize("hq,hkv,d,splits", [(8, 2, 64, 1), (8, 2, 64, 3), (6, 2, 128, 1)])
@pytest.mark.parametrize("lo,hi,vmul", [(1e4, 1e4, 1.0), (1e-6, 1e-6, 1e3), (1e-6, 1e4, 1.0), (-900.0, 900.0, 1.0)])
def test_prefill_fp16_weights_of_any_magnitude(dev, monkeypatch, hq, hkv, d, splits, lo, hi, vmul):
    """V weights far from 1 (constant, or rising or changing sign along the context): p * w leaves fp16's range."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", str(splits))
    _, pool, table, lens = decode_case(1, hq, hkv, d, 500, 16, torch.float16, dev, seed=9, ctx_lens=[500])
    pool = pool * vmul
    q = randn((1, 90, hq, d), torch.float16, dev, 10) / vmul
    ramp = torch.linspace(0, 1, 500, device=dev)
    w = (lo + (hi - lo) * ramp if lo * hi < 0 else lo * (hi / lo) ** ramp).float().view(1, -1)
    out = ops.fog_prefill(q, pool, table, lens, 500, fog_vscale=w)
    ref = paged_prefill_ref(q.cpu(), pool.cpu(), table.cpu(), lens.cpu(), w.cpu(), None, 0)
    _close(out, ref, torch.float16)


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (8, 2, 128), (6, 2, 128)])
@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, torch.finfo(torch.bfloat16).min, -1e38, -1e9, -65504.0,
                                 -float("inf")])
@pytest.mark.parametrize("splits", [1, 2])
def test_prefill_bias_masks(dev, monkeypatch, hq, hkv, d, low, splits):
    """Keys hidden by the lowest values a mask holds, and with the finite ones a sequence whose keys are all hidden
    alike."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", str(splits))
    _, pool, table, lens = decode_case(2, hq, hkv, d, 300, 16, torch.bfloat16, dev, seed=19, ctx_lens=[300, 300])
    q = randn((2, 70, hq, d), torch.bfloat16, dev, 20)
    bias = fog_bias(300, 0.5, 0.5, {3}, 0.1).to(dev).repeat(2, 1)
    bias[0, 5:100] = low
    if -float("inf") < low < -65504.0:  # (fp32 spacing there is above any score: all keys alike)
        bias[1] = low
    out = ops.fog_prefill(q, pool, table, lens, 300, fog_bias=bias)
    ref = paged_prefill_ref(q.cpu(), pool.cpu(), table.cpu(), lens.cpu(), None, bias.cpu(), 0)
    diff = (out.float().cpu() - ref).abs()
    assert bool((diff <= 2e-2 + 1e-2 * ref.abs()).all()), f"max diff {diff.max().item():.3e}"


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (8, 2, 128), (6, 2, 128)])
def test_prefill_large_common_bias(dev, hq, hkv, d):
    """A bias of -30,000 on every key leaves the softmax as it is but for one rounding of each logit, in base 2 to
    2^-9 at most: p to ln 2 * 2^-9 = 1.4e-3, independently from key to key."""
    from kessie_amd import ops

    n, c = 600, 90
    k, v = (torch.randn(n, hkv, d, generator=gen(dev, 31 + i), device=dev).half() for i in (0, 1))
    q = torch.randn(1, c, hq, d, generator=gen(dev, 33), device=dev).half()
    bias = torch.full((n,), -30000.0, device=dev)
    pool, table, lens = paged(k, v)
    out = ops.fog_prefill(q, pool, table, lens, n, fog_bias=bias)
    close_to_rounding(out[0], attend64(q[0], k, v, n - c), torch.float16, own=1.4e-3)


SHAPES = pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (6, 2, 128)])


def _kvq(dev, n, c, hq, hkv, d, dtype, seed):
    k, v = (torch.randn(n, hkv, d, generator=gen(dev, seed + i), device=dev).to(dtype) for i in (0, 1))
    return k, v, torch.randn(c, hq, d, generator=gen(dev, seed + 2), device=dev).to(dtype)


@SHAPES
@pytest.mark.parametrize("dt", ["fp16", "bf16"])
def test_prefill_small_probabilities(dev, monkeypatch, hq, hkv, d, dt):
    """One key 12 above all others, with a small V (an attention sink): the result rests on probabilities of e^-12,
    which 16-bit operands of fp16's range hold to a part in 1,000 only."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", "1")
    dtype, n, c = DT[dt], 4096, 70
    k = torch.zeros(n, hkv, d, device=dev, dtype=dtype)
    k[5] = 12 / d ** 0.5
    v = (1 + 0.1 * torch.randn(n, hkv, d, generator=gen(dev, 61), device=dev)).to(dtype)
    v[5] = 2.0 ** -10
    q = torch.ones(c, hq, d, device=dev, dtype=dtype)
    pool, table, lens = paged(k, v)
    close_to_rounding(ops.fog_prefill(q[None], pool, table, lens, n)[0], attend64(q, k, v, n - c), dtype)


@SHAPES
@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("where", ["faint", "window", "future"])
def test_prefill_fp16_one_large_weight(dev, monkeypatch, hq, hkv, d, splits, where):
    """A weight of 2^16 on a key whose probability is negligible, or that the window or the causal mask hides from
    some rows, costs those rows' other keys nothing."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", str(splits))
    n, c, window, at = 700, 64, 0, 190
    if where == "window":
        window, at = 100, 569  # the chunk's first 32 rows see it
    elif where == "future":
        at = 690  # the last ten rows see it, in the others' tile
    k, v, q = _kvq(dev, n, c, hq, hkv, d, torch.float16, 71)
    w, bias = torch.ones(n, device=dev), torch.zeros(n, device=dev)
    w[at] = 2.0 ** 16
    v[at] *= 2.0 ** -10  # (results of the rows that see it stay in fp16's range)
    if where == "faint":
        bias[at] = -60.0
    pool, table, lens = paged(k, v)
    out = ops.fog_prefill(q[None], pool, table, lens, n, fog_vscale=w, fog_bias=bias, window=window)[0]
    ref = attend64(q, k, v, n - c, w, bias, window)
    for r in range(c):
        close_to_rounding(out[r], ref[r], torch.float16)


@SHAPES
@pytest.mark.parametrize("splits", [1, 3])
def test_prefill_fp16_weights_under_a_mask(dev, monkeypatch, hq, hkv, d, splits):
    """Every key under a mask of -1e9: key tiles and splits, whose weights differ, still count alike."""
    from kessie_amd import ops

    monkeypatch.setenv("KESSIE_PREFILL_SPLITS", str(splits))
    n, c = 1000, 40
    k, v, q = _kvq(dev, n, c, hq, hkv, d, torch.float16, 75)
    k.zero_()
    w, bias = torch.logspace(-4, 0, n, device=dev), torch.full((n,), -1e9, device=dev)
    pool, table, lens = paged(k, v)
    out = ops.fog_prefill(q[None], pool, table, lens, n, fog_vscale=w, fog_bias=bias)[0]
    close_to_rounding(out, attend64(q, k, v, n - c, w, bias), torch.float16)


@SHAPES
@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("what", ["v", "-v", "weight", "hidden weight"])
def test_prefill_infinities(dev, hq, hkv, d, dt, what):
    """An infinity in V or in a weight shows as an infinity where its key takes part, and an infinite weight not at
    all where the probability is zero."""
    from kessie_amd import ops

    dtype, n, c = DT[dt], 300, 60
    k, v, q = _kvq(dev, n, c, hq, hkv, d, dtype, 78)
    w, bias = torch.ones(n, device=dev), torch.zeros(n, device=dev)
    if what.endswith("v"):
        v[130, :, 3] = float("-inf" if what == "-v" else "inf")
    else:
        w[130] = float("inf")
        if what == "hidden weight":
            bias[130] = -float("inf")
    pool, table, lens = paged(k, v)
    out = ops.fog_prefill(q[None], pool, table, lens, n, fog_vscale=w, fog_bias=bias)[0].double().cpu()
    ref = attend64(q, k, v, n - c, w, bias)
    finite = ref.isfinite()
    assert finite.all() == (what == "hidden weight") and not ref.isnan().any()
    assert torch.equal(out[~finite], ref[~finite])
    close_to_rounding(torch.where(finite, out, 0.0), torch.where(finite, ref, 0.0), dtype)


@SHAPES
def test_prefill_pages_before_the_window(dev, hq, hkv, d):
    """Pages wholly before the window may be anyone's, also where the first key tile covers them."""
    from kessie_amd import ops

    n, c, window = 300, 20, 40  # keys from 241 on; the tile begins at 192
    k, v, q = _kvq(dev, n, c, hq, hkv, d, torch.bfloat16, 82)
    pool, table, lens = paged(k, v)
    pool[:15] = float("nan")
    out = ops.fog_prefill(q[None], pool, table, lens, n, window=window)[0]
    close_to_rounding(out, attend64(q, k, v, n - c, window=window), torch.bfloat16)


def test_prefill_small_workspace(dev):
    """A workspace that the generic kernel, which ran head_dim 64 before, does without or is refused for."""
    from kessie_amd import ops

    tiny = torch.empty(16, dtype=torch.uint8, device=dev)
    for c, n, refused in ((512, 4096, False), (64, 512, True)):
        k, v, q = _kvq(dev, n, c, 32, 8, 64, torch.bfloat16, 85)
        pool, table, lens = paged(k, v)
        if refused:
            with pytest.raises(RuntimeError, match="workspace"):
                ops.fog_prefill(q[None], pool, table, lens, n, ws=tiny)
        else:
            out = ops.fog_prefill(q[None], pool, table, lens, n, ws=tiny)
            close_to_rounding(out[0, :40], attend64(q[:40], k[:n - c + 40], v[:n - c + 40], n - c), torch.bfloat16)
