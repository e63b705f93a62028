"""GPU parity of the dense launchers where H * N is no multiple of 16: the MFMA
instances whose probabilities keep fp32 precision.

Tolerance: the kernel's own error is that of fp32 sums (2e-5 of the result's
norm), so the distance from the oracle is that of rounding the oracle's result
to fp16, and no more."""
import pytest
import torch

from oracle.attention import fused_fog_attention_ref, windowed_attention_ref
from tests.exact64 import attend64, close_to_rounding
from tests.inputs import gen

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def mfma_only(monkeypatch):
    """A call that would run on the generic kernel is an error in this file."""
    monkeypatch.setenv("KESSIE_REQUIRE_MFMA", "1")


@pytest.mark.parametrize("b,h,n,d,splits", [
    (1, 1, 1, 64, 0), (1, 1, 1, 128, 0),        # one key
    (3, 1, 15, 64, 0), (2, 5, 17, 128, 0),      # around a page
    (1, 7, 63, 128, 0), (2, 3, 65, 64, 0),      # around a key tile
    (2, 1, 255, 64, 0), (1, 3, 257, 128, 0),    # around a query tile
    (2, 3, 517, 64, 3), (1, 5, 771, 128, 2),    # key splits
])
@pytest.mark.parametrize("window,causal,fog", [(0, True, True), (0, False, False), (50, True, False), (1, True, True)])
def test_dense_ragged(dev, monkeypatch, b, h, n, d, splits, window, causal, fog):
    from kessie_amd.kessie_hip_ctypes import KeSSieKernels

    assert h * n % 16
    if splits:
        monkeypatch.setenv("KESSIE_DENSE_SPLITS", str(splits))
    q, k, v = [torch.randn(b, h, n, d, generator=gen(dev, 40 + i), device=dev).half() for i in range(3)]
    kk = KeSSieKernels()
    qf, kf, vf = q.float().cpu(), k.float().cpu(), v.float().cpu()
    if fog:
        w = torch.rand(n, generator=gen(dev, 44), device=dev)
        out = kk.fused_fog_attention(q, k, v, w, window_size=window, causal=causal)
        ref = fused_fog_attention_ref(qf, kf, vf, w.cpu(), window)
    else:
        out = kk.windowed_attention(q, k, v, window_size=window, causal=causal)
        ref = windowed_attention_ref(qf, kf, vf, window, causal)
    err = (out.double().cpu() - ref.double()).norm()
    rounding = (ref.half().double() - ref.double()).norm()
    assert err <= 1.02 * rounding + 2e-5 * ref.double().norm(), f"error {err:.3e}, rounding alone {rounding:.3e}"


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("splits", [1, 3])
def test_dense_ragged_one_large_weight(dev, monkeypatch, d, splits):
    """A fog weight of 2^16 on a key that few rows see, beside weights of 1: the rows that do not see it keep their
    precision."""
    from kessie_amd.kessie_hip_ctypes import KeSSieKernels

    monkeypatch.setenv("KESSIE_DENSE_SPLITS", str(splits))
    h, n = 3, 517
    q, k, v = [torch.randn(1, h, n, d, generator=gen(dev, 90 + i), device=dev).half() for i in range(3)]
    w = torch.ones(n, device=dev)
    w[400] = 2.0 ** 16
    v[:, :, 400] *= 2.0 ** -10
    out = KeSSieKernels().fused_fog_attention(q, k, v, w, window_size=64, causal=True)
    ref = attend64(q[0].transpose(0, 1), k[0].transpose(0, 1), v[0].transpose(0, 1), 0, w, None, 64)
    for r in range(n):
        close_to_rounding(out[0, :, r], ref[r], torch.float16)
