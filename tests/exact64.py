"""Attention in 64 bits on the CPU, for tests that bound a kernel's own error."""
import torch


def attend64(q, k, v, first, weights=None, bias=None, window=0, sm_scale=None):
    """q [R, Hq, D] at positions first .. over k, v [N, Hkv, D], causal: [R, Hq, D] in float64.  A key with
    probability zero takes no part, whatever its weight."""
    q, k, v = (t.detach().double().cpu() for t in (q, k, v))
    r, hq, d = q.shape
    n, hkv = k.shape[:2]
    s = torch.einsum("rhgd,nhd->hgrn", q.view(r, hkv, hq // hkv, d), k) * (d ** -0.5 if sm_scale is None else sm_scale)
    if bias is not None:
        s = s + bias.detach().double().cpu()[:n]
    dist = (first + torch.arange(r))[:, None] - torch.arange(n)
    hide = dist < 0
    if window:
        hide |= dist >= window
    p = torch.softmax(s.masked_fill(hide, float("-inf")), -1)
    if weights is not None:
        p = torch.where(p == 0, p, p * weights.detach().double().cpu()[:n])
    return torch.einsum("hgrn,nhd->rhgd", p, v).reshape(r, hq, d)


def paged(k, v, page=16):
    """A native pool [pages, page, 2, Hkv, D] holding k, v [N, Hkv, D] in order, its table [1, pages] and length."""
    n, hkv, d = k.shape
    pages = -(-n // page)
    pool = torch.zeros(pages * page, 2, hkv, d, dtype=k.dtype, device=k.device)
    pool[:n, 0], pool[:n, 1] = k, v
    table = torch.arange(pages, dtype=torch.int32, device=k.device).view(1, -1)
    return pool.view(pages, page, 2, hkv, d), table, torch.tensor([n], dtype=torch.int32, device=k.device)


def close_to_rounding(out, ref, dtype, own=2e-5):
    """out is as far from ref (float64) as rounding ref to dtype, and a kernel's fp32 sums (`own` of the norm) besides."""
    err = (out.double().cpu() - ref).norm()
    rounding = (ref.to(dtype).double() - ref).norm()
    assert err <= 1.05 * rounding + own * ref.norm(), f"error {err:.3e}, rounding alone {rounding:.3e}, norm {ref.norm():.3e}"
