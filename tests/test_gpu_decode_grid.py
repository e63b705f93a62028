"""GPU parity of the decode's one-round grid: splits rounded down to the chip's
workgroup slots, balanced units that are no multiple of the batch, and splits
bounded by a window.  |gpu - ref| <= 2e-2 + 1e-2 * |ref| (bf16 probabilities
and outputs, fp32 sums), as tests/test_gpu_decode.py."""
import pytest
import torch

from oracle.attention import paged_decode_ref
from tests.inputs import decode_case, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hkv,ctx,lens,window", [
    (3, 8, 32768, [32768, 1, 9000], 0),                     # balanced: 256 units over 3 sequences
    (7, 2, 40000, [40000, 0, 17, 16, 15, 2500, 700], 0),    # balanced, one group of kv heads, an empty sequence
    (64, 8, 2048, [2048] * 5 + list(range(1, 60)), 0),      # balanced at the largest batch it takes
    (5, 8, 3000, [3000, 1500, 31, 2999, 16], 1024),         # a window bounds the splits
    (4, 1, 9000, [9000, 8999, 33, 1], 33),                  # ... to two of them
    (3, 1, 4000, [4000, 40, 17], 5),                        # ... and to one (no partials)
    (130, 8, 64, [64] * 100 + [1 + i for i in range(30)], 0),  # past half a round: two splits
    (12, 1, 5000, [5000] * 11 + [77], 4096),                # rounded up: few surplus workgroups
    (70, 8, 500, [500] * 3 + [7 * i + 1 for i in range(67)], 0),  # rounded up: a large batch of unknown lengths
])
def test_decode_one_round_grid(dev, b, hkv, ctx, lens, window):
    from kessie_amd import ops

    q, pool, table, lens_d = decode_case(b, 4 * hkv, hkv, 128, ctx, 16, torch.bfloat16, dev, seed=41, ctx_lens=lens)
    vs = torch.rand(ctx, generator=gen(dev, 42), device=dev)
    out = ops.fog_decode(q, pool, table, lens_d, ctx, fog_vscale=vs, window=window)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    for i, n in enumerate(lens):
        if n == 0:
            assert not out[i].any()
            continue
        row = table[i].long()[: -(-n // 16)]
        ref = paged_decode_ref(q[i:i + 1].cpu(), pool[row].cpu(), torch.arange(len(row), dtype=torch.int32)[None],
                               torch.tensor([n]), vs.cpu(), None, window)
        diff = (out[i:i + 1].float().cpu() - ref).abs()
        assert bool((diff <= 2e-2 + 1e-2 * ref.abs()).all()), f"sequence {i} ({n} tokens): {diff.max().item():.3e}"


@pytest.mark.parametrize("b,hq,hkv,d,dt,ctx,window", [
    (12, 32, 8, 128, torch.bfloat16, 3000, 0), (12, 32, 8, 64, torch.float16, 6000, 0),
    (24, 8, 2, 128, torch.float32, 4000, 0), (40, 32, 8, 128, torch.float32, 300, 0),  # fp32: rounded up
    (70, 32, 8, 128, torch.bfloat16, 500, 0),  # rounded up, or down by the total
    (24, 24, 8, 128, torch.bfloat16, 2000, 1000),
    (20, 32, 2, 128, torch.bfloat16, 9000, 0),  # 1,024 units a group of heads: the combine that loops
])
@pytest.mark.parametrize("total", ["sum", "one", "over"])
def test_decode_known_lengths(dev, b, hq, hkv, d, dt, ctx, window, total):
    """A total of the lengths given by the host chooses the balanced split below its size bound; any total
    (here also 1, and more than the batch holds) leaves the result that of the plain split."""
    from kessie_amd import ops

    lens = [ctx] + [1 + (37 * i * i) % (ctx // 3) for i in range(1, b)]
    q, pool, table, lens_d = decode_case(b, hq, hkv, d, ctx, 16, dt, dev, seed=43, ctx_lens=lens)
    seen = {"sum": sum(min(n, window or n) for n in lens), "one": 1, "over": 2 * b * ctx}[total]
    plain = ops.fog_decode(q, pool, table, lens_d, ctx, window=window)
    out = ops.fog_decode(q, pool, table, lens_d, ctx, window=window, seen_total=seen)
    diff = (out.float() - plain.float()).abs()
    if dt != torch.float32 and d == 128 and hq // hkv in (4, 16):
        # Probabilities rounded to the type against another running maximum (2^-9 each): this file's tolerance.
        assert bool((diff <= 2e-2 + 1e-2 * plain.float().abs()).all()), diff.max().item()
    else:
        # One rounding of the output apart: only the splits' fp32 sums meet in another order.
        tol = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10, torch.float32: 2e-5}[dt]
        assert bool((diff <= tol * (plain.float().abs() + 0.02)).all()), diff.max().item()


def test_layer_passes_the_lengths_of_each_step(dev, monkeypatch):
    """The serving layer's total of the lengths follows a metadata object that is refilled in place between steps, and a
    window; it is left out of steps too small for it and with the fog off."""
    from kessie_amd import kessie_attention as ka
    from kessie_amd import ops

    n, got = 4, []
    q, pool, table, lens = decode_case(n, 8, 2, 64, 16384, 16, torch.bfloat16, dev, seed=45)
    cache = pool.transpose(1, 2).contiguous()  # [pages, 2, page, heads, d]
    cpu, qsl = lens.cpu(), torch.arange(n + 1, dtype=torch.int32)
    meta = ka.KeSSieAttentionMetadata(n, 1, qsl.to(dev), 16384, lens, table, torch.zeros(n, dtype=torch.int64, device=dev),
                                      query_start_loc_cpu=qsl, seq_lens_cpu=cpu)
    real, state = ops.fog_decode, ka.KeSSieAttentionState()
    monkeypatch.setattr(ops, "fog_decode", lambda *a, **k: (got.append(k.get("seen_total", 0)), real(*a, **k))[1])
    monkeypatch.setattr(ka, "KESSIE_STATE", state)
    new = torch.zeros(n, 2, 64, dtype=torch.bfloat16, device=dev)
    for alpha, window, lengths in ((0.5, 0, [16384, 100, 40, 9]), (0.5, 0, [640, 200, 40, 9]),
                                   (0.5, 13000, [16384, 200, 40, 9]), (0.5, 64, [640, 200, 40, 9]), (0.0, 0, [640, 200, 40, 9])):
        state.update(fog_alpha=alpha, fog_start=0.5, prompt_len=16384)
        cpu.copy_(torch.tensor(lengths))
        lens.copy_(cpu)
        impl = ka.KeSSieAttentionImpl(8, 64, 0.125, 2, sliding_window=window or None)
        for _ in range(2):
            impl.forward(None, q, new, new, cache, meta)
    torch.cuda.synchronize()
    assert got == [16533] * 2 + [889] * 2 + [13249] * 2 + [0] * 2 + [0] * 2
