"""GPU: the launches small batches take.

Bar as in test_gpu_configs.py: 1e-5 (fp32) and 2e-2 (bf16), relative to
max |ref|, against a float64 computation on the same inputs.
"""

from __future__ import annotations

import pytest
import torch

from conftest import assert_close

pytestmark = pytest.mark.gpu

KIND = {torch.float32: "f32", torch.bfloat16: "bf16"}


@pytest.fixture(scope="module")
def ops():
    from asrback_amd import attention

    return attention


def say(*args):
    print(*args, flush=True)


def randn(*shape, seed, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype)


def attend(q, k, v, scale, visible):
    """float64 attention: q (B, n, H, d), k/v (B, m, Hkv, d), visible (B, n, m);
    rows that see no key are zeros."""
    group = q.shape[2] // k.shape[2]
    qd, kd, vd = (t.double().transpose(1, 2) for t in (q, k, v))
    kd, vd = (t.repeat_interleave(group, dim=1) for t in (kd, vd))
    s = (qd @ kd.transpose(2, 3)) * scale
    s = s.masked_fill(~visible[:, None], float("-inf"))
    p = s.softmax(-1).nan_to_num(0.0)
    return (p @ vd).transpose(1, 2)


@pytest.mark.parametrize("splits", [2, 3, 8, 9, 17, 64, 0])
@pytest.mark.parametrize("dtype,hd,heads_q,heads_kv", [
    (torch.bfloat16, 128, 4, 2), (torch.float32, 64, 3, 3), (torch.bfloat16, 512, 8, 1), (torch.float32, 256, 4, 1)])
def test_split_launch_over_any_workspace(ops, device, dtype, hd, heads_q, heads_kv, splits):
    """Split launches need no cleared workspace and leave it usable: over
    buffers of arbitrary bytes, back to back in one buffer, and replayed from
    a graph with other calls (and other bytes) in the buffer between replays.
    Split counts around the eight partials the fold reads at a time, and more
    splits than keys."""
    say("split launch", dtype, hd, heads_q, heads_kv, splits)
    length = 300
    q = randn(3, heads_q, hd, seed=1, dtype=dtype)
    k, v = (randn(3, length, heads_kv, hd, seed=s, dtype=dtype) for s in (2, 3))
    used = torch.tensor([300, 7, 131], dtype=torch.int32)
    visible = (torch.arange(length) < used[:, None])[:, None]
    ref = attend(q[:, None], k, v, hd**-0.5, visible)[:, 0]
    q, k, v, used = (t.to(device) for t in (q, k, v, used))
    need = ops.decode_workspace_size(3, heads_q, heads_kv, hd, length, dtype, splits)
    buffer = torch.empty(max(need, 256), dtype=torch.uint8, device=device)
    for fill in (255, 0, 7):
        buffer.fill_(fill)
        for _ in range(2):
            out = ops.decode(q, k, v, seqused_k=used, num_splits=splits, workspace=buffer)
            assert_close(out.float().cpu(), ref, KIND[dtype])
    graph = torch.cuda.CUDAGraph()
    held = torch.empty_like(q)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        for _ in range(2):
            ops.decode(q, k, v, seqused_k=used, num_splits=splits, workspace=buffer, out=held)
    for fill in (255, 0, 3):
        buffer.fill_(fill)
        ops.decode(q, k, v, seqused_k=used, num_splits=splits, workspace=buffer)
        held.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hd,heads_q,heads_kv", [(64, 8, 1), (128, 2, 2), (128, 8, 1), (256, 8, 1), (512, 8, 1)])
@pytest.mark.parametrize("norms,rotary,v_norm", [(True, True, True), (True, False, False), (False, True, True)])
def test_append_prologue_rows(ops, device, dtype, hd, heads_q, heads_kv, norms, rotary, v_norm):
    """The prologue's rows (query heads, new key, new value) shared by a
    workgroup: more rows than lane groups, fewer, and each of its parts alone,
    over split and unsplit launches.  The written key and value bound the
    prologue's own rounding: one unit in the last place (2^-7 relative in
    bf16, 1e-6 in fp32)."""
    if dtype == torch.float32 and hd == 512:
        pytest.skip("head_dim 512 decodes in bf16 only")
    say("append prologue", dtype, hd, heads_q, heads_kv, norms, rotary, v_norm)
    length, eps = 90, 1e-6
    positions = torch.tensor([0, 61, 89])
    q, k_new, v_new = (randn(3, h, hd, seed=s, dtype=dtype) for h, s in ((heads_q, 4), (heads_kv, 5), (heads_kv, 6)))
    keys, values = (randn(3, length, heads_kv, hd, seed=s, dtype=dtype) for s in (7, 8))
    wq, wk = ((1 + 0.2 * randn(hd, seed=s)).to(dtype) for s in (9, 10))
    angle = randn(3, hd // 2, seed=11)
    cos, sin = (torch.cat((f(angle), f(angle)), -1).to(dtype) for f in (torch.cos, torch.sin))

    def prologue(x, weight, norm, rotate):
        x = x.float()
        if norm:
            x = x * (x.square().mean(-1, keepdim=True) + eps).rsqrt()
            x = (x if weight is None else x * weight.float()).to(dtype).float()
        if rotate:
            swapped = torch.cat((-x[..., hd // 2:], x[..., : hd // 2]), -1)
            a, b = ((t * u.float()[:, None]).to(dtype).float() for t, u in ((x, cos), (swapped, sin)))
            x = (a + b).to(dtype).float()
        return x.to(dtype)

    qn, kn = prologue(q, wq, norms, rotary), prologue(k_new, wk, norms, rotary)
    vn = prologue(v_new, None, v_norm, False)
    rows = torch.arange(3)
    keys_ref, values_ref = keys.clone(), values.clone()
    keys_ref[rows, positions], values_ref[rows, positions] = kn, vn
    visible = (torch.arange(length) <= positions[:, None])[:, None]
    ref = attend(qn[:, None], keys_ref, values_ref, hd**-0.5, visible)[:, 0]
    for splits in (1, 3):
        kd, vd = keys.to(device), values.to(device)
        on = [t.to(device) for t in (q, k_new, v_new, wq, wk, cos, sin, positions)]
        out = ops.decode_append(
            on[0], on[1], on[2], kd, vd, on[7], eps=eps, num_splits=splits, v_norm=v_norm,
            **({"q_norm": on[3], "k_norm": on[4]} if norms else {}), **({"cos": on[5], "sin": on[6]} if rotary else {}))
        assert_close(out.float().cpu(), ref, KIND[dtype])
        for got, want in ((kd, keys_ref), (vd, values_ref)):
            ulp = 2.0**-7 if dtype == torch.bfloat16 else 1e-6
            worst = (got.cpu().float() - want.float()).abs() - ulp * want.float().abs()
            # Sums of rotated pairs may cancel: an absolute floor of one unit of the addends.
            assert float(worst.max()) <= ulp * 4.0
