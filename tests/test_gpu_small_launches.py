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
    (torch.bfloat16, 128, 4, 2), (torch.float32, 64, 3, 3), (torch.bfloat16, 512, 8, 1), (torch.float32, 256, 4, 1),
    (torch.bfloat16, 256, 8, 1), (torch.bfloat16, 512, 4, 1), (torch.float32, 64, 8, 1)])
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


@pytest.mark.parametrize("dtype,hd,heads_q,heads_kv", [
    (torch.bfloat16, 128, 4, 2), (torch.float32, 64, 3, 3), (torch.bfloat16, 512, 8, 1)])
@pytest.mark.parametrize("splits", [1, 2, 3, 8, 9, 17, 0])
def test_split_launch_with_infinite_values(ops, device, dtype, hd, heads_q, heads_kv, splits):
    """An infinite value of a key that every row sees is the output's infinity
    however the keys are split: in the last split's keys, which the fold's
    surplus slots repeat, and in the first's.  All keys alike, so that no
    weight is 0."""
    say("infinite values", dtype, hd, heads_q, heads_kv, splits)
    length = 600
    q = randn(2, heads_q, hd, seed=1, dtype=dtype).to(device)
    k = randn(1, 1, heads_kv, hd, seed=2, dtype=dtype).expand(2, length, -1, -1).contiguous().to(device)
    v = randn(2, length, heads_kv, hd, seed=3, dtype=dtype).to(device)
    v[:, -1, :, 5] = float("inf")
    v[:, 0, :, 9] = float("-inf")
    out = ops.decode(q, k, v, num_splits=splits)
    assert bool((out[..., 5] == float("inf")).all()) and bool((out[..., 9] == float("-inf")).all())
    keep = [i for i in range(hd) if i not in (5, 9)]
    ref = v.double().mean(1).repeat_interleave(heads_q // heads_kv, dim=1)
    assert_close(out[..., keep].float().cpu(), ref[..., keep].cpu(), KIND[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hd,heads_q,heads_kv", [(64, 8, 1), (128, 2, 2), (128, 8, 1), (256, 8, 1), (512, 8, 1)])
@pytest.mark.parametrize("norms,rotary,v_norm", [(True, True, True), (True, False, False), (False, True, True),
                                                 (False, False, False)])
def test_append_prologue_rows(ops, device, dtype, hd, heads_q, heads_kv, norms, rotary, v_norm):
    """The prologue's rows (query heads, new key, new value) shared by a
    workgroup: more rows than lane groups, fewer, each of its parts alone, and
    none (the rows as they are), over split and unsplit launches.  The written key and value bound the
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


def assert_ulps(got, want, dtype, scale):
    """Within one rounding of ``want`` (2^-7 relative in bf16, 1e-6 in fp32)
    plus one of addends of size ``scale`` (a rotated pair's sum may cancel),
    and nearly always the same value in bf16."""
    ulp = 2.0**-7 if dtype == torch.bfloat16 else 1e-6
    diff = (got.float() - want.float()).abs()
    assert float((diff - ulp * want.float().abs()).max()) <= ulp * scale
    if dtype == torch.bfloat16:
        assert float((diff > 0).float().mean()) < 0.02


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hd,heads,kv_heads,tokens,paged", [
    (64, 3, 1, 1, False), (128, 16, 8, 37, False), (128, 4, 2, 130, True), (256, 2, 2, 9, False), (512, 2, 1, 5, True)])
def test_prompt_rows_match_the_ops(device, dtype, hd, heads, kv_heads, tokens, paged, monkeypatch):
    """Qwen3's prompt pass with its rows prepared by the kernel against the
    ops it replaces: attention output, and the whole cache (slab, with rows
    and positions counted from the end; or pages, rows without a page writing
    to the sink)."""
    from asrback_amd import qwen3_asr

    say("prompt rows", dtype, hd, heads, kv_heads, tokens, paged)
    config = {"hidden_size": 128, "head_dim": hd, "num_attention_heads": heads, "num_key_value_heads": kv_heads,
              "rms_norm_eps": 1e-6, "rope_theta": 1e6, "num_hidden_layers": 1}
    torch.manual_seed(3)
    layer = qwen3_asr.TextAttention(config).to(device, dtype)
    with torch.no_grad():
        for norm in (layer.q_norm, layer.k_norm):
            norm.weight.normal_(1.0, 0.2)
    first = tokens // 2
    lengths = [n for n in (first, tokens - first) if n]
    x = randn(tokens, 128, seed=5, dtype=dtype).to(device)
    slots = [2, 0][: len(lengths)]
    rows = torch.cat([torch.full((n,), r) for n, r in zip(lengths, slots)]).to(device)
    positions = torch.cat([torch.arange(n) for n in lengths]).to(device)
    cos, sin = qwen3_asr.rope_tables(config, 1024, device, dtype)
    cos, sin = cos[positions], sin[positions]
    segments = qwen3_asr.Segments.from_lengths(lengths, device)
    results = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(qwen3_asr, "prompt_rows_takes", lambda *a: False)
        else:
            called = []
            real = qwen3_asr.prompt_rows
            monkeypatch.setattr(qwen3_asr, "prompt_rows", lambda *a, **k: called.append(1) or real(*a, **k))
        with torch.inference_mode():
            if paged:
                cache = qwen3_asr.PagedKVCache.allocate(config, 3, 40, 16, device, dtype)
                cache.assign(2, 24)  # a prompt past its row's pages writes to the sink
                cache.assign(0, 100)
                keys, values = cache.keys[0], cache.values[0]
                stored = [cache.pool_keys[0, :-1], cache.pool_values[0, :-1]]
                where = rows
            else:
                stored = [torch.zeros(3, 128, kv_heads, hd, dtype=dtype, device=device) for _ in range(2)]
                keys, values = stored
                where = rows - 3  # negative: from the end
            out = layer.prefill(x, keys, values, where, positions, segments, cos, sin)
        results.append((out, *stored))
    assert called
    (out, keys, values), (out_ref, keys_ref, values_ref) = results
    assert_ulps(keys, keys_ref, dtype, 4.0)
    assert torch.equal(values, values_ref) and bool(values.any())
    # q and k one rounding apart move the bf16 scores by 2^-8 of a few units.
    assert_close(out, out_ref, "module", 1e-4 if dtype == torch.float32 else 2e-2)


def prompt_layer(device, dtype=torch.float32):
    """A small Qwen3 attention layer and the rest of its prompt pass's
    arguments past the cache, five tokens of two prompts."""
    from asrback_amd import qwen3_asr

    config = {"hidden_size": 64, "head_dim": 64, "num_attention_heads": 2, "num_key_value_heads": 1,
              "rms_norm_eps": 1e-6, "rope_theta": 1e6, "num_hidden_layers": 1}
    layer = qwen3_asr.TextAttention(config).to(device, dtype).requires_grad_(False)
    positions = torch.tensor([0, 1, 2, 0, 1], device=device)
    cos, sin = (t[positions] for t in qwen3_asr.rope_tables(config, 8, device, dtype))
    rows = torch.tensor([0, 0, 0, 1, 1], device=device)
    return layer, (rows, positions, qwen3_asr.Segments.from_lengths([3, 2], device), cos, sin)


def test_prompt_rows_marks_the_cache_modified(device, monkeypatch):
    """The cache writes count as in-place writes, as the ops' do: a backward
    that saved the cache before them is refused, and so is a cache made in
    inference mode outside it."""
    from asrback_amd import qwen3_asr

    layer, rest = prompt_layer(device)
    called = []
    real = qwen3_asr.prompt_rows
    monkeypatch.setattr(qwen3_asr, "prompt_rows", lambda *a, **k: called.append(1) or real(*a, **k))
    x = torch.randn(5, 64, device=device)
    for which in (0, 1):
        cache = [torch.zeros(2, 4, 1, 64, device=device) for _ in range(2)]
        scale = torch.ones((), device=device, requires_grad=True)
        loss = (cache[which] * scale).sum()
        layer.prefill(x, *cache, *rest)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()
    assert len(called) == 2
    with torch.inference_mode():
        cache = [torch.zeros(2, 4, 1, 64, device=device) for _ in range(2)]
        layer.prefill(x, *cache, *rest)
    assert len(called) == 3
    with pytest.raises(RuntimeError, match="inference tensor"):
        layer.prefill(x, *cache, *rest)
    assert len(called) == 3


def test_prompt_rows_leaves_other_forms_to_the_ops(device, monkeypatch):
    """Rotation tables with a batch axis that packed prompts do not have, which
    the pass refuses; keys and values paged by different tables."""
    from asrback_amd import qwen3_asr

    layer, (rows, positions, segments, cos, sin) = prompt_layer(device)
    x = torch.randn(5, 64, device=device)
    cache = [torch.zeros(2, 4, 1, 64, device=device) for _ in range(2)]
    with pytest.raises((RuntimeError, ValueError, IndexError)):
        layer.prefill(x, *cache, rows, positions, segments, cos[None], sin[None])
    pools = [torch.zeros(5, 16, 1, 64, device=device) for _ in range(2)]
    tables = [qwen3_asr.PageTable(torch.tensor(t, dtype=torch.int32, device=device)) for t in ([[0], [1]], [[3], [2]])]
    layers = [qwen3_asr.PagedLayer(pool, qwen3_asr.PageTable(t.block_table, 16), 16) for pool, t in zip(pools, tables)]
    layer.prefill(x, *layers, rows, positions, segments, cos, sin)
    v = layer.qkv_proj(x).split(layer.sizes, dim=-1)[2].view(5, 1, 64)
    assert torch.equal(pools[1][3, :3], v[:3]) and torch.equal(pools[1][2, :2], v[3:])
    assert not bool(pools[1][:2].any()) and bool(pools[0][:2, 0].any()) and not bool(pools[0][2:4].any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layer_type", ["sliding_attention", "full_attention"])
def test_gemma_prompt_rows_match_the_ops(device, dtype, layer_type, monkeypatch):
    """Gemma 4's padded prompts (value norm, rotation tables shared by the
    batch, a shared layer's queries alone) through the kernel and the ops."""
    from asrback_amd import gemma4

    say("gemma prompt rows", dtype, layer_type)
    text = {"hidden_size": 128, "head_dim": 256, "global_head_dim": 512, "num_attention_heads": 2,
            "num_key_value_heads": 1, "sliding_window": 512, "rms_norm_eps": 1e-6}
    torch.manual_seed(4)
    own, shared = (gemma4.TextAttention(text, layer_type, s).to(device, dtype) for s in (False, True))
    with torch.no_grad():
        for norm in (own.q_norm, own.k_norm, shared.q_norm):
            norm.weight.normal_(0.1, 0.02)
    length, hd = 19, own.head_dim
    x = randn(2, length, 128, seed=6, dtype=dtype).to(device)
    angle = randn(length, hd // 2, seed=7)
    cos, sin = (torch.cat((f(angle), f(angle)), -1).to(device, dtype) for f in (torch.cos, torch.sin))
    sizes = gemma4.KeyPrefix(lengths=torch.tensor([19, 11], dtype=torch.int32, device=device))
    rows = torch.tensor([2, 0], device=device)
    results = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(gemma4, "prompt_rows_takes", lambda *a: False)
        else:
            called = []
            real = gemma4.prompt_rows
            monkeypatch.setattr(gemma4, "prompt_rows", lambda *a, **k: called.append(1) or real(*a, **k))
        with torch.inference_mode():
            cache = gemma4.LayerKV(*(torch.zeros(3, 40, 1, hd, dtype=dtype, device=device) for _ in range(2)))
            kv: dict = {}
            out = own.prefill(x, cache, rows, kv, sizes, cos, sin)
            out_shared = shared.prefill(x, cache, rows, kv, sizes, cos, sin)
        results.append((out, out_shared, cache.keys, cache.values))
    assert len(called) == 2
    for got, want in zip(results[0][2:], results[1][2:]):
        assert bool(want.any())
        assert_ulps(got, want, dtype, 4.0)
    for got, want in zip(results[0][:2], results[1][:2]):
        assert_close(got, want, "module", 1e-4 if dtype == torch.float32 else 2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,inputs,outputs", [
    (1, 8, (1,)), (1, 384, (384, 384, 384)), (2, 520, (7,)), (3, 1280, (5, 66)), (5, 1536, (384,)), (8, 2048, (9,)),
    (9, 3072, (13,)), (16, 1280, (1280,))])
def test_rows_linear(device, dtype, rows, inputs, outputs):
    """A step's linear layers: odd output counts (columns past the last),
    rows that fill no workgroup, reductions shorter and longer than a wave and
    past 512 threads, with and without bias, norm, activation and residual.
    Against float64 on the same inputs, rounded where the ops round: float32
    sums of k products (1e-5), or one bf16 rounding after another (2e-2)."""
    import torch.nn.functional as F
    from torch import nn

    from asrback_amd import layers

    say("rows linear", dtype, rows, inputs, outputs)
    torch.manual_seed(8)
    x = torch.randn(rows, 1, inputs, device=device).mul_(2.0).add_(0.5).to(dtype)
    linears = [nn.Linear(inputs, n, bias=i != 1) for i, n in enumerate(outputs)]
    linears = [m.to(device, dtype).requires_grad_(False) for m in linears]
    norm = nn.LayerNorm(inputs).to(device, dtype).requires_grad_(False)
    norm.weight.normal_(1.0, 0.2)
    norm.bias.normal_(0.0, 0.2)
    residual = torch.randn(rows, 1, outputs[0], device=device).to(dtype)
    assert layers.rows_linear_takes(x, linears, [norm], [])

    def exact(m, use_norm):
        h = x.double()
        if use_norm:
            h = F.layer_norm(h, (inputs,), norm.weight.double(), norm.bias.double(), norm.eps).to(dtype).double()
        return F.linear(h, m.weight.double(), None if m.bias is None else m.bias.double())

    for use_norm in (False, True):
        got = layers.rows_linear(x, linears, norm if use_norm else None)
        for out, m in zip(got, linears):
            assert_close(out.cpu(), exact(m, use_norm).cpu(), KIND[dtype])
        got = layers.rows_linear(x, linears, norm if use_norm else None, gelu=True)
        for out, m in zip(got, linears):
            assert_close(out.cpu(), F.gelu(exact(m, use_norm).to(dtype).double()).cpu(), KIND[dtype])
        (out,) = layers.rows_linear(x, linears[:1], norm if use_norm else None, residual=residual)
        assert_close(out.cpu(), (residual.double() + exact(linears[0], use_norm)).cpu(), KIND[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,inputs,outputs", [(1, 8, 5), (2, 384, 7), (4, 520, 9), (5, 1280, 6), (3, 3072, 5),
                                                 (4, 384, 16391), (1, 1280, 16387)])
def test_rows_linear_infinite_weights(device, dtype, rows, inputs, outputs):
    """An infinite weight in the first or last vector of its row gives its
    output the infinity, as the ops do, and touches no other output: reductions
    that end inside a wave's vectors, at a wave, and past one."""
    from torch import nn

    from asrback_amd import layers

    say("rows linear inf", dtype, rows, inputs, outputs)
    torch.manual_seed(12)
    x = torch.rand(rows, 1, inputs, device=device).add_(0.5).to(dtype)
    linear = nn.Linear(inputs, outputs, bias=False).to(device, dtype).requires_grad_(False)
    linear.weight[1, inputs - 1] = float("inf")
    linear.weight[3, 0] = float("-inf")
    assert layers.rows_linear_takes(x, [linear], [], [])
    (got,) = layers.rows_linear(x, [linear])
    ref = x.double() @ linear.weight.double().t().contiguous()
    assert bool((got[..., 1] == float("inf")).all()) and bool((got[..., 3] == float("-inf")).all())
    keep = [0, 2, *range(4, outputs)]
    assert_close(got[..., keep].cpu(), ref[..., keep].cpu(), KIND[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,inputs,outputs", [(1, 8, 16384), (1, 1280, 16387), (2, 384, 16389), (2, 1280, 16391),
                                                 (3, 520, 20001), (4, 640, 51865)])
def test_vocabulary_product(device, dtype, rows, inputs, outputs):
    """Few rows through a vocabulary's weights (eight or four columns a wave,
    counts that fill no wave), against float64: float32 sums of k products
    (1e-5), or one rounding (2e-2)."""
    from asrback_amd import layers

    say("vocabulary product", dtype, rows, inputs, outputs)
    torch.manual_seed(9)
    x = torch.randn(rows, inputs, device=device).to(dtype)
    weight = torch.randn(outputs, inputs, device=device).to(dtype)
    assert layers.rows_product_takes(x, weight)
    assert not layers.rows_product_takes(x[:, 1:], weight[:, 1:])
    assert not layers.rows_product_takes(x.requires_grad_(dtype == torch.float32), weight.t().contiguous().t())
    assert_close(layers.rows_product(x.detach(), weight).cpu(), (x.double() @ weight.double().t()).detach().cpu(),
                 KIND[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 384), (17, 1280), (2, 2056)])
def test_step_embeddings(device, dtype, rows, width):
    """The sum of token and position embeddings, to the bit, for tokens that
    are a column of a longer table; rows outside the tables are NaN."""
    from torch import nn

    from asrback_amd import layers

    torch.manual_seed(10)
    tables = [nn.Embedding(n, width).to(device, dtype).requires_grad_(False) for n in (101, 40)]
    tokens = torch.randint(101, (rows, 5), device=device)[:, 2:3]
    positions = torch.randint(40, (rows,), device=device)
    assert layers.embed_rows_takes(tokens, positions, *tables)
    got = layers.embed_rows(tokens, positions, *tables)
    assert torch.equal(got, tables[0](tokens) + tables[1](positions)[:, None])
    for bad in (tokens.int(), tokens.expand(rows, 2), tokens[:, 0], tokens.cpu()):
        assert not layers.embed_rows_takes(bad, positions, *tables)
    positions[0] = 40
    got = layers.embed_rows(tokens, positions, *tables)
    assert bool(got[0].isnan().all()) and not bool(got[1:].isnan().any())


def test_rows_linear_leaves_other_programs_to_the_ops(device):
    """Inputs whose ops something has to see, or the kernel does not address."""
    from torch import nn

    from asrback_amd import layers

    linear, norm = nn.Linear(64, 64).to(device), nn.LayerNorm(64).to(device)
    x = torch.randn(2, 1, 64, device=device)

    def takes(x=x):
        return layers.rows_linear_takes(x, [linear], [norm], [])

    assert not takes()  # weights that collect gradients
    with torch.no_grad():
        assert takes()
        assert not takes(x.double()) and not takes(x[:, :, 1:]) and not takes(x.expand(2, 3, 64))
        assert not takes(torch.randn(17, 1, 64, device=device)) and not takes(x.cpu())
        assert not takes(torch.randn(2, 1, 68, device=device)[..., 2:66])  # 8-byte aligned
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not takes()
        seen = []
        torch.vmap(lambda t: seen.append(takes(t)) or t)(x[None])
        assert seen == [False]
        hook = norm.register_forward_hook(lambda *a: None)
        assert not takes()
        hook.remove()
        hook = nn.modules.module.register_module_forward_hook(lambda *a: None)
        assert not takes()
        hook.remove()
        linear.forward = lambda t: t
        assert not takes()
        del linear.forward
        with torch.device("cuda"):  # a function mode
            assert not takes()
        assert takes()


@pytest.mark.parametrize("hd,window,causal", [(64, 33, 1), (128, 100, 2), (256, 0, 0), (256, 40, 1), (512, 0, 1), (512, 64, 2)])
@pytest.mark.parametrize("len_q,len_k,batch", [(1, 1, 1), (32, 32, 2), (33, 97, 2), (200, 200, 1), (1, 300, 3)])
@pytest.mark.parametrize("valu", [False, True])
def test_float32_wide_heads_and_windows(ops, device, hd, window, causal, len_q, len_k, batch, valu):
    """float32 attention on the matrix cores at head_dim 256 and 512 (a row
    block's dimensions split over waves) and within sliding windows, and on the
    vector-ALU twin (several lanes a row, keys from the window's start), around
    the 32-row and 32-key edges, with grouped heads and per-row key counts
    (zero keys among them)."""
    from asrback_amd import _lib

    say("f32 wide", hd, window, causal, len_q, len_k, batch, valu)
    q = randn(batch, len_q, 4, hd, seed=21)
    k, v = (randn(batch, len_k, 2, hd, seed=s) for s in (22, 23))
    used = torch.tensor([len_k, len_k // 2, 0][:batch], dtype=torch.int32)
    i, j, n = torch.arange(len_q)[:, None], torch.arange(len_k), used[:, None, None]
    last = i + (n - len_q if causal == _lib.CAUSAL_BOTTOM_RIGHT else 0)
    visible = (j < n).expand(batch, len_q, len_k)
    if causal:
        visible = visible & (j <= last)
    if window:
        visible = visible & (j > last - window)
    out = ops.flash(q.to(device), k.to(device), v.to(device), causal=causal, seqused_k=used.to(device),
                    window=window, force_valu=valu)
    assert_close(out.cpu(), attend(q, k, v, hd**-0.5, visible), "f32")


# heads, batch, rows, keys: the workgroups the launch rules take (csrc/fwd_f32row.hip).
F32_HEAD64 = [
    (2, 2, 97, 300),    # one 16-row block, eight key splits (28 workgroups)
    (8, 4, 70, 70),     # one block, four splits
    (5, 4, 200, 520),   # two blocks (140 workgroups against 260 of one and 100 of three)
    (8, 4, 150, 150),   # two (160; 320 of one cost more without a mask)
    (3, 4, 700, 520),   # three (180 workgroups; 264 of two take two rounds)
    (8, 4, 300, 300),   # three (224; 608 of one cost more without a mask)
    (20, 16, 40, 40),   # the 32-row kernel: 640 row blocks over two sub-tiles
    (12, 8, 200, 200),  # the same, two key splits: 1344 waves of 2048
    (12, 16, 200, 200),  # the same, unsplit: 1344 row blocks
]


@pytest.mark.parametrize("heads,batch,len_q,len_k", F32_HEAD64)
@pytest.mark.parametrize("form", ["none", "top-left", "bottom-right", "window", "padded"])
def test_float32_head64_workgroups(ops, device, heads, batch, len_q, len_k, form):
    """float32 attention at head_dim 64 through each workgroup size and mask,
    with per-row key counts that end inside a block (and an empty row), and
    NaN in the keys and values past them."""
    from asrback_amd import _lib

    say("f32 head_dim 64", heads, batch, len_q, len_k, form)
    causal = {"none": 0, "padded": 0, "bottom-right": _lib.CAUSAL_BOTTOM_RIGHT}.get(form, _lib.CAUSAL_TOP_LEFT)
    window = 33 if form == "window" else 0
    q = randn(batch, len_q, heads, 64, seed=61)
    k, v = (randn(batch, len_k, heads, 64, seed=s) for s in (62, 63))
    used = torch.tensor([(len_k, len_k - 9, len_k // 2 + 1, 0, 1)[b % 5] for b in range(batch)], dtype=torch.int32)
    i, j, n = torch.arange(len_q)[:, None], torch.arange(len_k), used[:, None, None]
    last = i + (n - len_q if form == "bottom-right" else 0)
    visible = (j < n).expand(batch, len_q, len_k)
    if causal:
        visible = visible & (j <= last)
    if window:
        visible = visible & (j > last - window)
    if form == "padded":
        visible = visible & (i < n)
    ref = attend(q, k, v, 0.125, visible)
    gone = (torch.arange(len_k) >= used[:, None])[..., None, None]
    k, v = (t.masked_fill(gone, float("nan")) for t in (k, v))
    out = ops.flash(q.to(device), k.to(device), v.to(device), causal=causal, seqused_k=used.to(device),
                    window=window, zero_padded_rows=form == "padded")
    assert_close(out.cpu(), ref, "f32")


@pytest.mark.parametrize("hd,heads,kv_heads,causal", [(64, 3, 3, 0), (64, 12, 12, 1), (128, 4, 4, 0), (128, 16, 8, 2)])
@pytest.mark.parametrize("len_q,len_k,batch", [
    (4, 129, 2), (4, 1500, 3), (33, 300, 2), (64, 65, 1), (65, 64, 1), (130, 257, 4), (300, 300, 1), (700, 700, 3),
    (128, 131, 8), (200, 300, 4), (200, 256, 4)])
def test_small_bf16_launches(ops, device, hd, heads, kv_heads, causal, len_q, len_k, batch):
    """bf16 launches around the lines where a workgroup's rows and key splits
    change (32, 64 and 128 rows; one workgroup per CU), with per-row key
    counts that end splits early or leave them empty."""
    say("small bf16", hd, heads, kv_heads, causal, len_q, len_k, batch)
    q = randn(batch, len_q, heads, hd, seed=31, dtype=torch.bfloat16)
    k, v = (randn(batch, len_k, kv_heads, hd, seed=s, dtype=torch.bfloat16) for s in (32, 33))
    used = torch.tensor([len_k, 1, len_k // 2, 0] * 2, dtype=torch.int32)[:batch]
    i, j, n = torch.arange(len_q)[:, None], torch.arange(len_k), used[:, None, None]
    visible = (j < n).expand(batch, len_q, len_k)
    if causal:
        visible = visible & (j <= i + (n - len_q if causal == 2 else 0))
    out = ops.flash(q.to(device), k.to(device), v.to(device), causal=causal, seqused_k=used.to(device))
    assert_close(out.float().cpu(), attend(q, k, v, hd**-0.5, visible), "bf16")


@pytest.mark.parametrize("hd,window", [(256, 0), (512, 0), (512, 40)])
@pytest.mark.parametrize("batch,length", [(1, 1), (1, 65), (4, 256), (5, 257), (12, 100)])
def test_wide_bf16_prompts(ops, device, hd, window, batch, length):
    """Prompts at head_dim 256 and 512 on both sides of the line between 32 and
    64 rows a workgroup (256 workgroups of 32 rows), with row ends inside a
    block and per-row key counts."""
    say("wide bf16", hd, window, batch, length)
    q = randn(batch, length, 8, hd, seed=51, dtype=torch.bfloat16)
    k, v = (randn(batch, length, 4, hd, seed=s, dtype=torch.bfloat16) for s in (52, 53))
    used = torch.tensor([max(length - 7 * b, 1) for b in range(batch)], dtype=torch.int32)
    i, j, n = torch.arange(length)[:, None], torch.arange(length), used[:, None, None]
    visible = ((j < n) & (j <= i)).expand(batch, length, length)
    if window:
        visible = visible & (j > i - window)
    out = ops.flash(q.to(device), k.to(device), v.to(device), causal=1, seqused_k=used.to(device), window=window)
    assert_close(out.float().cpu(), attend(q, k, v, hd**-0.5, visible), "bf16")


@pytest.mark.parametrize("frames,batch", [(65, 1), (100, 1), (300, 2), (504, 1), (130, 9)])
def test_small_sanm_launches(ops, device, frames, batch):
    """SAN-M attention with its memory in the launches of few utterances: the
    memory's row blocks follow the attention's."""
    say("small sanm", frames, batch)
    x = randn(batch, frames, 1536, seed=41, dtype=torch.bfloat16)
    weight = randn(512, 1, 11, seed=42, dtype=torch.bfloat16)
    used = torch.tensor([frames] + [1 + 17 * b for b in range(1, batch)], dtype=torch.int32)
    q, k, v = (t.view(batch, frames, 4, 128) for t in x.split(512, dim=-1))
    keep = torch.arange(frames) < used[:, None]
    ref = attend(q, k, v, 128**-0.5, keep[:, None].expand(batch, frames, frames)) * keep[..., None, None]
    inside = (v.reshape(batch, frames, 512).double() * keep[..., None]).transpose(1, 2)
    conv = torch.nn.functional.conv1d(torch.nn.functional.pad(inside, (5, 5)), weight.double(), groups=512)
    memory_ref = ((conv + inside) * keep[:, None]).transpose(1, 2)
    q, k, v = (t.view(batch, frames, 4, 128) for t in x.to(device).split(512, dim=-1))
    out, memory = ops.flash_fsmn(q, k, v, weight.to(device), seqused_k=used.to(device), zero_padded_rows=True)
    assert_close(out.float().cpu(), ref, "bf16")
    assert_close(memory.float().cpu(), memory_ref, "bf16")


@pytest.mark.parametrize("kernel_size", [11, 15])
@pytest.mark.parametrize("frames,batch", [(70, 3), (300, 2), (504, 9)])
def test_sanm_reads_nothing_past_a_count(ops, device, frames, batch, kernel_size):
    """Queries, keys and values of padded frames are NaN (the projection leaves
    them unwritten): the valid frames come out as over zeros there, bit for bit,
    and the padded ones finite.  Launches without and with key splits (300
    frames), of many utterances, and filters past what the attention's launch
    computes."""
    say("sanm nan", frames, batch, kernel_size)
    x = randn(batch, frames, 1536, seed=45, dtype=torch.bfloat16)
    weight = randn(512, 1, kernel_size, seed=46, dtype=torch.bfloat16).to(device)
    used = torch.tensor([(frames, frames - 1, frames // 2, 1, 64, 0, frames - 63)[b % 7] for b in range(batch)],
                        dtype=torch.int32)
    gone = (torch.arange(frames) >= used[:, None])[..., None]
    results = []
    for fill in (0.0, float("nan")):
        q, k, v = (t.view(batch, frames, 4, 128) for t in x.masked_fill(gone, fill).to(device).split(512, dim=-1))
        results.append(ops.flash_fsmn(q, k, v, weight, seqused_k=used.to(device), zero_padded_rows=True))
    for clean, dirty in zip(*results):
        clean, dirty = (t.reshape(batch, frames, 512) for t in (clean, dirty))
        assert bool(dirty.isfinite().all()) and torch.equal(clean, dirty)


@pytest.mark.parametrize("frames,batch", [(70, 3), (300, 2), (504, 12)])
def test_sanm_module_over_nan_padding(device, frames, batch):
    """The bf16 module with NaN in the padded frames of its input: the valid
    frames as over zeros there, and no NaN in the others."""
    from asrback_amd import sensevoice

    say("sanm module nan", frames, batch)
    torch.manual_seed(15)
    layer = sensevoice.SANMAttention(512, 512, 4, 11).to(device, torch.bfloat16).requires_grad_(False)
    lengths = torch.tensor([(frames, frames - 1, frames // 2, 1, 64, 0, frames - 63)[b % 7] for b in range(batch)],
                           dtype=torch.int32, device=device)
    mask = torch.arange(frames, device=device) < lengths[:, None]
    x = torch.randn(batch, frames, 512, device=device).bfloat16()
    clean, dirty = (layer(x.masked_fill(~mask[..., None], fill), mask, lengths) for fill in (0.0, float("nan")))
    assert bool(dirty.isfinite().all()) and torch.equal(clean[mask], dirty[mask])


@pytest.mark.parametrize("batch,rows,inputs", [(1, 8130, 64), (1, 8200, 192), (33, 250, 192), (65, 127, 128)])
def test_gemm_wide_tiles(device, batch, rows, inputs):
    """The 128 x 192 tiles of large outputs: 1536 outputs are 8 of 192, and 64 or
    65 tiles of 128 rows make 512 workgroups and more, the line.  Rows that end
    inside a tile, and row counts below, at and past 64 and 128 (waves without
    rows, tiles without any)."""
    from torch import nn

    from asrback_amd import layers

    say("gemm wide", batch, rows, inputs)
    assert -(-batch * rows // 128) * (1536 // 192) >= 512
    torch.manual_seed(16)
    linear = nn.Linear(inputs, 1536).to(device, torch.bfloat16).requires_grad_(False)
    x = torch.randn(batch, rows, inputs, device=device).bfloat16()
    counts = [min(n, rows) for n in (rows, 0, 1, 63, 64, 65, 127, 128, 129, 192, 193, rows - 1)]
    used = torch.tensor([counts[b % len(counts)] for b in range(batch)], dtype=torch.int32, device=device)
    keep = torch.arange(rows, device=device) < used[:, None]
    assert layers.gemm_takes(x, linear)
    ref = x.double() @ linear.weight.double().t().contiguous()
    got = layers.gemm(x, linear)
    assert_close(got.float().cpu(), (ref + linear.bias.double()).cpu(), "bf16")
    assert torch.equal(layers.gemm(x, linear, used)[keep], got[keep])
    held = torch.randn(batch, rows, 1536, device=device).bfloat16()
    into = held.clone()
    layers.gemm(x, linear, used, into=into)
    assert torch.equal(into[~keep], held[~keep])
    assert_close(into[keep].float().cpu(), (held.double() + ref)[keep].cpu(), "bf16")


@pytest.mark.parametrize("batch,rows,inputs,outputs", [
    (1, 1, 64, 8), (1, 33, 192, 40), (3, 17, 512, 512), (1, 300, 512, 1536), (2, 700, 128, 1000), (5, 504, 512, 1536),
    (1, 1500, 1280, 136),
    # 16 x 16 tiles, 32 x 16, and reductions of two, four and eight waves.
    (1, 32, 1280, 1280), (2, 31, 768, 760), (1, 5, 320, 24), (1, 100, 768, 768), (3, 50, 1024, 1000), (1, 90, 2048, 512)])
def test_gemm(device, batch, rows, inputs, outputs):
    """The bf16 linear layer over both tilings and their edges (rows, outputs
    and reductions that fill no tile), with and without bias, added to what the
    output holds, over strided rows, and with row counts, whose other rows stay
    as they were; against float64, one bf16 rounding (2e-2 of the largest)."""
    from torch import nn

    from asrback_amd import layers

    say("gemm", batch, rows, inputs, outputs)
    torch.manual_seed(9)
    linear = nn.Linear(inputs, outputs).to(device, torch.bfloat16).requires_grad_(False)
    wide = torch.randn(batch, rows, inputs + 64, device=device).to(torch.bfloat16)
    used = torch.tensor([rows, rows // 2, 0, 1, rows - 1][:batch], dtype=torch.int32, device=device)
    keep = torch.arange(rows, device=device) < used[:, None]
    for x in (wide[..., :inputs].contiguous(), wide[..., 64:]):
        assert layers.gemm_takes(x, linear)
        ref = x.double() @ linear.weight.double().T.contiguous()
        got = layers.gemm(x, linear)
        assert_close(got.float().cpu(), (ref + linear.bias.double()).cpu(), "bf16")
        part = layers.gemm(x, linear, used)
        assert torch.equal(part[keep], got[keep])
        held = torch.randn(batch, rows, outputs, device=device).to(torch.bfloat16)
        into = held.clone()
        assert layers.gemm(x, linear, used, into=into) is into
        assert torch.equal(into[~keep], held[~keep])
        assert_close(into[keep].float().cpu(), (held.double() + ref)[keep].cpu(), "bf16")


@pytest.mark.parametrize("where", ["module", "class"])
@pytest.mark.parametrize("name", ["project_key_value", "step", "attend", "_split_heads"])
def test_decoder_step_runs_replaced_methods(device, name, where, monkeypatch):
    """A method of a step's attention replaced on the module or its class takes
    effect in the decoder layer."""
    from asrback_amd import whisper
    from asrback_amd.attention import KeyPrefix

    config = {"d_model": 128, "decoder_attention_heads": 2, "decoder_ffn_dim": 256}
    layer = whisper.DecoderLayer(config).to(device).requires_grad_(False)
    x = torch.randn(3, 1, 128, device=device)
    cache = tuple(torch.randn(3, 2, 16, 64, device=device) for _ in range(4))
    positions = torch.tensor([0, 4, 15], device=device)
    mask = KeyPrefix(positions=positions)
    assert layer._rows_take(x)
    called = []
    method = getattr(whisper.MultiHeadAttention, name)
    if where == "class":
        monkeypatch.setattr(whisper.MultiHeadAttention, name,
                            lambda self, *a, **k: called.append(1) or method(self, *a, **k))
    else:
        module = layer.encoder_attn if name == "attend" else layer.self_attn
        monkeypatch.setattr(module, name, lambda *a, **k: called.append(1) or method(module, *a, **k), raising=False)
    assert not layer._rows_take(x)
    layer(x, cache, positions, None, mask)
    assert called


def test_replaced_class_forwards_run(device, monkeypatch):
    """A forward (or call) replaced on a module's class is not passed over by
    the kernels that compute it."""
    from torch import nn

    from asrback_amd import gemma4, layers, qwen3_asr

    linear = nn.Linear(64, 64).to(device, torch.bfloat16).requires_grad_(False)
    x = torch.randn(1, 4, 64, device=device, dtype=torch.bfloat16)
    assert layers.gemm_takes(x, linear)
    for cls in (nn.Linear, nn.LayerNorm, nn.Embedding, qwen3_asr.RMSNorm, gemma4.RMSNorm):
        module = cls(8, 8) if cls in (nn.Linear, nn.Embedding) else cls(8, eps=1e-6)
        assert layers.unhooked(module)
        with monkeypatch.context() as patch:
            patch.setattr(cls, "forward", lambda self, t: t)
            assert not layers.unhooked(module)
            if cls is nn.Linear:
                assert not layers.gemm_takes(x, linear)
        with monkeypatch.context() as patch:
            patch.setattr(nn.Module, "__call__", lambda self, *a: a)
            assert not layers.unhooked(module)
        assert layers.unhooked(module)


def test_layers_of_other_widths_are_refused(device):
    """An output layer whose width is not that of what it is added to is
    refused on the host, by the kernels and by the modules (as their ops
    refuse it)."""
    from torch import nn

    from asrback_amd import layers, sensevoice, whisper
    from asrback_amd.attention import KeyPrefix

    x = torch.randn(2, 1, 128, device=device)
    for outputs in (64, 256):
        linear = nn.Linear(128, outputs, bias=False).to(device).requires_grad_(False)
        with pytest.raises(ValueError, match="residual"):
            layers.rows_linear(x, [linear], residual=x)
        half = nn.Linear(128, outputs, bias=False).to(device, torch.bfloat16).requires_grad_(False)
        with pytest.raises(RuntimeError, match="added to"):
            layers.gemm(x.bfloat16(), half, into=torch.zeros(2, 1, 128, device=device, dtype=torch.bfloat16))

        config = {"d_model": 128, "decoder_attention_heads": 2, "decoder_ffn_dim": 256}
        cache = tuple(torch.randn(2, 2, 16, 64, device=device) for _ in range(4))
        positions = torch.tensor([0, 4], device=device)
        for module, name, inputs in (("self_attn", "out_proj", 128), ("encoder_attn", "out_proj", 128), (None, "fc2", 256)):
            layer = whisper.DecoderLayer(config)
            setattr(layer if module is None else getattr(layer, module), name, nn.Linear(inputs, outputs))
            layer = layer.to(device).requires_grad_(False)
            with pytest.raises(RuntimeError):
                layer(x, cache, positions, None, KeyPrefix(positions=positions))
        attention = sensevoice.SANMAttention(128, 128, 1, 11)
        attention.linear_out = nn.Linear(128, outputs, bias=False)
        attention = attention.to(device, torch.bfloat16).requires_grad_(False)
        with pytest.raises(RuntimeError):
            attention(torch.randn(2, 70, 128, device=device, dtype=torch.bfloat16), None, None)

    # The weight's own shape counts, as in F.linear, not what the module was built with.
    linear = nn.Linear(128, 128).to(device).requires_grad_(False)
    linear.weight = nn.Parameter(linear.weight[:64].clone(), requires_grad=False)
    assert not layers.rows_linear_takes(x, [linear], [], [])  # a bias of another length
    linear.bias = nn.Parameter(linear.bias[:64].clone(), requires_grad=False)
    assert layers.rows_linear_takes(x, [linear], [], [])
    (got,) = layers.rows_linear(x, [linear])
    assert_close(got.cpu(), linear(x).cpu(), "f32")
    half = linear.to(torch.bfloat16)
    assert_close(layers.gemm(x.bfloat16(), half).float().cpu(), half(x.bfloat16()).float().cpu(), "bf16")

    class Wrapped(nn.Module):  # a layer that is no nn.Linear and has its weight alone
        def __init__(self, linear):
            super().__init__()
            self.weight, self.bias = linear.weight, linear.bias

        def forward(self, t):
            return nn.functional.linear(t, self.weight, self.bias)

    layer = whisper.DecoderLayer(config).to(device).requires_grad_(False)
    want = layer(x, tuple(t.clone() for t in cache), positions, None, KeyPrefix(positions=positions))
    layer.self_attn.out_proj, layer.fc2 = Wrapped(layer.self_attn.out_proj), Wrapped(layer.fc2)
    got = layer(x, tuple(t.clone() for t in cache), positions, None, KeyPrefix(positions=positions))
    assert_close(got.cpu(), want.cpu(), "module", 1e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width,rows", [(384, 9), (768, 16), (1024, 13), (1280, 12), (1280, 13), (1280, 16)])
def test_decoder_layer_rows_match_the_ops(device, dtype, width, rows, monkeypatch):
    """A whole decoder layer's step at nine to sixteen rows through the row
    kernels against its ops (float32: the same sums in another order; bf16:
    every activation rounded at the same places), and the lines past which
    the ops run."""
    from asrback_amd import whisper
    from asrback_amd.attention import KeyPrefix

    say("decoder layer", dtype, width, rows)
    heads = width // 64
    config = {"d_model": width, "decoder_attention_heads": heads, "decoder_ffn_dim": 4 * width}
    torch.manual_seed(14)
    layer = whisper.DecoderLayer(config).to(device, dtype).requires_grad_(False)
    with torch.no_grad():
        for name, weight in layer.named_parameters():
            if "norm" in name:
                weight.normal_(float("weight" in name), 0.2)
    x = torch.randn(rows, 1, width, device=device).to(dtype)
    cache = [torch.randn(rows, heads, n, 64, device=device).to(dtype) for n in (64, 64, 90, 90)]
    positions = torch.arange(rows, device=device) * 3
    taken = layer._rows_take(x)
    # fc2's inputs: at most 1024 vectors of 16 bytes, and bf16 4096 past twelve rows.
    assert taken == (4 * width <= (4096 if dtype == torch.float32 or rows > 12 else 8192))
    results = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(whisper, "rows_linear_takes", lambda *a: False)
        copies = tuple(t.clone() for t in cache)
        results.append((layer(x, copies, positions, None, KeyPrefix(positions=positions)), *copies[:2]))
    tolerance = 1e-4 if dtype == torch.float32 else 2e-2
    for got, want in zip(*results):
        assert_close(got.float().cpu(), want.float().cpu(), "module", tolerance)


def test_vocabulary_product_lines(device):
    """Rows go to the kernel up to 2560 values, three and four bf16 ones up to
    640 inputs."""
    from asrback_amd import layers

    for dtype, rows, inputs, takes in ((torch.bfloat16, 3, 768, False), (torch.bfloat16, 4, 640, True),
                                       (torch.bfloat16, 2, 1280, True), (torch.float32, 3, 768, True),
                                       (torch.float32, 4, 768, False), (torch.bfloat16, 5, 384, False)):
        x, weight = (torch.randn(n, inputs, device=device).to(dtype) for n in (rows, 1000))
        assert layers.rows_product_takes(x, weight) == takes
