"""Decode attention with one workgroup per (request, KV head): the chunked grid's unsplit form
(bf16, head_dim 128, contexts below 2048 rows).

Against the float64 oracle (max-abs <= 2e-2, mean-abs <= 2e-3 for bf16 I/O with fp32
accumulation) over one, four and eight waves per workgroup, with lengths on and around the
16-key stages and the workgroup's whole stages, invalid positions, arenas read through
offsets, and masks of every type that hide keys in the middle, at the end or all but one.
The weights enter the products with all bits of their float32, so the result is as close to float64
as the split kernel's: its error norm is held to 1.02 times that kernel's, and outputs whose terms
cancel to what float32 weights leave."""
import numpy as np
import pytest
import torch

from oracle import attention as oatt
from oracle import bf16 as obf16
from oracle import rope as orope
from tests._util import assert_attention_close, bits, f64

pytestmark = pytest.mark.gpu

D = 128
# (batch, kv_heads, capacity): one wave; one wave with two stages; four waves (64 pairs and more);
# eight waves, one stage to sixteen
SHAPES = [(9, 8, 16), (5, 4, 32), (40, 8, 33), (64, 8, 300), (3, 8, 33), (7, 8, 130), (2, 2, 512), (5, 4, 1500), (2, 8, 2047)]


def _problem(batch, kv_heads, group, capacity, seed, device, tokens=1):
    gen = torch.Generator(device=device).manual_seed(seed)
    keys = torch.randn(batch, kv_heads, capacity, D, generator=gen, device=device, dtype=torch.bfloat16)
    values = torch.randn(keys.shape, generator=gen, device=device, dtype=torch.bfloat16)
    rows = torch.randn(batch, tokens, kv_heads * (group + 2), D, generator=gen, device=device, dtype=torch.bfloat16)
    q, k, v = rows.split([kv_heads * group, kv_heads, kv_heads], dim=2)
    host = torch.Generator().manual_seed(seed)
    positions = torch.randint(0, capacity, (batch,), generator=host)
    edge = torch.tensor([capacity - 1, 0, 15, 16, 17, 63, 64, 127, 128, 31, -1, capacity])
    edge = edge[(edge <= capacity)][:batch - 1]
    positions[:len(edge)] = edge
    return keys, values, q, k, v, positions


def _valid(positions, capacity):
    return ((positions >= 0) & (positions < capacity)).numpy()


@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("batch,kv_heads,capacity", SHAPES)
def test_attention_matches_the_oracle_and_the_split_kernel(pkg, device, batch, kv_heads, capacity, group):
    keys, values, q, _, _, positions = _problem(batch, kv_heads, group, capacity, 3 + capacity, device)
    assert pkg.decode_grid_for(batch, 1, kv_heads * group, kv_heads, D, capacity) == "chunked"
    dpos = positions.to(device)
    out = pkg.decode_attention(q, keys, values, dpos)
    split = pkg.decode_attention(q, keys, values, dpos, max_chunks=1)
    offsets = torch.arange(batch, device=device).flip(0) * keys.stride(0)
    moved = pkg.decode_attention(q, keys, values, dpos, kv_offsets=offsets)
    flipped = pkg.decode_attention(q, keys.flip(0).contiguous(), values.flip(0).contiguous(), dpos)
    ok = _valid(positions, capacity)
    assert bool((out[~torch.from_numpy(ok)] == 0).all())
    assert torch.equal(moved, flipped)
    expected = oatt.decode_attention(f64(q), f64(keys), f64(values), np.where(ok, positions.numpy(), 0), D ** -0.5)[ok]
    assert_attention_close(f64(out)[ok], expected)
    error, reference = (np.linalg.norm(f64(x)[ok] - expected) for x in (out, split))
    assert error <= 1.02 * reference


@pytest.mark.parametrize("group,tokens", [(1, 1), (2, 1), (4, 1), (2, 2), (4, 2)])
@pytest.mark.parametrize("batch,kv_heads,capacity", [(64, 8, 16), (64, 8, 40), (7, 8, 40)])
def test_cancelling_terms_keep_float32_weights(pkg, device, batch, kv_heads, capacity, group, tokens):
    """|out - exact| <= 2^-8 |exact| (the output's rounding to bf16: half of 2^-7) + 2^-21 times the
    mean |value| (float32 weights, sums and reciprocal: about 2^-23 each; the scores are kept small,
    so their rounding adds less).  Weights of 16 bits are off by up to 2^-18 of it, which shows in
    the outputs that cancel."""
    gen = torch.Generator(device=device).manual_seed(capacity + group)
    keys = torch.randn(batch, kv_heads, capacity, D, generator=gen, device=device, dtype=torch.bfloat16)
    values = torch.randn(keys.shape, generator=gen, device=device, dtype=torch.bfloat16)
    q = torch.randn(batch, tokens, kv_heads * group, D, generator=gen, device=device, dtype=torch.bfloat16) / 8
    positions = tokens + torch.arange(batch) % 13
    out = f64(pkg.decode_attention(q, keys, values, positions.to(device)))
    for t in range(tokens):
        last = positions.numpy() - tokens + 1 + t
        exact = oatt.decode_attention(f64(q[:, t:t + 1]), f64(keys), f64(values), last, D ** -0.5)
        size = oatt.decode_attention(f64(q[:, t:t + 1]), f64(keys), np.abs(f64(values)), last, D ** -0.5)
        over = np.abs(out[:, t:t + 1] - exact) - (2.0 ** -8 * np.abs(exact) + 2.0 ** -21 * size)
        assert over.max() <= 0, (over / size).max()


@pytest.mark.parametrize("tokens", [1, 2])
@pytest.mark.parametrize("batch,kv_heads,capacity", SHAPES)
def test_fused_step(pkg, device, batch, kv_heads, capacity, tokens):
    """RoPE, the paired write (bit-exact) and the attention, one and two tokens, against the
    rotated rows written by the oracle."""
    group = 2
    keys, values, q, k, v, positions = _problem(batch, kv_heads, group, capacity, 5 + capacity, device, tokens)
    positions[positions == 0] = tokens - 1  # every token has a position
    ok = _valid(positions, capacity)
    at = torch.where(torch.from_numpy(ok), positions, torch.full_like(positions, tokens - 1))
    where = (at[:, None] - tokens + 1 + torch.arange(tokens)).to(device)
    cos, sin = pkg.rope_tables(where, D)
    before_k, before_v = bits(keys).copy(), bits(values).copy()
    out = pkg.decode_step(q, k, v, keys, values, positions.to(device), cos, sin)
    cb, sb = bits(cos)[:, :, None, :], bits(sin)[:, :, None, :]
    q_rot, k_rot = orope.rope_bf16(bits(q), cb, sb), orope.rope_bf16(bits(k), cb, sb)
    for b in np.flatnonzero(ok):
        rows = where[b].cpu().numpy()
        before_k[b][:, rows] = k_rot[b].transpose(1, 0, 2)
        before_v[b][:, rows] = bits(v)[b].transpose(1, 0, 2)
    assert np.array_equal(bits(keys), before_k) and np.array_equal(bits(values), before_v)
    assert bool((out[~torch.from_numpy(ok)] == 0).all())
    kf, vf, qf = obf16.from_bits(before_k), obf16.from_bits(before_v), obf16.from_bits(q_rot)
    for t in range(tokens):
        last = np.where(ok, at.numpy() - tokens + 1 + t, 0)
        expected = oatt.decode_attention(qf[:, t:t + 1], kf, vf, last, D ** -0.5)[ok]
        assert_attention_close(f64(out)[ok][:, t:t + 1], expected)


@pytest.mark.parametrize("tokens", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bool, torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("batch,kv_heads,capacity", [(6, 8, 30), (33, 8, 131), (3, 8, 515), (2, 4, 2047)])
def test_masks(pkg, device, batch, kv_heads, capacity, dtype, tokens):
    """Rows that hide a random half, everything past a prefix, all but the last or the first
    key, and nothing; odd widths put the rows off their words' boundaries."""
    group = 2
    keys, values, q, _, _, _ = _problem(batch, kv_heads, group, capacity, 7 + capacity, device, tokens)
    gen = torch.Generator().manual_seed(capacity)
    seen = torch.rand(batch, tokens, capacity, generator=gen) < 0.5
    seen[..., 0] = True
    key = torch.arange(capacity)
    for b in range(batch):
        for t in range(tokens):
            kind = (b + t) % 5
            if kind == 1: seen[b, t] = key <= (37 * b) % capacity
            if kind == 2: seen[b, t] = key == capacity - 1
            if kind == 3: seen[b, t] = key == 0
            if kind == 4: seen[b, t] = True
    mask = seen if dtype == torch.bool else torch.zeros(seen.shape, dtype=dtype).masked_fill(~seen, torch.finfo(dtype).min)
    positions = torch.full((batch,), capacity - 1, device=device, dtype=torch.int64)
    out = pkg.decode_attention(q, keys, values, positions, mask=mask.to(device)[:, None])
    scores = np.einsum("bshgd,bhnd->bshgn", f64(q).reshape(batch, tokens, kv_heads, group, D), f64(keys)) * D ** -0.5
    scores = np.where(seen.numpy()[:, :, None, None], scores, -np.inf)
    weights = np.exp(scores - scores.max(-1, keepdims=True))
    weights /= weights.sum(-1, keepdims=True)
    expected = np.einsum("bshgn,bhnd->bshgd", weights, f64(values)).reshape(batch, tokens, -1, D)
    assert_attention_close(f64(out), expected)


def test_infinite_values_of_visible_keys_stay(pkg, device):
    keys, values, q, _, _, _ = _problem(4, 8, 2, 200, 11, device)
    mask = (torch.arange(200, device=device) < 50).expand(4, 200)[:, None, None, :].contiguous()
    positions = torch.full((4,), 199, device=device, dtype=torch.int64)
    expected = pkg.decode_attention(q, keys, values, positions, mask=mask)
    again = pkg.decode_attention(q, keys[:, :, :50], values[:, :, :50], torch.full_like(positions, 49))
    assert torch.equal(expected, again)
    values[:, :, 3, 5] = float("inf")  # a visible key: the dim is infinite, the others unchanged
    out = pkg.decode_attention(q, keys, values, positions, mask=mask)
    assert bool(torch.isposinf(out[..., 5]).all())
    keep = torch.arange(D, device=device) != 5
    assert torch.equal(out[..., keep], expected[..., keep])


@pytest.mark.parametrize("tokens", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bool, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch,kv_heads,capacity,visible", [
    (5, 8, 30, [7, 16, 30, 1, 21]), (16, 8, 200, [50, 1, 64, 100, 199]), (5, 8, 300, [50, 129, 257, 3, 300]),
    (2, 4, 1500, [70, 1003])])
def test_keys_behind_the_last_visible_one_do_not_reach_the_output(pkg, device, batch, kv_heads, capacity, visible, dtype, tokens):
    """One, four and eight waves; infinite keys and NaN values from the first hidden row on, of which
    a wave's first stages are read: bit for bit the outputs over finite rows there."""
    keys, values, q, _, _, _ = _problem(batch, kv_heads, 2, capacity, 17, device, tokens)
    ends = torch.tensor([visible[b % len(visible)] for b in range(batch)])
    seen = torch.arange(capacity) < ends[:, None]
    mask = seen if dtype == torch.bool else torch.zeros(seen.shape, dtype=dtype).masked_fill(~seen, torch.finfo(dtype).min)
    mask = mask.to(device)[:, None, None].expand(batch, 1, tokens, capacity).contiguous()
    positions = torch.full((batch,), capacity - 1, device=device, dtype=torch.int64)
    expected = pkg.decode_attention(q, keys, values, positions, mask=mask)
    hidden = (~seen).to(device)[:, None, :, None]
    out = pkg.decode_attention(q, keys.masked_fill(hidden, float("inf")), values.masked_fill(hidden, float("nan")),
                               positions, mask=mask)
    assert bool(torch.isfinite(expected).all()) and torch.equal(out, expected)


@pytest.mark.parametrize("tokens", [1, 2])
@pytest.mark.parametrize("batch,kv_heads,capacity", [(3, 8, 30), (16, 8, 131), (3, 8, 515)])
def test_a_row_that_hides_every_key_is_nan_and_alone(pkg, device, batch, kv_heads, capacity, tokens):
    """No weight to divide by: NaN, as on the split kernel; every other row as without that one."""
    keys, values, q, _, _, _ = _problem(batch, kv_heads, 2, capacity, 19, device, tokens)
    seen = torch.rand(batch, tokens, capacity, generator=torch.Generator().manual_seed(3)) < 0.5
    seen[..., capacity // 2] = True
    positions = torch.full((batch,), capacity - 1, device=device, dtype=torch.int64)
    full = pkg.decode_attention(q, keys, values, positions, mask=seen.to(device)[:, None])
    seen[1, tokens - 1] = False
    out = pkg.decode_attention(q, keys, values, positions, mask=seen.to(device)[:, None])
    split = pkg.decode_attention(q, keys, values, positions, mask=seen.to(device)[:, None], max_chunks=1)
    assert bool(torch.isnan(out[1, tokens - 1]).all()) and bool(torch.isnan(split[1, tokens - 1]).all())
    others = torch.ones(batch, tokens, dtype=torch.bool)
    others[1] = False
    assert torch.equal(out[others], full[others])
    if tokens == 2:
        assert_attention_close(f64(out[1, :1]), f64(full[1, :1]))


def test_step_in_a_graph_follows_rewritten_positions(pkg, device):
    keys, values, q, k, v, positions = _problem(6, 8, 2, 300, 13, device)
    positions = positions.clamp(0, 299).to(device)
    cos, sin = pkg.rope_tables(positions, D)
    out = torch.empty_like(q)
    pkg.decode_step(q, k, v, keys, values, positions, cos, sin, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.inference_mode(), torch.cuda.graph(graph):
        pkg.decode_step(q, k, v, keys, values, positions, cos, sin, out=out)
    for step in range(3):
        positions.copy_((positions * 7 + 13 + step) % 300)
        keys2, values2 = keys.clone(), values.clone()
        expected = pkg.decode_step(q, k, v, keys2, values2, positions, cos, sin)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, expected) and torch.equal(keys, keys2) and torch.equal(values, values2)


@pytest.mark.parametrize("batch,kv_heads,capacity,group,tokens,chunks", [
    (65, 8, 40, 1, 1, 1), (3, 8, 1100, 1, 1, 18), (513, 8, 33, 2, 1, 1), (513, 8, 40, 1, 2, 1)])
def test_many_pairs_of_few_rows_stay_split(pkg, device, batch, kv_heads, capacity, group, tokens, chunks):
    """Calls past the unsplit form's lines: bit for bit the split kernel's with its own chunk count, and
    one request fewer (or none past the line) as close to it."""
    keys, values, q, _, _, positions = _problem(batch, kv_heads, group, capacity, 23, device, tokens)
    positions = positions.clamp(tokens - 1, capacity - 1).to(device)
    out = pkg.decode_attention(q, keys, values, positions)
    assert torch.equal(out, pkg.decode_attention(q, keys, values, positions, max_chunks=chunks))
    fewer = pkg.decode_attention(q[1:], keys[1:], values[1:], positions[1:])
    assert_attention_close(f64(fewer), f64(out[1:]))


@pytest.mark.parametrize("batch,capacity,dtype,head_dim", [
    (6, 300, torch.bfloat16, 128), (64, 1024, torch.bfloat16, 128), (4, 2100, torch.bfloat16, 128),
    (5, 200, torch.float32, 128), (5, 200, torch.bfloat16, 64)])
def test_the_operator_call_attends_every_key_on_each_grid(pkg, device, batch, capacity, dtype, head_dim):
    """``attention`` without positions: the launch that reads no position vector, bit for bit the
    one given the last position of every request."""
    from types import SimpleNamespace
    module = SimpleNamespace(training=False, is_causal=True, sliding_window=None)
    gen = torch.Generator(device=device).manual_seed(capacity)
    query = torch.randn(batch, 16, 1, head_dim, generator=gen, device=device, dtype=dtype)
    keys, values = (torch.randn(batch, 8, capacity, head_dim, generator=gen, device=device, dtype=dtype) for _ in range(2))
    seen = torch.rand(batch, 1, 1, capacity, generator=gen, device=device) < 0.7
    last = torch.full((batch,), capacity - 1, device=device, dtype=torch.int64)
    for mask in (seen, None):
        out, _ = pkg.attention(module, query, keys, values, mask)
        assert torch.equal(out, pkg.decode_attention(query.transpose(1, 2), keys, values, last, mask=mask))
