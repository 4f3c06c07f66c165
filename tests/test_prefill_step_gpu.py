"""``prefill_step`` over its launch forms: one launch that rotates the keys itself (requests of up
to 64 rows), tiles of one and two 32-key blocks (launches that fill the card or not), work items
numbered by length or request by request, and more than 64 requests.

The arena is compared bit for bit with the prologue's (``prefill_rope_write`` of keys and values),
rows past the requests included; the outputs with float64 attention over the arena (max-abs <=
2e-2, mean-abs <= 2e-3 for bf16 I/O with fp32 accumulation)."""
import pytest
import torch

from tests._util import assert_attention_close, f64

pytestmark = pytest.mark.gpu


def _step(pkg, device, lengths, kv_heads, group, head_dim, capacity, seed):
    gen = torch.Generator(device=device).manual_seed(seed)
    batch, total = len(lengths), sum(lengths)
    rows = torch.randn(total, kv_heads * (group + 2), head_dim, generator=gen, device=device, dtype=torch.bfloat16)
    q, k, v = rows.split([kv_heads * group, kv_heads, kv_heads], dim=1)
    cu = torch.tensor([0] + lengths).cumsum(0).to(device=device, dtype=torch.int32)
    cos, sin = pkg.rope_tables(torch.cat([torch.arange(n) for n in lengths]).to(device), head_dim)
    slots = torch.randperm(batch, generator=torch.Generator().manual_seed(seed)).to(device)
    arena = torch.randn(2, batch, kv_heads, capacity, head_dim, generator=gen, device=device, dtype=torch.bfloat16)
    expected = arena.clone()
    q_rot = pkg.prefill_rope_write(q, k, v, cos, sin, cu, expected[0], expected[1], kv_slots=slots)
    out = pkg.prefill_step(q, k, v, cos, sin, cu, max(lengths), arena[0], arena[1], kv_slots=slots)
    torch.cuda.synchronize()
    assert torch.equal(arena.view(torch.int16), expected.view(torch.int16))
    want = torch.zeros(out.shape, device=device, dtype=torch.float64)
    at = 0
    for b, n in enumerate(lengths):
        keys, values = (arena[i, slots[b], :, :min(n, capacity)].double().repeat_interleave(group, 0) for i in (0, 1))
        scores = torch.bmm(q_rot[at:at + n].double().transpose(0, 1).contiguous(), keys.transpose(1, 2).contiguous()) * head_dim ** -0.5
        hidden = torch.ones(n, keys.shape[1], device=device, dtype=torch.bool).triu(1)
        weights = scores.masked_fill(hidden, float("-inf")).softmax(-1)
        want[at:at + n] = torch.bmm(weights, values).transpose(0, 1)
        at += n
    assert_attention_close(f64(out), want.cpu().numpy())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("lengths,capacity", [
    ([1], 1), ([64], 64), ([1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64], 80), ([64, 20], 40), ([5] * 70, 16)])
def test_short_requests(pkg, device, lengths, capacity, group, head_dim):
    _step(pkg, device, lengths, 4, group, head_dim, capacity, 3)


@pytest.mark.parametrize("group,head_dim", [(1, 128), (2, 128), (2, 64), (4, 128)])
@pytest.mark.parametrize("lengths,capacity", [
    ([65, 128, 129], 129), ([511, 3, 96], 512), ([300, 130], 200),      # few workgroups
    ([400 + 7 * i for i in range(14)], 512),                            # many, by length
    ([130 + 4 * i for i in range(40)], 512),                            # many, request by request
    ([66] * 65, 80)])                                                   # more than 64 requests
def test_longer_requests(pkg, device, lengths, capacity, group, head_dim):
    _step(pkg, device, lengths, 8, group, head_dim, capacity, 5)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("kv_heads,lengths,capacity", [
    (2, [66] * 65, 80), (2, [65, 300, 0, 129, 512, 64], 300), (1, [2000], 2048),    # blocks of 64 queries
    (8, [512] * 9, 512)])                                                            # of 128
def test_one_head_groups(pkg, device, kv_heads, lengths, capacity, head_dim):
    _step(pkg, device, lengths, kv_heads, 1, head_dim, capacity, 9)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("lengths", [[45], [200], [400 + 7 * i for i in range(14)]])
def test_output_rows_of_eight_byte_alignment(pkg, device, lengths, head_dim):
    """An output that starts 8 bytes off a 16-byte boundary: the same rows, nothing around them."""
    gen = torch.Generator(device=device).manual_seed(7)
    total = sum(lengths)
    q, k, v = (torch.randn(total, h, head_dim, generator=gen, device=device, dtype=torch.bfloat16) for h in (16, 8, 8))
    cu = torch.tensor([0] + lengths).cumsum(0).to(device=device, dtype=torch.int32)
    cos, sin = pkg.rope_tables(torch.cat([torch.arange(n) for n in lengths]).to(device), head_dim)
    arena = torch.zeros(2, len(lengths), 8, max(lengths), head_dim, device=device, dtype=torch.bfloat16)
    expected = pkg.prefill_step(q, k, v, cos, sin, cu, max(lengths), arena[0], arena[1])
    flat = torch.full((expected.numel() + 8,), 7.0, device=device, dtype=torch.bfloat16)
    out = flat[4:-4].view(expected.shape)
    assert out.data_ptr() % 16 == 8
    pkg.prefill_step(q, k, v, cos, sin, cu, max(lengths), arena[0], arena[1], out=out)
    assert torch.equal(out, expected) and bool((flat[:4] == 7).all()) and bool((flat[-4:] == 7).all())


@pytest.mark.parametrize("lengths,max_seqlen", [
    ([150] + [126] * 60, 128),      # request by request
    ([700] + [500] * 13, 512),      # by length
    ([300, 90, 60], 96)])           # few workgroups
def test_a_request_longer_than_max_seqlen_leaves_the_others_whole(pkg, device, lengths, max_seqlen):
    """``max_seqlen`` bounds the lengths; rows past it are not attended.  Every other request's rows
    are, as in a call that names the true maximum."""
    gen = torch.Generator(device=device).manual_seed(11)
    total = sum(lengths)
    q, k, v = (torch.randn(total, h, 128, generator=gen, device=device, dtype=torch.bfloat16) for h in (16, 8, 8))
    cu = torch.tensor([0] + lengths).cumsum(0).to(device=device, dtype=torch.int32)
    cos, sin = pkg.rope_tables(torch.cat([torch.arange(n) for n in lengths]).to(device), 128)
    arena = torch.zeros(2, len(lengths), 8, max(lengths), 128, device=device, dtype=torch.bfloat16)
    expected = pkg.prefill_step(q, k, v, cos, sin, cu, max(lengths), arena[0], arena[1])
    out = torch.zeros_like(expected)
    pkg.prefill_step(q, k, v, cos, sin, cu, max_seqlen, arena[0], arena[1], out=out)
    assert_attention_close(f64(out[:max_seqlen]), f64(expected[:max_seqlen]))
    assert_attention_close(f64(out[lengths[0]:]), f64(expected[lengths[0]:]))


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("lengths,max_seqlen,past,capacity", [
    ([20, 30], 32, 7, 64), ([200, 40, 0], 40, 3, 160), ([0], 8, 5, 16), ([30] * 70, 16, 90, 128),  # one launch
    ([70] * 64, 60, 9, 96), ([70] * 65, 60, 9, 96), ([70] * 128, 64, 9, 96),   # 64 requests a workgroup
    ([300, 100, 130], 128, 70, 260), ([150] + [126] * 60, 128, 1, 512), ([300] * 70, 100, 9, 320)])
def test_every_token_reaches_the_arena(pkg, device, lengths, max_seqlen, past, capacity, group, head_dim):
    """Tokens of requests longer than ``max_seqlen`` and past the last request's end: the arena bit for
    bit the prologue's."""
    gen = torch.Generator(device=device).manual_seed(13)
    total, batch = sum(lengths) + past, len(lengths)
    q, k, v = (torch.randn(total, 4 * h, head_dim, generator=gen, device=device, dtype=torch.bfloat16) for h in (group, 1, 1))
    cu = torch.tensor([0] + lengths).cumsum(0).to(device=device, dtype=torch.int32)
    cos, sin = pkg.rope_tables(torch.arange(total, device=device), head_dim)
    slots = torch.randperm(batch, generator=torch.Generator().manual_seed(5)).to(device)
    arena = torch.randn(2, batch, 4, capacity, head_dim, generator=gen, device=device, dtype=torch.bfloat16)
    expected = arena.clone()
    pkg.prefill_rope_write(q, k, v, cos, sin, cu, expected[0], expected[1], kv_slots=slots, rotate_query=False)
    pkg.prefill_step(q, k, v, cos, sin, cu, max_seqlen, arena[0], arena[1], kv_slots=slots)
    torch.cuda.synchronize()
    assert torch.equal(arena.view(torch.int16), expected.view(torch.int16))
