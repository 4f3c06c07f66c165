"""Decode attention over arenas of 65 to 2047 rows of the types that stay split (fp32, and bf16 rows of
64): against float64 (fp32: 1e-5; bf16: max-abs <= 2e-2, mean-abs <= 2e-3) with lengths around 64, 128,
256 and 512 keys, invalid positions, one and two query tokens and masks; fp32 also against another
number of chunks."""
import numpy as np
import pytest
import torch

from oracle import attention as oatt
from tests._util import assert_attention_close, f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,head_dim", [(torch.float32, 128), (torch.float32, 64), (torch.bfloat16, 64)])
@pytest.mark.parametrize("group,tokens", [(1, 1), (1, 2), (2, 1), (2, 2), (4, 1), (4, 2)])
@pytest.mark.parametrize("capacity", [65, 513, 2047])
def test_whole_requests(pkg, device, dtype, head_dim, group, tokens, capacity):
    batch, kv_heads = 12, 4
    gen = torch.Generator(device=device).manual_seed(capacity + group)
    keys, values = (torch.randn(batch, kv_heads, capacity, head_dim, generator=gen, device=device, dtype=dtype) for _ in range(2))
    q = torch.randn(batch, tokens, kv_heads * group, head_dim, generator=gen, device=device, dtype=dtype)
    lengths = [capacity - 1, 1, 63, 64, 127, 128, 255, 256, 511, 512, -1, capacity]
    positions = torch.tensor([n if n <= capacity else capacity // 2 for n in lengths])
    ok = ((positions >= 0) & (positions < capacity)).numpy()
    out = pkg.decode_attention(q, keys, values, positions.to(device))
    split = pkg.decode_attention(q, keys, values, positions.to(device), max_chunks=3)
    assert bool((out[~torch.from_numpy(ok)] == 0).all())
    expected = oatt.decode_attention(f64(q), f64(keys), f64(values), np.where(ok, positions.numpy(), 1), head_dim ** -0.5)
    if dtype == torch.float32:
        np.testing.assert_allclose(f64(out)[ok], expected[ok], atol=1e-5, rtol=0)
        np.testing.assert_allclose(f64(out), f64(split), atol=2e-6, rtol=0)
    else:
        assert_attention_close(f64(out)[ok], expected[ok])
    seen = torch.rand(batch, tokens, capacity, generator=gen, device=device) < 0.5
    seen[..., 0] = True
    masked = pkg.decode_attention(q, keys, values, positions.to(device), mask=seen[:, None])
    expected = oatt.decode_attention(f64(q), f64(keys), f64(values), np.where(ok, positions.numpy(), 1), head_dim ** -0.5,
                                     mask=seen.cpu().numpy())
    if dtype == torch.float32:
        np.testing.assert_allclose(f64(masked)[ok], expected[ok], atol=1e-5, rtol=0)
    else:
        assert_attention_close(f64(masked)[ok], expected[ok])
