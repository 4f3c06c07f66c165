"""The one-pass growth (``grow_arena``) bit for bit against torch: packed and per-layer arenas, every
slot, some and none in use, blocks of less and more than a workgroup's, row sizes that the pass
takes and sizes that it does not."""
from types import SimpleNamespace

import pytest
import torch


pytestmark = pytest.mark.gpu


def _random(shape, device, seed, dtype=torch.bfloat16):
    return torch.randn(shape, generator=torch.Generator(device=device).manual_seed(seed), device=device, dtype=dtype)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("head_dim,capacity,dtype", [(128, 64, torch.bfloat16), (128, 300, torch.bfloat16), (128, 96, torch.bfloat16), (64, 16, torch.float32),
                                                     (20, 3, torch.bfloat16)])
@pytest.mark.parametrize("active", [None, 0, 2, 5])
def test_growth(pkg, device, packed, head_dim, capacity, dtype, active):
    weight = torch.empty(1, device=device, dtype=dtype)
    reference = SimpleNamespace(parameters=lambda: iter([weight]), layers=[None] * 3,
                                config=SimpleNamespace(num_key_value_heads=4, head_dim=head_dim))
    old = pkg.SlotArena(reference, 5, capacity, packed_kv=packed)
    for i, plane in enumerate(old.planes()):
        plane.copy_(_random(plane.shape, device, 10 + i, dtype))
    junk = torch.full((1 << 22,), 7.0, device=device)  # memory that a new arena may be given
    del junk
    new = pkg.grow_arena(old, capacity, active=active)
    used = 5 if active is None else active
    assert new.capacity == max(2 * capacity, 1 << capacity.bit_length()) and new.packed_kv == packed
    for target, source in zip(new.planes(), old.planes()):
        expected = torch.zeros_like(target)
        expected[:used, :, :capacity] = source[:used]
        assert torch.equal(target, expected)
    if packed:
        assert new.keys[0].data_ptr() == new.packed.data_ptr()


def test_growth_to_32_gib(pkg, device):
    """Offsets past 32 bits of bytes and of vectors, every word compared."""
    weight = torch.empty(1, device=device, dtype=torch.bfloat16)
    reference = SimpleNamespace(parameters=lambda: iter([weight]), layers=[None],
                                config=SimpleNamespace(num_key_value_heads=4, head_dim=128))
    old = pkg.SlotArena(reference, 4, 1 << 21, packed_kv=True)
    words = old.packed.view(torch.int64)
    torch.arange(words.numel(), device=device, out=words.view(-1))
    new = pkg.grow_arena(old, 1 << 21, active=3)
    assert pkg.packed_kv.can_grow_blocks(new.packed, old.packed) and new.packed.nbytes == 32 << 30
    for plane in range(2):
        for slot in range(4):
            for head in range(4):
                block, source = new.packed[plane, slot, head], old.packed[plane, slot, head]
                kept = block[:1 << 21].view(torch.int64)
                assert torch.equal(kept, source.view(torch.int64)) if slot < 3 else not bool(kept.any())
                assert not bool(block[1 << 21:].view(torch.int64).any())
