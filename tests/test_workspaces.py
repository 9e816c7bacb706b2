"""The device workspaces that the Python layer keeps for decode and prefill: how they grow, who
shares them, and what a captured graph holds."""

import pytest
import torch

from kavor_amd.layers import attention
from tests.helpers import gen, randn_bf16

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


@pytest.fixture
def fresh(cuda_device, monkeypatch):
    """Starts a test without workspaces; those of graphs captured earlier stay alive."""
    for name in ("_workspaces", "_prefill_workspaces"):
        monkeypatch.setattr(attention, name, {})
    monkeypatch.setattr(attention, "_retired_workspaces", [])
    return cuda_device


def _decode(d, B, hq, hkv, width, bs=256, seed=1):
    """An eager decode of B one-page sequences under a block table of `width` pages."""
    g = gen(seed)
    kc, vc = (randn_bf16((4, bs, hkv, 128), g).to(d) for _ in range(2))
    bt = torch.zeros(B, width, dtype=torch.int32, device=d)
    ctx = torch.full((B,), 40, dtype=torch.int32, device=d)
    return attention.paged_decode(randn_bf16((B, hq, 128), g).to(d), kc, vc, ctx, bt, SCALE)


def test_growing_step_by_step_retires_less_than_is_held(fresh):
    """Calls whose block tables widen page by page, then whose batches grow: the buffers that
    were outgrown add up to less than the one in use."""
    d = fresh
    for width in range(1, 129):
        _decode(d, 1, 64, 8, width)
    for batch in range(1, 65):
        _decode(d, batch, 64, 8, 36)
    held = attention._workspaces[d.index].numel()
    assert sum(t.numel() for t in attention._retired_workspaces) < held
    need = attention.decode_workspace_bytes(64, 64, 128, 4 * 36, 256)
    assert need <= held <= 2 * need
