"""What a call keeps of its groups' tokens until their outputs are put together (no GPU needed)."""
import types

import pytest
import torch
from torch import nn


class Scaled(nn.Module):
    """A block that somebody put in a block's place: twice its input, in place or not."""

    def __init__(self, in_place):
        super().__init__()
        self.in_place, self.norm1 = in_place, nn.Identity()

    def forward(self, x, normed=None, next_norm=None, **kw):
        x = x.mul_(2) if self.in_place else 2 * x
        return x if next_norm is None else (x, None)


@pytest.mark.parametrize("selected", [None, [0, 2]])
@pytest.mark.parametrize("stacked", [False, True])
def test_replaced_blocks_that_work_in_place(selected, stacked):
    """A frame block that overwrites its input leaves the outputs of the groups before it as they were."""
    from lingbot_map_amd import HipAggregatorStream
    torch.manual_seed(0)
    model = HipAggregatorStream(embed_dim=64, depth=3, num_heads=1)
    model.kv_cache_manager = types.SimpleNamespace(num_frames=0)
    model.frame_blocks = nn.ModuleList([Scaled(i > 0) for i in range(3)])
    model.global_blocks = nn.ModuleList([Scaled(False) for _ in range(3)])
    images = torch.rand(1, 1, 3, 28, 42)
    with torch.no_grad():
        tokens = model._embed_images(images)[0][None]
        outs, _ = model(images, selected_idx=selected, stacked=stacked)
    assert torch.is_tensor(outs) == stacked
    groups = range(3) if selected is None else selected
    assert len(outs) == len(groups)
    for out, g in zip(outs, groups):
        assert torch.equal(out, torch.cat([tokens * 2.0 ** (2 * g + 1), tokens * 2.0 ** (2 * g + 2)], dim=-1)), g
