"""What the native host side of an attention call does not recognise is left to the general way (no GPU needed)."""
import torch


def test_other_tensors_are_not_recognised():
    from lingbot_map_amd import _native as N
    t = torch.zeros(8, 2, 64)
    assert N.host.frames_key(t, t, t, 1) is None                       # on the CPU
    assert N.host.frames_key(None, t, t, 1) is None and N.host.frames_key(t, "k", 3, 1) is None
    assert N.host.frames_key(t, t, t) is None and N.host.frames_key(t, t, t, 1 << 80) is None
    assert N.host.rows_fit(t, t, t, 8, 2, 64, True) is False and N.host.rows_fit(None, None, None, 8, 2, 64, True) is False


def test_attend_refuses_what_was_not_recognised():
    import pytest
    from lingbot_map_amd import _native as N
    t = torch.zeros(8, 2, 64)
    with pytest.raises(TypeError):
        N.host.attend(t, t, t, t, 0, 0, 0, 0, t, 1.0, b"")
