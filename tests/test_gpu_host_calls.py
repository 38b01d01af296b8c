"""The native host side of attention calls against Python's general way, which tensors of a subclass still take: the same
results, the same refusals, on whatever stream is current."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Rows(torch.Tensor):
    """Not recognised by the native way; otherwise a tensor."""


def _general(*tensors):
    return [t.as_subclass(Rows) for t in tensors]


def _rows(n, H, D, dtype, seed, count=3):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return [torch.randn(n, H, D, generator=g, device=DEV).to(dtype) for _ in range(count)]


@pytest.mark.parametrize("n,streams,H,D,dtype", [(64, 1, 4, 64, torch.bfloat16), (261, 1, 16, 64, torch.bfloat16), (300, 3, 2, 64, torch.bfloat16),
                                                 (70, 2, 3, 64, torch.float32), (4, 4, 16, 128, torch.float32)])
def test_dense_attention_both_ways(n, streams, H, D, dtype):
    from lingbot_map_amd import dense_attention
    from lingbot_map_amd._native import host, scratch_lane
    q, k, v = _rows(n, H, D, dtype, n)
    assert host.frames_key(q, k, v, streams) == (n, H, D, streams, int(dtype == torch.float32), 0)
    for prescaled in (False, True):
        want = dense_attention(*_general(q, k, v), num_streams=streams, q_prescaled=prescaled).as_subclass(torch.Tensor)
        assert torch.equal(dense_attention(q, k, v, num_streams=streams, q_prescaled=prescaled), want)
        with scratch_lane(5):
            assert torch.equal(dense_attention(q, k, v, num_streams=streams, q_prescaled=prescaled), want)
    want = dense_attention(q, k, v, num_streams=streams)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = dense_attention(q * 1, k, v, num_streams=streams)
    side.synchronize()
    assert torch.equal(got, want)
    # views: laid out as the kernels want them first, as before
    views = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in (q, k, v)]
    assert host.frames_key(*views, streams) is None or n == 1 or H == 1
    assert torch.equal(dense_attention(*views, num_streams=streams), want)
    grad = dense_attention(q.clone().requires_grad_(), k, v, num_streams=streams)
    assert torch.equal(grad, want) and not grad.requires_grad


def test_dense_attention_refuses_what_it_refused():
    from lingbot_map_amd import dense_attention
    from lingbot_map_amd._native import LbmError
    q, k, v = _rows(12, 2, 64, torch.bfloat16, 1)
    for bad in ((q, k[:6], v), (q, k, v.float()), (q.half(), k.half(), v.half()), (q.cpu(), k.cpu(), v.cpu()), (q[0], k[0], v[0])):
        with pytest.raises(AssertionError):
            dense_attention(*bad)
    for streams in (0, 5, 17, -1):
        with pytest.raises(AssertionError):
            dense_attention(q, k, v, num_streams=streams)
    with pytest.raises(LbmError):
        dense_attention(*_rows(12, 2, 32, torch.bfloat16, 1))


@pytest.mark.parametrize("tokens,D,dtype,streams", [(40, 64, torch.bfloat16, 1), (40, 64, torch.bfloat16, 2), (1, 128, torch.float32, 1)])
def test_step_both_ways(tokens, D, dtype, streams):
    from lingbot_map_amd import HipPagedKVCacheManager
    H, blocks = 4, 2
    make = lambda: HipPagedKVCacheManager(blocks, 24, tokens, H, D, dtype, torch.device(DEV), num_special_tokens=1 if tokens > 1 else 0, scale_frames=1,
                                          sliding_window=[2, 4][:streams] if streams > 1 else 2, max_total_frames=64, force_fp32=dtype == torch.float32,
                                          page_size=16, layout="frame_pages", num_streams=streams)
    a, b = make(), make()
    for f, flags in enumerate([None, None, [True] * streams, [False] * streams, [f == 0 for f in range(streams)], None, None]):
        for block in range(blocks):
            q, k, v = _rows(tokens * streams, H, D, dtype, 10 * f + block)
            got = a.step(block, q, k, v, keyframe=flags)
            want = b.step(block, *_general(q, k, v), keyframe=flags)
            assert torch.equal(got, want.as_subclass(torch.Tensor)), (f, block)
    assert all(torch.equal(x, y) for x, y in zip(a.kv_caches, b.kv_caches))
    q, k, v = _rows(tokens * streams, H, D, dtype, 99)
    before = list(a.frame_count)
    with pytest.raises((AssertionError, ValueError)):
        a.step(0, q, k[:, :2], v)
    assert a.frame_count == before
    got = a.step(0, q.to(torch.float64).to(dtype), k.double(), v.double())     # cast, as before
    assert torch.equal(got, b.step(0, *_general(q, k, v)).as_subclass(torch.Tensor))
