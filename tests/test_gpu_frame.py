"""The kernels around the blocks of a frame against the torch operations they stand for, bit for bit."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def ptr(t):
    return C.c_void_p(t.data_ptr())


def _native_calls(monkeypatch, *names):
    """How often each of the library's entry points is called."""
    from lingbot_map_amd import _native as N
    count = dict.fromkeys(names, 0)
    for name in names:
        def counted(*args, name=name, own=getattr(N.lib, name)):
            count[name] += 1
            return own(*args)
        monkeypatch.setattr(N.lib, name, counted)
    return count


@pytest.mark.parametrize("pairs,shape,dtype", [(1, (1, 1, 1, 8), torch.bfloat16), (4, (1, 1, 261, 1024), torch.bfloat16),
                                               (3, (2, 1, 37, 768), torch.float32), (33, (1, 2, 5, 24), torch.bfloat16), (2, (1, 1, 9, 12), torch.bfloat16)])
def test_group_outputs(pairs, shape, dtype, monkeypatch):
    """One pair, more than one launch takes, last workgroups that are nearly empty, rows that are no whole pieces (left to
    torch), and one tensor for all."""
    from lingbot_map_amd import _native as N
    from lingbot_map_amd.aggregator import _group_outputs
    count = _native_calls(monkeypatch, "lbm_group_outputs")
    launches = -(-pairs // N.MAX_GROUPS) if shape[-1] * torch.finfo(dtype).bits // 8 % 16 == 0 else 0
    parts = [(torch.randn(shape, device="cuda").to(dtype), torch.randn(shape, device="cuda").to(dtype)) for _ in range(pairs)]
    want = [torch.cat(p, dim=-1) for p in parts]
    with torch.no_grad():
        got, whole = _group_outputs(parts), _group_outputs(parts, stacked=True)
        assert count["lbm_group_outputs"] == 2 * launches
        apart = _group_outputs([(f.transpose(1, 2), g.transpose(1, 2)) for f, g in parts])
    assert len(got) == pairs and all(torch.equal(a, b) and a._base is None for a, b in zip(got, want))
    assert torch.equal(whole, torch.stack(want))
    assert all(torch.equal(a, torch.cat((f.transpose(1, 2), g.transpose(1, 2)), dim=-1)) for a, (f, g) in zip(apart, parts))
    if shape[1] > 1:
        assert count["lbm_group_outputs"] == 2 * launches      # (the transposed are not contiguous)
    before = count["lbm_group_outputs"]
    f, g = (t.clone().requires_grad_() for t in parts[0])      # somebody differentiates: torch's own operations
    _group_outputs([(f, g)])[0].float().sum().backward()
    assert count["lbm_group_outputs"] == before and (f.grad == 1).all() and (g.grad == 1).all()


@pytest.mark.parametrize("selected", [None, [0, 2, 3]])
def test_group_outputs_of_a_call(selected, monkeypatch):
    """The chosen groups' parts are held up to a number of bytes: one launch for all groups of a small frame, one per group
    where the bound is passed each time, the same bits, as a list and as one tensor; and where the parts are not held the
    call's peak is lower by them."""
    from lingbot_map_amd import HipAggregatorStream
    from lingbot_map_amd.aggregator import _GroupOutputs
    torch.manual_seed(1)
    model = HipAggregatorStream(embed_dim=128, depth=16, num_heads=2, aa_block_size=2, kv_cache_sliding_window=4, kv_cache_scale_frames=1,
                                page_size=16, layout="frame_pages").cuda().to(torch.bfloat16).eval()
    images = torch.rand(1, 1, 3, 14 * 9, 14 * 13, device="cuda").to(torch.bfloat16)
    count = _native_calls(monkeypatch, "lbm_group_outputs")
    groups = 8 if selected is None else len(selected)
    results, launches, peaks = [], [], []
    for held in (1 << 30, 0):
        monkeypatch.setattr(_GroupOutputs, "HELD_BYTES", held)
        for stacked in (False, True):
            model.clean_kv_cache()
            with torch.no_grad():
                model(images, selected_idx=selected, stacked=stacked)     # (whatever is kept is there)
                model.clean_kv_cache()
                before = count["lbm_group_outputs"]
                torch.cuda.synchronize()
                torch.cuda.reset_peak_memory_stats()
                base = torch.cuda.memory_allocated()
                out = model(images, selected_idx=selected, stacked=stacked)[0]
                peaks.append(torch.cuda.max_memory_allocated() - base)
            assert torch.is_tensor(out) == stacked and len(out) == 2 * groups
            launches.append(count["lbm_group_outputs"] - before)
            results.append(list(out))
            del out
    assert launches == [1, 1, groups, groups]
    assert all(torch.equal(a, b) for r in results[1:] for a, b in zip(r, results[0]))
    part = 2 * 128 * (9 * 13 + 6)
    # All 4 x groups parts are there at the held call's peak, beside all results.  The other's peak is inside a block, beside its
    # scratch memory: less than half of them here.  (Of three groups the parts are less than the call's other memory.)
    assert peaks[0] - peaks[2] >= (2 * groups * part if selected is None else 0), peaks


@pytest.mark.parametrize("frames,rows,cols,streams", [(1, 16, 16, 1), (1, 27, 37, 4), (8, 3, 5, 1)])
@pytest.mark.parametrize("f0", [0, 1, 9_999])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_stream_table(frames, rows, cols, streams, f0, dtype):
    """The blocks' table against the public one in float64, at the stream's first frames and far into it."""
    from lingbot_map_amd import HipAggregatorStream
    from lingbot_map_amd.aggregator import _plain
    model = HipAggregatorStream(embed_dim=128, depth=2, num_heads=2, enable_3d_rope=True, max_frame_num=10_100, num_streams=streams).cuda().to(dtype)
    model.total_frames_processed = f0
    with torch.no_grad():
        want = model.stream_table(frames, 14 * rows, 14 * cols, "cuda:0").to(torch.complex64).expand(streams, -1, -1, -1)
        got = model._stream_table64(frames, 14 * rows, 14 * cols, "cuda:0", streams)
        base = model._table_base(frames, rows, cols, "cuda:0")
        assert _plain(*base) and all(t.dtype == torch.float64 for t in base)      # (the kernel's path is the one that ran)
    assert got.shape == want.shape and got.is_contiguous() and torch.equal(torch.view_as_real(got), torch.view_as_real(want.contiguous()))


def test_stream_table_of_the_instance():
    """A ``stream_table`` set on the model itself is the one that the blocks and the replayed frames take."""
    from lingbot_map_amd import HipAggregatorStream
    from lingbot_map_amd.aggregator import _graph_table
    model = HipAggregatorStream(embed_dim=128, depth=2, num_heads=2, enable_3d_rope=True, num_streams=2).cuda().to(torch.bfloat16)
    own = model.stream_table
    model.stream_table = lambda *args, **kwargs: own(*args, **kwargs).conj()
    with torch.no_grad():
        want = own(1, 28, 42, "cuda:0").conj().to(torch.complex64).expand(2, -1, -1, -1)
        assert torch.equal(torch.view_as_real(model._stream_table64(1, 28, 42, "cuda:0", 2)), torch.view_as_real(want.resolve_conj()))
        assert torch.equal(_graph_table(model, (28, 42), "cuda:0"), torch.view_as_real(want[:1].resolve_conj()))


@pytest.mark.parametrize("shape", [(1, 1, 3, 14, 14), (2, 3, 3, 28, 42), (1, 1, 3, 378, 518), (1, 1, 3, 7, 9)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_normalised_images(shape, dtype, monkeypatch):
    """The kernel's values where planes are whole fours, torch's where they are not and where images are strided."""
    from lingbot_map_amd import HipAggregatorStream
    count = _native_calls(monkeypatch, "lbm_normalise_images")
    model = HipAggregatorStream(embed_dim=128, depth=2, num_heads=2).cuda().to(dtype)
    images = torch.rand(shape, device="cuda").to(dtype)
    images[0, 0, 0, 0, :3] = torch.tensor([float("inf"), float("-inf"), 0.0])
    with torch.no_grad():
        want = (images - model._resnet_mean.to(dtype)) / model._resnet_std.to(dtype)
        assert torch.equal(model._normalised(images), want) and count["lbm_normalise_images"] == (shape[-1] * shape[-2] % 4 == 0)
        wide = torch.rand(*shape[:-1], 2 * shape[-1], device="cuda").to(dtype)[..., ::2]     # strided: torch's own operations
        assert torch.equal(model._normalised(wide), (wide - model._resnet_mean.to(dtype)) / model._resnet_std.to(dtype))
    assert count["lbm_normalise_images"] == (shape[-1] * shape[-2] % 4 == 0)


@pytest.mark.parametrize("name", ["_resnet_mean", "_resnet_std"])
@pytest.mark.parametrize("shape", [(), (1, 1, 1, 1, 1), (1, 1, 1, 14, 1), (1, 1, 1, 3, 1), (3, 1, 1), (2, 1, 3, 1, 1)])
def test_normalised_images_with_another_mean_or_deviation(name, shape):
    """Replaced statistics broadcast as torch broadcasts them: one value for all colours, one per row, one set per stream."""
    from lingbot_map_amd import HipAggregatorStream
    model = HipAggregatorStream(embed_dim=128, depth=2, num_heads=2).cuda().to(torch.bfloat16)
    images = torch.rand(2, 1, 3, 14 if shape != (1, 1, 1, 3, 1) else 3, 28, device="cuda").to(torch.bfloat16)
    setattr(model, name, (0.25 + torch.rand(shape, device="cuda")).to(torch.bfloat16))
    with torch.no_grad():
        assert torch.equal(model._normalised(images), (images - model._resnet_mean) / model._resnet_std)


@pytest.mark.parametrize("n,rows,cols,channels", [(1, 1, 1, 64), (1, 9, 9, 1024), (2, 8, 8, 768), (3, 13, 5, 128), (1, 27, 37, 1024)])
def test_patch_tokens(n, rows, cols, channels, monkeypatch):
    """One patch, one short and one more than whole tiles, against the module's own operations."""
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, channels).cuda().to(torch.bfloat16)
    images = torch.randn(n, 3, 14 * rows, 14 * cols, device="cuda").to(torch.bfloat16)
    want = conv.proj(images).flatten(2).transpose(1, 2)
    with torch.no_grad():
        count = _native_calls(monkeypatch, "lbm_patch_tokens")
        got = conv(images)
        assert got.is_contiguous() and torch.equal(got, want) and count["lbm_patch_tokens"] == 1
        seen = []
        handle = conv.proj.register_forward_hook(lambda m, a, o: seen.append(o.shape))
        assert torch.equal(conv(images), want) and len(seen) == 1      # somebody listens to the convolution
        handle.remove()
    conv(images).float().sum().backward()
    assert conv.proj.bias.grad is not None and count["lbm_patch_tokens"] == 1


@pytest.mark.parametrize("bias,channels", [(1, 64), (63, 64), (128, 64), (64, 128)])
def test_patch_tokens_with_another_bias(bias, channels):
    """A bias that is not one value per channel is refused, as the convolution refuses it, and never read by the kernel."""
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, channels).cuda().to(torch.bfloat16)
    conv.proj.bias = torch.nn.Parameter(torch.zeros(bias, device="cuda", dtype=torch.bfloat16))
    with torch.no_grad(), pytest.raises(RuntimeError):
        conv(torch.randn(1, 3, 28, 28, device="cuda").to(torch.bfloat16))


@pytest.mark.parametrize("autocast", [torch.float16, torch.bfloat16])
def test_patch_tokens_under_autocast(autocast):
    """The type that the convolution gives under autocast, and its values."""
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, 128).cuda().to(torch.bfloat16)
    images = torch.randn(2, 3, 42, 28, device="cuda").to(torch.bfloat16)
    with torch.no_grad(), torch.autocast("cuda", dtype=autocast):
        want = conv.proj(images).flatten(2).transpose(1, 2)
        got = conv(images)
        assert got.dtype == want.dtype == autocast and torch.equal(got, want)


@pytest.mark.parametrize("name", ["forward", "_conv_forward", "_compiled_call_impl"])
def test_patch_tokens_with_a_method_of_the_instance(name):
    """A wrapper set on the convolution itself is what a call of it runs."""
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, 64).cuda().to(torch.bfloat16)
    images = torch.randn(1, 3, 28, 28, device="cuda").to(torch.bfloat16)
    own = conv.proj.forward if name == "_compiled_call_impl" else getattr(conv.proj, name)
    with torch.no_grad():
        plain = conv.proj(images).flatten(2).transpose(1, 2)
        setattr(conv.proj, name, lambda *args: 2 * own(*args))
        assert torch.equal(conv(images), 2 * plain)


@pytest.mark.parametrize("n,rows,cols,channels", [(1, 16, 16, 1024), (2, 27, 37, 128)])
def test_patch_tokens_of_another_convolution(n, rows, cols, channels):
    """With the convolution library switched off the bits are those of torch's own convolution, which need not round before
    its bias."""
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, channels).cuda().to(torch.bfloat16)
    images = torch.randn(n, 3, 14 * rows, 14 * cols, device="cuda").to(torch.bfloat16)
    with torch.no_grad(), torch.backends.cudnn.flags(enabled=False):
        assert torch.equal(conv(images), conv.proj(images).flatten(2).transpose(1, 2))


def test_patch_tokens_of_no_image():
    from lingbot_map_amd.aggregator import PatchConv
    conv = PatchConv(14, 64).cuda().to(torch.bfloat16)
    with torch.no_grad():
        assert conv(torch.empty(0, 3, 28, 42, device="cuda", dtype=torch.bfloat16)).shape == (0, 6, 64)


class _Dispatched(torch.utils._python_dispatch.TorchDispatchMode):
    def __init__(self, seen):
        super().__init__()
        self.seen = seen

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(func.overloadpacket.__name__)
        return func(*args, **(kwargs or {}))


class _Called(torch.overrides.TorchFunctionMode):
    def __init__(self, seen):
        super().__init__()
        self.seen = seen

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(func.__name__)
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("mode", [_Dispatched, _Called])
def test_modes_see_the_operations(mode, monkeypatch):
    """Inside a mode that counts or records torch's operations they are torch's, with the same results; a default device,
    which is a mode as well, changes nothing."""
    from lingbot_map_amd import HipAggregatorStream
    from lingbot_map_amd.aggregator import _group_outputs
    model = HipAggregatorStream(embed_dim=128, depth=2, num_heads=2, enable_3d_rope=True).cuda().to(torch.bfloat16)
    images = torch.rand(1, 1, 3, 28, 42, device="cuda").to(torch.bfloat16)
    f, g = (torch.randn(1, 1, 6, 128, device="cuda").to(torch.bfloat16) for _ in range(2))
    count = _native_calls(monkeypatch, "lbm_normalise_images", "lbm_patch_tokens", "lbm_group_outputs", "lbm_stream_table")

    def run():
        return (model._normalised(images), model.patch_embed(images[0]), _group_outputs([(f, g)])[0],
                torch.view_as_real(model._stream_table64(1, 28, 42, "cuda:0", 1)))

    with torch.no_grad():
        want = run()
        assert set(count.values()) == {1}
        with torch.device("cuda"):
            again = run()
        assert set(count.values()) == {2} and all(torch.equal(a, b) for a, b in zip(again, want))
        seen = []
        with mode(seen):
            got = run()
        assert set(count.values()) == {2} and all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(any(op in name for name in seen) for op in ("sub", "div", "conv", "cat", "polar")), seen


def test_refusals():
    from lingbot_map_amd import _native as N
    t = torch.zeros(64, device="cuda")
    two, one = (C.c_void_p * 2)(t.data_ptr(), t.data_ptr()), (C.c_void_p * 1)(t.data_ptr())
    off = (C.c_void_p * 1)(t.data_ptr() + 4)
    bad = lambda *a: N.lib.lbm_group_outputs(*a, None) == N.ERR_INVALID
    assert bad(None, one, 1, 1, 16) and bad(two, None, 1, 1, 16) and bad(two, off, 1, 1, 16) and bad(two, one, 0, 1, 16)
    assert bad(two, one, N.MAX_GROUPS + 1, 1, 16) and bad(two, one, 1, 0, 16) and bad(two, one, 1, 1, 24) and bad(two, one, 1, 1 << 31, 32)
    bad = lambda *a: N.lib.lbm_stream_table(*a, None) == N.ERR_INVALID
    assert bad(None, ptr(t), 0, ptr(t), 1, 1, 1) and bad(ptr(t), ptr(t), 0, ptr(t), 0, 1, 1) and bad(ptr(t), ptr(t), 0, ptr(t), 1 << 16, 1 << 15, 1)
    bad = lambda *a: N.lib.lbm_patch_tokens(*a, None) == N.ERR_INVALID
    assert bad(None, ptr(t), ptr(t), 1, 64, 1) and bad(ptr(t), ptr(t), ptr(t), 0, 64, 1) and bad(ptr(t), ptr(t), ptr(t), 1, 60, 1)
    assert bad(ptr(t), ptr(t), ptr(t), 1, 64, 0) and bad(ptr(t), ptr(t), C.c_void_p(t.data_ptr() + 2), 1, 64, 1)
    bad = lambda *a: N.lib.lbm_normalise_images(*a, None) == N.ERR_INVALID
    assert bad(ptr(t), ptr(t), ptr(t), None, 0, 1, 4) and bad(ptr(t), ptr(t), ptr(t), ptr(t), 7, 1, 4) and bad(ptr(t), ptr(t), ptr(t), ptr(t), 0, 1, 6)
