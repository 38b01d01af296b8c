"""The streaming branch of the block on the GPU: outputs against the same block evaluated
with a dense dict cache (the reference SDPA path's semantics) and torch SDPA in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class ReferenceSurfaceOnly:
    """Hides everything but the reference manager's call surface
    (lingbot_map/layers/flashinfer_cache.py:202-560)."""

    def __init__(self, m):
        object.__setattr__(self, "_m", m)

    def __getattr__(self, name):
        if name in ("step", "step_qkv", "set_active_streams"):
            raise AttributeError(name)
        return getattr(self._m, name)

    def __setattr__(self, name, value):
        setattr(self._m, name, value)


@pytest.mark.parametrize("reference_calls,rope", [(False, False), (True, False), (False, True), (True, True)])
def test_block_stream_matches_dense_cache(reference_calls, rope):
    """reference_calls=False takes the fused producer + `step_qkv`; True the reference's own
    method sequence.  rope=True adds the global blocks' 3-D rotary embedding (interleaved pairs,
    complex table per frame)."""
    from lingbot_map_amd import (HipPagedBlock, HipPagedKVCacheManager, RotaryPositionEmbedding3D, keyframe_flags,
                                 set_skip_append)
    from oracle.sdpa_cache import DictCacheOracle
    torch.manual_seed(5)
    rope3d = RotaryPositionEmbedding3D(attention_head_dim=64)
    dev = torch.device("cuda:0")
    dim, H, T, n_sp, scale, window, blocks = 256, 4, 53, 5, 1, 3, 2
    mods = [HipPagedBlock(dim, H, init_values=0.1, qk_norm=True, rope=True if rope else None,
                          kv_cache_sliding_window=window,
                          kv_cache_scale_frames=scale).to(dev, torch.bfloat16).eval() for _ in range(blocks)]
    for mod in mods:   # non-trivial LayerNorm parameters
        for ln in (mod.attn.q_norm, mod.attn.k_norm):
            ln.weight.data.uniform_(0.5, 1.5)
            ln.bias.data.uniform_(-0.2, 0.2)
    m = HipPagedKVCacheManager(blocks, scale + window + 16, T, H, 64, torch.bfloat16, dev, num_special_tokens=n_sp,
                               scale_frames=scale, sliding_window=window, max_total_frames=64, page_size=16,
                               layout="frame_pages")
    cache = ReferenceSurfaceOnly(m) if reference_calls else m
    dense = [DictCacheOracle(scale, window, n_sp) for _ in range(blocks)]
    flags = keyframe_flags(14, scale, 3)
    with torch.no_grad():
        for f, kf in enumerate(flags):
            x = torch.randn(1, T, dim, device=dev).to(torch.bfloat16)
            pos = None
            if rope:   # complex128 table of frame f: 5 special tokens + a 6 x 8 patch grid
                pos = rope3d(ppf=1, pph=6, ppw=8, patch_start_idx=n_sp, device=dev, f_start=f, f_end=f + 1)
                assert pos.shape == (1, 1, T, 32) and pos.dtype == torch.complex128
            set_skip_append(cache, not kf)
            y, y_ref = x, x
            for b, mod in enumerate(mods):
                y = mod(y, pos=pos, enable_3d_rope=rope, kv_cache=cache, global_idx=b, num_frames=1)
                q, k, v = mod.attn_pre(y_ref, pos=pos, enable_3d_rope=rope)
                kk, vv = dense[b].visible(k, v, keyframe=kf)
                a = torch.nn.functional.scaled_dot_product_attention(
                    q.float().permute(1, 0, 2)[None], kk.float().permute(1, 0, 2)[None], vv.float().permute(1, 0, 2)[None])
                a = a[0].permute(1, 0, 2).reshape(1, T, dim).to(torch.bfloat16)
                y_ref = mod.ffn_residual(y_ref + mod.ls1(mod.attn.proj(a)))
            set_skip_append(cache, False)
            err = (y.float() - y_ref.float()).abs()
            assert err.max().item() <= 3e-2 and err.mean().item() <= 2e-3, (f, err.max().item(), err.mean().item())
    assert m.frame_count == [sum(flags)] * blocks and m.device_header()["error"] == 0


def test_two_streams_through_one_block():
    from lingbot_map_amd import HipPagedBlock, HipPagedKVCacheManager
    torch.manual_seed(6)
    dev = torch.device("cuda:0")
    dim, H, T = 256, 4, 53
    mod = HipPagedBlock(dim, H, qk_norm=True, kv_cache_sliding_window=2, kv_cache_scale_frames=1).to(dev, torch.bfloat16).eval()
    both = HipPagedKVCacheManager(1, 19, T, H, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=1,
                                  sliding_window=2, max_total_frames=32, page_size=16, layout="frame_pages", num_streams=2)
    single = [HipPagedKVCacheManager(1, 19, T, H, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=1,
                                     sliding_window=2, max_total_frames=32, page_size=16, layout="frame_pages")
              for _ in range(2)]
    with torch.no_grad():
        for f in range(6):
            x = torch.randn(2, T, dim, device=dev).to(torch.bfloat16)
            y = mod(x, kv_cache=both, global_idx=0, num_frames=1)
            for s in range(2):
                ys = mod(x[s:s + 1], kv_cache=single[s], global_idx=0, num_frames=1)
                assert (y[s:s + 1].float() - ys.float()).abs().max().item() <= 1e-2


@pytest.mark.parametrize("rope", ["none", "2d", "interleaved"])
def test_frame_block_without_cache_matches_torch_path(rope):
    """Cache-less frames (the aggregator's frame blocks): fused producer + paged kernel over a
    trivial row table against the same module's torch operations and SDPA in fp32."""
    import torch.nn.functional as F
    from lingbot_map_amd import HipPagedBlock, RotaryPositionEmbedding2D, dense_attention
    torch.manual_seed(8)
    dev = torch.device("cuda:0")
    dim, H, T, B = 256, 4, 333, 3
    mod = HipPagedBlock(dim, H, init_values=0.1, qk_norm=True,
                        rope={"none": None, "2d": RotaryPositionEmbedding2D(), "interleaved": True}[rope]).to(dev, torch.bfloat16).eval()
    for ln in (mod.attn.q_norm, mod.attn.k_norm):
        ln.weight.data.uniform_(0.5, 1.5)
        ln.bias.data.uniform_(-0.2, 0.2)
    x = torch.randn(B, T, dim, device=dev).to(torch.bfloat16)
    pos, e3 = None, False
    if rope == "2d":
        pos = torch.stack([torch.randint(0, 20, (1, T), device=dev), torch.randint(0, 20, (1, T), device=dev)], -1).expand(B, -1, -1).contiguous()
    if rope == "interleaved":
        ang = torch.rand(1, 1, T, 32, device=dev) * 6.283185
        pos, e3 = torch.polar(torch.ones_like(ang), ang), True
    with torch.no_grad():
        assert mod.attn.can_fuse_dense(mod.norm1(x), pos, e3)
        y = mod(x, pos=pos, enable_3d_rope=e3)
        q, k, v = mod.attn._qkv(mod.norm1(x), pos, e3)
        a = F.scaled_dot_product_attention(q.float(), k.float(), v.float()).transpose(1, 2).reshape(B, T, dim).to(torch.bfloat16)
        y_ref = mod.ffn_residual(x + mod.ls1(mod.attn.proj(a)))
        # the kernel alone, three independent groups in one launch
        nhd = lambda t: t.permute(0, 2, 1, 3).reshape(B * T, H, 64).contiguous()
        o = dense_attention(nhd(q), nhd(k), nhd(v), num_streams=B).reshape(B, T, dim)
    err = (o.float() - a.float()).abs()
    assert err.max().item() <= 2e-2 and err.mean().item() <= 2e-3
    err = (y.float() - y_ref.float()).abs()
    assert err.max().item() <= 3e-2 and err.mean().item() <= 2e-3


def test_camera_trunk_blocks_one_token_per_frame_fp32():
    """The camera head's trunk (lingbot_map/heads/camera_head.py:212-219, :296-346): blocks of 128-wide
    heads in fp32 over one camera token per frame at coordinates (f, 0, 0), the anchor frames in
    one call and every later frame on its own, nothing ever evicted (attention.py:307).  Checked
    against attention over the concatenation of every frame's K/V in float64."""
    from lingbot_map_amd import HipPagedBlock, HipPagedKVCacheManager, RotaryPositionEmbedding3D
    torch.manual_seed(9)
    dev = torch.device("cuda:0")
    dim, H, D, blocks, anchor, frames = 256, 2, 128, 4, 3, 45
    rope3d = RotaryPositionEmbedding3D(attention_head_dim=D, patch_size=(1024, 1, 1), fhw_dim=(40, 44, 44))
    mods = [HipPagedBlock(dim, H, init_values=0.5, qk_norm=True, rope=True, kv_cache_sliding_window=frames,
                          kv_cache_scale_frames=anchor).to(dev).eval() for _ in range(blocks)]
    m = HipPagedKVCacheManager(blocks, frames + 8, 1, H, D, torch.float32, dev, num_special_tokens=0,
                               scale_frames=anchor, sliding_window=frames, max_total_frames=frames + 8,
                               force_fp32=True, page_size=16, layout="frame_pages")
    seen_k = [[] for _ in range(blocks)]
    seen_v = [[] for _ in range(blocks)]
    f = 0
    with torch.no_grad():
        while f < frames:
            S = anchor if f == 0 else 1
            x = torch.randn(1, S, dim, device=dev)
            pos = rope3d(ppf=S, pph=1, ppw=1, patch_start_idx=0, device=dev, f_start=f, f_end=f + S)
            y, y_ref = x, x
            for b, mod in enumerate(mods):
                y = mod(y, pos=pos, enable_3d_rope=True, kv_cache=m, global_idx=b, num_frames=S)
                q, k, v = mod.attn_pre(y_ref, pos=pos, enable_3d_rope=True)      # [S, H, D]
                seen_k[b].append(k.double()); seen_v[b].append(v.double())
                K, V = torch.cat(seen_k[b]), torch.cat(seen_v[b])
                s = torch.einsum("qhd,khd->hqk", q.double(), K) / D ** 0.5
                a = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), V).reshape(1, S, dim).float()
                y_ref = mod.ffn_residual(y_ref + mod.ls1(mod.attn.proj(a)))
            err = (y - y_ref).abs().max().item()
            assert err <= 2e-5, (f, err)
            f += S
    assert m.frame_count == [frames] * blocks and m.device_header()["error"] == 0


@pytest.mark.parametrize("reference_calls", [False, True])
def test_anchor_pass_over_several_frames_then_streaming(reference_calls):
    """Phase 1 of the streaming model (attention.py:475-511): the anchor frames arrive in one call,
    attend to one another densely, and are appended frame by frame, each block in turn, so block 0
    is several frames ahead of the others while they write.  Later frames stream one at a time
    and must see exactly the anchor frames and the window."""
    from lingbot_map_amd import HipPagedBlock, HipPagedKVCacheManager, keyframe_flags, set_skip_append
    from oracle.sdpa_cache import DictCacheOracle
    torch.manual_seed(11)
    dev = torch.device("cuda:0")
    dim, H, T, n_sp, scale, window, blocks = 256, 4, 37, 5, 3, 2, 3
    mods = [HipPagedBlock(dim, H, init_values=0.1, qk_norm=True, kv_cache_sliding_window=window,
                          kv_cache_scale_frames=scale).to(dev, torch.bfloat16).eval() for _ in range(blocks)]
    m = HipPagedKVCacheManager(blocks, scale + window + 16, T, H, 64, torch.bfloat16, dev, num_special_tokens=n_sp,
                               scale_frames=scale, sliding_window=window, max_total_frames=64, page_size=16,
                               layout="two_stream")
    cache = ReferenceSurfaceOnly(m) if reference_calls else m
    dense = [DictCacheOracle(scale, window, n_sp) for _ in range(blocks)]
    sdpa = lambda q, k, v: torch.nn.functional.scaled_dot_product_attention(
        q.float().permute(1, 0, 2)[None], k.float().permute(1, 0, 2)[None], v.float().permute(1, 0, 2)[None])[0].permute(1, 0, 2)
    flags = [True] * scale + keyframe_flags(9, 0, 2)
    with torch.no_grad():
        f = 0
        while f < len(flags):
            S = scale if f == 0 else 1
            kf = flags[f]
            x = torch.randn(1, S * T, dim, device=dev).to(torch.bfloat16)
            set_skip_append(cache, not kf)
            y, y_ref = x, x
            for b, mod in enumerate(mods):
                y = mod(y, kv_cache=cache, global_idx=b, num_frames=S)
                q, k, v = mod.attn_pre(y_ref)                                      # [S * T, H, D]
                if S > 1:
                    a = sdpa(q, k, v)
                    for i in range(S):
                        dense[b].visible(k[i * T:(i + 1) * T], v[i * T:(i + 1) * T], keyframe=True)
                else:
                    a = sdpa(q, *dense[b].visible(k, v, keyframe=kf))
                a = a.reshape(1, S * T, dim).to(torch.bfloat16)
                y_ref = mod.ffn_residual(y_ref + mod.ls1(mod.attn.proj(a)))
            set_skip_append(cache, False)
            err = (y.float() - y_ref.float()).abs()
            assert err.max().item() <= 3e-2 and err.mean().item() <= 2e-3, (f, err.max().item(), err.mean().item())
            f += S
    assert m.frame_count == [sum(flags)] * blocks and m.device_header()["error"] == 0 and not m._rows_log


def test_blocks_out_of_step_raise_with_shared_tables():
    """With one page table for all blocks a block may lag only while appending (the anchor pass);
    anything else out of step raises instead of reading or writing another frame's rows."""
    from lingbot_map_amd import HipPagedKVCacheManager
    dev = torch.device("cuda:0")
    H, D, T = 2, 64, 9
    mk = lambda **kw: HipPagedKVCacheManager(2, 24, T, H, D, torch.bfloat16, dev, num_special_tokens=1, scale_frames=1,
                                             sliding_window=2, max_total_frames=32, page_size=4, **kw)
    t = lambda: torch.randn(T, H, D, device=dev).to(torch.bfloat16)
    m = mk()
    with pytest.raises(RuntimeError, match="block 0 goes first"):
        m.append_frame(1, t(), t())
    m.append_frame(0, t(), t())
    assert m.compute_attention(1, t()).abs().max().item() == 0      # an empty block attends to nothing
    m.append_frame(0, t(), t())          # block 0 two frames ahead: allowed, rows of frame 0 are kept
    m.append_frame(1, t(), t())
    with pytest.raises(RuntimeError, match="compute_attention"):
        m.compute_attention(1, t())
    m.append_frame(1, t(), t())
    m.compute_attention(1, t())
    m.append_frame(0, t(), t())
    with pytest.raises(RuntimeError, match="block 0 starts a frame"):
        m.step(0, t(), t(), t())
    m.append_frame(1, t(), t())
    m.step(0, t(), t(), t())
    with pytest.raises(RuntimeError, match="block 0 goes first|no longer known"):
        m.append_frame(1, t(), t()); m.append_frame(1, t(), t())
    # per-block tables: any order
    p = mk(per_block_tables=True)
    p.append_frame(1, t(), t()); p.compute_attention(1, t()); p.append_frame(0, t(), t())
    assert p.device_header(0)["error"] == 0 and p.device_header(1)["error"] == 0


@pytest.mark.parametrize("rope", [False, True])
def test_chained_blocks_agree_with_the_separate_launches(rope):
    """Three blocks handing each other their row statistics (norm1 / norm2 folded into the qkv
    projection and fc1, proj / fc2 with LayerScale + residual in their store, lbm_linear_norm)
    against the same blocks run through the separate launches (LayerNorm + residual kernels,
    library GEMMs): streamed frames through a shared cache and a cache-less frame block.  The two
    paths round in different places, so the bar is the accumulated bf16 noise of three blocks, a
    small fraction of the activations' scale; the caches end up with the same page tables."""
    import math
    from lingbot_map_amd.block import HipPagedBlock, Mlp, RowStats, RotaryPositionEmbedding3D
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    T, H, D, NS, frames = 70, 2, 64, 5, 4
    C = H * D
    torch.manual_seed(17)
    dev = torch.device("cuda:0")
    blocks = [HipPagedBlock(dim=C, num_heads=H, qk_norm=True, init_values=0.5, kv_cache_sliding_window=2, kv_cache_scale_frames=1,
                            rope=object() if rope else None).to(dev).to(torch.bfloat16).eval() for _ in range(3)]
    for b in blocks:
        for m in (b.norm1, b.norm2):
            m.weight.data.add_(0.2 * torch.randn_like(m.weight)); m.bias.data.add_(0.1 * torch.randn_like(m.bias))
    rope3d = RotaryPositionEmbedding3D(attention_head_dim=D, patch_size=(1, 14, 14), max_seq_len=64) if rope else None

    def manager():
        return HipPagedKVCacheManager(num_blocks=3, max_num_frames=6, tokens_per_frame=T, num_heads=H, head_dim=D,
                                      dtype=torch.bfloat16, device=dev, num_special_tokens=NS, scale_frames=1, sliding_window=2,
                                      max_total_frames=32)

    def run(chained: bool):
        limit = Mlp.FUSED_MAX_ROWS
        Mlp.FUSED_MAX_ROWS = limit if chained else 0     # no fused launch qualifies: the separate ones run
        try:
            m, outs, kinds = manager(), [], []
            for f in range(frames):
                x = torch.randn(1, T, C, generator=torch.Generator().manual_seed(100 + f)).to(dev).to(torch.bfloat16)
                pos = rope3d(ppf=1, pph=5, ppw=13, patch_start_idx=NS, device=dev, f_start=f, f_end=f + 1) if rope else None
                normed = None
                with torch.no_grad():
                    for i, b in enumerate(blocks):
                        nxt = blocks[i + 1].norm1 if i + 1 < len(blocks) else None
                        r = b(x, pos=pos, kv_cache=m, global_idx=i, enable_3d_rope=rope, normed=normed, next_norm=nxt,
                              num_frames=1, num_register_tokens=NS - 1)
                        x, normed = r if nxt is not None else (r, None)
                        kinds.append(type(normed).__name__)
                outs.append(x.float().cpu())
            tables = [m.build_visible_page_table(i) for i in range(3)]
            return outs, kinds, tables
        finally:
            Mlp.FUSED_MAX_ROWS = limit

    got, kinds, tables = run(True)
    ref, ref_kinds, ref_tables = run(False)
    assert "RowStats" in kinds and "RowStats" not in ref_kinds       # the chain really ran, and only there
    assert tables == ref_tables
    for a, b in zip(got, ref):
        assert torch.isfinite(a).all()
        scale = b.abs().mean().item()
        assert (a - b).abs().mean().item() <= 0.01 * scale, ((a - b).abs().mean().item(), scale)
        assert (a - b).abs().max().item() <= 0.1 * max(scale, 1.0)
    # a frame block (no cache) fed with statistics, against the same block fed with norm1(x)
    blk = HipPagedBlock(dim=C, num_heads=H, qk_norm=True, init_values=0.5).to(dev).to(torch.bfloat16).eval()
    x = torch.randn(2, T, C, generator=torch.Generator().manual_seed(5)).to(dev).to(torch.bfloat16)
    with torch.no_grad():
        lin = torch.nn.Linear(C, C).to(dev).to(torch.bfloat16)
        x0 = torch.randn_like(x)
        # statistics of x as a residual launch leaves them: x = x0 + lin(h) recomputed through the chain's own helper
        xr, st = blk._linear_residual(x0, lin, torch.nn.Identity(), x0, True)
        y_stats, _ = blk(xr, normed=st, next_norm=blocks[1].norm1)
        y_norm, _ = blk(xr, normed=blk.norm1(xr), next_norm=blocks[1].norm1)
    assert isinstance(st, RowStats)
    d = (y_stats.float() - y_norm.float()).abs()
    assert d.mean().item() <= 0.01 * y_norm.float().abs().mean().item()


@pytest.mark.parametrize("native", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("streams,frames,tokens", [(1, 3, 70), (2, 2, 33), (1, 5, 20)])
def test_anchor_pass_in_one_launch_per_block(streams, frames, tokens, native):
    """The anchor pass whose producer stores all frames' rows (``begin_frames``), block by block mixed
    with the separate launches, against the separate launches alone: same page tables, pool rows and
    outputs within the bf16 noise of the two roundings, and the next streamed frame on top."""
    from lingbot_map_amd.block import HipPagedBlock, Mlp
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, H, C = torch.device("cuda:0"), 2, 128
    torch.manual_seed(3)
    blocks = [HipPagedBlock(dim=C, num_heads=H, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval() for _ in range(2)]
    g = torch.Generator().manual_seed(4)
    first = torch.randn(streams, frames * tokens, C, generator=g).to(dev, torch.bfloat16)
    later = torch.randn(streams, tokens, C, generator=g).to(dev, torch.bfloat16)

    def run(chained):
        m = HipPagedKVCacheManager(2, 24, tokens, H, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=2,
                                   sliding_window=4, max_total_frames=32, page_size=16, layout="frame_pages", num_streams=streams)
        limit, outs = Mlp.FUSED_MAX_ROWS, []
        try:
            with torch.no_grad():
                for x, n in ((first, frames), (later, 1)):
                    for i, b in enumerate(blocks):
                        Mlp.FUSED_MAX_ROWS = limit if chained[i] else 0
                        x = b(x, kv_cache=m, global_idx=i, num_frames=n)
                    outs.append(x.float())
        finally:
            Mlp.FUSED_MAX_ROWS = limit
        assert m.device_header()["error"] == 0
        return outs, [c.float() for c in m.kv_caches], [m.build_visible_page_table(0, s) for s in range(streams)]

    (a, pools_a, tables_a), (b, pools_b, tables_b) = run(native), run((False, False))
    assert tables_a == tables_b
    for x, y in zip(a + pools_a, b + pools_b):
        assert (x - y).abs().mean().item() <= 0.01 * y.abs().mean().item()
        assert ((x != 0).any() == (y != 0).any()) and torch.isfinite(x).all()


@pytest.mark.parametrize("where", ["norm1", "attn", "attn.proj", "mlp"])
def test_anchor_pass_runs_the_hooks_of_its_sub_modules(where):
    """A block whose sub-modules carry forward hooks calls them module by module in the anchor pass."""
    from lingbot_map_amd.block import HipPagedBlock
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens, frames = torch.device("cuda:0"), 40, 3
    torch.manual_seed(5)
    block = HipPagedBlock(dim=128, num_heads=2, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval()
    m = HipPagedKVCacheManager(1, 24, tokens, 2, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames, sliding_window=4,
                               max_total_frames=32, page_size=16, layout="frame_pages")
    seen = []
    block.get_submodule(where).register_forward_hook(lambda mod, args, out: seen.append(out))
    with torch.no_grad():
        block(torch.randn(1, frames * tokens, 128, device=dev).to(torch.bfloat16), kv_cache=m, global_idx=0, num_frames=frames)
    assert len(seen) == 1


@pytest.mark.parametrize("windows", [4, [4, 2]])
@pytest.mark.parametrize("own", [0, 1, 2, 3])
def test_anchor_pass_keeps_to_the_blocks_window(own, windows):
    """The anchor pass evicts by the block's own ``kv_cache_sliding_window`` (by the streams' own windows where
    the manager has one per stream), whatever the manager's: page tables, counts and the frame after it
    as ``append_frame`` + ``evict_frames`` frame by frame leave them, with the fewest frames the window
    holds and more.  (One table set per block: with shared ones a pass that evicts is refused.)"""
    from lingbot_map_amd.block import HipPagedBlock, Mlp
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens, frames, scale, H = torch.device("cuda:0"), 40, 5, 2, 2
    streams = len(windows) if isinstance(windows, list) else 1
    torch.manual_seed(own)
    blocks = [HipPagedBlock(dim=128, num_heads=H, qk_norm=True, init_values=0.5,
                            kv_cache_sliding_window=own).to(dev, torch.bfloat16).eval() for _ in range(2)]
    first = torch.randn(streams, frames * tokens, 128, device=dev).to(torch.bfloat16)
    later = torch.randn(streams, tokens, 128, device=dev).to(torch.bfloat16)

    def run(native):
        m = HipPagedKVCacheManager(2, 24, tokens, H, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=scale,
                                   sliding_window=windows, max_total_frames=32, page_size=16, layout="frame_pages",
                                   num_streams=streams, per_block_tables=True)
        limit, seen = Mlp.FUSED_MAX_ROWS, []
        Mlp.FUSED_MAX_ROWS = limit if native else 0
        try:
            with torch.no_grad():
                for x, n in ((first, frames), (later, 1)):
                    for i, b in enumerate(blocks):
                        x = b(x, kv_cache=m, global_idx=i, num_frames=n)
                    seen += [[m.build_visible_page_table(0, s), m.build_visible_page_lens(0, s), m.get_cache_stats(0, s)]
                             for s in range(streams)]
        finally:
            Mlp.FUSED_MAX_ROWS = limit
        assert m.device_header()["error"] == 0
        return seen, x.float()

    (seen, x), (ref, y) = run(True), run(False)
    assert seen == ref
    for s in range(streams):
        kept = min(frames - scale, windows[s] if streams > 1 else own)     # (what is asked for, not only that both agree)
        assert seen[s][2]["live_pages"] == kept * 3
    assert (x - y).abs().mean().item() <= 0.01 * y.abs().mean().item()     # bf16 noise, as in the pass without evictions


@pytest.mark.parametrize("heads", [1, 4])
@pytest.mark.parametrize("frames", [1, 3])
def test_manager_of_another_geometry_is_refused_untouched(heads, frames):
    """A block of two heads on a manager of fewer or more: an AssertionError before anything is stored, streaming
    and in the anchor pass."""
    from lingbot_map_amd.block import HipPagedBlock
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens = torch.device("cuda:0"), 40
    block = HipPagedBlock(dim=128, num_heads=2, qk_norm=True).to(dev, torch.bfloat16).eval()
    m = HipPagedKVCacheManager(1, 24, tokens, heads, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames,
                               sliding_window=4, max_total_frames=32, page_size=16, layout="frame_pages")
    with torch.no_grad(), pytest.raises(AssertionError):
        block(torch.randn(1, frames * tokens, 128, device=dev).to(torch.bfloat16), kv_cache=m, global_idx=0, num_frames=frames)
    assert m.frame_count == [0] and m.device_header()["frame_count"] == 0 and not m.kv_caches[0].any()


@pytest.mark.parametrize("rope", [False, True])
def test_cacheless_attention_of_float32_rows_under_autocast(rope):
    """Autocast projects float32 rows to bfloat16: the producer has to read the projection in the type that it
    came in.  Against the same attention written out in float32 on the projection's bfloat16 values."""
    from lingbot_map_amd.block import HipPagedAttention, RotaryPositionEmbedding2D, PositionGetter
    dev, B, h, w, C = torch.device("cuda:0"), 2, 5, 9, 128
    torch.manual_seed(11)
    attn = HipPagedAttention(dim=C, num_heads=2, qk_norm=True, rope=RotaryPositionEmbedding2D() if rope else None)
    attn = attn.to(dev, torch.bfloat16).eval()
    x = torch.randn(B, h * w, C, device=dev)
    pos = PositionGetter()(B, h, w, dev) if rope else None
    with torch.no_grad():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            got = attn.dense_attend_fused(x, pos)
            qkv = attn.qkv(x)
        assert qkv.dtype == torch.bfloat16 and got.dtype == torch.float32
        q, k, v = qkv.float().reshape(B, h * w, 3, 2, 64).permute(2, 0, 3, 1, 4).unbind(0)
        q, k = (torch.nn.functional.layer_norm(t, (64,), m.weight.float(), m.bias.float(), m.eps)
                for t, m in ((q, attn.q_norm), (k, attn.k_norm)))
        if rope:
            q, k = attn.rope(q, pos), attn.rope(k, pos)
        ref = (torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) / 8, -1) @ v).transpose(1, 2).reshape(B, h * w, C)
    # The producer rounds the LayerNorm and the rotation to the projection's type, 2^-9 of each of the 64 products of
    # a score four times over: sqrt(64 x 4) x 2^-9 / 8 = 0.004 of a score, which moves a mean of values below 2
    # by 0.004 times their spread; a projection read in the wrong type is off by the values themselves (0.3).
    assert (got - ref).abs().max().item() <= 1e-2


@pytest.mark.parametrize("kind", ["dense", "streamed", "anchor"])
def test_block_under_autocast_and_with_foreign_norms(kind):
    """norm1's result reaches the native call only as bfloat16 of the input's shape: under autocast LayerNorm gives
    float32, and a caller may hand in a float32 ``normed``, which a bfloat16 projection refuses outside of
    autocast.  The block under autocast against the block without, which round in different places (bf16 noise), and
    a refusal leaves the cache untouched."""
    from lingbot_map_amd.block import HipPagedBlock
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens, C = torch.device("cuda:0"), 40, 128
    torch.manual_seed(12)
    frames = 3 if kind == "anchor" else 1
    block = HipPagedBlock(dim=C, num_heads=2, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval()
    x = torch.randn(1, frames * tokens, C, device=dev).to(torch.bfloat16)

    def run(autocast, **kw):
        m = None if kind == "dense" else HipPagedKVCacheManager(
            1, 24, tokens, 2, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames, sliding_window=4,
            max_total_frames=32, page_size=16, layout="frame_pages")
        try:
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
                out = block(x, kv_cache=m, global_idx=0, num_frames=frames, **kw)
            return out.float(), None if m is None else m.kv_caches[0].float()
        except RuntimeError:
            assert m is None or (m.frame_count == [0] and m.device_header()["frame_count"] == 0 and not m.kv_caches[0].any())
            raise

    (y, pool), (z, pool_z) = run(True), run(False)
    for a, b in ((y, z), (pool, pool_z)):
        if a is not None:
            assert (a - b).abs().mean().item() <= 0.01 * b.abs().mean().item()
    with torch.no_grad():
        n1 = block.norm1(x)
    assert torch.equal(run(False, normed=n1)[0], z)
    with pytest.raises(RuntimeError):
        run(False, normed=n1.float())
    with pytest.raises((RuntimeError, AssertionError)):
        run(False, normed=n1[:, :-1])


def test_parameters_of_other_sizes_do_not_reach_the_native_call():
    """Parameters whose sizes the heads do not mean (a projection swapped for another, a LayerScale or q/k
    LayerNorm of another length) are left to the module-by-module calls, which name what does not fit."""
    from torch import nn
    from lingbot_map_amd.block import HipPagedBlock, LayerScale, _NativeBlock
    dev, make = torch.device("cuda:0"), lambda **kw: HipPagedBlock(dim=128, num_heads=2, qk_norm=True, init_values=0.5, **kw)
    swaps = {"attn.proj": nn.Linear(128, 256), "attn.qkv": nn.Linear(128, 128), "mlp.fc1": nn.Linear(256, 512),
             "mlp.fc2": nn.Linear(512, 256), "attn.q_norm": nn.LayerNorm(128), "ls1": LayerScale(64), "ls2": LayerScale(1)}
    assert _NativeBlock.possible(make().to(dev, torch.bfloat16))
    for name, other in swaps.items():
        block = make()
        parent, _, leaf = name.rpartition(".")
        setattr(block.get_submodule(parent), leaf, other)
        assert not _NativeBlock.possible(block.to(dev, torch.bfloat16)), name


@pytest.mark.parametrize("frames", [1, 3])
@pytest.mark.parametrize("how", ["override", "wrap", "plain"])
def test_managers_that_change_the_calls_are_called(how, frames):
    """A manager that overrides ``step_qkv`` or ``append_frame``, or wraps another and shows the reference's call
    surface only, gets those calls; one that leaves them alone is driven by the native call."""
    from lingbot_map_amd.block import HipPagedBlock
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    calls = []

    class Counting(HipPagedKVCacheManager):
        def step_qkv(self, *a, **kw):
            calls.append("step_qkv")
            return super().step_qkv(*a, **kw)

        def append_frame(self, *a, **kw):
            calls.append("append_frame")
            return super().append_frame(*a, **kw)

    class Extended(HipPagedKVCacheManager):
        def begin_block(self, *a, **kw):
            calls.append("native")
            return super().begin_block(*a, **kw)

        def begin_frames(self, *a, **kw):
            calls.append("native")
            return super().begin_frames(*a, **kw)

    dev, tokens = torch.device("cuda:0"), 40
    torch.manual_seed(13)
    block = HipPagedBlock(dim=128, num_heads=2, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval()
    m = (Counting if how == "override" else Extended)(
        1, 24, tokens, 2, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames, sliding_window=4,
        max_total_frames=32, page_size=16, layout="frame_pages")
    with torch.no_grad():
        block(torch.randn(1, frames * tokens, 128, device=dev).to(torch.bfloat16),
              kv_cache=ReferenceSurfaceOnly(m) if how == "wrap" else m, global_idx=0, num_frames=frames)
    assert m.frame_count == [frames]
    assert calls == {"override": ["step_qkv"] if frames == 1 else ["append_frame"] * frames, "wrap": [], "plain": ["native"]}[how]


@pytest.mark.parametrize("kind", ["dense", "streamed", "anchor"])
def test_settings_changed_after_the_first_call_hold(kind):
    """The settings that a forward pass reads from its sub-modules (epsilons, GELU's approximation) and the class of
    the attention may change between calls: each result is a new block's with the same settings, bit for bit."""
    from lingbot_map_amd.block import HipPagedAttention, HipPagedBlock
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens, C = torch.device("cuda:0"), 40, 128
    torch.manual_seed(14)
    frames = 3 if kind == "anchor" else 1
    block = HipPagedBlock(dim=C, num_heads=2, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval()
    x = 0.1 * torch.randn(1, frames * tokens, C, device=dev).to(torch.bfloat16)     # (small enough for an epsilon to show)

    def run(b):
        m = None if kind == "dense" else HipPagedKVCacheManager(
            1, 24, tokens, 2, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames, sliding_window=4,
            max_total_frames=32, page_size=16, layout="frame_pages")
        with torch.no_grad():
            return b(x, kv_cache=m, global_idx=0, num_frames=frames)

    last = run(block)
    for name, field, value in (("norm2", "eps", 0.5), ("attn.q_norm", "eps", 0.5), ("attn.k_norm", "eps", 0.5), ("mlp.act", "approximate", "tanh"),
                               ("norm1", "eps", 0.5)):
        setattr(block.get_submodule(name), field, value)
        new = HipPagedBlock(dim=C, num_heads=2, qk_norm=True, init_values=0.5).to(dev, torch.bfloat16).eval()
        new.load_state_dict(block.state_dict())
        for n in ("norm1", "norm2", "attn.q_norm", "attn.k_norm"):
            new.get_submodule(n).eps = block.get_submodule(n).eps
        new.mlp.act.approximate = block.mlp.act.approximate
        out = run(block)
        assert torch.equal(out, run(new)), name
        # (one q_scale and one epsilon for q and k: the producer takes q's, so k's alone changes nothing)
        assert name in ("mlp.act", "attn.k_norm") or not torch.equal(out, last), name
        last = out

    seen = []

    class Watched(HipPagedAttention):
        def stream_attend_fused(self, *a, **kw):
            seen.append("streamed")
            return super().stream_attend_fused(*a, **kw)

        def dense_attend_fused(self, *a, **kw):
            seen.append("dense")
            return super().dense_attend_fused(*a, **kw)

    block.attn.__class__ = Watched
    run(block)
    assert seen == ["streamed" if kind == "streamed" else "dense"]


def test_anchor_pass_runs_hooks_of_all_modules():
    """A hook registered for all modules sees the block's sub-modules in the anchor pass."""
    from torch.nn.modules.module import register_module_forward_hook
    from lingbot_map_amd.block import HipPagedAttention, HipPagedBlock, Mlp
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, tokens, frames, seen = torch.device("cuda:0"), 40, 3, []
    block = HipPagedBlock(dim=128, num_heads=2, qk_norm=True).to(dev, torch.bfloat16).eval()
    m = HipPagedKVCacheManager(1, 24, tokens, 2, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames,
                               sliding_window=4, max_total_frames=32, page_size=16, layout="frame_pages")
    hook = register_module_forward_hook(lambda mod, args, out: seen.append(type(mod)))
    try:
        with torch.no_grad():
            block(torch.randn(1, frames * tokens, 128, device=dev).to(torch.bfloat16), kv_cache=m, global_idx=0, num_frames=frames)
    finally:
        hook.remove()
    assert {HipPagedAttention, Mlp, HipPagedBlock} <= set(seen)


@pytest.mark.parametrize("spread", [0.0, 0.3])
def test_anchor_pass_with_folded_norms_is_no_farther_from_float64(spread):
    """The anchor pass of twelve blocks as native calls (LayerNorms folded into bf16 weights, sums of the row
    statistics) and as separate launches (LayerNorm rounded to bf16 in front of the projections), both against
    float64: the roundings differ in place, not in size.  LayerNorm weights of one and spread around it.  The errors
    are norms over 54,000 values of independent roundings; 1 % is five times what their difference varies by."""
    import torch.nn.functional as F
    from lingbot_map_amd.block import HipPagedBlock, Mlp
    from lingbot_map_amd.manager import HipPagedKVCacheManager
    dev, H, tokens, frames, depth = torch.device("cuda:0"), 4, 70, 3, 12
    C = 64 * H
    torch.manual_seed(21)
    blocks = [HipPagedBlock(C, H, qk_norm=True, init_values=0.1).to(dev, torch.bfloat16).eval() for _ in range(depth)]
    for b in blocks:
        for m in (b.norm1, b.norm2, b.attn.q_norm, b.attn.k_norm):
            m.weight.data.add_(spread * torch.randn_like(m.weight)); m.bias.data.add_(spread * torch.randn_like(m.bias))
    x0 = torch.randn(1, frames * tokens, C, device=dev).to(torch.bfloat16)

    def run(native):
        m = HipPagedKVCacheManager(depth, 24, tokens, H, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=frames,
                                   sliding_window=4, max_total_frames=32, page_size=16, layout="frame_pages")
        limit, x, normed = Mlp.FUSED_MAX_ROWS, x0, None
        Mlp.FUSED_MAX_ROWS = limit if native else 0
        try:
            with torch.no_grad():
                for i, b in enumerate(blocks):
                    x, normed = b(x, kv_cache=m, global_idx=i, num_frames=frames, normed=normed, next_norm=blocks[(i + 1) % depth].norm1)
        finally:
            Mlp.FUSED_MAX_ROWS = limit
        return x.double()

    with torch.no_grad():
        x = x0[0].double()
        ln = lambda t, m: F.layer_norm(t, m.normalized_shape, m.weight.double(), m.bias.double(), m.eps)
        lin = lambda t, m: t @ m.weight.double().t() + m.bias.double()
        for b in blocks:
            q, k, v = lin(ln(x, b.norm1), b.attn.qkv).reshape(-1, 3, H, 64).unbind(1)
            q, k = ln(q, b.attn.q_norm), ln(k, b.attn.k_norm)
            heads = [torch.softmax(q[:, h] @ k[:, h].t() / 8, -1) @ v[:, h] for h in range(H)]
            x = x + b.ls1.gamma.double() * lin(torch.stack(heads, 1).reshape(-1, C), b.attn.proj)
            x = x + b.ls2.gamma.double() * lin(F.gelu(lin(ln(x, b.norm2), b.mlp.fc1)), b.mlp.fc2)
    err = {native: (run(native)[0] - x).norm().item() for native in (True, False)}
    assert err[True] <= 1.01 * err[False], err


@pytest.mark.parametrize("rows,kv", [(261, 2349), (261, 4437), (90, 90)])
def test_block_as_one_call_equals_its_parts(rows, kv):
    """``lbm_block_run`` against the launches that its declaration names, bit for bit: the attention over a cache is
    the flagged call, whose order of sums is fixed."""
    import ctypes as C
    from lingbot_map_amd import _native as N
    dev, H, hidden, S = torch.device("cuda:0"), 16, 2048, 16
    dim = 64 * H
    g = torch.Generator(device=dev).manual_seed(rows + kv)
    rand = lambda *shape, s=1.0: (torch.randn(*shape, generator=g, device=dev) * s)
    bf = lambda t: t.to(torch.bfloat16)
    x, a = bf(rand(rows, dim)), bf(rand(rows, dim))
    ws = {n: bf(rand(*shape, s=shape[1] ** -0.5)) for n, shape in (("qkv", (3 * dim, dim)), ("proj", (dim, dim)), ("fc1", (hidden, dim)), ("fc2", (dim, hidden)))}
    fc1_sum, ls = ws["fc1"].float().sum(1).contiguous(), rand(dim, s=0.1)
    pages = -(-kv // S)
    pool = bf(rand(pages, 2, S, H, 64))
    t = torch.arange(kv, dtype=torch.int32, device=dev)
    table = (t // S * 2 * S + t % S).to(torch.int32).contiguous()
    append = table[-rows:].contiguous()
    arr = (N.AttnStream * 1)(N.AttnStream(0, rows, 0, kv, 0))
    need = int(N.lib.lbm_attn_workspace_bytes(arr, 1, H, 64))
    attn_ws, split_bytes = torch.empty(max(need, 16), dtype=torch.uint8, device=dev), int(N.lib.lbm_linear_workspace_bytes(rows, dim, hidden, N.LINEAR_BIAS_RESIDUAL))
    split = torch.zeros(max(split_bytes, 16), dtype=torch.uint8, device=dev)
    scale, tiles = N.q_scale_log2(0.125), int(N.lib.lbm_linear_stats_tiles(rows, dim))
    st = N.stream_handle(dev)
    p = lambda t: t.data_ptr()

    one, pool_one = torch.empty_like(x), pool.clone()
    scratch = torch.empty(int(N.lib.lbm_block_scratch_bytes(rows, H, hidden)), dtype=torch.uint8, device=dev)
    weights = N.BlockWeights(p(ws["qkv"]), p(ws["proj"]), p(ws["fc1"]), p(ws["fc2"]), None, None, None, None, None, p(fc1_sum), p(ls), p(ls),
                             None, None, None, None, 0.0, 1e-6, 1e-5, H, hidden)
    call = N.BlockCall(p(x), p(a), None, p(one), None, p(scratch), None, p(pool_one), p(append), p(table), None, C.addressof(arr),
                       p(attn_ws), p(split), scratch.numel(), attn_ws.numel(), split_bytes, scale, rows, 0, 0, False, 1, S,
                       (None,) * 4, (0,) * 4, 0)
    N.check(N.lib.lbm_block_run(weights, call, st))

    q, heads, x1, parts, pool_parts = (torch.empty_like(t) for t in (x, x, x, x, pool))
    pool_parts.copy_(pool)
    mid, stats = torch.empty(rows, hidden, dtype=torch.bfloat16, device=dev), torch.empty(rows, tiles, 2, device=dev)
    N.check(N.lib.lbm_qkv_linear_prepare_norm(p(a), None, p(ws["qkv"]), None, rows, dim, None, None, None, None, 1e-5, scale, None, 0, p(q),
                                              None, None, p(pool_parts), p(append), H, 64, S, st))
    N.check(N.lib.lbm_attn_run_call(
        N.ATTN_CALL_HEAD.pack(p(q), p(pool_parts), p(heads), 0, 0, p(table), 0, 0, C.addressof(arr), p(attn_ws), attn_ws.numel(), 0.0)
        + N.attn_call_tail(0, 1, H, 64, S, N.DTYPE_BF16, N.ATTN_FIXED_ORDER), st))
    N.check(N.lib.lbm_linear_norm(p(heads), None, p(ws["proj"]), None, p(ls), p(x), p(x1), p(stats), rows, dim, dim,
                                  N.LINEAR_BIAS_RESIDUAL, None, 0, st))
    N.check(N.lib.lbm_linear_norm(p(x1), N.RowNorm(p(stats), p(fc1_sum), tiles, 1e-6), p(ws["fc1"]), None, None, None, p(mid), None,
                                  rows, hidden, dim, N.LINEAR_BIAS_GELU, None, 0, st))
    N.check(N.lib.lbm_linear_norm(p(mid), None, p(ws["fc2"]), None, p(ls), p(x1), p(parts), None, rows, dim, hidden,
                                  N.LINEAR_BIAS_RESIDUAL, p(split), split_bytes, st))
    torch.cuda.synchronize()
    assert torch.isfinite(one.float()).all() and torch.equal(pool_one, pool_parts) and torch.equal(one, parts)


@pytest.mark.parametrize("rows", [20, 261, 600])
def test_weights_asked_for_ahead_change_no_result(rows, monkeypatch):
    """A block's launches ask for the weights of those behind them, the attention among them where it leaves CUs idle: a frame
    block's and a streamed block's results with and without."""
    from lingbot_map_amd import HipPagedBlock, HipPagedKVCacheManager
    torch.manual_seed(rows)
    dev, heads = torch.device("cuda:0"), 16
    blocks = [HipPagedBlock(64 * heads, heads, init_values=0.1).to(dev, torch.bfloat16).eval() for _ in range(2)]
    frames = [torch.randn(1, rows, 64 * heads, device=dev).to(torch.bfloat16) for _ in range(3)]
    got = []
    for hints in (False, True):
        monkeypatch.setattr(HipPagedBlock, "PREFETCH_HINTS", hints)
        m = HipPagedKVCacheManager(1, 20, rows, heads, 64, torch.bfloat16, dev, num_special_tokens=5, scale_frames=1,
                                   sliding_window=2, max_total_frames=32, page_size=16, layout="frame_pages")
        outs = []
        with torch.no_grad():
            for x in frames:
                x, normed = blocks[0](x, next_norm=blocks[1].norm1)
                outs.append(blocks[1](x, kv_cache=m, global_idx=0, num_frames=1, normed=normed))
        got.append(outs)
    for a, b in zip(*got):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


def test_eager_frames_below_a_line_name_no_weights(monkeypatch):
    """``HipPagedBlock.HINT_ROWS``, 0 unless it is set: eager frames of fewer rows give no hints, others do."""
    from lingbot_map_amd import HipPagedBlock
    from lingbot_map_amd.block import _NativeBlock
    dev, asked = torch.device("cuda:0"), []
    block = HipPagedBlock(1024, 16).to(dev, torch.bfloat16).eval()
    hints_with = _NativeBlock.hints_with
    monkeypatch.setattr(_NativeBlock, "hints_with", lambda self, next_norm: asked.append(1) or hints_with(self, next_norm))
    counts = []
    for line in (None, 100, 101):
        if line is not None:
            monkeypatch.setattr(HipPagedBlock, "HINT_ROWS", line)
        with torch.no_grad():
            block(torch.randn(1, 100, 1024, device=dev).to(torch.bfloat16))
        counts.append(len(asked))
    assert counts == [1, 2, 2]
