"""Which launch of a block asks for which of the weights ahead (csrc/touch_logic.h, ``lbm_attention_asks``): a hint goes to
a launch that asks for it, whenever one of those that may can."""
import ctypes as C
import itertools
import os
import subprocess
import tempfile

import pytest

from lingbot_map_amd import _native as N

HERE = os.path.dirname(os.path.abspath(__file__))
NOT, WAVES, IDLE, WIDE_IDLE = range(4)


@pytest.fixture(scope="module")
def host():
    so = os.path.join(tempfile.mkdtemp(prefix="lbm_hints_host_"), "hints_host.so")
    lib = os.path.dirname(N.LIB_PATH)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", "-w", "-o", so,
                           os.path.join(HERE, "native", "hints_host.cpp"), f"-L{lib}", "-llbm_paged_attn", f"-Wl,-rpath,{lib}"])
    return C.CDLL(so)


def test_every_hint_goes_to_a_launch_that_asks(host):
    """All 1,024 ways in which a block's launches can ask (qkv projection, attention, proj, fc1, fc2): what launch 2 + r reads is
    asked for by one of the three before it, by none only if none of them asks, and by wavefronts only if no tile of 256 columns
    has idle CUs for it."""
    by = (C.c_int * 4)()
    for asks in itertools.product(range(4), repeat=5):
        host.lbm_hints_deal((C.c_int * 5)(*asks), by)
        for r in range(4):
            may = range(max(r - 1, 0), r + 2)
            if by[r] < 0:
                assert all(asks[l] == NOT for l in may)
                continue
            assert by[r] in may and asks[by[r]] != NOT
            later = [asks[l] for l in may if l > by[r]]
            assert all(a == NOT for a in later) or (asks[by[r]] == WIDE_IDLE and next(a for a in reversed(later) if a != NOT) == WAVES)
            assert asks[by[r]] != WAVES or all(asks[l] != WIDE_IDLE for l in may)


@pytest.mark.parametrize("H,frames,rows", [(16, 1, 86), (16, 1, 1004), (16, 2, 666), (16, 4, 1004), (16, 5, 821), (16, 5, 1004), (16, 6, 593), (16, 6, 1004),
                                           (16, 7, 450), (16, 8, 450), (16, 8, 1004), (12, 6, 1004), (12, 8, 593), (8, 16, 100)])
@pytest.mark.parametrize("kv", [None, 5000])
def test_attention_asks_where_its_kernel_does(host, H, frames, rows, kv):
    """The kernels of own rows in order - one split of every stream, or two of every stream of more than 256 rows - have no
    workgroups that ask; the short-KV kernel and the one that goes by the table do, where 32 CUs or more are idle."""
    arr = (N.AttnStream * frames)(*[N.AttnStream(i * rows, rows, i * (kv or rows), kv or rows, 0) for i in range(frames)])
    small, wgs, splits = C.c_int(), C.c_int(), (C.c_int * frames)()
    asks = [host.lbm_hints_attention(arr, frames, H, own, C.byref(small), C.byref(wgs), splits) for own in (0, 1)]
    idle = -wgs.value % 256 >= 32
    own_kernel = not small.value and (all(s == 1 for s in splits) or (all(s == 2 for s in splits) and rows > 256))
    assert asks == [idle, idle and not own_kernel]


def test_attention_of_several_frames_leaves_hints_to_others(host):
    """Frames whose own rows go by those kernels with 32 idle CUs or more: the case in which a hint was lost."""
    small, wgs, splits = C.c_int(), C.c_int(), (C.c_int * 6)()
    arr = (N.AttnStream * 6)(*[N.AttnStream(i * 1004, 1004, i * 1004, 1004, 0) for i in range(6)])
    assert host.lbm_hints_attention(arr, 6, 16, 0, C.byref(small), C.byref(wgs), splits) == 1 and not small.value
    assert host.lbm_hints_attention(arr, 6, 16, 1, C.byref(small), C.byref(wgs), splits) == 0


def _pending(host):
    at, lines = (C.c_longlong * 4)(), (C.c_uint * 4)()
    host.lbm_hints_pending(at, lines)
    return [(a, n) for a, n in zip(at, lines) if n]


def _refused_block(hints):
    """A block of one head, whose 64 columns the first linear refuses; nothing is launched and no address read."""
    p = 1 << 40
    w = N.BlockWeights(*[p] * 8, None, p, *[None] * 6, 0.0, 1e-5, 1e-5, 1, 256)
    call = N.BlockCall(p, p, None, p, None, p, None, None, None, p, None, None, p, None, 1 << 30, 0, 0, 1.0, 4, 0, 0, 1, 0, 16, hints, (4096,) * 4, 1)
    assert N.lib.lbm_block_run(w, call, None) != N.OK
    assert b"multiple of 128" in N.lib.lbm_last_error()


def test_a_refused_block_leaves_no_hint_of_its_own(host):
    N.lib.lbm_linear_prefetch_hint(None, 0)
    _refused_block(tuple((2 << 40) + i * 4096 for i in range(4)))
    assert _pending(host) == []
    _refused_block((None,) + tuple((2 << 40) + i * 4096 for i in range(3)))
    assert _pending(host) == []


def test_a_hint_given_before_a_block_is_its_first_linears(host):
    """A block with no hint for proj does not withdraw it: refused, it leaves it as it was."""
    for own in ((None,) * 4, (None, 3 << 40, 3 << 40, 3 << 40)):
        N.lib.lbm_linear_prefetch_hint(2 << 40, 8192)
        _refused_block(own)
        assert _pending(host) == [(2 << 40, 64)]
    _refused_block((3 << 40,) + (None,) * 3)      # (the block's own takes its place)
    assert _pending(host) == []
    N.lib.lbm_linear_prefetch_hint(None, 0)


@pytest.mark.gpu
def test_a_block_refused_at_its_last_linear_leaves_no_hint(host):
    """192 hidden columns: fc1 takes them, fc2 does not; the first three launches have run.  And a hint given beforehand has been taken."""
    import torch
    dev = torch.device("cuda:0")
    rows, dim, hidden = 8, 128, 192
    mem = torch.zeros(1 << 22, dtype=torch.uint8, device=dev)
    p = mem.data_ptr()
    w = N.BlockWeights(*[p] * 4, None, None, None, None, None, p, *[None] * 6, 0.0, 1e-5, 1e-5, 2, hidden)
    need = int(N.lib.lbm_block_scratch_bytes(rows, 2, hidden))
    scratch = torch.zeros(need, dtype=torch.uint8, device=dev)
    out = torch.zeros(rows, dim, dtype=torch.bfloat16, device=dev)
    for hints in ((p,) * 4, (None,) * 4):
        N.lib.lbm_linear_prefetch_hint(p, 4096)
        call = N.BlockCall(p, p, None, out.data_ptr(), None, scratch.data_ptr(), None, None, None, p, None, None, None, None, need, 0, 0, 1.0,
                           rows, 0, 0, 1, 0, 16, hints, (4096,) * 4, 1)
        assert N.lib.lbm_block_run(w, call, None) != N.OK and b"multiple of 128" in N.lib.lbm_last_error()
        torch.cuda.synchronize()
        assert _pending(host) == []
