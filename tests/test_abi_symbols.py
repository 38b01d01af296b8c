"""The built library exports every function include/lbm_paged_attn.h declares, and the
Python binding's constants agree with the header.  No GPU, no compute calls."""
import ctypes as C
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "lbm_paged_attn.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lbm_[a-z_0-9]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    for n in ("lbm_tables_step", "lbm_rows_from_pages", "lbm_kv_append", "lbm_qkv_prepare", "lbm_attn_run",
              "lbm_attn_workspace_bytes", "lbm_tables_words", "lbm_abi_version", "lbm_last_error"):
        assert n in names


def test_library_exports_every_declared_symbol():
    from lingbot_map_amd import _native as N
    lib = C.CDLL(N.LIB_PATH)
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} declared in the header but not exported"
    assert set(N.SYMBOLS) == set(declared_functions())
    assert N.lib.lbm_abi_version() == N.ABI_VERSION


def test_binding_constants_match_header():
    from lingbot_map_amd import _native as N
    text = open(HEADER).read()
    defs = {m.group(1): int(m.group(2)) for m in re.finditer(r"#define\s+(LBM_[A-Z_0-9]+)\s+(\d+)\b", text)}
    assert defs["LBM_ABI_VERSION"] == N.ABI_VERSION
    assert defs["LBM_MAX_STREAMS"] == N.MAX_STREAMS and defs["LBM_MAX_GROUPS"] == N.MAX_GROUPS
    assert defs["LBM_STATIC_SCRATCH_MIB"] == N.STATIC_SCRATCH_MIB
    assert (defs["LBM_OP_RESET"], defs["LBM_OP_ROLLBACK"], defs["LBM_OP_APPEND"], defs["LBM_OP_EVICT"],
            defs["LBM_OP_PLAN"]) == (N.OP_RESET, N.OP_ROLLBACK, N.OP_APPEND, N.OP_EVICT, N.OP_PLAN)
    assert defs["LBM_HDR_WORDS"] == N.HDR_WORDS
    for k, i in N.HDR.items():
        assert defs["LBM_HDR_" + k.upper()] == i
    assert (defs["LBM_DTYPE_BF16"], defs["LBM_DTYPE_F32"]) == (N.DTYPE_BF16, N.DTYPE_F32)
    assert (defs["LBM_LAYOUT_TWO_STREAM"], defs["LBM_LAYOUT_FRAME_PAGES"]) == (N.LAYOUT_TWO_STREAM, N.LAYOUT_FRAME_PAGES)
    # struct sizes: plain int32 fields, no padding
    assert C.sizeof(N.CacheGeom) == 9 * 4 and C.sizeof(N.StepOp) == 8 * 4 and C.sizeof(N.AttnStream) == 5 * 4
    # lbm_attn_call: ten pointers, a size, a float and seven ints without holes
    assert N.ATTN_CALL_HEAD.size == 11 * 8 + 4 and len(N.attn_call_tail(0, 1, 2, 3, 4, 5, 6)) == 7 * 4
    assert (defs["LBM_ATTN_OWN_ROWS"], defs["LBM_ATTN_APPEND_APART"]) == (N.ATTN_OWN_ROWS, N.ATTN_APPEND_APART)
    assert defs["LBM_ATTN_FIXED_ORDER"] == N.ATTN_FIXED_ORDER


def test_host_side_argument_checks_need_no_gpu():
    from lingbot_map_amd import _native as N
    g = N.CacheGeom(0, 7, 3, 4, 1, 19, 21, 0, 40)
    assert N.lib.lbm_tables_words(C.byref(g)) == 16 + 19 + 21 + 1 + 19 + 21 + 0 + 1 + 1
    bad = N.CacheGeom(0, 3, 3, 4, 1, 19, 21, 0, 40)   # no patch tokens
    assert N.lib.lbm_tables_words(C.byref(bad)) == 0
    s = (N.AttnStream * 1)(N.AttnStream(0, 1004, 0, 17068))
    # 4 query tiles x 16 heads x 8 splits = 512 workgroups -> 8 partial results per row
    assert N.lib.lbm_attn_workspace_bytes(s, 1, 16, 64) == 8 * 1004 * 16 * (64 * 2 + 4)
    s1 = (N.AttnStream * 1)(N.AttnStream(0, 9, 0, 64))      # one workgroup per head, nothing to merge
    assert N.lib.lbm_attn_workspace_bytes(s1, 1, 16, 64) == 0
    # at most 8 query rows: partials of the fp32 few-query path, (D + 2) floats per chunk, row and head
    s8 = (N.AttnStream * 1)(N.AttnStream(0, 8, 0, 64))
    assert N.lib.lbm_attn_workspace_bytes(s8, 1, 16, 64) == 1 * 8 * 16 * (64 + 2) * 4
    s9 = (N.AttnStream * 1)(N.AttnStream(0, 1, 0, 10000))
    assert N.lib.lbm_attn_workspace_bytes(s9, 1, 16, 128) == 40 * 1 * 16 * (128 + 2) * 4
    rc = N.lib.lbm_attn_run(None, None, None, None, None, None, s, 1, 16, 64, 16, 0, 0.125, None, 0, None)
    assert rc == N.ERR_INVALID and b"null" in N.lib.lbm_last_error()
    # two streams whose append_rows ranges overlap (an idle stream left at q_begin 0) are refused
    ops = (N.StepOp * 2)(N.StepOp(N.OP_APPEND, 0, 0, 0, 0, 0, 0, 0), N.StepOp(0, 0, 0, 0, 0, 0, 0, 0))
    fake = C.c_void_p(256)   # never dereferenced: the call fails in the argument checks
    rc = N.lib.lbm_tables_step(fake, C.byref(g), 2, ops, fake, None, None, None, None)
    assert rc == N.ERR_INVALID and b"overlap" in N.lib.lbm_last_error()


def test_schedule_leaves_whole_what_the_upper_estimate_leaves_whole():
    """Partial results are rounded to bf16 on their way through memory, so a stream of a ragged launch is split only
    where the upper estimate splits it; the fitted costs choose among such splits.  Rows of partials show it:
    (splits x rows of every split stream) x heads x (64 bf16 values + a float)."""
    from lingbot_map_amd import _native as N

    def partial_rows(heads, *streams):
        arr, at = (N.AttnStream * len(streams))(), 0
        for i, (rows, kv) in enumerate(streams):
            arr[i] = N.AttnStream(at, rows, 0, kv, 0)
            at += rows
        per_row = heads * (64 * 2 + 4)
        size = int(N.lib.lbm_attn_workspace_bytes(arr, len(streams), heads, 64))
        assert size % per_row == 0
        return size // per_row

    # 520 rows x 2,787 tokens, 200 x 776 and 530 x 6,222 stay whole beside streams ten times as long
    assert partial_rows(16, (128, 19598), (520, 2787), (9, 12085)) == 7 * 128 + 5 * 9
    assert partial_rows(8, (333, 9), (487, 24626), (113, 3), (10, 1), (284, 90), (200, 776)) == 12 * 487
    assert partial_rows(12, (15, 5868), (530, 6222), (17, 63013), (14, 40299)) == 10 * 17 + 7 * 14


def test_workspace_query_is_zero_where_nothing_is_split():
    """Eight streams of 1,004 rows x 5,000 tokens: 256 workgroups of the split-KV kernel, each with the whole KV
    list, no partial results; one frame of 1,004 x 1,004 on the short-KV kernel."""
    from lingbot_map_amd import _native as N
    arr = (N.AttnStream * 8)(*[N.AttnStream(i * 1004, 1004, i * 5000, 5000, 0) for i in range(8)])
    assert N.lib.lbm_attn_workspace_bytes(arr, 8, 16, 64) == 0
    assert N.lib.lbm_attn_workspace_bytes((N.AttnStream * 1)(N.AttnStream(0, 1004, 0, 1004, 0)), 1, 16, 64) == 0


def test_one_hip_runtime_whichever_is_imported_first():
    """Imported before torch the package still uses torch's HIP runtime: of two in a process one finds no device."""
    import subprocess
    import sys
    show = "import os; print(*{os.path.realpath(l.split()[-1]) for l in open('/proc/self/maps') if 'libamdhip64' in l}, sep='\\n')"
    seen = [subprocess.run([sys.executable, "-c", f"import sys; sys.path.insert(0, {os.path.join(ROOT, 'lingbot-map_amd')!r}); {first}; {show}"],
                           stdout=subprocess.PIPE, text=True, check=True).stdout.split() for first in ("import lingbot_map_amd", "import torch, lingbot_map_amd")]
    assert len(seen[0]) == 1 and seen[0] == seen[1]
