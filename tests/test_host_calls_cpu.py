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


def test_the_extension_module_has_no_thread_locals():
    """A thread-local that nobody touches, in the library loaded last, slows down every other one of the process (glibc up
    to 2.38): no PT_TLS (7) among the module's program headers (64-bit ELF: their offset, size and number at 32, 54 and 56)."""
    import struct
    from lingbot_map_amd.build import HOST_PATH
    with open(HOST_PATH, "rb") as f:
        elf = f.read()
    assert elf[:5] == b"\x7fELF\x02"
    at, (size, count) = struct.unpack_from("<Q", elf, 32)[0], struct.unpack_from("<HH", elf, 54)
    assert count > 0 and all(struct.unpack_from("<I", elf, at + i * size)[0] != 7 for i in range(count))


def test_a_module_of_another_abi_version_is_refused(monkeypatch):
    import pytest
    from lingbot_map_amd import _native as N
    assert N._load_host().ABI_VERSION == N.ABI_VERSION == N.lib.lbm_abi_version()
    monkeypatch.setattr(N, "ABI_VERSION", N.ABI_VERSION + 1)
    with pytest.raises(RuntimeError, match="ABI version"):
        N._load_host()


def test_a_build_that_fails_leaves_no_old_module(monkeypatch, tmp_path):
    import pytest
    from lingbot_map_amd import build
    for name, value in (("LIB_DIR", str(tmp_path)), ("LIB_PATH", str(tmp_path / "lib.so")), ("HOST_PATH", str(tmp_path / "host.so"))):
        monkeypatch.setattr(build, name, value)
    old = tmp_path / "host.so"
    old.write_bytes(b"old")
    monkeypatch.setattr(build, "HIPCC", "false")
    with pytest.raises(RuntimeError):
        build.build()
    assert not old.exists()
    old.write_bytes(b"old")                        # the library is built, the module is not
    monkeypatch.setattr(build, "HIPCC", "true")
    monkeypatch.setenv("CXX", "false")
    with pytest.raises(RuntimeError):
        build.build()
    assert not old.exists()
