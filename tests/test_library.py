"""The kernel library and its sources: a library built from other sources than those beside it is
never called (entry points gain parameters; an old binary would read shifted arguments)."""
import pytest

from bare_cuda_4gib_amd.csrc import build, library
from bare_cuda_4gib_amd.errors import KernelError


def test_the_built_library_carries_the_digest_of_its_sources():
    if not build.is_built():
        pytest.skip("the kernel library is not built here")
    assert len(build.sources_digest()) == 64
    assert build.built_digest() == build.sources_digest() and not build.is_stale()


def test_a_stale_library_is_rebuilt_or_refused(monkeypatch):
    if not build.is_built():
        pytest.skip("the kernel library is not built here")
    monkeypatch.setattr(library, "_lib", None)
    monkeypatch.setattr(build, "sources_digest", lambda: "0" * 64)          # as if a source had been edited
    assert build.is_stale()
    with pytest.raises(KernelError, match="other sources"):
        library.load(build_if_missing=False)
    monkeypatch.setattr(build, "can_build", lambda: False)                  # no compiler on this machine
    with pytest.raises(KernelError, match="other sources"):
        library.load()
    calls = []
    monkeypatch.setattr(build, "can_build", lambda: True)
    monkeypatch.setattr(build, "build", lambda verbose=True: calls.append(1))
    with pytest.raises(KernelError, match="digest"):                        # "rebuilt" (here: not really), checked again
        library.load()
    assert calls == [1]


def test_where_the_library_lives(monkeypatch, tmp_path):
    """Beside its sources, where that folder can be written or already holds a library of these sources; else in a
    folder that belongs to this user alone under the temporary folder -- and never in one that others can write."""
    import os
    import tempfile
    in_tree = (os.path.join(build.HERE, "_build"), os.path.join(build.HERE, "libbc4g.so"))
    monkeypatch.setattr(build, "BUILD_DIR", in_tree[0])
    monkeypatch.setattr(build, "LIB_PATH", in_tree[1])
    monkeypatch.setattr(tempfile, "tempdir", str(tmp_path))
    monkeypatch.setattr(os, "access", lambda path, mode: True)
    build._settle()
    assert (build.BUILD_DIR, build.LIB_PATH) == in_tree
    monkeypatch.setattr(os, "access", lambda path, mode: False)          # a checkout that belongs to someone else
    monkeypatch.setattr(build, "built_digest", lambda path="": build.sources_digest())
    build._settle()                                                      # ... with a library of these sources
    assert (build.BUILD_DIR, build.LIB_PATH) == in_tree
    monkeypatch.setattr(build, "built_digest", lambda path="": "")       # ... without
    build._settle()
    home = os.path.join(str(tmp_path), f"bc4g-{os.getuid()}")
    assert build.LIB_PATH == os.path.join(home, "libbc4g.so") and build.BUILD_DIR == os.path.join(home, "_build")
    assert os.stat(home).st_mode & 0o777 == 0o700
    monkeypatch.setattr(build, "BUILD_DIR", in_tree[0])
    monkeypatch.setattr(build, "LIB_PATH", in_tree[1])
    os.chmod(home, 0o777)
    with pytest.raises(KernelError, match="nowhere to build"):
        build._settle()


def test_latent_prepare_refuses_absorbed_queries_without_a_place_or_whole_rows():
    """Whatever else is asked for, and also where nothing is rotated: refused before anything is launched."""
    if not build.is_built():
        pytest.skip("the kernel library is not built here")
    at, heads, plain, rank = 1 << 20, 4, 16, 32                # (no call gets as far as reading from this address)

    def prepare(q=at, q_lat=at, rot=0, q_row=heads * 16, rows=8, dtype=1, cache=None, absorb=at):
        library.call("bc4g_latent_prepare", q, at, dtype, at, 1e-5, at, at, cache, q_lat, rows, heads, plain, rot, rank, 0, q_row, rank + rot, 0,
                     None, None, None, 0, 0, absorb, None)

    for wrong in (dict(q_lat=None), dict(q_lat=None, cache=at), dict(q=None), dict(q=None, cache=at), dict(q_row=heads * 16 - 8), dict(q_row=heads * 16 - 8, cache=at),
                  dict(rows=33), dict(dtype=0), dict(q=at + 8), dict(absorb=at + 8), dict(q_row=heads * 16 + 4)):
        with pytest.raises(KernelError, match="absorbed queries"):
            prepare(**wrong)
    prepare(rows=0)
