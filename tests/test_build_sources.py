"""build() compiles the package's and the oracle's sources only: it passes
beside a tests/ of another revision, whose sources need not compile against
this package's internals, and beside none."""
import ctypes
import os
import shutil

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("tests_tree", [True, False])
def test_build_takes_no_source_from_tests(tmp_path, monkeypatch, tests_tree):
    import __graft_entry__ as g
    pkg = os.path.basename(g.PKG_DIR)
    for d in (pkg, "oracle", "include"):
        shutil.copytree(os.path.join(ROOT, d), tmp_path / d, ignore=shutil.ignore_patterns("build", "__pycache__"))
    if tests_tree:
        (tmp_path / "tests" / "emu").mkdir(parents=True)
        (tmp_path / "tests" / "emu" / "psf_emu.cpp").write_text("#error another revision\n")
    run, makes = g._run, []

    def only_host_library(cmd, cwd):        # the device library takes minutes and is built anyway
        makes.append(cmd)
        run(cmd + (["build/libpsf_emu.so"] if cmd[0] == "make" and pkg in cmd[3] else []), cwd)

    monkeypatch.setattr(g, "ROOT", str(tmp_path))
    monkeypatch.setattr(g, "PKG_DIR", str(tmp_path / pkg))
    monkeypatch.setattr(g, "_run", only_host_library)
    monkeypatch.setattr(g, "load_package", lambda: None)
    g.build()
    assert len(makes) == 2 and all(c[0] == "make" for c in makes)
    assert (tmp_path / "tests").is_dir() == tests_tree
    built = tmp_path / ("tests/emu" if tests_tree else pkg + "/build") / "libpsf_emu.so"
    assert ctypes.CDLL(str(built)).emu_bin_cmd_smooth
