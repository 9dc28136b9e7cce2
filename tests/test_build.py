"""The build without what only the torch wrappers' C++ call path needs."""
import importlib.util
import os
import sysconfig

import pytest

from fastmlx_amd import build


@pytest.fixture
def here(monkeypatch, tmp_path):
    """The module's outputs in an empty folder."""
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "FAST", str(tmp_path / os.path.basename(build.FAST)))
    return tmp_path


def test_without_torch(monkeypatch, here):
    monkeypatch.setattr(importlib.util, "find_spec", lambda name: None)
    assert build.build_fast(verbose=False) is None


def test_without_a_compiler(monkeypatch, here):
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    monkeypatch.setenv("ROCM_PATH", str(here))
    assert build.build_fast(verbose=False) is None


def test_module_carries_the_abi_tag():
    assert build.FAST.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    from fastmlx_amd import ops

    if ops._fast is not None:
        assert ops._fast.__file__ == build.FAST
