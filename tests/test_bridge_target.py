"""A bridge module left from other sources, another PyTorch or another Python is refused: it reads their
objects inline."""

import types

import pytest
import torch

from gguf_train_amd import _C, _srchash


def _module(**other):
    kept = {"SOURCE_HASH": _C.bridge.SOURCE_HASH, "BUILT_FOR": _C.bridge.BUILT_FOR, "__file__": "_gt_bridge.so"}
    return types.SimpleNamespace(**{**kept, **other})


def test_the_loaded_bridge_names_what_it_was_built_for():
    assert _C.bridge.BUILT_FOR == _srchash.bridge_target()
    assert f"torch {torch.__version__} {torch.version.git_version}" in _C.bridge.BUILT_FOR
    _C._check_bridge(_module())


@pytest.mark.parametrize("now,then", [(torch.__version__, "1.0.0"), (torch.version.git_version, "0" * 40),
                                      ("cpython-", "cpython-9"), ("python 3", "python 4")])
def test_a_bridge_for_something_else_is_refused(now, then):
    built_for = _C.bridge.BUILT_FOR.replace(now, then)
    assert built_for != _C.bridge.BUILT_FOR
    with pytest.raises(ImportError, match="was built for"):
        _C._check_bridge(_module(BUILT_FOR=built_for))


def test_a_bridge_from_other_sources_is_refused():
    with pytest.raises(ImportError, match="other sources"):
        _C._check_bridge(_module(SOURCE_HASH="0" * 64))
