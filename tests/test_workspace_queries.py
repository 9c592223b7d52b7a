"""The workspace queries of the Python layer keep answers by plain whole numbers only.  CPU only: the
queries compute on the host."""
import ctypes
import os

import pytest
import torch

import syntropy_amd.gemv as S
from syntropy_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="the library is not built")


def test_a_changed_tensor_is_asked_again():
    rows = torch.tensor(5)
    small = S.workspace_bytes(S.WeightType.Q8_0, rows, 64)
    assert small == S.workspace_bytes(S.WeightType.Q8_0, 5, 64)
    rows += 60
    assert S.workspace_bytes(S.WeightType.Q8_0, rows, 64) == S.workspace_bytes(S.WeightType.Q8_0, 65, 64) > small


def test_a_float_is_refused_whatever_was_asked_before():
    S.workspace_bytes(S.WeightType.Q8_0, 6, 64)
    with pytest.raises(ctypes.ArgumentError):
        S.workspace_bytes(S.WeightType.Q8_0, 6.0, 64)
