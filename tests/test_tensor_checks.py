"""The check of a device tensor argument: what it refuses, and that a call
after the first imports nothing (an import statement costs more than the rest
of the check, four times in a small ``Psource``)."""
import builtins

import pytest
import torch

from anelastic_solve_amd import mg


@pytest.mark.parametrize("t", [
    torch.zeros((4, 3, 2), dtype=torch.float32),
    torch.zeros((4, 3, 2), dtype=torch.int64),
    torch.zeros((4, 2, 3), dtype=torch.float64),
    torch.zeros((24,), dtype=torch.float64),
    torch.zeros((2, 3, 4), dtype=torch.float64).permute(2, 1, 0),
    torch.zeros((4, 3, 4), dtype=torch.float64)[:, :, ::2],
    torch.zeros((4, 3, 2), dtype=torch.float64),          # not on a device
])
def test_refused(t):
    with pytest.raises(ValueError, match="U: "):
        mg._dev_ptr(t, (4, 3, 2), "U")


class _Device:
    """Stands in for a device tensor."""
    shape, dtype, is_cuda = (4, 3, 2), torch.float64, True

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 4096


def test_no_import_per_call(monkeypatch):
    assert mg._dev_ptr(_Device(), (4, 3, 2), "U").value == 4096
    seen = []
    real = builtins.__import__
    monkeypatch.setattr(builtins, "__import__", lambda name, *a, **k: (seen.append(name), real(name, *a, **k))[1])
    mg._dev_ptr(_Device(), (4, 3, 2), "U")
    assert seen == []
