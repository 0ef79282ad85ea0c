"""The launch results that a compact layer's degrees carry serve only the tensor as it
was launched: a provider that writes into the degrees, derives others from them or asked
for other rows gets the rows it returns."""
import pytest
import torch

from cast_amd.closed_loop import _carried, _carry

ROWS = (10, 2, 4)


def _degrees():
    base = torch.arange(10)
    current = base[2:].view(2, 4)
    _carry(current, "results", ROWS)
    return base, current


def test_carried_as_launched():
    _, current = _degrees()
    assert _carried(current) == _carried(current, ROWS) == "results"


@pytest.mark.parametrize("change", [lambda b, c: c.clamp_(max=5), lambda b, c: b.add_(1),
                                    lambda b, c: c[0].zero_()])
def test_written_degrees_carry_nothing(change):
    base, current = _degrees()
    change(base, current)
    assert _carried(current) is None


def test_other_tensors_and_rows_carry_nothing():
    _, current = _degrees()
    assert _carried(current.flip(0)) is None and _carried(current + 0) is None
    assert _carried(current, (10, 3, 4)) is None and _carried(current, (10, 2, 5)) is None
    with torch.inference_mode():
        untracked = torch.arange(8)
        _carry(untracked, "results", ROWS)
    assert _carried(untracked) is None
