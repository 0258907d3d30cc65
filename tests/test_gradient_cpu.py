"""Host side of the phase gradients: the forms in which targets may be given."""
import numpy as np
import pytest

from perceval_amd.gradient import _target_rows


@pytest.mark.parametrize("targets", [
    [[1, 0], [0, 1]], ((2, 0),), np.array([[1, 2], [3, 4]]), np.array([[1, 2], [3, 4]], dtype=np.int8).T,
    np.arange(6).reshape(2, 3)[:, ::-1], np.array([[2 ** 31 - 1, 0]], dtype=np.uint64), np.array([[1.5, 2.0]]),
    np.array([[True, False]]), np.array([[1, 2]], dtype=object), np.zeros((0, 3), dtype=int)])
def test_target_rows_as_from_lists(targets):
    rows = _target_rows(targets)
    ref = np.asarray([list(t) for t in targets], dtype=np.int32)
    assert rows.dtype == np.int32 and rows.flags.c_contiguous and rows.tolist() == ref.tolist()


@pytest.mark.parametrize("targets", [
    np.array([[2 ** 32 + 1, 0]]), np.array([[-2 ** 40, 0]]), np.array([[2 ** 31, 0]], dtype=np.uint32),
    np.array([[2 ** 64 - 1, 0]], dtype=np.uint64), np.array([[np.nan, 0.0]]), np.array([[1e10, 0.0]]),
    np.ma.array([[1, 2]], mask=[[1, 0]])])
def test_target_rows_out_of_range_are_refused(targets):
    """Numbers that int32 does not hold are refused as in lists, and not wrapped."""
    with pytest.raises((OverflowError, ValueError, np.ma.MaskError)):
        _target_rows(targets)
