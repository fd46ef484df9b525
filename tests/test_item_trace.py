"""The item trace says so when a launch left no records, instead of summing up none."""
import numpy as np
import pytest

from mpserve_amd.item_trace import _require_records


def test_no_records():
    with pytest.raises(RuntimeError, match="outside the trace"):
        _require_records(np.zeros((256, 128), dtype=bool))
    _require_records(np.eye(4, dtype=bool))
