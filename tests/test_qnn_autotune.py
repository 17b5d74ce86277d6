"""What QNNBatch.autotune may choose: nothing that changes results."""
import pytest

from quict_amd.gradient.qnn import DEFAULT_CONFIG, QNNBatch


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("fuse", [1, 2, 3])
def test_the_order_of_rounding_is_not_chosen_by_time(precision, fuse):
    qb = QNNBatch.__new__(QNNBatch)
    qb.precision, qb.config = precision, {**DEFAULT_CONFIG, "fuse_qubits": fuse}
    space = list(qb.search_space())
    assert space and all(c["fuse_qubits"] == fuse for c in space)
    assert space[0] is not qb.config
