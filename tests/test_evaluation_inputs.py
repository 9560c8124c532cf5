"""What the evaluation calls take for entity ids and counts: the integers torch.as_tensor takes, no more and no less."""
import numpy as np
import pytest
import torch

from smore_amd import _lib

VALUES = {
    "ints": [3, 4], "tuple": (3, 4), "range": range(3), "set": {3, 4}, "keys": {3: 1}.keys(), "empty": [], "array": np.array([3, 4]),
    "int32": np.array([3, 4], dtype=np.int32), "uint8": np.array([3, 4], dtype=np.uint8), "tensor": torch.tensor([3, 4]),
    "scalars": [torch.tensor(3), torch.tensor(4)], "one-element tensors": [torch.tensor([3]), torch.tensor([4])],
    "floats": [1.5, 2.0], "bools": [True, False], "objects": np.array([3, 4], dtype=object), "numpy scalars": [np.int64(3), np.int32(4)],
    "strings": ["3", "4"], "string": "34", "bytes": b"34", "string array": np.array(["3"]), "dates": np.array(["2020-01-01"], "M8[D]"),
    "float tensor": torch.tensor([1.5]), "too large": [2 ** 63], "uint64": np.array([2 ** 63 + 1], dtype=np.uint64), "nan": [float("nan")],
    "none": [None], "ragged": [[1], [2, 3]], "negative": [-1, 2],
}


def _either(f):
    try:
        return f().tolist()
    except Exception as e:
        return "refused" if isinstance(e, (TypeError, ValueError, RuntimeError, OverflowError)) else e


@pytest.mark.parametrize("kind", VALUES)
def test_answer_ids(kind):
    from smore_amd.evaluation.ranking import _int64
    x = VALUES[kind]
    want = _either(lambda: torch.as_tensor(list(x), dtype=torch.int64))
    assert _either(lambda: _int64(x)) == want
    assert want == "refused" or _int64(x).dtype == np.int64


@pytest.mark.parametrize("kind", [*VALUES, "scalar", "too large for 32 bits"])
def test_hard_answer_counts(kind):
    from smore_amd.evaluation.ranking import _counts
    x = {"scalar": 3, "too large for 32 bits": [2 ** 31]}.get(kind, VALUES.get(kind))
    want = _either(lambda: torch.as_tensor(x, dtype=torch.int32).reshape(-1))
    assert _either(lambda: _counts(x)) == want
    assert want == "refused" or _counts(x).dtype == torch.int32


@pytest.mark.parametrize("kind", VALUES)
def test_answer_lists_in_one_array(kind):
    """Lists taken together give what each would alone, or are left to be taken one by one."""
    from smore_amd.evaluation.ranking import _int64, _one_array
    lists = [[7, 8], VALUES[kind], (), [9]]
    flat = _one_array(lists)
    if flat is not None:
        assert flat.dtype == np.int64 and flat.tolist() == [int(v) for x in lists for v in _int64(x)]
    else:
        assert kind not in ("ints", "tuple", "empty", "numpy scalars", "negative")


def test_counts_on_another_device_are_brought_to_the_table():
    """Counts that are on a device already are those of the table's device, whichever they came from."""
    from smore_amd.evaluation.ranking import _counts_on

    class Counts:
        device, dtype = torch.device("cuda", 1), torch.int32

        def to(self, device):
            return "counts on", device

    for index in (0, 1):
        dev = torch.device("cuda", index)
        assert _counts_on(Counts(), dev) == ("counts on", dev)


@pytest.mark.parametrize("easy,hard,error,message", [([[9]], [[1]], IndexError, "outside the entity table"),
                                                     ([[1]], [[1]], _lib.SmxError, "listed twice"),
                                                     ([[2]], [[1]], _lib.SmxError, "fp32 device tensor")])
def test_a_table_on_the_host_is_refused_for_the_reason_it_always_was(easy, hard, error, message):
    """Pinned memory is for copies to a device: none is asked for (and none is needed) where the table is on the host."""
    from smore_amd.evaluation.ranking import filtered_ranks
    table, q = torch.rand(5, 4), torch.rand(1, 4)
    with pytest.raises(error, match=message):
        filtered_ranks("l1", table, q, None, None, easy, hard)


def test_candidates_on_the_host_are_refused_for_the_reason_they_always_were():
    from smore_amd.evaluation.ranking import candidate_ranks
    with pytest.raises(_lib.SmxError, match="fp32 device tensor"):
        candidate_ranks("l1", torch.rand(5, 4), torch.rand(1, 4), None, None, torch.tensor([[1, 2]]), [1])
