"""The arrays of a segment plan are stretches of one allocation: what the kernels are handed has to be the arrays that the plan holds now."""
import copy

import pytest
import torch

ARRAYS = ("order", "sorted_ids", "seg_of_pos", "seg_start", "uniq_buf", "n_uniq_dev", "pair_seg")
FIELDS = dict(zip(ARRAYS, range(len(ARRAYS))))


def _addresses(plan):
    view = plan.view()
    return [getattr(view, name) for name, _ in view._fields_][: len(ARRAYS)]


@pytest.mark.parametrize("n_pairs", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("want_inverse", [False, True])
def test_arrays_do_not_overlap(n_pairs, want_inverse):
    from smore_amd.fused import SegmentPlan
    plan = SegmentPlan(n_pairs, 10_000, torch.device("cpu"), want_inverse)
    names = ARRAYS + (("inverse",) if want_inverse else ())
    for i, name in enumerate(names):
        getattr(plan, name).fill_(i + 1)
    for i, name in enumerate(names):
        t = getattr(plan, name)
        assert t.numel() == (1 if name == "n_uniq_dev" else n_pairs + (name == "seg_start"))
        assert t.dtype == (torch.int64 if name in ("uniq_buf", "inverse") else torch.int32)
        assert (t == i + 1).all() and t.data_ptr() % 8 == 0
    assert want_inverse or plan.inverse is None
    assert _addresses(plan) == [getattr(plan, name).data_ptr() for name in ARRAYS]


@pytest.mark.parametrize("touched", [False, True])
def test_a_deep_copy_has_memory_of_its_own(touched):
    from smore_amd.fused import SegmentPlan
    plan = SegmentPlan(100, 1000, torch.device("cpu"), True)
    plan.order.copy_(torch.arange(100, dtype=torch.int32)) if touched else None
    other = copy.deepcopy(plan)
    assert not set(_addresses(plan)) & set(_addresses(other))
    assert _addresses(other) == [getattr(other, name).data_ptr() for name in ARRAYS]
    if touched:
        assert torch.equal(other.order, plan.order)
        plan.order.zero_()
        assert other.order[99] == 99


def test_an_array_that_the_caller_replaced_is_the_one_handed_out():
    from smore_amd.fused import SegmentPlan
    plan = SegmentPlan(100, 1000, torch.device("cpu"), False)
    plan.pair_seg = torch.zeros(100, dtype=torch.int32)
    assert _addresses(plan)[FIELDS["pair_seg"]] == plan.pair_seg.data_ptr()


@pytest.mark.parametrize("touched", [False, True])
@pytest.mark.parametrize("name", ARRAYS)
def test_an_array_that_the_caller_took_away_is_a_null_pointer(name, touched):
    """pair_seg may be missing (the one-pair fast path is not used then); without another array the library refuses the plan."""
    from smore_amd.fused import SegmentPlan
    plan = SegmentPlan(100, 1000, torch.device("cpu"), True)
    if touched:
        getattr(plan, name)
    setattr(plan, name, None)
    assert getattr(plan, name) is None and _addresses(plan)[FIELDS[name]] is None
    assert all(a for n, a in zip(ARRAYS, _addresses(plan)) if n != name)
