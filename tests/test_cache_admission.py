"""Requests admitted together: their states cleared a run of neighbouring slots at a time, and nobody else's touched."""
import pytest
import torch

from infernum_amd.cache import CacheConfig, CacheManager, PageError
from infernum_amd.parts import StateSpec


def manager(slots):
    needs = [(None, StateSpec((3, 2), torch.float32)), (None, None), (None, StateSpec((5,), torch.float32))]
    return CacheManager(needs, [None] * len(needs), CacheConfig(page_size=4, num_pages=4, num_state_slots=slots),
                        dtype=torch.float32, device=torch.device("cpu"))


@pytest.mark.parametrize("leave", [(), (2,), (1, 3, 4), (0, 1, 2, 3, 4, 5)])
def test_states_of_requests_admitted_together_are_cleared(leave):
    m = manager(8)
    assert m.admit_many(range(6)) == 6 and m.admit_many([]) == 0
    for r in leave:
        m.release(r)
    for st in m.state:
        if st is not None:
            st.fill_(7.0)
    new = [f"n{i}" for i in range(len(leave) + 1)]
    assert m.admit_many(new) == len(new)
    cleared = {m.state_slot(r) for r in new}
    for st in m.state:
        if st is not None:
            for slot in range(8):
                assert bool((st[slot] == (0.0 if slot in cleared else 7.0)).all()), slot


def test_admitted_together_with_too_few_slots_and_twice():
    m = manager(3)
    assert m.admit_many("abcd") == 3 and not m.has("d") and not m.admit("d")
    m.release("a"), m.release("b")
    for st in (m.state[0], m.state[2]):
        st.fill_(7.0)
    with pytest.raises(PageError, match="twice"):
        m.admit_many(["e", "c", "f"])
    assert m.has("e") and not m.has("f") and bool((m.state[2][m.state_slot("e")] == 0.0).all())    # as one after the other
    assert bool((m.state[2][m.state_slot("c")] == 7.0).all())
