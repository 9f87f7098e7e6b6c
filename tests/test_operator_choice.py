"""The operator a timing picks does not hang on one launch that something else held up."""
import pytest


class _Timed:
    def __init__(self, ms, held_up=()):
        self.ms, self.held_up, self.turn = ms, held_up, 0

    def time_ms(self, X, **kw):
        self.turn += 1
        return self.ms * (10.0 if self.turn in self.held_up else 1.0)


@pytest.mark.parametrize("held_up", [(), (1,), (2,), (3,), (1, 3)])
def test_a_held_up_turn_does_not_decide(held_up):
    from paramspmm_ae_amd.GNN import _fastest

    slow, fast = _Timed(0.15), _Timed(0.11, held_up)
    assert _fastest([slow, fast], None) is fast and _fastest([_Timed(0.11, held_up), _Timed(0.15)], None).ms == 0.11
    same = [_Timed(0.1), _Timed(0.1)]
    assert _fastest(same, None) is same[0]  # a tie keeps the first
