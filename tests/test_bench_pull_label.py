"""bench.py names the pull that ran, not the one that was asked for (no GPU)."""
from types import SimpleNamespace

import pytest

import bench


class _Graph:
    def __init__(self, regrouped):
        self.regrouped = regrouped

    def info(self):
        return [0] * 11 + ([9, 4, 5, 0] if self.regrouped else [0] * 4) + [0]


@pytest.mark.parametrize("asked,regrouped,ran", [("hotcold", True, "hotcold"), ("hotcold", False, "plain"),
                                                 ("plain", False, "plain"), ("segmented", True, "segmented")])
def test_pull_that_ran(asked, regrouped, ran):
    assert bench.pull_run(SimpleNamespace(pull=asked), _Graph(regrouped)) == ran
    assert ran in bench.PULL_KERNELS
