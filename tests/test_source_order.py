"""Orders of host calls that no result shows reliably, read from the sources."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "exahype_amd", "csrc")


def _body(source, function):
    with open(os.path.join(CSRC, source)) as f:
        return re.search(r'^extern "C" int %s\(.*?^}' % function, f.read(), re.M | re.S).group()


@pytest.mark.parametrize("source,function", [("capi.hip", "exa_grid_create"), ("capi.hip", "exa_ensemble_create"),
                                             ("fv_capi.hip", "exa_fv_grid_create"),
                                             ("amr_grid.hip", "exa_amr_grid_create")])
def test_creation_waits_for_its_clearing(source, function):
    """Objects that clear device memory on the null stream and then work on a
    non-blocking stream of their own, which does not wait for the null stream:
    creation waits for the clearing before it returns."""
    body = _body(source, function)
    memsets = [m.start() for m in re.finditer(r"hipMemset\(", body)]
    assert memsets
    assert body.rfind("hipStreamSynchronize(nullptr)") > memsets[-1]


def test_timed_phases_of_a_patch_grid_hold_their_launches():
    """The events around the ghost layers, the update and the time step stand
    on both sides of a launch; a pair around nothing reads 5 us as well, as
    much as the short launches."""
    body = _body("fv_capi.hip", "exa_fv_grid_step")
    marks = [re.search(r"hipEventRecord\(m\[%d\]" % k, body).start() for k in range(5)]
    assert marks == sorted(marks)
    for k, launch in ((0, "k_fv_ghosts"), (2, "launch_fv_update("), (3, "k_fv_dt_advance")):
        assert launch in body[marks[k]:marks[k + 1]]
