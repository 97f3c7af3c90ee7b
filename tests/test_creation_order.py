"""Objects that clear device memory on the null stream and then work on a
non-blocking stream of their own, which does not wait for the null stream:
their creation has to wait for the clearing before it returns.  Read from the
sources, since a lost wait shows on the device only now and then."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "exahype_amd", "csrc")


@pytest.mark.parametrize("source,function", [("capi.hip", "exa_grid_create"), ("capi.hip", "exa_ensemble_create"),
                                             ("fv_capi.hip", "exa_fv_grid_create"),
                                             ("amr_grid.hip", "exa_amr_grid_create")])
def test_creation_waits_for_its_clearing(source, function):
    with open(os.path.join(CSRC, source)) as f:
        text = f.read()
    body = re.search(r'^extern "C" int %s\(.*?^}' % function, text, re.M | re.S).group()
    memsets = [m.start() for m in re.finditer(r"hipMemset\(", body)]
    assert memsets
    assert body.rfind("hipStreamSynchronize(nullptr)") > memsets[-1]
