"""Candidate values of the tuning parameters of the multi-kernel refinement and
of the general contraction, with the one-launch team paths off (wg_max_n = 0:
with the default the levels of these graphs hardly reach those kernels). Every
value gives the partitions of the defaults, bit for bit."""
import numpy as np
import pytest

import jet_amd
from jet_amd import autotune
from test_gpu_tuning import reference  # noqa: F401 (the graphs and their partitions with the defaults)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("knob", sorted(set(autotune.SPACE) - {"wg_max_n", "wg_big_deg"}))
def test_candidate_values_on_the_kernels(knob, reference):  # noqa: F811
    for v in autotune.SPACE[knob]:
        with jet_amd.tuned(**{knob: v, "wg_max_n": 0}):
            for name, g, cfg, (p0, c0) in reference:
                print(knob, v, name, flush=True)
                p, c = jet_amd.partition_csr(g, cfg, seed=3)
                assert c == c0, (knob, v, name)
                assert np.array_equal(p, p0), (knob, v, name)
