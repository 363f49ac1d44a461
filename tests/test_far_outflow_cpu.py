"""Outflow cells whose extrapolation source is more than one cell away (far_outflow_patterns)."""

import numpy as np

import xlb_amd as xa
from xlb_amd.operator.stepper.nse_stepper import far_outflow_patterns


def test_every_set_of_missing_directions_of_d2q9():
    """Against the definition: n = -c of the first missing axis direction, sources x - c_l - n."""
    c = np.asarray(xa.velocity_set.D2Q9(xa.PrecisionPolicy.FP32FP32, xa.ComputeBackend.MI355X).c)
    main = [l for l in range(9) if np.abs(c[:, l]).sum() == 1]
    got = far_outflow_patterns(c)
    assert got.shape == (512,)
    for bits in range(512):
        missing = [l for l in range(9) if bits >> l & 1]
        normal = next((-c[:, l] for l in main if l in missing), np.zeros(2, dtype=c.dtype))
        assert got[bits] == any(np.abs(c[:, l] + normal).max() > 1 for l in missing), bits
