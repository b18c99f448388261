"""GPU: registers that are one tile, whose workgroup brings its descriptors to the
device itself: flush after flush on one register, each with other descriptors of another
length (one load per thread, several, more than fit a slot), against the oracle.

A line of an earlier flush read in place of a new one would be another circuit.  Allowed
are 4 roundings for each gate on the amplitudes (at most 1), over all gates so far.
"""
import numpy as np
import pytest

from dgquest_amd import circuits
from oracle.binding import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shape", [(10, (4, 3, 1)), (11, (5, 3, 2)), (12, (6, 3, 3)), (13, (7, 4, 3)), (12, (6, 4, 2))])
@pytest.mark.parametrize("prec", [1, 2])
def test_flush_after_flush(n, shape, prec, quest, env, quest32, env32):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    ref = np.zeros(1 << n, dtype=np.complex128)
    ref[0] = 1.0
    q = api.createQureg(n, e)
    gates = 0
    try:
        api.dgq_set_tuning(q, *shape, 4096)
        for i, depth in enumerate((1, 12, 2, 40, 3, 1, 6)):
            circ = circuits.hea(n, depth, i) if i % 2 else circuits.layered_u3_cz(n, depth, i)
            gates += len(circ)
            Oracle().run(ref, circ)
            api.apply_circuit(q, circ)
            err = np.abs(api.state_vector(q) - ref).max()
            assert err <= 4 * gates * (2.0 ** -53 if prec == 2 else 2.0 ** -24), (i, err)
    finally:
        api.destroyQureg(q, e)
