"""GPU: circuits whose blocks have so many exchanges that no swizzle serves all of
them without bank conflicts, and their neighbours that one serves, in split and
whole-amplitude exchanges, against the oracle.

Any swizzle is a bijection, so a wrong slot would move amplitudes: errors of the size
of an amplitude.  Allowed are 4 roundings for each gate on the amplitudes (at most
1): 4 * gates * 2^-53, in FP32 * 2^-24.
"""
import numpy as np
import pytest

from dgquest_amd import circuits
from oracle.binding import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shape", [(8, (2, 2, 0)), (10, (4, 3, 1)), (12, (6, 3, 3)), (12, (6, 4, 2)), (13, (7, 4, 3)),
                                     (13, (4, 4, 0))])
@pytest.mark.parametrize("family", ["hea", "layered"])
@pytest.mark.parametrize("prec", [1, 2])
def test_many_exchanges(n, shape, family, prec, quest, env, quest32, env32):
    api, e = (quest, env) if prec == 2 else (quest32, env32)
    circ = circuits.hea(n, 10, 3) if family == "hea" else circuits.layered_u3_cz(n, 16, 2)
    ref = np.zeros(1 << n, dtype=np.complex128)
    ref[0] = 1.0
    Oracle().run(ref, circ)
    q = api.createQureg(n, e)
    try:
        api.dgq_set_tuning(q, *shape, 4096)
        api.apply_circuit(q, circ)
        err = np.abs(api.state_vector(q) - ref).max()
        assert err <= 4 * len(circ) * (2.0 ** -53 if prec == 2 else 2.0 ** -24)
    finally:
        api.destroyQureg(q, e)
