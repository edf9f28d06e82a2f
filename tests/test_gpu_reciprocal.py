"""The parts of the short division that are results themselves in the
hydrodynamic pair terms: the reciprocal after its Newton step (2/b is taken
as twice it) and the short square root, against IEEE 1/b and sqrt(b) for
every float b they are used on.  The one numerator is zero, whose quotient
is zero whatever the reciprocal, so each mismatch counted is theirs."""
import numpy as np
import pytest

import sopgpu as S

pytestmark = pytest.mark.gpu


def test_reciprocal_and_square_root_equal_ieee_over_all_operands():
    print("case: every b in [2^-64, 2^62]", flush=True)
    assert S.check_division(0x1F800000, 0x5E800001, np.zeros(1, np.float32)) == 0
