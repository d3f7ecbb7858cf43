"""The undefined-scalar-register check of test_isa_guard.py on the tile-expansion kernels."""
import os

import pytest

import test_isa_guard


@pytest.mark.skipif(not os.path.exists(test_isa_guard.HIPCC), reason="hipcc not available")
def test_far_kernels():
    test_isa_guard.test_no_undefined_scalar_registers_in_kernels("lt_far.hip")
