"""The property lookup on both sides of 1,048,576 cells with tables in global
memory whose knots leave a CU two blocks of 256 (3400 knots) or one (4096):
bit for bit the CPU oracle's, as the other forms."""
import pytest

import test_gpu_property_forms as forms

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("knots", [3400, 4096])
@pytest.mark.parametrize("cells", [(1 << 20) - 1, 1 << 20])
def test_large_tables(knots, cells):
    forms.test_lookup_forms_bitwise(knots, cells, True)
