"""A block a polygon's triplet ranking at its edges: one partition or none (20
triplets, 6 vertices), a full round of 256 threads and just past it (12 and 13
vertices), the last size whose triplets lie in LDS and the first that does not
(24 and 25), against the oracle.  The caps are
regular, so that most triplets tie with others."""
import pytest

from test_gpu_big_polygons import prism
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [6, 7, 12, 13, 24, 25, 48])
def test_prisms(ctx, n):
    compare(ctx, prism(n), prism(max(6, n - 5), r=0.7, h=1.4, centre=(0.2, 0.1, 0.3), twist=0.37))
