"""The float32 scans at the edges of the rules that choose vectors and splits by the number of columns: rows just past one wave of single elements, just below two
vectors a lane, a first and a last shape of each rule, with time left over, against the sequential reference in double precision."""
import pytest

from test_gpu_scan_plans import test_scan_plans as check_plan

pytestmark = pytest.mark.gpu

SHAPES = [
    (504, 33, 65), (505, 33, 65), (702, 70, 67), (300, 257, 111), (293, 257, 112),    # rows of 65 to 111, four and eight waves
    (512, 70, 96), (513, 70, 96), (1025, 70, 97), (512, 256, 101), (341, 255, 102),                   # from 96 floats on: eight waves up to 512 rows
    (400, 1023, 83), (400, 1024, 83),                                                 # the longest sequence of that rule
    # MinGRU backward streaming, but for rows of one workgroup and 341 to 512 workgroups; short sequences
    (342, 64, 193), (342, 63, 193), (341, 70, 191), (130, 97, 1007), (134, 66, 1007), (340, 64, 193), (512, 70, 193), (513, 70, 193), (513, 256, 193), (340, 256, 193),
    (150, 255, 700), (150, 256, 700), (171, 70, 700),
    (255, 128, 129), (255, 127, 129), (64, 131, 515), (127, 150, 515), (128, 150, 515),   # four elements per lane
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["f32", "mingru"])
def test_scan_plan_edges(kind, shape):
    # the bound of the other plans' test: float32 sums of products of at most one, over the memory of decays of 0.8 to 1
    check_plan(kind, shape)
