"""A batch's gradient takes the histogram of the objective at the same points, as a pair's does, and
computes it anew when anything came between: other points, another histogram of one of the pairs,
or no objective at all.  Every way gives each pair exactly the gradient it computes alone.
"""
import numpy as np
import pytest

from niftyreg_amd.f3d import F3dBatch
from test_gpu_batch import SIZES, alone, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("between", ["objective", "nothing", "other points", "another histogram", "autotune"])
def test_gradient_after(gpu, between):
    pairs = [make_pair(d, 30 + i) for i, d in enumerate(SIZES[:3])]
    try:
        want = [alone(h, c) for h, c in pairs]
        b = F3dBatch([h for h, _ in pairs])
        try:
            for h, c in pairs:
                h.set_control_points(c)
            if between != "nothing":
                b.objective()
            if between == "other points":
                h, c = pairs[1]
                h.set_control_points(c + np.float32(0.75))
                b.objective()
                h.set_control_points(c)
            elif between == "another histogram":
                h, c = pairs[1]
                h.set_control_points(c + np.float32(0.75))
                h.GetDeformationField()
                h.ResampleImage()
                h.set_control_points(c)
                b.objective()
                h.GetSimilarityMeasureValue()  # of the warped image, which is that of the moved points
            elif between == "autotune":
                b.autotune()
            for _ in range(2):  # the second pass finds points that the first one's round trip touched
                maxlens = b.gradient(normalise=True)
                for q, (h, c) in enumerate(pairs):
                    assert maxlens[q] == want[q][2], q
                    assert np.array_equal(h.node_gradient(), want[q][3]), q
                    h.set_control_points(c)
        finally:
            b.close()
    finally:
        for h, _ in pairs:
            h.close()
