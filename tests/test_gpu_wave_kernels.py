"""A batch's waves run the smallest kernel that holds their phases (WaveNeed,
wave.hpp): plain stamps, stamps on canvas column/row 0, anything.  Each of
those waves gives what the job's list gives alone, to the bit."""
import numpy as np
import pytest
import torch  # noqa: F401  (before the library: it brings the HIP runtime up)

from painty_amd import _lib
from painty_amd import workload as W
from tests.test_gpu_batch import _layers, _setup, restore_config  # noqa: F401

pytestmark = pytest.mark.gpu


def _job(place, radius, seed):
    """20 stamps in two strokes: inside, over column 0, over row 0, or over
    the corner; fractional centres, the last stroke away from the edges."""
    wl = W.small(150, 170, 20, radius, seed, pickup=True, noisy=True, reach=0.1)
    rs = np.random.RandomState(seed)
    st = wl.stamps
    n = len(st)
    for k in range(n):
        edge = k < n // 2
        x, y = 80.0 + rs.uniform(-9, 9), 70.0 + rs.uniform(-9, 9)
        if edge and place in ("column", "corner"):
            x = rs.uniform(0.2, 0.8 * radius + 0.3)
        if edge and place in ("row", "corner"):
            y = rs.uniform(0.2, 0.8 * radius + 0.3)
        st["cx"][k], st["cy"][k] = x, y
    return wl


@pytest.mark.parametrize("radius", [1, 7, 16])
@pytest.mark.parametrize("places,snap,dry", [
    (("inside", "inside"), True, False),
    (("inside", "column"), True, False),
    (("row", "corner"), True, False),
    (("corner", "inside"), True, True),
    (("column", "row"), False, False),
])
def test_waves_of_each_need_equal_the_list_alone(hip, restore_config, radius, places, snap, dry):
    hip.batch_set_config(16, 1, 1, 1)
    wls = [_job(p, radius, 31 + i) for i, p in enumerate(places)]
    if dry:
        wls[0].stamps["flags"][9] |= W.DRY_AFTER
    jobs, alone = [], []
    for wl in wls:
        cv, br, out = _setup(hip, wl, snap)
        jobs.append((cv, br, wl.stamps, out))
        cv2, br2, _ = _setup(hip, wl, snap)
        br2.imprintStamps(wl.stamps, cv2, mode=_lib.EXEC_FUSED)
        alone.append((cv2, br2))
    hip.batch_run(jobs)
    for (cv, br, _, _), (cv2, br2) in zip(jobs, alone):
        for a, b in zip(_layers(cv), _layers(cv2)):
            np.testing.assert_array_equal(a, b)
        for a, b in zip(br.getPickupMap(), br2.getPickupMap()):
            np.testing.assert_array_equal(a, b)
