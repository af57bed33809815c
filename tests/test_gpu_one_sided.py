"""The masks' one-sided distance test, taken above 65,536 particles: lattices
whose neighbours lie at exactly the cut, where it lets slots pass that the exact
test does not, on either side of the size at which the exact test ends."""
import pytest

from helpers import announce
from test_gpu_fast_arithmetic import _check, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65536, 65537, 68921])
@pytest.mark.parametrize("centred,r2", [(True, 0.35 * 0.35), (False, 0.04), (True, 0.03)])
def test_neighbours_at_the_cut_bitexact(n, centred, r2):
    announce("one-sided", n, centred, r2)
    pos, vel, p = _scene(0.2, n=n, jitter=0.0, centred=centred)
    p.prefilter_r2 = r2
    _check(pos, vel, p, True)
