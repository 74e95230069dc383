"""MVN over many short groups, either side of the lines at which their kernel and the groups a workgroup takes change."""
import pytest

from test_gpu_mvn_groups import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups,len_", [((1 << 18) - 1, 24), (1 << 18, 24), ((1 << 18) + 5, 72), ((1 << 18) + 9, 96), ((1 << 18) + 1, 104), ((1 << 17) - 1, 129), ((1 << 17) + 3, 129),
                                         ((1 << 17) + 15, 255), ((1 << 17) + 1, 257)])
def test_groups(rt, dev, groups, len_):
    run(rt, dev, (1, groups, 1, len_), False)
