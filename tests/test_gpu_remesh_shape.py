"""The remesh launch shape where none is set: the getter answers what runs, and
putting an answer back leaves the context as it was."""
import ctypes as C

import pytest

from voxplat_amd import abi

pytestmark = pytest.mark.gpu

BIG, SMALL = abi.WorldDesc.make(6, (1, 1, 1)), abi.WorldDesc.make(5, (1, 1, 1))
OF_BIG = {"block": 1024, "wg_per_cu": 1, "records_in_flight": 4}
OF_SMALL = {"block": 512, "wg_per_cu": 2, "records_in_flight": 4}


@pytest.fixture
def fresh():
    """A context nobody has set a shape in."""
    from voxplat_amd import GPU

    g = GPU(0)
    yield g
    g.close()


def _unset(g):
    return (g.get_remesh_shape(), g.get_remesh_shape(BIG), g.get_remesh_shape(SMALL),
            tuple(g.get_launch())) == (OF_BIG, OF_BIG, OF_SMALL, (1024, 1))


def test_the_default_is_restored_by_its_own_answer(fresh):
    assert _unset(fresh)
    keep = fresh.get_remesh_shape()
    fresh.set_remesh_shape(None, 256, 2, 2)
    assert fresh.get_remesh_shape(SMALL) == fresh.get_remesh_shape(BIG) == \
        {"block": 256, "wg_per_cu": 2, "records_in_flight": 2}
    fresh.set_remesh_shape(None, keep["block"], keep["wg_per_cu"], keep["records_in_flight"])
    assert _unset(fresh)
    launch = fresh.get_launch()
    fresh.set_launch(512, 2)
    assert tuple(fresh.get_launch()) == (512, 2)
    assert fresh.get_remesh_shape(BIG) == OF_SMALL
    fresh.set_launch(*launch)
    assert _unset(fresh)


@pytest.mark.parametrize("w", [BIG, SMALL])
def test_a_world_is_restored_by_its_own_answer(fresh, w):
    keep = fresh.get_remesh_shape(w)
    fresh.set_remesh_shape(w, 256, 1, 2)
    assert fresh.get_remesh_shape(w)["block"] == 256
    fresh.set_remesh_shape(w, keep["block"], keep["wg_per_cu"], keep["records_in_flight"])
    assert _unset(fresh)


def test_a_failed_tuning_leaves_the_shape(fresh):
    """No voxels: the first launch is refused and the shape goes back."""
    best, ms, timed = abi.RemeshShape(), C.c_float(), C.c_int()
    rc = fresh.lib.vp_host_autotune_remesh(fresh.ctx, C.byref(BIG), None, None, None, None, 1, 0,
                                           None, 1, None, C.byref(best), C.byref(ms),
                                           C.byref(timed))
    assert rc == -1                      # VP_ERR_ARG
    assert _unset(fresh)
