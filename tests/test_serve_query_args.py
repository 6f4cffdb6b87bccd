"""ResidentScene.sdf_query's arguments: the tile's origin is three numbers, which the kernel's call
reads from a host array; any other number of them is refused before the call."""
import pytest

from voxurf_amd import serve


@pytest.mark.parametrize("origin", [(), (1,), (1, 2), (1, 2, 3, 4)])
def test_origin_of_three(origin):
    scene = serve.ResidentScene.__new__(serve.ResidentScene)
    with pytest.raises(ValueError):
        scene.sdf_query(8, origin, 4)


def test_negative_tile():
    scene = serve.ResidentScene.__new__(serve.ResidentScene)
    with pytest.raises(ValueError):
        scene.sdf_query(8, (0, 0, 0), -1)
