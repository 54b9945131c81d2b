"""Host side of the operators (no GPU)."""
import numpy as np

from opymize_amd.linear import GradientOp


def test_grid_description_follows_its_attributes():
    """Kept between calls, formed again when an attribute changes, whatever
    sequence the spacing is assigned as."""
    A = GradientOp((3, 5), 2, imageh=(0.5, 2.0))
    g = A._grid()
    assert A._grid() is g and (g.ndims, g.nchannels, list(g.dims[:2]), list(g.h[:2])) == (2, 2, [3, 5], [0.5, 2.0])
    for h in ([1.0, 3.0], (1.5, 3.0), np.array([4.0, 0.25]), np.array([2, 3])):
        A.imageh = h
        assert list(A._grid().h[:2]) == [float(v) for v in h]
    A.imageh[1] = 7
    assert A._grid().h[1] == 7.0
    A.imagedims, A.nchannels = [4, 6], 1
    assert list(A._grid().dims[:2]) == [4, 6] and A._grid().nchannels == 1
