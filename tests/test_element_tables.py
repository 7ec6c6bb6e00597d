"""The element tables that the filter and the interpolation form on the device are the host's."""
import numpy as np
import pytest


@pytest.mark.parametrize("ne", [(1, 1, 1), (2, 3, 5), (5, 1, 4), (4, 4, 4)])
@pytest.mark.parametrize("N", [3, 4])
def test_element_tables(ne, N):
    from cmdg import closure
    from cmdg.grid import uniform_brick
    mk = lambda n: uniform_brick(n, (0, 0, 0), (1, 1, 1), N=N, lean=True)  # noqa: E731
    coarse, fine = mk(ne), mk(tuple(2 * n for n in ne))
    for got, ref in ((closure._children_on(coarse, fine, "cpu"), closure.children_map(coarse, fine)),
                     (closure._element_ijk_on(coarse, "cpu"), closure.element_ijk(coarse))):
        assert got.is_contiguous() and got.numpy().dtype == ref.dtype
        assert np.array_equal(got.numpy(), ref)
    with pytest.raises(ValueError):
        closure._children_on(coarse, coarse, "cpu")
    assert np.array_equal(closure._projection_words(N), closure.filter_projection(N).ravel())
    assert np.array_equal(closure._interpolation_words(N, 3), closure.interpolation_matrix(N, 3).ravel())
