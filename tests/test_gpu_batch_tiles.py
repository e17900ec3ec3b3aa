"""Which tile a batch takes, and FP64 Kennedy-Gruber and Ismail-Roe solves in a batch and in a stream:
these run in kernels of their own, beside Chandrashekar solves of the same shape.  Bar: the bits of the
same solve alone."""
import numpy as np
import pytest

import philip_amd as P

pytestmark = pytest.mark.gpu
SMALL_2D = {1: 16, 2: 10, 3: 8, 4: 6, 5: 5, 6: 4}  # elements of the small meshes' block, by degree


def params(dim, p, n, tp=P.CH, precision=P.FP64, cf=P.TWO_POINT_ROE):
    kw = dict(dim=dim, poly_degree=p, n_cells_1d=n, use_split_form=1, two_point_flux=tp, conv_flux=cf, mach_inf=0.3,
              precision=precision)
    if dim == 2:
        kw.update(domain_left=-5.0, domain_right=5.0, mach_inf=1.195228609334)
    return kw


def start(d, dim):
    d.set_initial_condition_vortex() if dim == 2 else d.set_initial_condition_tgv()


def batch(cases, tile=-1, steps=0):
    """Batch of the cases after `steps` RK4 steps."""
    b = P.Batch(cases)
    for d, kw in zip(b.instances, cases):
        start(d, kw["dim"])
    b.set_tile(tile)
    b.allocate("rk4", [d.constant_time_step(0.01) for d in b.instances])
    if steps:
        b.step_in_time(steps)
        b.synchronize()
    return b


def test_no_tile_for_a_block_that_single_solves_do_not_take():
    """FP64 3D p=6: the small meshes' block (768 threads) would spill."""
    b = batch([params(3, 6, 3)] * 2, tile=2)
    assert b.tile(0)[2] != 768
    b.close()


@pytest.mark.parametrize("precision", [P.FP64, P.MIXED])
@pytest.mark.parametrize("first", ["tiny", "large"])
def test_tile_follows_the_batch_and_not_what_ran_before(first, precision):
    """A batch that leaves most of the chip idle takes the small meshes' tile, one that fills it a timed
    tile, in either order and again."""
    p = 1 if first == "tiny" else 4  # a shape of its own for each order
    tiny, large = [params(2, p, 8, precision=precision)] * 2, [params(2, p, 128, precision=precision)] * 4
    order = [tiny, large, tiny, large] if first == "tiny" else [large, tiny, large]
    for cases in order:
        b = batch(cases)
        print(first, precision, len(cases), b.tile(0), flush=True)
        assert (b.tile(0)[0] == SMALL_2D[p]) == (cases is tiny)
        b.close()
