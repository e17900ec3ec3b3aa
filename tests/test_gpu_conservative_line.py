"""The FP64 conservative form on meshes of more than two blocks per compute unit, which take the line
kernel's default block: against the oracle, bar as in the other residual parity tests."""
import pytest

import philip_amd as P
from test_gpu_line64 import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,n", [(1, 26), (2, 17), (3, 13), (4, 11), (5, 9)])
@pytest.mark.parametrize("cf", [P.LXF, P.ROE])
def test_default_block_conservative(p, n, cf):
    check(dict(dim=3, poly_degree=p, n_cells_1d=n, use_split_form=0, conv_flux=cf, mach_inf=0.3), 23 * p + n)
