"""The maps are cleared to the last word, whatever they held: maps of less than one piece of 4 KB, of pieces with a remainder,
and of more pieces than the clearing blocks (4 M, 17 GB); with the clear beside the tiles' preparation (small grids)
and by itself (192^3)."""
import numpy as np
import pytest
import torch

import crime_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


class _View:
    def __init__(self, gh):
        ptr, _ = gh.device_maps()
        self.__cuda_array_interface__ = dict(shape=(gh.n_nu, gh.npix), typestr="<f4" if gh.precision == crime_amd.FP32 else "<f8",
                                             data=(ptr, False), version=2, strides=None)


@pytest.mark.parametrize("n_grid, n_side, n_nu, precision", [(16, 1, 3, "single"), (16, 3, 5, "single"), (12, 17, 7, "double"),
                                                            (192, 33, 16, "single"), (16, 1024, 400, "single")])
def test_old_contents_go(cfgdir, n_grid, n_side, n_nu, precision):
    par = small_params(cfgdir, f"clr_{n_side}_{n_nu}", n_grid=n_grid, n_side=n_side, n_nu=n_nu, precision=precision,
                       l_box=600.0)
    with crime_amd.GetHI(par) as gh:
        gh.run()
        maps = torch.as_tensor(_View(gh), device="cuda")
        hit = int(torch.count_nonzero(maps))
        assert 0 < hit <= n_grid ** 3 * gh.n_sub
        maps.fill_(7.0)
        torch.cuda.synchronize()
        gh.mk_T_maps()
        assert int(torch.count_nonzero(maps)) == hit
        del maps
