"""The public array of an ensemble's kernel times keeps its size and order."""
import os
import re

import pytest

NAMES = ["kb_cfl", "kb_dispersion", "kb_wave", "kb_wave_rows", "kb_flow_nuh", "kb_flow_u", "kb_flow_v", "kb_flow_uvcorr",
         "kb_flow_zsall", "kb_flow_uvvu", "kb_sed_flux", "kb_sed_conc", "kb_sed_morph"]


def test_names_keep_their_places():
    from xbeach_gpu_amd import lib

    L = lib()
    assert [L.xbg_ens_kernel_name(k).decode() for k in range(len(NAMES))] == NAMES
    assert L.xbg_ens_kernel_name(len(NAMES)) is None and L.xbg_ens_kernel_name(-1) is None
    h = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "xbg.h")).read()
    assert re.search(r"#define XBG_ENS_NKERNELS (\d+)", h).group(1) == str(len(NAMES))


@pytest.mark.gpu
def test_times_of_the_classes(need_gpu):
    from test_gpu_wave_tiles import CASES, build
    from xbeach_gpu_amd.ensemble import Ensemble, RunSetup

    d, _, _, _, Trep = build(3, *CASES[3][:3], CASES[3][3])
    ens = Ensemble([d], [RunSetup(150.0, 0.05, 1e9, 150.0, 1.0, Trep)])
    us = ens.kernel_times(3)
    assert list(us) == NAMES and us["kb_wave_rows"] == 0.0
    assert all(v > 0.0 for k, v in us.items() if k != "kb_wave_rows")
    ens.step(1)
    assert (ens.status()[2] == 4).all()
    ens.close()
    d.close()
