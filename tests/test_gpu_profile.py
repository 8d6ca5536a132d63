"""athmi_profile_steps times the kernels that the step launches, and names the
path a batch takes: the paired predictor, the merged sweeps, the march that
holds the corrector and the final update (at the sizes whose results the tests of
those kernels check), or the separate kernels."""
import ctypes

import pytest

from helpers import load_pkg
from test_gpu_corr_final import BCS, EDGES, FILLER, FILLERS
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu

SEPARATE = ["k_begin", "k_pred_x1", "k_pred_x2", "k_corner<pred>", "k_corr<1>", "k_corr<2>",
            "k_corner<corr>", "k_final", "k_ghost", "k_end"]


def profile(pkg, g, nslots, steps=2):
    L = pkg.lib()
    L.athmi_step_kernel_name.restype = ctypes.c_char_p
    avg = (ctypes.c_double * 20)(*[-1.0] * 20)
    n0 = g.clock(0)[2]
    rc = L.athmi_profile_steps(g._h, ctypes.c_int(steps), avg, ctypes.c_int(nslots))
    assert rc == 0 and g.clock(0)[2] == n0 + steps
    names = [L.athmi_step_kernel_name(k).decode() for k in range(20)]
    assert names[:10] == SEPARATE and names[14:] == [""] * 6
    shown = 14 if nslots >= 14 else 10
    assert all(t >= 0.0 for t in avg[:shown]) and all(t == -1.0 for t in avg[shown:])
    return {names[k] for k in range(shown) if avg[k] > 0.0}


def ready(pkg, descs):
    g = pkg.Grid(descs)
    for k, d in enumerate(descs):
        g.upload(k, *state(d["nx1"], d["nx2"], k))
        g.set_clock(k, 1e-4 / max(d["nx1"], d["nx2"]), 0.0, 1)
    g.set_bvals()
    g.set_limits(1e30, -1)
    return g


@pytest.mark.parametrize("nx,ny,flux,shape,want", [
    (64, 64, "roe", None, {"k_pred_pair", "k_corr_both", "k_final"}),
    (300, 200, "hlle", None, {"k_pred", "k_corr_both", "k_final"}),
    (1301, 1001, "hlle", (3, 0), {"k_pred", "k_corr_final"}),
    (1240, 1040, "hlle", (3, 0), {"k_pred", "k_corr_final"}),
    (1985, 1701, "roe", (3, 0), {"k_pred", "k_corr_final"}),
    (1985, 1701, "roe", (3, 1), {"k_pred_x1", "k_pred_x2", "k_corr<1>", "k_corr<2>", "k_final"}),
    (3, 40, "roe", None, {"k_pred_pair", "k_corr_both", "k_final", "k_ghost"}),
])
def test_the_steps_own_kernels(nx, ny, flux, shape, want):
    pkg = load_pkg()
    g = ready(pkg, [desc(nx, ny, flux, (4, 4, 1, 2))])
    if shape:
        g.set_shape(*shape)
    assert profile(pkg, g, 16) == want | {"k_begin", "k_corner<pred>", "k_end"}
    # a caller with the ten slots only: the separate kernels (corners inside k_final)
    for nslots in (10, 13):
        assert profile(pkg, g, nslots) == set(SEPARATE) - {"k_corner<corr>"}
    assert pkg.lib().athmi_profile_steps(g._h, 1, (ctypes.c_double * 20)(), 9) != 0
    g.close()


@pytest.mark.parametrize("main,others", [("hlle", 0), ("hlle", 3), ("roe", 0), ("roe", 3)])
def test_ensembles_take_the_march(main, others):
    pkg = load_pkg()
    other = "roe" if main == "hlle" else "hlle"
    descs = [desc(*n, main, b) for k, n in enumerate(EDGES) for b in (BCS[k % 5], BCS[(k + 2) % 5])]
    descs += [desc(*FILLER, main, BCS[1])] * FILLERS[main] + [desc(*FILLER, other, BCS[4])] * others
    g = ready(pkg, descs)
    got = profile(pkg, g, 14)
    assert "k_corr_final" in got
    assert ("k_corr_both" in got) == ("k_final" in got) == (others > 0)
    g.close()
