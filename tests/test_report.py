"""The per-configuration report's account of one F^H d, by the path it took."""
import json

import pytest


def _records(**given):
    return lambda name: given.get(name, (0.0, 0))


def test_fhd_account_by_path():
    from impatient.report import fhd_account
    nk, nv, nz = 8192 * 16, 64 * 64 * 16, 16
    for rec, want in (
            (dict(nufft_stack=(0.5, 1)), (0.5, "separable", 0.0)),
            (dict(nufft_adjoint=(7.0, 1)), (7.0, "separable", 0.0)),
            (dict(k_nudft_stack=(1.0, 2), k_reduce_stack=(0.25, 1)),
             (1.25, "stacked (z-separable)", 2.0 * 8192 * nv)),
            (dict(k_nudft_mfma=(3.0, 1)), (3.0, "direct", float(nk) * nv)),
            (dict(k_nudft_valu=(2.0, 1)), (2.0, "direct", float(nk) * nv))):
        ms, path, evaluated, parts = fhd_account(_records(**rec), nk, nv, nz)
        assert (ms, path, evaluated) == want
        assert {k: v for k, v in parts.items() if v[1]} == rec


@pytest.mark.gpu
@pytest.mark.parametrize("config", [0, 1])
def test_report_runs(ctx, config, capsys):
    """64^2 x 1 coil (direct) and 64^2 x 16 x 4 coils (a stack in separable
    form), a few iterations of each solver."""
    from impatient import report
    assert report.main(["--config", str(config), "--cg-max-iter", "5"]) == 0
    out = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert out["fhd_path"] == ("separable" if config == 1 else "direct")
    assert out["fhd_ms"] > 0 and out["fhd_gsample_vox_s"] > 0
