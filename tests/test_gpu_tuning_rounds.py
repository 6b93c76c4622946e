"""The tuned variant of the one-kernel QR and the batches that run in rounds: the
variant does not keep a small batch out of the rounds, and a small batch does not
choose the variant."""
import numpy as np
import pytest

from openrcwa_amd import engine, workloads

pytestmark = pytest.mark.gpu


def _solve(w, count, line, tmp_path, tune=False):
    ctx = engine.Context(0)
    f = tmp_path / "tune.txt"
    f.write_text(line)
    try:
        ctx.set_tuning_file(f, append=True)
        plan = engine.Plan(ctx, w["nX"], w["nY"], w["coord_x"], w["coord_y"], w["thickness"],
                           w["lam"][:count], w["kx0"][:count], w["ky0"][:count], w["eps"],
                           w["pols"][:count])
        choice = plan.autotune() if tune else None
        plan.execute()
        plan.sync()
        res = plan.results()
        plan.close()
    finally:
        ctx.close()
    assert not res.status.any()
    return res, choice, f.read_text()


# n = 162, 4 patterned layers: rounds for up to 22 matrices
def test_variant_does_not_shut_the_rounds_out(gpu_ctx, tmp_path):
    w = workloads.pillar2d(n_freq=2, nX=4, nY=4)
    plain, _, _ = _solve(w, 3, "gfx950 162 0 0 1.0\n", tmp_path)
    tuned, _, _ = _solve(w, 3, "gfx950 162 2 0 1.0\n", tmp_path)
    assert np.array_equal(plain.amp, tuned.amp)
    # the variant does reach a batch that is solved in one kernel
    plain, _, _ = _solve(w, 16, "gfx950 162 0 0 1.0\n", tmp_path)
    tuned, _, _ = _solve(w, 16, "gfx950 162 2 0 1.0\n", tmp_path)
    assert not np.array_equal(plain.amp, tuned.amp)


@pytest.mark.parametrize("variant", [0, 1, 2])
def test_small_plan_keeps_the_variant(gpu_ctx, tmp_path, variant):
    w = workloads.pillar2d(n_freq=2, nX=4, nY=4)
    _, (qr, tile), table = _solve(w, 2, f"gfx950 162 {variant} 0 1.0\n", tmp_path, tune=True)
    assert qr == variant
    assert table.splitlines()[-1].split()[1:4] == ["162", str(variant), str(tile)]
