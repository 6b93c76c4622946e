"""The cascade's column chain (blocks of 32 rows solved by waves with their own
roles) against the oracle: matrix orders around its block edges, with several
patterned layers so that every link of the chain runs."""
import numpy as np
import pytest

from oracle import rcwa_oracle as o
from openrcwa_amd import ofd

pytestmark = pytest.mark.gpu


def layer(e1, e2=None, fill=0.5, d=0.0):
    return dict(eps1=e1, eps2=e1 if e2 is None else e2, eps1i=0.0, eps2i=0.0, fill=fill,
                fill_y=1.0, thickness=d)


# n = 2 (2 nX + 1) rows: one block and less, an edge on either side, several blocks
@pytest.mark.parametrize("nX", [0, 7, 8, 15, 16, 24, 31])
def test_chain_matches_oracle(gpu_ctx, nX):
    grating = [layer(1.0), layer(4.0, 1.0, 0.4, 2.5e-7), layer(2.25, 1.5, 0.6, 1.2e-7),
               layer(3.0, 1.2, 0.5, 0.8e-7), layer(2.25)]
    freqs = [4.7e14, 5.9e14]
    got = ofd.solve_ofd(gpu_ctx, nX, 6e-7, grating, freqs, 12.0, 0.0)
    assert not got["status"].any()
    for f, freq in enumerate(freqs):
        ref = o.ofd_solve_frequency(nX, 6e-7, grating, freq, 12.0, 0.0, 0, None, None)
        for p in range(2):
            # both solve to a few hundred n u; far below 1e-10
            assert np.abs(got["REF"][f, p] - ref["REF"][p]).max() < 1e-10
            assert np.abs(got["TRN"][f, p] - ref["TRN"][p]).max() < 1e-10
