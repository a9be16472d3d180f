"""A context's pinned memory is bounded whatever its L: lattices on both sides
of the sizes where ln W and the site tables leave it give the oracle's chain,
and a large context maps no more than its device buffers."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [228, 229, 294, 295, 296, 400])
@pytest.mark.parametrize("prec", [M.REF32, M.FP64])
def test_copies_on_both_sides_of_the_bound(orc, L, prec):
    W, N, seed = 3, L * L, 6
    lnw = -2.0 * np.arange(N + 1) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    lat = orc.init_lattice(M.KEYING_WEIGHT, L, W, seed=seed)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=1.6, precision=prec) as ctx:
        ctx.init_lattice(seed=seed)
        ctx.compute_state()
        for it in range(2):   # the second ln W replaces the first
            ctx.set_log_weight(lnw)
            hist, _ = ctx.run(it, seed, 50, 101)
            ref = orc.mcs(L, lat, E, D, Mg, keying=0, fp64=prec == M.FP64,
                          lnw32=lnw.astype(np.float32), lnw64=lnw, iter=it, seed=seed, therm=50,
                          nupdates=101, beta=1.6)
            assert np.array_equal(hist, ref)
            lnw = lnw[::-1].copy()
        assert np.array_equal(ctx.get_lattice(), lat.T)


def _mapped():
    line = [q for q in open("/proc/self/status") if q.startswith("VmSize")][0]
    return int(line.split()[1]) * 1024


def test_a_large_context_pins_little():
    """41 bytes a site of device buffers (tables, ln W, histogram, one walker's
    lattice), mapped into the process with the driver's own; 20 bytes a site
    of pinned memory on top took it to 72.  The second context is looked at:
    the first also maps what the runtime keeps."""
    L = 4000
    with M.Context(L, 1):
        before = _mapped()
        with M.Context(L, 1) as ctx:
            assert _mapped() - before < 60 * ctx.N
