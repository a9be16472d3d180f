"""Which kernel MUCA_KERNEL_AUTO takes, on both sides of each line drawn by the
measured times (walkers per compute unit, odd L, joint histogram, moments)."""
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu

T, G, K = M.KERNEL_TEAM, M.KERNEL_GENERIC, M.KERNEL_LANE


@pytest.fixture(scope="module")
def cus():
    with M.Context(8, 1) as ctx:
        return ctx.info.cus


def _choice(L, W, prec, blocks=0, obs=M.OBS_JOINT):
    with M.Context(L, W, precision=prec, joint_blocks=blocks, observables=obs) as ctx:
        return ctx.info.kernel


@pytest.mark.parametrize("prec", [M.REF32, M.FP64])
@pytest.mark.parametrize("L,per_cu,below,above", [
    (9, 96, T, G), (11, 128, T, G), (31, 128, T, G), (33, 256, T, G), (51, 256, T, G),
    (57, 192, T, G), (63, 192, T, G), (79, 192, T, G), (36, 256, T, K), (72, 128, T, K)])
def test_weights(cus, prec, L, per_cu, below, above):
    assert _choice(L, per_cu * cus, prec) == below
    assert _choice(L, per_cu * cus + 1, prec) == above


@pytest.mark.parametrize("L,per_cu,above", [(9, 32, G), (11, 32, G), (13, 96, G), (17, 128, G),
                                            (33, 128, G), (16, 128, K)])
def test_joint(cus, L, per_cu, above):
    assert _choice(L, per_cu * cus, M.FP64, 2) == T
    assert _choice(L, per_cu * cus + 1, M.FP64, 2) == above


@pytest.mark.parametrize("L,per_cu,kernel", [(9, 512, T), (16, 512, T), (63, 300, T), (65, 256, T),
                                             (65, 257, G)])
def test_moments(cus, L, per_cu, kernel):
    assert _choice(L, per_cu * cus, M.FP64, 2, M.OBS_MOMENTS) == kernel


@pytest.mark.parametrize("L,W,kernel,lds_lattice", [
    # odd lattices that fit in LDS where no histogram is kept there
    (81, 4096, T, 1), (83, 4096, T, 1), (85, 4096, G, 0),
    # even ones: in LDS likewise, and in HBM once walkers outnumber the resident
    (80, 4096, T, 1), (66, 4096, T, 1), (66, 4100, T, 0)])
def test_moments_layout_is_the_launch_s(cus, L, W, kernel, lds_lattice):
    W += 16 * (cus - 256)
    with M.Context(L, W, precision=M.FP64, joint_blocks=2, observables=M.OBS_MOMENTS) as ctx:
        assert (ctx.info.kernel, ctx.info.lds_lattice) == (kernel, lds_lattice)


@pytest.mark.parametrize("prec", [M.REF32, M.FP64])
@pytest.mark.parametrize("L,n,W,tiles", [
    (12, 8, 4096, K), (22, 2, 16384, K), (28, 2, 16384, T), (14, 4, 4096, K), (20, 4, 4096, T),
    (10, 8, 1024, K), (14, 8, 1024, T), (10, 1, 2048, T), (16, 8, 4096, T), (100, 4, 4096, T)])
def test_batch_tiles(cus, prec, L, n, W, tiles):
    with M.Batch([dict(L=L, walkers=W * cus // 256, seed=i) for i in range(n)], precision=prec) as b:
        assert b.tiles == tiles
