"""Camera vertices (GPU): occlusion rays as a list of their own and point merges shared by a wave, at
path counts around a wave's 64 and photon maps from one primitive up, against the oracle on the same
random streams."""
import numpy as np
import pytest

from gpuupbp_amd import capi
from gpuupbp_amd import renderer as gpu
from oracle import oracle_py

pytestmark = pytest.mark.gpu

SIX = "upbp_bpt+surf+pp3d+pb2d+bb1d+bp2d"


@pytest.mark.parametrize("res", ["1x1", "9x7", "64x1", "65x1", "33x31"])
@pytest.mark.parametrize("paths,length,alg,radius", [(1, 6, SIX, 0.3), (3, 2, SIX, 0.3), (50, 16, SIX, 0.1),
                                                     (2000, 6, SIX, 0.1), (300, 8, "upbp_bpt", 0.1),
                                                     (2000, 6, "upbp_surf+pp3d+bp2d", 0.1)])
def test_small_frames_match_the_oracle(boxfog_obj, res, paths, length, alg, radius):
    rc, cfg = capi.parse_args(["-s", "-1", boxfog_obj, "-r", res, "-l", str(length), "-pcpi", str(paths), "-a", alg,
                               "-r_initial", str(radius), "-r_alpha", "1"])
    assert rc == 0
    if alg == "upbp_surf+pp3d+bp2d":  # the parser adds to the defaults only for upbp_all
        assert not cfg.algorithm_flags & 4
    sh = capi.SceneHandle(boxfog_obj, cfg.res_x, cfg.res_y)
    with gpu.Renderer(sh.ptr, cfg) as r:
        st = [r.run_iteration(i) for i in range(2)]
        g = r.read_accum(2)
    o, _ = oracle_py.render(sh.ptr, cfg, 0, 2)
    sh.close()
    assert all(s.path_errors == 0 for s in st) and np.isfinite(g).all()
    # same streams: all but the few pixels whose path takes another turn (a transcendental's last bit)
    rel = np.abs(g - o) / np.maximum(np.abs(o), 1e-3 * max(o.max(), 1e-6))
    assert np.mean(rel < 2e-3) >= (1.0 if g.size <= 3 else 0.95), float(np.mean(rel < 2e-3))


@pytest.mark.parametrize("res,paths", [("32x32", 512), ("1025x1", 513), ("64x64", 4097), ("181x181", 16384),
                                       ("241x272", 16385)])
@pytest.mark.parametrize("alg", ["upbp_bpt", SIX])
def test_shared_lists_match_the_oracle(boxfog_obj, res, paths, alg):
    """Lists whose waves take 1 to 64 entries (the share changes where the count passes the waves
    that share it times a power of two)."""
    rc, cfg = capi.parse_args(["-s", "-1", boxfog_obj, "-r", res, "-l", "5", "-pcpi", str(paths), "-a", alg,
                               "-r_initial", "0.01", "-r_alpha", "1"])
    assert rc == 0
    sh = capi.SceneHandle(boxfog_obj, cfg.res_x, cfg.res_y)
    with gpu.Renderer(sh.ptr, cfg) as r:
        st = r.run_iteration(0)
        g = r.read_accum(1)
    o, _ = oracle_py.render(sh.ptr, cfg, 0, 1)
    sh.close()
    assert st.path_errors == 0 and np.isfinite(g).all()
    rel = np.abs(g - o) / np.maximum(np.abs(o), 1e-3 * max(o.max(), 1e-6))
    assert np.mean(rel < 2e-3) >= 0.95, float(np.mean(rel < 2e-3))
