"""Parts of the segment merges (GPU): with few query pieces or bundles each walk is cut into 8 or 64
parts by the tree's first children. The packet walk, which is never cut, accepts the same pairs, on
trees from one primitive to many and on piece counts on either side of the rule's bounds."""
import os
import shutil

import numpy as np
import pytest

from gpuupbp_amd import capi
from gpuupbp_amd import renderer as gpu
from gpuupbp_amd import workloads as wl
from oracle import oracle_py

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def workdir(tmp_path_factory):
    return str(tmp_path_factory.mktemp("parts"))


def _render(workdir, scene, args, tuning):
    head = ["-s", str(scene)] if isinstance(scene, int) else ["-s", "-1", wl.scene(workdir, scene, 0)]
    rc, cfg = capi.parse_args(head + args)
    assert rc == 0
    sh = capi.SceneHandle(scene if isinstance(scene, int) else head[2], cfg.res_x, cfg.res_y)
    with gpu.Renderer(sh.ptr, cfg) as r:
        r.set_tuning(**tuning)
        st = [r.run_iteration(i) for i in range(2)]
        img = r.read_accum(2)
    sh.close()
    return img, st


# light paths 1, 2, 7 and 40 leave trees of a few primitives (leaves at the root and below it); the
# others put the pieces per bounce below, between and above the rule's bounds
CASES = [("boxfog", ["-r", "48x48", "-l", "6", "-pcpi", str(n), "-r_initial", "0.05", "-a", "upbp_all"])
         for n in (1, 2, 7, 40)]
CASES += [("boxfog", ["-r", "64x64", "-l", "8", "-r_initial", "0.03", "-a", "upbp_all"]),
          ("boxfog", ["-r", "211x157", "-l", "6", "-r_initial", "0.01", "-a", "upbp_all"]),
          (27, ["-r", "160x120", "-l", "4", "-pcpi", "800", "-r_initial", "0.004", "-a", "upbp_all"])]


@pytest.mark.parametrize("scene,args", CASES)
@pytest.mark.parametrize("tuning", [dict(), dict(bundle_bounces=0), dict(bundle_bounces=0, merge_blocks_per_cu=1),
                                    dict(bundle_bounces=64, bundle_factor=1e6)])
def test_parts_accept_the_packet_walks_pairs(workdir, scene, args, tuning):
    ref, rst = _render(workdir, scene, args, dict(packet_bounces=64))
    img, st = _render(workdir, scene, args, tuning)
    print("pieces", [s.seg_pieces for s in st], "bundles", [s.bundles for s in st], "accepts",
          [(s.pb2d_accepts, s.bb1d_accepts) for s in st])
    assert [(s.pb2d_accepts, s.bb1d_accepts, s.merge_accepts) for s in st] == \
           [(s.pb2d_accepts, s.bb1d_accepts, s.merge_accepts) for s in rst]
    assert all(s.path_errors == 0 for s in st)
    # the same pairs in another order of FP32 sums: at most a few thousand terms per pixel
    assert np.allclose(img, ref, rtol=1e-4, atol=1e-6 * max(ref.max(), 1e-3))


@pytest.mark.parametrize("sub", [0.0, 0.05, 0.3])
@pytest.mark.parametrize("lean", [0.003, 0.0035, 0.01, 0.05, 0.0999, 0.1001, 0.3, 1.0])
def test_leaf_cull_keeps_what_the_predicate_accepts(sub, lean):
    """Segment queries over beams at a set angle to them (from the predicate's parallel cut-off up)
    and nearly perpendicular ones, through the wide walk with its leaf cull."""
    rng = np.random.default_rng(int(lean * 1e4) + int(sub * 100))
    n, r = 3000, 0.02
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = rng.uniform(-2, 2, (n, 3))
    beams = np.hstack([o, d, rng.uniform(0.2, 3, (n, 1))]).astype(np.float32)
    k = rng.integers(0, n, 1500)
    side = rng.normal(size=(1500, 3))
    side -= (side * d[k]).sum(1, keepdims=True) * d[k]
    side /= np.linalg.norm(side, axis=1, keepdims=True)
    across = np.cross(d[k], side)
    q = d[k] + lean * side
    perp = rng.uniform(size=1500) < 0.3
    q[perp] = side[perp] + rng.choice([1e-4, 1e-3, 1e-2, 0.04, 0.06], (perp.sum(), 1)) * d[k[perp]]
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    at = o[k] + d[k] * rng.uniform(0, 1, (1500, 1)) + across * rng.uniform(-1.05 * r, 1.05 * r, (1500, 1))
    back = rng.uniform(0.1, 1.5, (1500, 1))
    queries = np.hstack([at - q * back, q, np.zeros((1500, 1)), back + rng.uniform(0.1, 1.5, (1500, 1))]).astype(np.float32)
    narrow = gpu.range_query(3, beams, queries, r, subbeam_len=sub)
    wide = gpu.range_query(3, beams, queries, r, subbeam_len=sub, wide=True)
    assert narrow[0][-1] > 1000
    assert np.array_equal(narrow[0], wide[0])
    for i in range(1500):
        a, b = narrow[0][i], narrow[0][i + 1]
        assert np.array_equal(np.sort(narrow[1][a:b]), np.sort(wide[1][a:b]))


def _far_scene(workdir, radii):
    """The fog box in a thin global fog, its camera so many scene radii away and as many times narrower."""
    src = os.path.dirname(wl.scene(workdir, "boxfog", 0))
    dst = os.path.join(workdir, "far%d" % radii)
    shutil.copytree(src, dst, dirs_exist_ok=True)
    aux = os.path.join(dst, "boxfog.obj.aux")
    z = 1.7320508 * radii
    text = open(aux).read().replace("3.200000", "%f" % z).replace("CAMERA_FOV 0.6981317",
                                                                  "CAMERA_FOV %f" % (0.6981317 * 3.2 / z))
    text += "\nmedium thin\nabsorption 0.001 0.001 0.001\nemission 0 0 0\nscattering 0.02 0.02 0.02\ng 0\n\n" \
            "globalMediumId thin\n"
    open(aux, "w").write(text)
    return os.path.join(dst, "boxfog.obj")


@pytest.mark.parametrize("radii", [4, 20])
@pytest.mark.parametrize("tuning", [dict(), dict(bundle_bounces=0), dict(packet_bounces=64)])
def test_cameras_far_from_the_scene_match_the_oracle(workdir, radii, tuning):
    rc, cfg = capi.parse_args(["-s", "-1", _far_scene(workdir, radii), "-r", "48x36", "-l", "5", "-pcpi", "2000",
                               "-r_initial", "0.02", "-r_alpha", "1", "-a", "upbp_all"])
    assert rc == 0
    sh = capi.SceneHandle(_far_scene(workdir, radii), cfg.res_x, cfg.res_y)
    with gpu.Renderer(sh.ptr, cfg) as r:
        r.set_tuning(**tuning)
        st = r.run_iteration(0)
        g = r.read_accum(1)
    o, _ = oracle_py.render(sh.ptr, cfg, 0, 1)
    sh.close()
    assert st.path_errors == 0 and st.bb1d_accepts > 10000 and np.isfinite(g).all()
    rel = np.abs(g - o) / np.maximum(np.abs(o), 1e-3 * max(o.max(), 1e-6))
    assert np.mean(rel < 2e-3) >= 0.95, float(np.mean(rel < 2e-3))
