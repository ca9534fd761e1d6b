"""Motions without a GPU: the oracle's restatement of Transformation / Quaternion / Motion
(src/Transformation.cu, src/Quaternion.cu, src/Motion.cu) pinned by closed forms and a
library rotation, the product's host evaluation (cs_motion_eval, cs_scene_motion) bit-exact
against it, and the scene loader's motion forms (keyframe lists, .mot files, obstacle
sequences).

  Hermite       two keys: x0 + (x1 - x0)(3 s^2 - 2 s^3) (zero end tangents); every key hit;
                interior tangent = (x[i+1] - x[i-1]) / (t[i+1] - t[i-1]) (finite difference);
                after the last key: the last key exactly; a first key after t = 0 gets an
                identity key at t = 0
  rotation      unit quaternions against scipy.spatial.transform.Rotation; a quaternion of
                norm r rotates and scales by r^2 (the reference never renormalises)
  inverse       T^-1(T(p)) = p;  composition: (A * B)(p) = A(B(p)) for unit scales, and
                the reference's s_a s_b R_a R_b p + t_a + R_a(s_b t_b) in general
"""
import json
import os
import re

import numpy as np
import pytest

import clothsimulator_amd as cs
import oracle
from clothsimulator_amd import ClothError

REF = "/root/reference"


def key(scale=1.0, t=(0.0, 0.0, 0.0), q=(1.0, 0.0, 0.0, 0.0)):
    return np.array([scale, *t, *q], dtype=np.float32)


def test_two_key_hermite_is_smoothstep():
    k0 = key(1.0, (0.5, -1.0, 2.0))
    k1 = key(2.0, (1.5, 3.0, -2.0), (0.5, 0.5, 0.5, 0.5))
    for s in np.linspace(0.0, 1.0, 11):
        time = np.float32(1.5 * s)
        got = oracle.motion_eval([0.0, 1.5], [k0, k1], time)
        s64 = float(time) / 1.5
        want = k0 + (k1.astype(np.float64) - k0) * (3 * s64 ** 2 - 2 * s64 ** 3)
        assert np.allclose(got, want, atol=2e-6), (s, got, want)


def test_keys_hit_and_after_last_key():
    rng = np.random.default_rng(3)
    t = np.array([0.0, 0.4, 1.1, 1.5, 2.75], dtype=np.float32)
    keys = rng.normal(size=(5, 8)).astype(np.float32)
    for i in range(5):
        assert np.allclose(oracle.motion_eval(t, keys, t[i]), keys[i], atol=1e-5)
    for late in (2.75001, 3.0, 100.0):
        assert np.array_equal(oracle.motion_eval(t, keys, late), keys[-1])


def test_interior_tangent_is_central_difference():
    rng = np.random.default_rng(4)
    t = np.array([0.0, 0.5, 1.25, 2.0], dtype=np.float32)
    keys = rng.normal(size=(4, 8)).astype(np.float32)
    for i in (1, 2):
        h = 2e-3
        fd = (oracle.motion_eval(t, keys, t[i] + h).astype(np.float64) -
              oracle.motion_eval(t, keys, t[i] - h)) / (2 * h)
        want = (keys[i + 1].astype(np.float64) - keys[i - 1]) / (t[i + 1] - t[i - 1])
        assert np.allclose(fd, want, rtol=2e-2, atol=2e-2), (i, fd, want)
    # zero tangent at both ends
    for tt, sgn in ((0.0, 1), (2.0, -1)):
        h = 1e-3
        d = (oracle.motion_eval(t, keys, tt + sgn * h).astype(np.float64) - oracle.motion_eval(t, keys, tt)) / h
        assert np.abs(d).max() < 0.05


def test_identity_key_inserted_before_late_first_key():
    k = key(3.0, (1.0, 2.0, 3.0))
    assert np.array_equal(oracle.motion_eval([1.0, 2.0], [k, k], 0.0), key())
    # keys I, k, k at t = 0, 1, 2: tangent 0 at t = 0 and (k - I) / 2 at t = 1, so on [0, 1]
    # the cubic Hermite basis gives I + (h01(s) + h11(s) / 2)(k - I), h01 = 3s^2 - 2s^3, h11 = s^3 - s^2
    for s in (0.25, 0.5, 0.75):
        got = oracle.motion_eval([1.0, 2.0], [k, k], s)
        w = (3 * s * s - 2 * s ** 3) + (s ** 3 - s * s) / 2
        assert np.allclose(got, key() + (k - key()) * w, atol=1e-6), s


def test_single_key_is_constant():
    k = key(0.5, (1.0, 0.0, 0.0))
    for tt in (0.0, 1.0, 10.0):
        assert np.array_equal(oracle.motion_eval([0.0], [k], tt), k)
    with pytest.raises(RuntimeError):
        oracle.motion_eval([0.0, 0.0], [k, k], 0.5)


def test_rotation_matches_scipy_and_scales_by_norm():
    from scipy.spatial.transform import Rotation
    rng = np.random.default_rng(5)
    p = rng.normal(size=(20, 3))
    for _ in range(10):
        q = rng.normal(size=4)
        q /= np.linalg.norm(q)
        a = key(1.0, (0, 0, 0), q)
        want = Rotation.from_quat([q[1], q[2], q[3], q[0]]).apply(p)
        assert np.allclose(oracle.transform_points(a, p), want, atol=1e-6)
        # norm r quaternion: r^2 times the rotation, then scale and translate
        r = 1.7
        b = key(0.5, (1.0, -2.0, 0.25), q * r)
        want_b = 0.5 * r * r * want + np.array([1.0, -2.0, 0.25])
        assert np.allclose(oracle.transform_points(b, p), want_b, atol=1e-5)


def test_inverse_and_composition():
    """T^-1(T(p)) = p.  A * B applies B then A when both scales are 1; with scales the
    reference composes the translation as t_a + R_a(s_b t_b) (src/Transformation.cu:58-64),
    not t_a + s_a R_a(t_b), and that is kept."""
    from scipy.spatial.transform import Rotation
    rng = np.random.default_rng(6)
    p = rng.normal(size=(20, 3))
    for _ in range(10):
        qa, qb = rng.normal(size=4), rng.normal(size=4)
        qa, qb = qa / np.linalg.norm(qa), qb / np.linalg.norm(qb)
        sa, sb = rng.uniform(0.5, 2, 2)
        ta, tb = rng.normal(size=3), rng.normal(size=3)
        a, b = key(sa, ta, qa), key(sb, tb, qb)
        assert np.allclose(oracle.transform_points(a, oracle.transform_points(a, p), op=1), p, atol=1e-5)
        Ra = Rotation.from_quat([qa[1], qa[2], qa[3], qa[0]])
        Rb = Rotation.from_quat([qb[1], qb[2], qb[3], qb[0]])
        want = np.float32(sa) * np.float32(sb) * (Ra * Rb).apply(p) + np.float32(ta) + Ra.apply(np.float32(sb) * np.float32(tb))
        ab = oracle.transform_points(a, p, op=2, b=b)
        assert np.allclose(ab, want, atol=1e-5)
        assert np.allclose(oracle.transform_points(oracle.transform_compose(a, b), p), ab, atol=1e-6)
        a1, b1 = key(1.0, ta, qa), key(1.0, tb, qb)
        assert np.allclose(oracle.transform_points(a1, p, op=2, b=b1),
                           oracle.transform_points(a1, oracle.transform_points(b1, p)), atol=1e-5)


def test_product_motion_eval_bitexact_with_oracle():
    rng = np.random.default_rng(7)
    checked = 0
    for _ in range(100):
        n = int(rng.integers(1, 7))
        t = (np.cumsum(rng.uniform(0.05, 1.0, n)) - rng.uniform(0.0, 0.3)).astype(np.float32)
        keys = rng.normal(size=(n, 8)).astype(np.float32)
        for time in rng.uniform(-0.2, float(t[-1]) + 0.5, 4).astype(np.float32):
            a = cs.motion_eval(t, keys, time).as_array()
            b = oracle.motion_eval(t, keys, time)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (t, time, a, b)
            checked += 1
    assert checked == 400


def test_product_rejects_bad_keys():
    with pytest.raises(ClothError, match="CS_E_ARG"):
        cs.motion_eval([0.0, 1.0, 1.0], [key()] * 3, 0.5)
    with pytest.raises(ClothError, match="CS_E_ARG"):
        cs.motion_eval([], [], 0.5)


# ---------------------------------------------------------------- scene files
SHEET = "v 0 0 0\nv 1 0 0\nv 0 1 0\nv 1 1 0\nf 1 2 4 3\n"
TRI = "v -1 -1 0\nv 1 -1 0\nv 0 1 0\nf 1 2 3\n"


def write(d, name, text):
    with open(os.path.join(d, name), "w") as f:
        f.write(text)
    return os.path.join(d, name)


def material_json():
    return json.dumps({"density": 0.2, "stretching": [[1e3, 0, 1e3, 0]] * 6, "bending": [[1e-6] * 5] * 3})


def motion_scene(d, motions, obstacles, handles="[]"):
    write(d, "mat.json", material_json())
    write(d, "sheet.obj", SHEET)
    write(d, "tri.obj", TRI)
    return write(d, "scene.json", """{
    "frame_time": 0.04, "frame_steps": 8,
    "cloths": [{"mesh": "sheet.obj", "materials": {"data": "mat.json"}}],
    "motions": %s,
    "obstacles": %s,
    "handles": %s,
    "gravity": [0, 0, -9.8]
}""" % (motions, obstacles, handles))


KEYS = """[[{"time": 0, "transform": {"translate": [0, 0, 0]}},
             {"time": 1, "transform": {"translate": [0, 0, 1], "rotate": [90, 0, 0, 1]}},
             {"time": 2, "transform": {"scale": 2, "translate": [1, 0, 1]}}]]"""


def keys_from_json(motion):
    t, k = [], []
    for e in motion:
        tr = e["transform"]
        rot = tr.get("rotate", [0, 1, 0, 0])
        t.append(e["time"])
        k.append(key(tr.get("scale", 1.0), tr.get("translate", [0, 0, 0]), cs.axis_angle(rot[1:], rot[0])))
    return np.array(t, dtype=np.float32), np.array(k)


def test_scene_keyframe_motion_matches_oracle(tmp_path):
    d = str(tmp_path)
    path = motion_scene(d, KEYS, '[{"mesh": "tri.obj", "motion": 0}]', '[{"cloth": 0, "nodes": [2, 3], "motion": 0}]')
    info = cs.scene_info(path, d)
    assert (info.n_motions, info.n_moving_obstacles, info.n_obstacles, info.n_handles) == (1, 1, 1, 1)
    t, k = keys_from_json(json.loads(KEYS)[0])
    for time in (0.0, 0.3, 1.0, 1.7, 2.0, 3.0):
        a = cs.scene_motion(path, 0, time, d).as_array()
        assert np.array_equal(a, oracle.motion_eval(t, k, time)), time
    with pytest.raises(ClothError, match="CS_E_ARG"):
        cs.scene_motion(path, 1, 0.0, d)


def write_mot(d, frames, bodies):
    lines = ["NumFrames: %d" % len(frames)]
    for b in range(bodies):
        lines.append("body[%d] position" % b)
        lines += [" ".join("%.9g" % float(v) for v in f[b][:3]) for f in frames]
        lines.append("body[%d] rotation" % b)
        lines += [" ".join("%.9g" % float(v) for v in f[b][3:]) for f in frames]
    return write(d, "walk.mot", "\n".join(lines) + "\n")


def test_scene_mot_file_motion_composes_transform(tmp_path):
    d = str(tmp_path)
    rng = np.random.default_rng(8)
    frames = [[np.concatenate([rng.normal(size=3), rng.normal(size=4)]).astype(np.float32) for _ in range(2)]
              for _ in range(4)]
    write_mot(d, frames, 2)
    motions = '{"motfile": "walk.mot", "fps": 10, "transform": {"translate": [0, 0, -1], "rotate": [-90, 0, 0, 1]}}'
    write(d, "body0000.obj", TRI)
    write(d, "body0001.obj", TRI)
    path = motion_scene(d, motions, '"body%04d.obj"')
    info = cs.scene_info(path, d)
    assert (info.n_motions, info.n_obstacles, info.n_moving_obstacles) == (2, 2, 2)
    T = key(1.0, (0, 0, -1), cs.axis_angle((0, 0, 1), -90))
    dt = np.float32(1.0) / np.float32(10.0)
    for b in range(2):
        # keys = transform * (position, rotation) at i / fps (src/Motion.cu:22-37)
        keys = []
        for f in frames:
            body = key(1.0, f[b][:3], f[b][3:])
            keys.append(oracle.transform_compose(T, body))
        times = np.array([np.float32(i) * dt for i in range(len(frames))], dtype=np.float32)
        for time in (0.0, 0.05, 0.1, 0.17, 0.3, 0.5):
            a = cs.scene_motion(path, b, time, d).as_array()
            assert np.array_equal(a, oracle.motion_eval(times, keys, time)), (b, time)


def test_obstacle_sequence_pattern(tmp_path):
    d = str(tmp_path)
    write(d, "p00.obj", TRI)
    write(d, "p01.obj", TRI)
    write(d, "p02.obj", TRI)
    two = KEYS[:-1] + ", " + KEYS[1:]
    path = motion_scene(d, two, '"p%02d.obj"')
    with pytest.raises(ClothError, match="CS_E_FORMAT.*no motion 2"):
        cs.scene_info(path, d)
    three = KEYS[:-1] + ", " + KEYS[1:-1] + ", " + KEYS[1:]
    path = motion_scene(d, three, '"p%02d.obj"')
    info = cs.scene_info(path, d)
    assert (info.n_obstacles, info.n_moving_obstacles, info.n_motions) == (3, 3, 3)
    path = motion_scene(d, three, '"p%s.obj"')
    with pytest.raises(ClothError, match="CS_E_FORMAT.*%d"):
        cs.scene_info(path, d)


def test_missing_motion_index_is_refused(tmp_path):
    d = str(tmp_path)
    path = motion_scene(d, KEYS, '[{"mesh": "tri.obj", "motion": 1}]')
    with pytest.raises(ClothError, match="CS_E_FORMAT.*missing motion"):
        cs.scene_info(path, d)
    path = motion_scene(d, KEYS, "[]", '[{"cloth": 0, "nodes": [0], "motion": 3}]')
    with pytest.raises(ClothError, match="CS_E_FORMAT.*missing motion"):
        cs.scene_info(path, d)


def strip_comments(text):
    return re.sub(r"^\s*//[^\n]*$", "", text, flags=re.M)


@pytest.mark.skipif(not os.path.isdir(os.path.join(REF, "conf")), reason="reference tree not present")
def test_reference_scene_motions():
    """conf/funnel.json moves the ball by a two-key smoothstep; conf/sphere.json's eight keys and
    conf/dress-blue.json's .mot bodies evaluate bit-exactly as the oracle evaluates them."""
    funnel = os.path.join(REF, "conf", "funnel.json")
    for time, z in ((0.0, 0.0), (2.5, -0.75), (5.0, -1.5), (6.0, -1.5)):
        assert cs.scene_motion(funnel, 0, time, REF).as_array()[3] == pytest.approx(z, abs=1e-6)
    sphere = os.path.join(REF, "conf", "sphere.json")
    t, k = keys_from_json(json.loads(strip_comments(open(sphere).read()))["motions"][0])
    for time in (0.0, 1.5, 2.25, 3.0, 4.6, 7.0, 8.0):
        assert np.array_equal(cs.scene_motion(sphere, 0, time, REF).as_array(), oracle.motion_eval(t, k, time))
    dress = os.path.join(REF, "conf", "dress-blue.json")
    a = cs.scene_motion(dress, 3, 1.0, REF).as_array()
    assert np.all(np.isfinite(a)) and a[0] == 1.0
