"""The wave speed of csrc/swe_kernels.h (swe::lambda_vacc, with its sign test that skips phi) against the
oracle, bit for bit, on states of every case and at the edges of that test; and the divisions that share a
refined reciprocal (swe::div_shared) against the division.  tests/hip/lambda_check is built by
__graft_entry__.build() (make -C tests/hip)."""
import os
import subprocess

import numpy as np
import pytest

import pyoracle as O
from conftest import REPO

pytestmark = pytest.mark.gpu

CHECK = os.path.join(REPO, "tests", "hip", "_build", "lambda_check")
built = pytest.mark.skipif(not os.path.exists(CHECK), reason="tests/hip/_build/lambda_check is not built")


def states(kind, htiny, n, rng):
    """Records (hl, qxl, qyl, hr, qxr, qyr, n1, n2): kind picks the depths and velocities."""
    th = rng.uniform(0.0, 2.0 * np.pi, n)
    hl = 10.0 ** rng.uniform(-3, 1, n)
    hr = hl * 10.0 ** rng.uniform(-0.02, 0.02, n)
    speed, ab = 0.3, rng.uniform(0.4, 0.6, n)
    if kind == "ratio":            # around and past the depth ratio (2 sqrt 2 - 1)^2 where the test stops applying
        x0 = (2.0 * np.sqrt(2.0) - 1.0) ** 2
        hr = hl * x0 ** rng.choice([-1.0, 1.0], n) * (1.0 + rng.choice([0.0, 1e-16, -2.2e-16, 1e-3, -1e-3, 5.0], n))
    elif kind == "separating":     # velocities around the test's bound, 1.65 sqrt(g h), and the true 1.8884, and vacuum
        speed = rng.choice([1.63, 1.645, 1.65, 1.66, 1.88, 1.8884, 1.89, 2.5, 5.0], n)
        ab = 0.5
    elif kind == "dry":            # exact zeros, depths at and under htiny
        hl = rng.choice([0.0, htiny, 0.5 * htiny, np.nextafter(htiny, 0), 1e-30, 1e-200, 0.7], n)
        hr = rng.choice([0.0, htiny, 0.5 * htiny, np.nextafter(htiny, 1), 1e-30, 1e-200, 0.7], n)
        hr = np.where(rng.random(n) < 0.5, hl * rng.uniform(1.0, 2.0, n), hr)
        speed = 10.0 ** rng.uniform(-3, 1, n)
    elif kind == "extreme":        # depths of any size
        hl = 10.0 ** rng.uniform(-140, 140, n)
        hr = hl * rng.choice([1.0, 1.5, 3.0, 4.0], n)
    c = np.sqrt(9.81 * np.maximum(hl, hr))
    sgn = rng.choice([-1.0, 1.0], n)
    ul, ur = -sgn * speed * c * ab, sgn * speed * c * ab
    nx, ny = np.cos(th), np.sin(th)
    tl, tr = rng.normal(size=n), rng.normal(size=n)
    return np.column_stack([hl, hl * (ul * nx - tl * ny), hl * (ul * ny + tl * nx),
                            hr, hr * (ur * nx - tr * ny), hr * (ur * ny + tr * nx), nx, ny])


@built
@pytest.mark.parametrize("htiny", [1.0e-4, 1.0e-12])
@pytest.mark.parametrize("kind", ["smooth", "ratio", "separating", "dry", "extreme"])
def test_wave_speed_matches_the_oracle_bit_for_bit(kind, htiny, tmp_path):
    rec = states(kind, htiny, 200_000, np.random.default_rng(5))
    src, dst = tmp_path / "in.bin", tmp_path / "out.bin"
    np.concatenate([[9.81, htiny], rec.ravel()]).tofile(src)
    r = subprocess.run([CHECK, str(src), str(dst)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    got = np.fromfile(dst)
    with np.errstate(all="ignore"):
        ref, _ = O.lambda_batch(rec, 9.81, htiny)
    same = (got == ref) | (np.isnan(got) & np.isnan(ref))
    assert same.all(), (int((~same).sum()), rec[~same][:3], got[~same][:3], ref[~same][:3])


@built
def test_shared_divisions_match_the_division_bit_for_bit():
    r = subprocess.run([CHECK, "24"], capture_output=True, text=True, timeout=120)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = [l for l in r.stdout.splitlines() if l.startswith("class")]
    assert len(lines) == 5 and all(" 0 of " in l for l in lines)
