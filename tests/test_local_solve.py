"""The product's local update (cufim-nvlink_amd/csrc/local_solve.hpp),
compiled for the host with g++, against the oracle's restatement on random
element geometries and node times.  FP64 must agree to rounding; the
reference update (compat mode) must agree bit for bit; the FP32 exact path
must agree to FP32 accuracy.  CPU only."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import pyoracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cufim-nvlink_amd", "csrc")

SHIM = r"""
#include "local_solve.hpp"
extern "C" {
double ls_exact64(const double *g, const double *ph, int t) {
  const double inf = 1e300;
  switch (t) {
    case 0: return fim::cand_exact<0, double>(g, ph, inf);
    case 1: return fim::cand_exact<1, double>(g, ph, inf);
    case 2: return fim::cand_exact<2, double>(g, ph, inf);
    default: return fim::cand_exact<3, double>(g, ph, inf);
  }
}
float ls_exact32(const float *g, const float *ph, int t) {
  const float inf = 3.0e38f;
  switch (t) {
    case 0: return fim::cand_exact<0, float>(g, ph, inf);
    case 1: return fim::cand_exact<1, float>(g, ph, inf);
    case 2: return fim::cand_exact<2, float>(g, ph, inf);
    default: return fim::cand_exact<3, float>(g, ph, inf);
  }
}
double ls_ref(const double *g, const double *ph, int t) { return fim::cand_ref(g, ph, t); }
void ls_bounds(const double *g, unsigned char *b, float *scale) { fim::cand_bounds(g, b, scale); }
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("ls")
    src = d / "shim.cpp"
    src.write_text(SHIM)
    so = d / "shim.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                    f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    pd, pf = C.POINTER(C.c_double), C.POINTER(C.c_float)
    lib.ls_exact64.restype = C.c_double
    lib.ls_exact64.argtypes = [pd, pd, C.c_int]
    lib.ls_exact32.restype = C.c_float
    lib.ls_exact32.argtypes = [pf, pf, C.c_int]
    lib.ls_ref.restype = C.c_double
    lib.ls_ref.argtypes = [pd, pd, C.c_int]
    return lib


def _cases(n, seed):
    """Geometry of random well-shaped tets (a regular tet of side ~600 um,
    vertices moved by up to 30 % of a side, random orientation) under a
    random transversely anisotropic metric (speeds 0.2-0.6 um/us, as in
    cardiac tissue), node times spread so that every branch (edge,
    triangle, face, unusable node) is taken."""
    rng = np.random.default_rng(seed)
    base = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.5, np.sqrt(3) / 2, 0.0],
                     [0.5, np.sqrt(3) / 6, np.sqrt(2.0 / 3.0)]]) * 600.0
    out = []
    while len(out) < n:
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        x = (base + rng.uniform(-0.3, 0.3, (4, 3)) * 600.0) @ q
        if abs(np.linalg.det(x[1:] - x[0])) < 1e6:
            continue
        r, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        v = rng.uniform(0.2, 0.6, 3)
        M = r @ np.diag(1.0 / v ** 2) @ r.T
        packed = np.array([M[0, 0], M[0, 1], M[0, 2], M[1, 1], M[1, 2], M[2, 2]])
        g = O.geo_elem(x, np.arange(4), packed)
        assert np.all(g > 0)  # SPD metric: positive squared lengths
        ph = rng.uniform(0, 2000.0, 4)
        if rng.random() < 0.15:
            ph[rng.integers(4)] = 1e300
        out.append((np.ascontiguousarray(g), ph))
    return out


def _ptr(a, t):
    return a.ctypes.data_as(C.POINTER(t))


def test_exact_fp64_matches_oracle(shim):
    worst = 0.0
    for g, ph in _cases(3000, 1):
        for t in range(4):
            ours = shim.ls_exact64(_ptr(g, C.c_double), _ptr(ph, C.c_double), t)
            ref = O.local(O.LOCAL_EXACT, g, ph, t)
            if ref >= 1e299:
                assert ours >= 1e299
                continue
            worst = max(worst, abs(ours - ref) / max(1.0, abs(ref)))
    assert worst < 1e-9, worst


def test_reference_update_bit_identical(shim):
    for g, ph in _cases(3000, 2):
        ph = np.where(ph >= 1e299, np.finfo(np.float64).max, ph)
        for t in range(4):
            ours = shim.ls_ref(_ptr(g, C.c_double), _ptr(ph, C.c_double), t)
            ref = O.local(O.LOCAL_REF, g, ph, t)
            assert ours == ref or (np.isnan(ours) and np.isnan(ref))


def test_exact_fp32_close_to_oracle(shim):
    worst = 0.0
    for g, ph in _cases(3000, 3):
        gf = g.astype(np.float32)
        pf = np.where(ph >= 1e299, np.float32(3.0e38), ph).astype(np.float32)
        for t in range(4):
            ours = shim.ls_exact32(_ptr(gf, C.c_float), _ptr(pf, C.c_float), t)
            ref = O.local(O.LOCAL_EXACT, g, ph, t)
            if ref >= 1e299:
                continue
            assert ours < 3.0e38  # an edge candidate always exists here
            worst = max(worst, abs(ours - ref) / max(1.0, abs(ref)))
    assert worst < 2e-4, worst


SHIM_SH = r"""
#include "local_solve.hpp"
extern "C" int ls_shared_equal(const float *g, const float *ph) {
  float sq[6], rc[6];
  for (int k = 0; k < 6; ++k) { sq[k] = fim::csqrt(g[k]); rc[k] = 1.0f / g[k]; }
  const float inf = 3.0e38f;
  const float a[4] = {fim::cand_exact<0, float>(g, ph, inf), fim::cand_exact<1, float>(g, ph, inf),
                      fim::cand_exact<2, float>(g, ph, inf), fim::cand_exact<3, float>(g, ph, inf)};
  const float b[4] = {fim::cand_exact_sh<0, float>(g, sq, rc, ph, inf),
                      fim::cand_exact_sh<1, float>(g, sq, rc, ph, inf),
                      fim::cand_exact_sh<2, float>(g, sq, rc, ph, inf),
                      fim::cand_exact_sh<3, float>(g, sq, rc, ph, inf)};
  int bad = 0;
  for (int k = 0; k < 4; ++k) {
    const float tol = 1e-4f * (a[k] < inf ? a[k] : 1.0f);
    if (!((a[k] >= inf && b[k] >= inf) || (a[k] - b[k] <= tol && b[k] - a[k] <= tol))) ++bad;
  }
  return bad;
}
"""


def test_shared_root_candidate_equals_plain_candidate(tmp_path):
    """the variant with per-element square roots and reciprocals (device
    path) gives the same candidates.  On the host a/b and a*(1/b) round
    differently, so a validity test at a face or edge boundary can flip and
    select the neighbouring candidate, which is continuous there: 1e-4
    relative; a wrong edge or reciprocal would be off by far more."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src = tmp_path / "sh.cpp"
    src.write_text(SHIM_SH)
    so = tmp_path / "sh.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", f"-I{CSRC}",
                    str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    pf = C.POINTER(C.c_float)
    lib.ls_shared_equal.argtypes = [pf, pf]
    bad = 0
    for g, ph in _cases(2000, 7):
        gf = g.astype(np.float32)
        pf_ = np.where(ph >= 1e299, np.float32(3.0e38), ph).astype(np.float32)
        bad += lib.ls_shared_equal(_ptr(gf, C.c_float), _ptr(pf_, C.c_float))
    assert bad == 0


def test_candidate_bounds_lie_below_every_candidate(shim):
    """cand_bounds on ordinary, strongly anisotropic, flat and needle-shaped
    elements: for random times of the other nodes (some unreached, some equal,
    some far apart) the bound is at most the exact candidate.  The bound has a
    margin of 1e-4 of an edge, so nothing is allowed for rounding."""
    shim.ls_bounds.restype = None
    shim.ls_bounds.argtypes = [C.POINTER(C.c_double), C.POINTER(C.c_uint8), C.POINTER(C.c_float)]
    rng = np.random.default_rng(11)
    pd = C.POINTER(C.c_double)
    tight = 0
    for k in range(4000):
        x = rng.normal(size=(4, 3)) * [1.0, rng.choice([1.0, 0.2, 1e-3]), rng.choice([1.0, 0.1, 1e-4])]
        if k % 7 == 0:
            x[3] = x[:3].mean(0) + 1e-5 * rng.normal(size=3)  # target in the face's centroid
        x *= 10.0 ** rng.uniform(-2, 5)
        g = np.array([np.sum((x[a] - x[b]) ** 2) for a, b in ((0, 1), (0, 2), (1, 2), (0, 3), (1, 3), (2, 3))])
        b = np.zeros(12, np.uint8)
        sc = C.c_float()
        shim.ls_bounds(g.ctypes.data_as(pd), b.ctypes.data_as(C.POINTER(C.c_uint8)), C.byref(sc))
        v = (b.astype(np.float64) - 128.0) * sc.value
        size = np.sqrt(g.max())
        for t in range(4):
            ph = rng.uniform(0, size, 4) * rng.choice([0.0, 0.1, 1.0, 3.0])
            if rng.random() < 0.2:
                ph[rng.integers(4)] = 1e300
            o = [(t + 1 + j) % 4 for j in range(3)]
            bound = min(ph[o[j]] + v[3 * t + j] for j in range(3))
            c = shim.ls_exact64(g.ctypes.data_as(pd), ph.ctypes.data_as(pd), t)
            assert bound <= c, (k, t, bound, c, g, ph)
            tight += bound > min(ph[o]) + 0.3 * (c - min(ph[o]))
    assert tight > 4000  # they do bound: most lie well above the earliest node


SHIM_LATE = r"""
#include "local_solve.hpp"
// smallest difference FP32 candidate - FP32 bound, and the number of
// (element, target) pairs whose candidate lies below its bound
extern "C" int ls_late(int n, const double *g, const float *ph, float *least) {
  int bad = 0;
  *least = 3e38f;
  for (int i = 0; i < n; ++i) {
    unsigned char b[12];
    float scale, g32[6], sq[6], rc[6], v[4];
    fim::cand_bounds(g + 6 * i, b, &scale);
    uint32_t w[3] = {0, 0, 0};
    for (int k = 0; k < 12; ++k) w[k / 4] |= (uint32_t)b[k] << 8 * (k % 4);
    for (int k = 0; k < 6; ++k) {
      g32[k] = (float)g[6 * i + k];
      sq[k] = fim::csqrt(g32[k]);
      rc[k] = 1.0f / g32[k];
    }
    const float *p = ph + 4 * i, inf = 3.0e38f;
    fim::cand_bounds32(w, scale, p, v);
    const float c[8] = {fim::cand_exact<0, float>(g32, p, inf), fim::cand_exact<1, float>(g32, p, inf),
                        fim::cand_exact<2, float>(g32, p, inf), fim::cand_exact<3, float>(g32, p, inf),
                        fim::cand_exact_sh<0, float>(g32, sq, rc, p, inf), fim::cand_exact_sh<1, float>(g32, sq, rc, p, inf),
                        fim::cand_exact_sh<2, float>(g32, sq, rc, p, inf), fim::cand_exact_sh<3, float>(g32, sq, rc, p, inf)};
    for (int k = 0; k < 8; ++k) {
      if (!(v[k & 3] <= c[k])) ++bad;
      if (c[k] - v[k & 3] < *least) *least = c[k] - v[k & 3];
    }
  }
  return bad;
}
"""


@pytest.mark.parametrize("edges", [0, 30, 1e3, 1e4, 1e6])
def test_bounds_in_single_precision_lie_below_every_candidate_at_late_times(tmp_path, edges):
    """the kernel's form of the bounds against the FP32 candidates, on
    well-shaped elements under anisotropic metrics whose times lie `edges` edge
    lengths after the start.  A candidate's additions round by at most 2.5 ulp
    of its time together with the bound's, which has a margin of at least 4:
    nothing is allowed for rounding."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src = tmp_path / "late.cpp"
    src.write_text(SHIM_LATE)
    so = tmp_path / "late.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", f"-I{CSRC}",
                    str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.ls_late.argtypes = [C.c_int, C.POINTER(C.c_double), C.POINTER(C.c_float), C.POINTER(C.c_float)]
    rng = np.random.default_rng(int(edges) + 3)
    n = 200000
    base = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.5, np.sqrt(3) / 2, 0.0],
                     [0.5, np.sqrt(3) / 6, np.sqrt(2.0 / 3.0)]])
    x = base + rng.uniform(-0.25, 0.25, (n, 4, 3))
    f = rng.normal(size=(n, 3))
    f /= np.linalg.norm(f, axis=1, keepdims=True)
    slow = rng.uniform(1.0, 3.0, n)  # slowness along the fibre 1, across it up to 3
    pairs = ((0, 1), (0, 2), (1, 2), (0, 3), (1, 3), (2, 3))
    g = np.empty((n, 6))
    for k, (a, b) in enumerate(pairs):
        d = x[:, a] - x[:, b]
        along = np.sum(d * f, axis=1)
        g[:, k] = slow ** 2 * (np.sum(d * d, axis=1) - along ** 2) + along ** 2
    g *= 600.0 ** 2
    # times within a front's reach of each other, so that faces, triangles and
    # edges all occur
    ph = (600.0 * (edges + rng.uniform(0.0, 1.0, (n, 4)) * rng.choice([0.0, 0.1, 0.5, 1.5], (n, 1)))).astype(np.float32)
    g = np.ascontiguousarray(g)
    least = C.c_float()
    bad = lib.ls_late(n, _ptr(g, C.c_double), _ptr(ph, C.c_float), C.byref(least))
    assert bad == 0, (bad, least.value)
