"""Rules that leave work out, compiled for the host from the headers that the
kernels include, against the general path they stand in for."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from fastipc_amd import build as B
from oracle import lib as O

SOURCE = r'''
#include "fipc_math.h"
// the box of n points in single precision, outward by one unit or more
static void box(const double* p, int n, float* lo, float* hi)
{
    for (int d = 0; d < 3; d++) {
        double l = p[d], h = p[d];
        for (int k = 1; k < n; k++) { l = fmin(l, p[3 * k + d]); h = fmax(h, p[3 * k + d]); }
        lo[d] = nextafterf((float)l, -INFINITY);
        hi[d] = nextafterf((float)h, INFINITY);
    }
}
// pairs of segment (2 points) and triangle (3): is the pair left out, is it accepted
extern "C" void seg_tri_pairs(int n, const double* p, int* apart, int* hit)
{
    for (int k = 0; k < n; k++, p += 15) {
        float slo[3], shi[3], tlo[3], thi[3];
        box(p, 2, slo, shi);
        box(p + 6, 3, tlo, thi);
        apart[k] = fipc::seg_tri_apart(slo, shi, tlo, thi);
        hit[k] = fipc::seg_tri(fipc::ld3(p), fipc::ld3(p + 3), fipc::ld3(p + 6), fipc::ld3(p + 9), fipc::ld3(p + 12));
    }
}
'''


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.hip", d / "rules.so"
    src.write_text(SOURCE)
    subprocess.run([B.HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I", B.CSRC, str(src), "-o", str(so)], check=True, capture_output=True)
    return C.CDLL(str(so))


def _nearly_coplanar(rng, n, size, offset):
    """A triangle with edges of about ``size`` and a segment beside it, in one
    plane of random orientation up to rounding."""
    q = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
    uv = np.empty((n, 5, 2))
    uv[:, 2:] = [[0, 0], [1, 0], [0, 1]]
    uv[:, 2:] *= rng.uniform(0.05, 1, (n, 1, 2))
    uv[:, 0] = rng.uniform(-1.2, 1.2, (n, 2))
    uv[:, 1] = uv[:, 0] + rng.uniform(-1, 1, (n, 2)) * 10 ** rng.uniform(-2, 0.5, (n, 1))
    p = uv @ q[:, :2] * size + offset * size * rng.uniform(-1, 1, (n, 1, 3))
    return np.ascontiguousarray(p.reshape(n, 15))


@pytest.mark.parametrize("offset", [0.0, 30.0])
@pytest.mark.parametrize("size", [1e-3, 0.1, 1.0, 30.0, 100.0, 1e3, 1e5, 1e9])
def test_pairs_left_out_of_the_collision_test_would_be_rejected(rules, size, offset):
    """The collision check's segment-triangle test is not run on pairs whose
    boxes are too far apart for it; every pair that it accepts, correctly or by
    its rounding error alone, is run."""
    rng = np.random.default_rng(int(size * 1e3) % 1000003)
    p = _nearly_coplanar(rng, 200_000, size, offset)
    apart, hit = np.zeros(len(p), np.int32), np.zeros(len(p), np.int32)
    rules.seg_tri_pairs(len(p), O.dptr(p), apart.ctypes.data_as(C.c_void_p), hit.ctypes.data_as(C.c_void_p))
    assert not (apart & hit).any()
    # the rule leaves out what it is for, and the pairs of long edges that are
    # accepted with their boxes apart exist
    s, t = p[:, :6].reshape(-1, 2, 3), p[:, 6:].reshape(-1, 3, 3)
    gap = np.maximum(s.min(1) - t.max(1), t.min(1) - s.max(1)).max(1)
    if size <= 0.1:
        assert apart[gap > 0.01 * size].all()
    if size >= 1e3:
        assert hit[gap > 0.05 * size].any()
    for k in range(0, len(p), 2000):
        assert hit[k] == O.seg_tri(*p[k].reshape(5, 3))
