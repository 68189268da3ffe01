"""The exact transpose's candidate ranges: the FP32 shadow with its margin
(matched_margin, compiled for the host) against the shadow in FP64, from ordinary
scans to a source close above the volume, where the cancellation in the depth
moves a shadow end by many bins. The FP32 shadow is the kernel's, with the
reciprocal off by its 1 ulp either way. A ray that meets a voxel is a candidate,
or, where the margin does not cover the error, its segment is within the
rounding of the slice's faces: two of half an ulp of the source's height, times
the ray's length per unit of height."""
import subprocess

import numpy as np
import pytest

from newrecon_amd.build import CSRC, HIPCC
from newrecon_amd.geometry import Geometry

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "matched_device.h"
int main(int argc, char** argv) {
    double a[20];
    for (int k = 1; k < argc; ++k) a[k] = atof(argv[k]);
    ostr::DevGeom g = {};
    g.nx = (int)a[1], g.ny = (int)a[2], g.nz = (int)a[3];
    g.dx = a[4], g.dy = a[5], g.dz = a[6], g.x_p0 = a[7], g.y_p0 = a[8], g.z_p0 = a[9];
    g.nbx = (int)a[10], g.nby = (int)a[11], g.dbx = a[12], g.dby = a[13];
    g.x_d0 = a[14], g.y_d0 = a[15], g.det_r = a[16], g.src_y = a[17];
    ostr::ViewTab v = {};
    v.x0 = a[18], v.z0 = a[19];
    printf("%.9g %.9g\\n", ostr::matched_margin(g, &v, 1, true), ostr::matched_margin(g, &v, 1, false));
}
"""
F = np.float32
# nx, ny, nz, voxel, dz, z of the volume's floor, nbx, nby, bin, source x, covered
CASES = {
    "ordinary": (200, 100, 20, 0.5, 1.0, 0.0, 256, 128, 0.56, 85.0, True),
    "fine-bins": (200, 100, 20, 0.5, 1.0, 0.0, 9000, 4000, 0.002, 85.0, True),
    "below": (64, 48, 8, 1.0, 7.25, 600.0, 1500, 1000, 0.05, 3.0007, True),
    "close": (64, 48, 8, 1.0, 7.499897003173828, 600.0, 1500, 1000, 0.05, 3.00003, False),
    "closer": (64, 48, 8, 1.0, 7.499988555908203, 600.0, 1500, 1000, 0.05, 3.000004, False),
}
SZ = 660.0


@pytest.fixture(scope="module")
def margin(tmp_path_factory):
    d = tmp_path_factory.mktemp("margin")
    (d / "m.hip").write_text(PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-host-only", "-I", CSRC, str(d / "m.hip"),
                    "-o", str(d / "m")], check=True, capture_output=True)

    def call(g, sx, sz):
        args = [g.nx, g.ny, g.nz, g.dx, g.dy, g.dz, g.x_p0, g.y_p0, g.z_p0, g.nbx, g.nby, g.dbx,
                g.dby, g.x_d0, g.y_d0, g.detector_r, g.source_y, sx, sz]
        out = subprocess.run([str(d / "m")] + [repr(float(a)) for a in args], check=True,
                             capture_output=True, text=True).stdout
        return [F(v) for v in out.split()]
    return call


def left_out(n, v, p0, s, z, bins, b, d0, m, ulp):
    """Per voxel of the axis the rays of the exact shadow outside the FP32 range:
    their longest part of the voxel (x and z slabs), 0 where none is left out."""
    i = np.arange(n)
    x = [float(F(p0)) + (i + k) * float(F(v)) for k in (0, 1)]
    s64, b64, d64 = float(F(s)), float(F(b)), float(F(d0))
    ends = [s64 + (e - s64) * (-SZ / (q - SZ)) for e in x for q in z]
    q0 = np.ceil((np.minimum.reduce(ends) - d64) / b64 - 0.5).clip(0, bins).astype(int)
    q1 = np.floor((np.maximum.reduce(ends) - d64) / b64 - 0.5).clip(-1, bins - 1).astype(int)
    t = [-F(SZ) * np.nextafter(F(1.0) / (F(q) - F(SZ)), F(ulp) * F(np.inf), dtype=F) for q in z]
    ends = [np.asarray(float(F(s)) + (F(e) - F(s)).astype(float) * float(r), F) for e in x for r in t]
    inv = F(1.0) / F(b)
    b0 = np.ceil((np.minimum.reduce(ends) - F(d0)) * inv - F(0.5) - m).clip(0, bins).astype(int)
    b1 = np.floor((np.maximum.reduce(ends) - F(d0)) * inv + (m - F(0.5))).clip(-1, bins - 1).astype(int)
    longest = np.zeros(n)
    for k in np.nonzero((q0 <= q1) & ((b0 > q0) | (b1 < q1)))[0]:
        j = np.r_[q0[k]:min(b0[k], q1[k] + 1), max(b1[k] + 1, q0[k]):q1[k] + 1]
        e = d64 + (j + 0.5) * b64
        c = np.sort([(x[0][k] - e) / (s64 - e), (x[1][k] - e) / (s64 - e)], axis=0)
        part = np.minimum(c[1], z[1] / SZ) - np.maximum(c[0], z[0] / SZ)
        longest[k] = max(0.0, (part * SZ).max())   # per unit of height
    return longest


@pytest.mark.parametrize("name", CASES)
def test_candidates_hold_the_rays(margin, name):
    nx, ny, nz, v, dz, z0, nbx, nby, b, sx, covered = CASES[name]
    g = Geometry(nx=nx, ny=ny, nz=nz, dx=v, dy=v, dz=dz, x_p0=-nx * v / 2, y_p0=-ny * v,
                 z_p0=z0, nbx=nbx, nby=nby, dbx=b, dby=b, x_d0=-nbx * b / 2, y_d0=-nby * b,
                 detector_r=0.0, source_r=SZ, source_y=0.0)
    mx, my = margin(g, sx, SZ)
    assert (max(mx, my) < 0.5) == covered
    rounding = float(np.spacing(F(SZ)))
    for iz in range(nz):
        z = [float(F(z0)) + k * float(F(dz)) for k in (iz, iz + 1)]
        for ulp in (-1, 1):
            for axis in ((nx, v, g.x_p0, sx, z, nbx, b, g.x_d0, mx),
                         (ny, v, g.y_p0, 0.0, z, nby, b, g.y_d0, my)):
                out = left_out(*axis, ulp)
                assert out.max() <= (0.0 if covered else rounding)
