"""A launch's error is reported, not cleared by the questions asked around it (on the host, against a stand-in for
the HIP runtime: nothing reaches a GPU)."""
import os
import shutil
import subprocess
import sys

import pytest

from dmgs_amd import _native as N

STAND_IN = r"""
/* The first kernel launch fails, all else succeeds; the last error is kept as HIP keeps it. */
static int last, launches;
int hipLaunchKernel() { return launches++ ? 0 : (last = 2); }
int hipPointerGetAttributes() { return last = 1; } /* plain host memory */
int hipGetLastError(void) { int e = last; last = 0; return e; }
int hipPeekAtLastError(void) { return last; }
int hipMemcpyAsync() { return 0; }
int __hipPushCallConfiguration() { return 0; }
int __hipPopCallConfiguration() { return 0; }
"""
CALL = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[2])
ctypes.CDLL(sys.argv[3], ctypes.RTLD_GLOBAL)  # before the HIP runtime: the library's calls bind to it
from dmgs_amd import _native as N
lib = ctypes.CDLL(sys.argv[1])
fake = ctypes.c_void_p(0x1000)
s, g = N.DmgsSettings(), N.DmgsGaussians()
s.image_width = s.image_height = 64
s.tanfovx = s.tanfovy = s.scale_modifier = 1.0
s.viewmatrix = s.projmatrix = s.campos = s.bg = 0x1000
g.count = 10
g.means3D = g.opacities = g.colors_precomp = g.cov3D_precomp = 0x1000
counts = (ctypes.c_uint32 * 2)()
print("rc", lib.dmgs_view_geometry(ctypes.byref(s), ctypes.byref(g), 0, fake, fake, counts, None))
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_view_geometry_reports_a_failed_launch(tmp_path):
    (tmp_path / "hip.c").write_text(STAND_IN)
    so = tmp_path / "hip.so"
    subprocess.run(["gcc", "-w", "-std=gnu89", "-shared", "-fPIC", "-o", so, tmp_path / "hip.c"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CALL, N.library_path(), root, str(so)], capture_output=True, text=True,
                       timeout=120, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"))
    assert "rc -2" in r.stdout, (r.stdout, r.stderr[-2000:])
