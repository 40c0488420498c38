"""The hop launchers' checks of the launch shape (host code, no GPU): a launch
whose kernel would leave its operands is refused before it starts.  A launch
that passes them goes on to the runtime, which answers with another error
where there is no device."""
import os
import shutil
import subprocess

import pytest

import cps_public_amd as C

CSRC = os.path.join(os.path.dirname(os.path.abspath(C.__file__)), "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include "hop.h"
using namespace cpship;

static HopParams shape(int kind, int prec, int clov, int Vcb, int nb, int nrhs) {
  HopParams P;
  std::memset((void*)&P, 0, sizeof P);
  P.geom.Vcb = Vcb;
  P.geom.L[3] = 4;
  P.kind = kind;
  P.prec = prec;
  P.clov = clov;
  P.nb = nb;
  P.nrhs = nrhs;
  P.nsites_out = kind == KIND_DWF ? 2 * Vcb : Vcb;
  P.ls = 2 * nb;
  P.perm_S = kind == KIND_DWF ? Vcb / 4 : Vcb / 8;
  P.block = pick_block((long long)P.nsites_out * nb);
  P.rhs_per_set = 1;
  return P;
}

// 1: refused for its shape, 0: not
static int refused(HopParams P) {
  static double mem[8];
  P.in.data = P.out.data = P.X.data = P.R.data = mem;
  P.clover.data = mem;
  P.kscale = P.ralpha = mem;
  P.ractive = (const int*)mem;
  P.gauge.data = mem;
  return launch_hop(P, nullptr) == hipErrorInvalidValue;
}

int main() {
  static double part[8];
  static uint32_t perm[8];
  int count = 0;
  if (hipGetDeviceCount(&count) == hipSuccess && count > 0) { printf("device\n"); return 0; }
  // partials per block: blocks of the default size only (a domain-wall field
  // of two slices, 256 elements per rhs, in one block or in four)
  HopParams P = shape(KIND_DWF, PREC_D_D18, CLOV_NONE, 128, 1, 3);
  P.dag = P.rupd = 1;
  P.partial = part;
  printf("partials %d", refused(P));
  P.block = 64;
  printf(" %d\n", refused(P));
  // partials per chunk do not depend on the block
  P = shape(KIND_WILSON, PREC_D_D18, CLOV_NONE, 256, 1, 3);
  P.dag = P.rupd = 1;
  P.partial = part;
  printf("chunks %d", refused(P));
  P.block = 64;
  printf(" %d\n", refused(P));
  // the spatial order without its table, with it, in hardware block order,
  // and with blocks that straddle two spatial blocks
  for (int clov : {(int)CLOV_NONE, (int)CLOV_S5X}) {
    P = shape(KIND_WILSON, PREC_D_D18, clov, 256, 8, 2);
    P.flags = HOP_SPATIAL;
    printf("spatial %d", refused(P));
    P.perm = perm;
    printf(" %d", refused(P));
    P.flags |= HOP_NO_XCD_REMAP;
    printf(" %d", refused(P));
    P = shape(KIND_WILSON, PREC_D_D18, clov, 256, 12, 2);
    P.flags = HOP_SPATIAL;
    P.perm = perm;
    printf(" %d\n", refused(P));   // 256 * 12 / 8 = 384 elements, blocks of 256
  }
  return 0;
}
"""


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="no hipcc")
def test_launch_shape_checks(tmp_path):
    src = tmp_path / "checks.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "checks")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-I", CSRC, "-I",
                    os.path.join(CSRC, "..", "..", "include"), str(src), "-x", "none", C.LIB_PATH, "-o", exe,
                    f"-Wl,-rpath,{os.path.dirname(C.LIB_PATH)}"], check=True, capture_output=True, timeout=100)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout.split("\n")
    if out[0] == "device":
        pytest.skip("a GPU is there: the accepted shapes would be launched")
    assert out[:4] == ["partials 0 1", "chunks 0 0", "spatial 1 0 1 1", "spatial 1 0 1 1"]
