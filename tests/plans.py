"""The kernel choice rules of csrc/plan.h, compiled for the CPU: which kernel a call takes and how it splits k."""
import ctypes
import subprocess
from pathlib import Path

from oracle import oracle as O

CSRC = Path(__file__).resolve().parent.parent / "qxotic_amd" / "csrc"
SHIM = """
#include "plan.h"
using namespace jamhip;
extern "C" void q_wide(int dt, int k, int m, int n, size_t act, int* o) {
    const WidePlan p = wide_plan(dt, k, m, n, 256, act);
    o[0] = p.wide, o[1] = p.k.ns, o[2] = p.k.per;
}
extern "C" void q_mx4(int m, int k, int n, int* o) { const Mx4Plan p = mx4_plan(m, k, n); o[0] = p.rt, o[1] = p.tiles, o[2] = p.k.ns, o[3] = p.k.per; }
extern "C" int q_big(int dt, int m, int k, int n) {
    const int units = up_div(k, 64);
    return dense_big(dt, units, m, n, split_plan(up_div(m, 128) * up_div(n, 64), units), 256);
}
extern "C" void q_prep_grid(int n, int Kp, int* o) { const PrepGrid g = dense_prep_grid(n, Kp); o[0] = g.x, o[1] = g.y; }
extern "C" int q_few(int dt, int k, int n) { return dense_prep_few(dt, k, n); }
extern "C" int q_tile32(int m, int n) { return dense_tile32(m, n); }
extern "C" long long q_pitch(long long bytes) { return dense_row_pitch(bytes); }
extern "C" void q_split(int total, int units, int* o) { const Split s = split_plan(total, units); o[0] = s.ns, o[1] = s.per; }
extern "C" int q_tail(int total, int cus) { return tail_tiles(total, cus); }
"""


class Plans:
    def __init__(self, so):
        self.lib = ctypes.CDLL(str(so))
        self.lib.q_pitch.restype, self.lib.q_pitch.argtypes = ctypes.c_longlong, [ctypes.c_longlong]

    def _get(self, name, size, *args):
        o = (ctypes.c_int * size)()
        getattr(self.lib, name)(*args, o)
        return list(o)

    def wide(self, dt, k, m, n):
        np_, sums = (n + 63) // 64 * 64, 16 if dt == O.Q6_K else 8
        act = k * np_ * 2 + k // 32 * np_ * 4 + 2 * (k // 256 * np_ * sums * 2) + 4 * np_
        return self._get("q_wide", 3, dt, k, m, n, ctypes.c_size_t(act))

    def mx4(self, m, k, n):
        return self._get("q_mx4", 4, m, k, n)

    def prep_grid(self, n, kp):
        return self._get("q_prep_grid", 2, n, kp)

    def split(self, total, units):
        return self._get("q_split", 2, total, units)


def build(folder):
    (folder / "plans.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(folder / "plans.cpp"), "-o",
                    str(folder / "plans.so")], check=True)
    return Plans(folder / "plans.so")
