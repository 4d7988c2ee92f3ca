"""The grid coordinate of an atom anywhere: the loops that wrap it end, with
the exact remainder, however far the atom is (run in a process of its own, so
that an endless loop ends with the test)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CODE = r'''
import ctypes as C, math, random, sys
from fractions import Fraction
lib = C.CDLL(sys.argv[1])
lib.grid_coordinate.argtypes = [C.c_double, C.c_double, C.c_int, C.c_int, C.POINTER(C.c_int), C.POINTER(C.c_double)]

def coord(x, hr, K, off):
    b, w = C.c_int(), C.c_double()
    lib.grid_coordinate(x, hr, K, off, C.byref(b), C.byref(w))
    return b.value, w.value

rng = random.Random(5)
for _ in range(20000):
    K, order = rng.choice([4, 30, 64, 216, 4096]), rng.choice([2, 4, 6, 8])
    hr, off = rng.uniform(0.01, 40.0), -((order - 1) // 2) + K
    x = rng.choice([-1, 1]) * 10.0 ** rng.uniform(-3, 11)
    u = Fraction(x * hr)
    if abs(u) >= 2 ** 40:
        continue
    r = u % K
    b, w = coord(x, hr, K, off)
    if r < K - Fraction(1, 2 ** 20):  # (next to K the last addition may round up to it: place 0)
        # a negative place loses what K + u rounds off
        assert abs((b - off) % K + Fraction(w) - r) <= Fraction(1, 2 ** 40), (x, hr, K, b, w)
for x in (1e16, -1e16, 1e300, -1e300, math.inf, -math.inf):
    b, w = coord(x, 1.0, 64, 63)
    assert 0 <= b < 64 and w == 0.0
assert math.isnan(coord(math.nan, 1.0, 64, 63)[1])
print("done")
'''


def test_the_place_of_an_atom_far_from_the_box():
    lib = os.path.join(ROOT, "tests", "native", "libpairfunctions.so")
    r = subprocess.run([sys.executable, "-c", CODE, lib], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "done" in r.stdout, r.stderr[-2000:]
