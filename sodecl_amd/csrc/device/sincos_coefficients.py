"""Derivation of the constants in sincos.hip (run: python sincos_coefficients.py).

Reduction x = q pi/2 + r, |r| <= pi/4: 2/pi rounded to double; pi/2 split as
P1 + P2, P1 = pi/2 rounded to double, P2 the remainder rounded.  On
0 <= z = r^2 <= (pi/4)^2 (slightly widened) by Chebyshev interpolation at 60
significant digits (mpmath.chebyfit, near-minimax):
  * S of degree 5 approximating (sin r - r) / r^3,
  * C of degree 5 approximating (cos r - 1 + r^2/2) / r^4.
Hex literals are printed in the order the source uses them."""
import mpmath as mp

mp.mp.dps = 60


def hexd(v):
    return float.hex(float(mp.mpf(v)))


def s_of_z(z):
    if z == 0:
        return -mp.mpf(1) / 6
    r = mp.sqrt(z)
    return (mp.sin(r) - r) / r ** 3


def c_of_z(z):
    if z == 0:
        return mp.mpf(1) / 24
    r = mp.sqrt(z)
    return (mp.cos(r) - 1 + r ** 2 / 2) / r ** 4


def main():
    p1 = mp.mpf(float(mp.pi / 2))
    p2 = mp.mpf(float(mp.pi / 2 - p1))
    print("2/pi", hexd(2 / mp.pi), "P1", hexd(p1), "P2", hexd(p2), "left over", mp.nstr(mp.pi / 2 - p1 - p2, 3))
    hi = (mp.pi / 4) ** 2 * mp.mpf("1.0001")
    for name, fn, degree in (("S", s_of_z, 5), ("C", c_of_z, 5)):
        poly, err = mp.chebyfit(fn, [0, hi], degree + 1, error=True)
        print(name, "degree", degree, "error", mp.nstr(err, 3))
        for c in poly:
            print("   ", hexd(c))


if __name__ == "__main__":
    main()
