"""Tables of the tile expansions of lt_far.hip (lt_cheb_tables.h), derived with mpmath at 50 digits
and printed as C hexadecimal floating-point literals. Not part of the build: run
`python gen_cheb.py > lt_cheb_tables.h` to reproduce the header.

  kNode[i]      the 16 Chebyshev nodes cos((2 i + 1) pi / 32)
  kDct[k][i]    c_k = sum_i kDct[k][i] f(node_i): the Chebyshev coefficients of the interpolant
  kShift[s][m][k]  T_k(-1/2 + t/2) (s = 0), T_k(1/2 + t/2) (s = 1) = sum_m kShift[s][m][k] T_m(t): the
                coefficients of a parent tile's expansion on its left / right (lower / upper) half
"""
import mpmath as mp

mp.mp.dps = 50
P = 16
NODE = [mp.cos((2 * i + 1) * mp.pi / (2 * P)) for i in range(P)]
DCT = [[mp.cos(k * (2 * i + 1) * mp.pi / (2 * P)) * (1 if k == 0 else 2) / P for i in range(P)] for k in range(P)]


def shift(s):
    # exact: T_k of degree k <= 15 is interpolated by 16 nodes
    off = mp.mpf(-1) / 2 if s == 0 else mp.mpf(1) / 2
    return [[mp.fsum(DCT[m][i] * mp.cos(k * mp.acos(off + NODE[i] / 2)) for i in range(P)) if m <= k else mp.mpf(0)
             for k in range(P)] for m in range(P)]


def rows(name, t):
    print(f"__constant__ const double {name}[{len(t) * len(t[0])}] = {{")
    for r in t:
        print("    " + ", ".join(float(v).hex() for v in r) + ",")
    print("};")


def main():
    print("// lt_cheb_tables.h -- printed by gen_cheb.py: Chebyshev nodes, transform and half-tile shifts of order 16.")
    print("#pragma once\n\nnamespace lt {\n")
    rows("kNode", [NODE])
    rows("kDct", DCT)
    rows("kShift", shift(0) + shift(1))
    print("\n}  // namespace lt")


if __name__ == "__main__":
    main()
