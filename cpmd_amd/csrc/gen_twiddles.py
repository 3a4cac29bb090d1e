"""Generates twiddle_consts.h: exp(-2 pi i j / R) for the in-register DFT sizes,
evaluated with 50-digit decimal arithmetic and rounded once to float64.
Run: python cpmd_amd/csrc/gen_twiddles.py > cpmd_amd/csrc/twiddle_consts.h"""
from decimal import Decimal, getcontext

getcontext().prec = 60
SIZES = (6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 28)


def pi():
    # Machin's formula
    def arctan_inv(x):
        x = Decimal(x)
        s, t, n, k = Decimal(0), 1 / x, 1, 0
        x2 = x * x
        while True:
            term = t / n
            if term == 0 or abs(term) < Decimal(10) ** -58:
                break
            s += term if k % 2 == 0 else -term
            t /= x2
            n += 2
            k += 1
        return s
    return 4 * (4 * arctan_inv(5) - arctan_inv(239))


PI = pi()


def cos_sin(a):
    c, s, term, n = Decimal(0), Decimal(0), Decimal(1), 0
    while True:
        if n % 2 == 0:
            c += term * (1 if (n // 2) % 2 == 0 else -1)
        else:
            s += term * (1 if (n // 2) % 2 == 0 else -1)
        n += 1
        term = term * a / n
        if abs(term) < Decimal(10) ** -58:
            break
    return c, s


def main():
    print("// Generated by gen_twiddles.py: W_R^j = exp(-2 pi i j/R) = (c[j], -s[j]).")
    print("#pragma once")
    print("namespace mc {")
    print("template <int R> struct TwC;")
    for r in SIZES:
        cs, ss = [], []
        for j in range(r):
            c, s = cos_sin(2 * PI * j / r)
            cs.append(repr(float(c)) if abs(c) > Decimal(10) ** -40 else "0.0")
            ss.append(repr(float(s)) if abs(s) > Decimal(10) ** -40 else "0.0")
        print(f"template <> struct TwC<{r}> {{")
        print(f"  static constexpr double c[{r}] = {{{', '.join(cs)}}};")
        print(f"  static constexpr double s[{r}] = {{{', '.join(ss)}}};")
        print("};")
    print("}  // namespace mc")


if __name__ == "__main__":
    main()
