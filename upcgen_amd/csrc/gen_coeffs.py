"""Generate upc_coeffs.h: Chebyshev / power-series coefficients for the device
Bessel functions J0, J1, K0, K1 used by the photon-flux kernels.

The functions are defined by the mathematics (DLMF 10.2, 10.17, 10.25, 10.31,
10.40); the coefficients are computed here with mpmath at 50 digits and
rounded to double.  Run:  python gen_coeffs.py > upc_coeffs.h
"""
import mpmath as mp

mp.mp.dps = 50
TOL = mp.mpf("1e-19")


def cheb_coeffs(f, a, b, n=96, atol=None):
    """Chebyshev coefficients of f on [a, b] (first kind), c0 with full weight.
    Trailing coefficients below TOL times the leading scale are dropped, or
    below atol when it is given."""
    xs = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / n) for k in range(n)]
    fx = [f((b - a) / 2 * x + (b + a) / 2) for x in xs]
    cs = []
    for j in range(n):
        s = mp.fsum(fx[k] * mp.cos(mp.pi * j * (k + mp.mpf(1) / 2) / n) for k in range(n))
        cs.append(2 * s / n)
    cs[0] /= 2
    scale = max(abs(c) for c in cs[:4])
    m = len(cs)
    lim = TOL * scale if atol is None else atol
    while m > 1 and abs(cs[m - 1]) < lim:
        m -= 1
    return cs[:m]


def econ_poly(g, a, n, N=64):
    """Monomial coefficients (in z) of the degree n-1 Chebyshev interpolant of
    g on z in [0, a] (Chebyshev economisation: near-minimax on a short range)."""
    xs = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / N) for k in range(N)]
    fz = [g((x + 1) * a / 2) for x in xs]
    cs = []
    for j in range(n):
        s = mp.fsum(fz[k] * mp.cos(mp.pi * j * (k + mp.mpf(1) / 2) / N) for k in range(N))
        cs.append(2 * s / N)
    cs[0] /= 2
    T = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]
    for j in range(2, n):
        p = [mp.mpf(0)] * (j + 1)
        for i, c in enumerate(T[j - 1]):
            p[i + 1] += 2 * c
        for i, c in enumerate(T[j - 2]):
            p[i] -= c
        T.append(p)
    tpoly = [mp.mpf(0)] * n
    for j in range(n):
        for i, c in enumerate(T[j]):
            tpoly[i] += cs[j] * c
    zpoly = [mp.mpf(0)] * n  # t = 2 z / a - 1
    for i, c in enumerate(tpoly):
        for k in range(i + 1):
            zpoly[k] += c * mp.binomial(i, k) * (2 / a) ** k * (-1) ** (i - k)
    return zpoly


def cheb_to_mono(c):
    """Monomial coefficients of sum c_k T_k(v) (exact, at the working precision)."""
    n = len(c)
    T = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]
    for j in range(2, n):
        p = [mp.mpf(0)] * (j + 1)
        for i, x in enumerate(T[j - 1]):
            p[i + 1] += 2 * x
        for i, x in enumerate(T[j - 2]):
            p[i] -= x
        T.append(p)
    a = [mp.mpf(0)] * n
    for j in range(n):
        for i, x in enumerate(T[j]):
            a[i] += c[j] * x
    return a


def emit(name, cs):
    body = ",\n  ".join(mp.nstr(c, 25, min_fixed=-1, max_fixed=-1) if c != 0 else "0.0" for c in cs)
    return f"static constexpr int {name}_N = {len(cs)};\n__constant__ static const double {name}[{len(cs)}] = {{\n  {body}}};\n"


def main():
    out = ["// Generated by gen_coeffs.py (mpmath, 50 digits). Do not edit by hand.",
           "#pragma once", ""]
    # J1(x)/x on [0, 8] as a function of u = x^2/32 - 1 in [-1, 1]; the
    # dropped tail costs J1 at most 8 x its sum (< 1e-17 absolute).
    j1s = cheb_coeffs(lambda u: (lambda x: mp.besselj(1, x) / x if x != 0 else mp.mpf(1) / 2)(
        mp.sqrt(32 * (u + 1))), -1, 1, atol=mp.mpf("1e-18"))
    out.append("// J1(x)/x = sum c_k T_k(x^2/32 - 1), 0 <= x <= 8")
    out.append(emit("kJ1Small", j1s))

    # J0 likewise (J1' = J0 - J1/x).
    j0s = cheb_coeffs(lambda u: mp.besselj(0, mp.sqrt(32 * (u + 1))), -1, 1, atol=mp.mpf("1e-17"))
    out.append("// J0(x) = sum c_k T_k(x^2/32 - 1), 0 <= x <= 8")
    out.append(emit("kJ0Small", j0s))

    # Hankel modulus/phase form for x >= 8, s = 64/x^2 in (0, 1] -> v = 2 s - 1.
    def pq(x, nu=1):
        chi = x - (2 * nu + 1) * mp.pi / 4
        j, y = mp.besselj(nu, x), mp.bessely(nu, x)
        f = mp.sqrt(mp.pi * x / 2)
        P = f * (j * mp.cos(chi) + y * mp.sin(chi))
        Q = f * (y * mp.cos(chi) - j * mp.sin(chi))
        return P, Q

    def P_of_v(v):
        s = (v + 1) / 2
        if s == 0:
            return mp.mpf(1)
        return pq(8 / mp.sqrt(s))[0]

    def Q_of_v(v):
        s = (v + 1) / 2
        if s == 0:
            return mp.mpf(3) / 64
        x = 8 / mp.sqrt(s)
        return pq(x)[1] * x / 8

    # P ~ 1 and Q (8/x) <= 0.05: Chebyshev tails below 1e-17 each (J1 error <
    # 1e-17 absolute), then re-expanded in powers of v for Horner evaluation:
    # sum |p_k v^k| <= 1.002 and sum |q_k v^k| <= 0.047 on [-1, 1], so the
    # monomial form loses nothing against Clenshaw (both within 1 ulp).
    pc = cheb_coeffs(P_of_v, -1, 1, atol=mp.mpf("1e-17"))
    qc = cheb_coeffs(Q_of_v, -1, 1, atol=mp.mpf("1e-17"))
    n = max(len(pc), len(qc))  # padded to one length: evaluated together
    pc, qc = pc + [mp.mpf(0)] * (n - len(pc)), qc + [mp.mpf(0)] * (n - len(qc))
    out.append("// J1(x) = (P (sin x - cos x) + Q (sin x + cos x)) / sqrt(pi x), x >= 8,")
    out.append("// P = sum p_k v^k, Q = (8/x) sum q_k v^k, v = 128/x^2 - 1")
    out.append(emit("kJ1P", cheb_to_mono(pc)))
    out.append(emit("kJ1Q", cheb_to_mono(qc)))

    def P0_of_v(v):
        s = (v + 1) / 2
        return mp.mpf(1) if s == 0 else pq(8 / mp.sqrt(s), 0)[0]

    def Q0_of_v(v):
        s = (v + 1) / 2
        if s == 0:
            return -mp.mpf(1) / 64
        x = 8 / mp.sqrt(s)
        return pq(x, 0)[1] * x / 8

    pc = cheb_coeffs(P0_of_v, -1, 1, atol=mp.mpf("1e-17"))
    qc = cheb_coeffs(Q0_of_v, -1, 1, atol=mp.mpf("1e-17"))
    n = max(len(pc), len(qc))
    pc, qc = pc + [mp.mpf(0)] * (n - len(pc)), qc + [mp.mpf(0)] * (n - len(qc))
    out.append("// J0(x) = (P (sin x + cos x) - Q (sin x - cos x)) / sqrt(pi x), x >= 8, P, Q in v as for J1")
    out.append(emit("kJ0P", cheb_to_mono(pc)))
    out.append(emit("kJ0Q", cheb_to_mono(qc)))

    # sin r = r + r^3 S(r^2), cos r = 1 - r^2/2 + r^4 C(r^2) on |r| <= pi/4
    # (after reduction by pi/2); absolute errors 1.4e-17 and 9e-19.
    a = (mp.pi / 4) ** 2
    sp = econ_poly(lambda z: (mp.sin(mp.sqrt(z)) - mp.sqrt(z)) / (z * mp.sqrt(z)) if z > 0 else -mp.mpf(1) / 6,
                   a, 6)
    cp = econ_poly(lambda z: (mp.cos(mp.sqrt(z)) - 1 + z / 2) / (z * z) if z > 0 else mp.mpf(1) / 24, a, 6)
    out.append("// sin r = r + r^3 S(r^2), cos r = 1 - r^2/2 + r^4 C(r^2), |r| <= pi/4: S, C in powers of r^2")
    out.append(emit("kSinPoly", sp))
    out.append(emit("kCosPoly", cp))

    # Power series for K0, K1 at 0 < x <= 1 in y = x^2/4 (DLMF 10.25.2, 10.31.1).
    NS = 16
    i0 = [1 / mp.factorial(k) ** 2 for k in range(NS)]
    s0 = [mp.harmonic(k) / mp.factorial(k) ** 2 for k in range(NS)]
    i1 = [1 / (mp.factorial(k) * mp.factorial(k + 1)) for k in range(NS)]
    s1 = [(mp.digamma(k + 1) + mp.digamma(k + 2)) / (mp.factorial(k) * mp.factorial(k + 1))
          for k in range(NS)]
    out.append("// Series in y = x^2/4: I0 = sum a_k y^k, S0 = sum H_k y^k/(k!)^2,")
    out.append("// I1 = (x/2) sum y^k/(k!(k+1)!), S1 = sum (psi(k+1)+psi(k+2)) y^k/(k!(k+1)!)")
    out.append("// K0 = -(ln(x/2)+gamma) I0 + S0 ; K1 = 1/x + ln(x/2) I1 - (x/4) S1")
    for nm_, cs in (("kI0Ser", i0), ("kS0Ser", s0), ("kI1Ser", i1), ("kS1Ser", s1)):
        out.append(emit(nm_, cs))

    # Scaled K_nu(x) e^x sqrt(x) for x > 1, two pieces in t = 1/x.
    for nu in (0, 1):
        f = lambda t, nu=nu: (mp.besselk(nu, 1 / t) * mp.exp(1 / t) * mp.sqrt(1 / t)) if t > 0 \
            else mp.sqrt(mp.pi / 2)
        for tag, a, b in (("A", mp.mpf(1) / 4, 1), ("B", 0, mp.mpf(1) / 4)):
            cs = cheb_coeffs(f, a, b, n=128)
            out.append(f"// K{nu}(x) e^x sqrt(x) on 1/x in [{mp.nstr(a, 3)}, {mp.nstr(b, 3)}]"
                       f" = sum c_k T_k((2/x - {mp.nstr(a + b, 4)})/{mp.nstr(b - a, 4)})")
            out.append(emit(f"kK{nu}{tag}", cs))
    print("\n".join(out))


if __name__ == "__main__":
    main()
