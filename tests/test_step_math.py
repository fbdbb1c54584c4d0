"""The step's square root, divisions, logarithm and sine/cosine (csrc/pt_math.h), compiled
for the host with approximations of 1/x and 1/sqrt(x) of the hardware's quality, against
IEEE arithmetic (bit for bit) and 80-bit long double.

Error bounds.  log: half an ulp of the last sum, plus the roundings of r^2 p (2^-7 of the
result at most, two roundings and the polynomial's 2^-57) and, beside 1, half of the last
bit that r can lose: 0.6 ulp.  Sine and cosine: half an ulp, plus the term that is added
last (at most a fifth of the result, with up to three roundings): 0.8 ulp."""
import os
import subprocess
import sys

SRC = r"""
#include "pt_math.h"
#include <cmath>
#include <cstdio>
using namespace pt;
static const double T[] = {PT_MATH_TABLE};
static_assert(sizeof(T) == sizeof(double) * MATH_DOUBLES, "table");
static uint64_t s0 = 0x9E3779B97F4A7C15ull, s1 = 0xD1B54A32D192ED03ull;
static uint64_t rnd() {
    uint64_t a = s0, b = s1;
    s0 = b;
    a ^= a << 23;
    s1 = a ^ b ^ (a >> 17) ^ (b >> 26);
    return s1 + b;
}
static double uni() { return ((double)(rnd() >> 12) + 0.5) * 0x1p-52; }
static double ulp(long double v) {
    int e;
    frexpl(fabsl(v), &e);
    return ldexp(1.0, e - 53);
}
static bool same(double a, double b) { return a == b || (a != a && b != b); }
int main() {
    double el = 0, es = 0, ec = 0;
    long sq = 0, dv = 0, iv = 0, sp = 0;
    const double *t = T;
    for (long i = 0; i < 3000000; i++) {
        double u = uni();
        if (i % 4 == 1) u = 1.0 - ldexp(uni(), -(int)(rnd() % 50));
        if (i % 4 == 2) u = ldexp(1.0 + uni(), (int)(rnd() % 200) - 100);
        if (i % 4 == 3) u = exp(uni() * 0.04 - 0.02);
        const long double l = logl((long double)u);
        if (l != 0) el = fmax(el, (double)(fabsl(log_tab(u, t) - l) / ulp(l)));
        else if (log_tab(u, t) != 0) sp++;
        double x = 6.283185307179586 * uni(), sn, cs;
        if (i % 8 == 0) x = fabs(1.5707963267948966 * (rnd() % 5) - ldexp(uni(), -(int)(rnd() % 40)));
        if (x > 6.283185307179586) x = 6.283185307179586;
        sincos_turn(x, sn, cs, t);
        const long double ls = sinl((long double)x), lc = cosl((long double)x);
        es = fmax(es, (double)(fabsl(sn - ls) / ulp(ls)));
        ec = fmax(ec, (double)(fabsl(cs - lc) / ulp(lc)));
        const double a = ldexp(1.0 + uni(), (int)(rnd() % 600) - 300), b = ldexp(1.0 + uni(), (int)(rnd() % 300) - 150);
        sq += qsqrt(a) != sqrt(a);
        dv += qdiv(a, b) != a / b || qdiv(-a, b) != -a / b;
        iv += Recip(b).inverse() != 1.0 / b;
    }
    const double inf = HUGE_VAL, v[] = {0.0, 1.0, inf, -inf, NAN, -3.0, 1e-300};
    for (double a : v)
        for (double b : v) sp += !same(qdiv_any(a, b), a / b);
    for (double a : v) sp += !same(qsqrt(a), sqrt(a));
    double sn, cs;
    sincos_turn(0.0, sn, cs, t);
    sp += sn != 0.0 || cs != 1.0;
    printf("%.4f %.4f %.4f %ld %ld %ld %ld\n", el, es, ec, sq, dv, iv, sp);
    return 0;
}
"""


def test_step_math(tmp_path):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, exe = tmp_path / "m.cpp", tmp_path / "m"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-I",
                    os.path.join(root, "particulator.jl_amd", "csrc"), "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    print(out, file=sys.stderr)
    log, sin, cos = (float(v) for v in out[:3])
    assert log <= 0.6 and sin <= 0.8 and cos <= 0.8
    assert [int(v) for v in out[3:]] == [0, 0, 0, 0]  # sqrt, quotients, reciprocals, special values
