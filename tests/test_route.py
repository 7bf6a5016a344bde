"""How a batch is launched (csrc/route.h), compiled for the host: the estimate
of a launch's time against its workgroups taken one by one, and the choices
against measured times."""
import heapq
import os
import subprocess

import pytest

from conftest import PKG

ROW_BYTES = {2: 4096, 3: 4096, 4: 2048, 5: 2048, 6: 1024, 7: 512}
MAX_T = {2: 1, 3: 2, 4: 4, 5: 8, 6: 8, 7: 8}
NCU = 256

DRIVER = r"""
#include <stdio.h>
#include "route.h"
int main() {
    char f;
    int K, a, n, ncu, pivot, n1;
    double rb;
    while (scanf(" %c %d %d %d %d", &f, &K, &a, &n, &ncu) == 5) {
        if (f == 's') printf("%.17g\n", xtq::forward_step_us(K, a));
        if (f == 'c') printf("%.17g\n", xtq::forward_cost_us(K, a, n, ncu));
        if (f == 'g') printf("%d\n", xtq::forward_group(K, a, n, ncu));
        if (f == 'f' && scanf("%d %d %lf", &pivot, &n1, &rb) == 3)
            printf("%d\n", (int)xtq::fused_ends_first(K, a, rb, n, n1, pivot, 256, ncu));
    }
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    """route(queries) -> one number per query (function, K, T or max T, n, CUs)"""
    tmp = tmp_path_factory.mktemp("route")
    (tmp / "route.cpp").write_text(DRIVER)
    exe = str(tmp / "route")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    "-I" + os.path.join(PKG, "csrc"), str(tmp / "route.cpp"), "-o", exe],
                   check=True, capture_output=True)

    def ask(queries):
        text = "".join(" ".join(map(str, q)) + "\n" for q in queries)
        out = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout
        return [float(v) for v in out.split()]

    return ask


@pytest.mark.parametrize("K", range(2, 8))
def test_cost_is_the_end_of_the_last_workgroup(route, K):
    """Each CU takes the next workgroup as soon as it is free.  A last one of
    fewer than T sequences is shorter than the others, so it never costs a
    round of T sequences."""
    for ncu in (1, 5, NCU):
        for T in [t for t in (1, 2, 4, 8) if t <= MAX_T[K]]:
            us1, us = route([("s", K, 1, 0, 0), ("s", K, T, 0, 0)])
            ns = sorted({n for r in (1, 2, 3) for n in range(r * T * ncu - T, r * T * ncu + 2 * T)
                         if n > 0} | {1, 2, 3, 7, 100})
            got = route([("c", K, T, n, ncu) for n in ns])
            for n, g in zip(ns, got):
                cus = [0.0] * ncu
                for q in range(0, n, T):
                    r = min(T, n - q)
                    t = T * us if r == T else min(T * us, 1.2 * r * us1)
                    heapq.heappush(cus, heapq.heappop(cus) + t)
                assert g == pytest.approx(max(cus), rel=1e-12), (K, T, n, ncu)


# Microseconds per step of the forwards of a tail-bite of n sequences on 256
# CUs, by sequences per workgroup (1, 2, 4, 8).
MEASURED = {
    (3, 513): (3.574, 3.781), (3, 1025): (5.960, 6.247), (3, 2049): (10.872, 11.184),
    (4, 257): (2.370, 2.423, 4.455), (4, 513): (3.382, 3.825, 4.437),
    (4, 1025): (5.667, 6.247, 6.016), (4, 1026): (5.706, 7.187, 7.351),
    (4, 1537): (7.960, 8.666, 9.221), (4, 2049): (10.470, 11.129, 10.702),
    (4, 2053): (10.662, 12.449, 14.340),
    (5, 1025): (5.790, 6.249, 5.992, 8.767), (5, 2049): (10.833, 11.265, 10.808, 10.850),
    (5, 2053): (10.864, 12.636, 14.502, 16.960), (5, 3073): (15.806, 16.618, 15.945, 18.855),
    (6, 1025): (6.215, 6.661, 6.392, 9.413), (6, 2049): (11.417, 11.854, 11.421, 11.225),
    (7, 1025): (6.430, 6.729, 6.615, 9.560), (7, 2049): (11.725, 11.997, 11.721, 11.321),
    (7, 2048): (10.482, 10.457, 10.090, 9.842), (7, 3073): (16.990, 17.195, 16.964, 19.912),
}


def test_group_choice_against_measured_times(route):
    """Around whole rounds, where a larger group's last workgroup may be short:
    the chosen group's time is the least measured, within the 3.5 % by which
    two runs of one size differ here."""
    got = route([("g", K, MAX_T[K], n, NCU) for K, n in MEASURED])
    for (key, us), T in zip(MEASURED.items(), got):
        assert us[int(T).bit_length() - 1] <= 1.035 * min(us), (key, T)


# Microseconds of whole tail-bite calls on 256 CUs, (K, sequences, pivot,
# margin): as separate launches at the best group, and as one fused launch.
ROUTES = {
    (2, 64, 128, 0): (754, 789), (2, 128, 128, 0): (765, 840), (2, 192, 128, 0): (780, 1186),
    (2, 257, 128, 0): (1401, 1168), (2, 300, 128, 0): (1435, 1185), (2, 400, 128, 0): (1466, 1571),
    (2, 512, 128, 0): (1559, 1599), (2, 513, 128, 0): (2138, 1943), (2, 600, 128, 0): (2221, 1977),
    (2, 1003, 128, 0): (3094, 3135), (2, 1025, 128, 0): (3693, 3539),
    (2, 1537, 128, 0): (5199, 5094), (2, 2049, 128, 0): (6451, 6752), (2, 64, 128, 16): (579, 628),
    (2, 257, 128, 16): (1094, 1018), (2, 600, 128, 16): (1720, 1637), (3, 64, 128, 0): (712, 751),
    (3, 256, 128, 0): (790, 815), (3, 257, 128, 0): (1318, 1136), (3, 300, 128, 0): (1343, 1141),
    (3, 400, 128, 0): (1374, 1497), (3, 513, 128, 0): (2016, 1850), (3, 600, 128, 0): (2073, 1856),
    (3, 768, 128, 0): (2180, 2237), (3, 1003, 128, 0): (2851, 2943),
    (3, 1200, 128, 0): (3554, 3693), (3, 1500, 128, 0): (4271, 4447),
    (3, 2300, 128, 0): (6027, 6769), (4, 64, 128, 0): (670, 713), (4, 256, 128, 0): (708, 804),
    (4, 257, 128, 0): (1273, 1084), (4, 300, 128, 0): (1259, 1080), (4, 400, 128, 0): (1258, 1422),
    (4, 513, 128, 0): (1828, 1765), (4, 600, 128, 0): (1873, 1752), (4, 768, 128, 0): (1960, 2105),
    (4, 1003, 128, 0): (2507, 2737), (4, 1200, 128, 0): (3189, 3436),
    (4, 1500, 128, 0): (3836, 4177), (4, 2300, 128, 0): (5746, 6266), (5, 64, 128, 0): (676, 721),
    (5, 256, 128, 0): (746, 844), (5, 257, 128, 0): (1310, 1128), (5, 300, 128, 0): (1283, 1151),
    (5, 400, 128, 0): (1314, 1511), (5, 513, 128, 0): (1881, 1871), (5, 600, 128, 0): (1916, 1880),
    (5, 768, 128, 0): (2050, 2249), (5, 1003, 128, 0): (2529, 2837),
    (5, 1200, 128, 0): (3282, 3556), (5, 1500, 128, 0): (3945, 4242),
    (5, 2300, 128, 0): (5923, 6507), (6, 64, 128, 0): (707, 763), (6, 256, 128, 0): (771, 877),
    (6, 257, 128, 0): (1378, 1187), (6, 300, 128, 0): (1355, 1183), (6, 400, 128, 0): (1361, 1577),
    (6, 513, 128, 0): (1972, 1944), (6, 600, 128, 0): (2003, 1933), (6, 768, 128, 0): (2097, 2299),
    (6, 1003, 128, 0): (2633, 2959), (6, 1200, 128, 0): (3365, 3694),
    (6, 1500, 128, 0): (4053, 4449), (6, 2300, 128, 0): (6180, 6767), (7, 64, 128, 0): (736, 787),
    (7, 256, 128, 0): (784, 902), (7, 257, 128, 0): (1386, 1197), (7, 300, 128, 0): (1378, 1217),
    (7, 400, 128, 0): (1385, 1603), (7, 513, 128, 0): (2026, 1948), (7, 600, 128, 0): (2055, 2007),
    (7, 768, 128, 0): (2107, 2342), (7, 1003, 128, 0): (2668, 3036),
    (7, 1200, 128, 0): (3435, 3728), (7, 1500, 128, 0): (4113, 4491),
    (7, 2300, 128, 0): (6281, 6775), (4, 600, 128, 16): (1455, 1438),
    (5, 600, 128, 16): (1491, 1550), (7, 600, 128, 16): (1610, 1655),
}


def test_fused_choice_against_measured_times(route):
    """The faster of the two, within the 4.5 % by which two runs of one size
    on one route differ here (K=5, 512 sequences, T = 2: 1339 and 1401 us)."""
    got = route([("f", K, MAX_T[K], n, NCU, p, p + m if m and p + m < 256 else 256, ROW_BYTES[K])
                 for K, n, p, m in ROUTES])
    for (key, us), fused in zip(ROUTES.items(), got):
        assert us[int(fused)] <= 1.045 * min(us), (key, us, fused)


def test_fused_only_where_rounds_count(route):
    """Not up to one sequence per CU, nor from 16; any CU count is taken."""
    for K in MAX_T:
        for ncu in (1, 3, NCU):
            ns = [1, ncu, 16 * ncu, 40 * ncu]
            assert route([("f", K, MAX_T[K], n, ncu, 128, 256, ROW_BYTES[K]) for n in ns]) == [0] * 4
    assert route([("f", 4, 4, 5, 0, 128, 256, 2048)]) in ([0], [1])
