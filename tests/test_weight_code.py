"""The library's own functions that decide when a pair's weight is exactly 1.0
(score_amd/csrc/gm_weight.h), compiled for the host: the device's disorientation against
the largest of Grimmer's 24 candidates, bit for bit, and the threshold against the
weights of all angles and pairs it covers."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "gm_weight.h"
#include "score_orient.h"

static uint64_t s = 88172645463325252ull;
static uint64_t nx() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }
static double ur() { return (double)(nx() >> 11) * (1.0 / 9007199254740992.0); }
static double gauss() { return sqrt(-2.0 * log(1.0 - ur())) * cos(2.0 * kPi * ur()); }
static void unit(double *q) {
    double n = 0.0;
    for (int i = 0; i < 4; i++) { q[i] = gauss(); n += q[i] * q[i]; }
    for (int i = 0; i < 4; i++) q[i] /= sqrt(n);
}
static double weight(const score_gm_params &p, double th) {
    return 1.0 - (p.rh_cut * exp(-1.0 * p.rh_trans * pow((th / kLagbHagb), p.rh_exponent)));
}

int main(int argc, char **argv) {
    const double fac = 1.0 / sqrt(2.0);
    /* the disorientation: random, near, equal and coarse pairs */
    for (long k = 0; k < 400000; k++) {
        double p[4], q[4];
        unit(p);
        unit(q);
        if (k % 4 == 1) for (int i = 0; i < 4; i++) q[i] = p[i] + 1e-7 * gauss();
        if (k % 4 == 2) memcpy(q, p, sizeof(q));
        if (k % 4 == 3) for (int i = 0; i < 4; i++) { p[i] = rint(p[i] * 4.0) / 4.0; q[i] = rint(q[i] * 4.0) / 4.0; }
        const double a = grimmer_omega(p, q, fac), b = score_orient::disori_omega(p, q);
        if (memcmp(&a, &b, sizeof(a))) { printf("omega %a %a\n", a, b); return 1; }
    }
    /* the threshold */
    score_gm_params p;
    memset(&p, 0, sizeof(p));
    p.mobility_model = SCORE_GM_MOB_ROLLETTHOLM;
    long used = 0, below = 0;
    for (int k = 0; k < 600; k++) {
        if (k == 0) { p.rh_cut = 0.9; p.rh_trans = 5.0; p.rh_exponent = 9.0; }
        else if (k == 1) { p.rh_cut = 1.0; p.rh_trans = 3.0; p.rh_exponent = 4.0; }
        else {
            p.rh_cut = pow(10.0, -12.0 + 18.0 * ur());
            p.rh_trans = pow(10.0, -2.0 + 4.5 * ur());
            p.rh_exponent = pow(10.0, -0.5 + 3.7 * ur());
        }
        const double om = rh_omega_threshold(p);
        if (om < 0.0) {
            if (k < 2) { printf("no threshold for %g %g %g\n", p.rh_cut, p.rh_trans, p.rh_exponent); return 1; }
            continue;
        }
        used++;
        /* every angle from the threshold's on: close by in small steps, then to pi */
        const double th0 = 2.0 * acos(om);
        for (int i = 0; i < 2000; i++) {
            const double th = i < 1000 ? th0 + i * 1e-9 : th0 + (kPi - th0) * (i - 1000) / 999.0;
            if (weight(p, th) != 1.0) { printf("angle %.17g: %.17g\n", th, weight(p, th)); return 1; }
        }
        for (int i = 0; i < 200; i++) {
            double a[4], b[4];
            unit(a);
            unit(b);
            if (grimmer_omega(a, b, fac) > om) continue;
            below++;
            if (weight(p, score_orient::disori_angle(a, b)) != 1.0) { printf("pair\n"); return 1; }
        }
    }
    /* refused: other models and settings that are no weight's */
    for (int k = 0; k < 4; k++) {
        p.rh_cut = k == 0 ? -0.9 : 0.9;
        p.rh_trans = k == 1 ? -5.0 : 5.0;
        p.rh_exponent = k == 2 ? -9.0 : 9.0;
        p.mobility_model = k == 3 ? SCORE_GM_MOB_SEBALDGOTTSTEIN : SCORE_GM_MOB_ROLLETTHOLM;
        if (rh_omega_threshold(p) != -1.0) { printf("accepted %d\n", k); return 1; }
    }
    printf("%ld %ld\n", used, below);
    return 0;
}
"""


def test_disorientation_and_threshold(tmp_path):
    cxx = shutil.which(os.environ.get("CXX", "g++"))
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(HARNESS)
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "score_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), str(src), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    used, below = (int(v) for v in out.stdout.split())
    assert used >= 100 and below >= 1000
