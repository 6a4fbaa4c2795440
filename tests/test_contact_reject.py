"""The cheap rejections of the repulsion items (csrc/contact_reject.h), compiled for the CPU:
whatever they reject, the full sign tests reject too, over random, grazing, parallel,
degenerate, tiny, huge and non-finite edge and vertex-face pairs; and they reject most of what
fails."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "xrtailor_amd" / "csrc"

DRIVER = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include "contact_reject.h"
using namespace xrt::cm;
static std::mt19937_64 gen(12345);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); }
static double Nm() { return std::normal_distribution<double>()(gen); }
struct P { double x, y, z; };
static P R(double s) { return P{s * Nm(), s * Nm(), s * Nm()}; }
static P Add(P a, P b, double s = 1) { return P{a.x + s * b.x, a.y + s * b.y, a.z + s * b.z}; }
static F3 F(P a) { return F3{float(a.x), float(a.y), float(a.z)}; }
int main(int argc, char** argv) {
  const long n = atol(argv[1]);
  long open_ee = 0, fail_ee = 0, rej_ee = 0, open_vf = 0, fail_vf = 0, rej_vf = 0, pass_ee = 0, pass_vf = 0;
  const float special[8] = {0.0f, -0.0f, NAN, INFINITY, -INFINITY, 1e-42f, 3e38f, -1e20f};
  for (long i = 0; i < n; ++i) {
    const int kind = static_cast<int>(i % 9);
    const double scale = std::pow(10.0, U(-8, 4)), off = kind == 7 ? std::pow(10.0, U(-2, 3)) * scale : 0.0;
    P o = R(off);
    P x0 = R(scale), e = R(scale), x1, y0, y1, y2;
    const double tiny = std::pow(10.0, U(-9, 0));
    P f = R(scale);
    x1 = Add(x0, e);
    if (kind == 1 || kind == 5) f = Add(P{e.x * U(-2, 2), e.y, e.z}, R(scale), tiny);  // nearly parallel
    if (kind == 5) f = Add(P{0, 0, 0}, Add(e, R(scale), tiny), U(-2, 2));
    y0 = R(scale);
    if (kind == 2 || kind == 5) {  // the lines cross near an end of a segment, at a small distance
      const double s = std::round(U(0, 1)) + tiny * Nm(), t = U(-0.1, 1.1);
      y0 = Add(Add(Add(x0, e, s), f, -t), R(scale), 0.1 * tiny);
    }
    if (kind == 3) {  // one plane
      x0.y = x1.y = y0.y = 0.1 * scale;
      f.y = 0;
    }
    if (kind == 4) y0 = Add(x0, R(scale), tiny);  // nearly shared vertex
    if (kind == 8) {  // all in a line but for tiny, apart or overlapping, of unlike lengths
      f = Add(P{0, 0, 0}, Add(e, R(scale), tiny), std::pow(10.0, U(-4, 4)));
      y0 = Add(Add(x0, e, U(-3, 3)), R(scale), tiny * std::pow(10.0, U(-3, 0)));
    }
    y1 = Add(y0, f);
    y2 = Add(y0, R(scale));
    if (kind == 6) y2 = Add(y0, Add(f, R(scale), tiny), U(-1, 2));  // sliver
    F3 p[5] = {F(Add(x0, o)), F(Add(x1, o)), F(Add(y0, o)), F(Add(y1, o)), F(Add(y2, o))};
    if (i % 97 == 0) (&p[gen() % 5].x)[gen() % 3] = special[gen() % 8];
    if (kind == 2 && i % 3 == 0) p[2] = p[0];
    float4 num;
    const int2 a = make_int2(0, 1), b = make_int2(2, 3);
    const bool ee = EESigns(a, b, p[0], p[1], p[2], p[3], false, Nz(S(p[1], p[0])), Nz(S(p[3], p[2])), num);
    const bool er = EeReject(p[0], p[1], p[2], p[3]);
    if (ee && er) { printf("EE rejected but passes, kind %d case %ld\n", kind, i); return 1; }
    if (er && EESigns(b, a, p[2], p[3], p[0], p[1], false, Nz(S(p[3], p[2])), Nz(S(p[1], p[0])), num)) {
      printf("EE rejected but passes the other way round, kind %d case %ld\n", kind, i);
      return 1;
    }
    pass_ee += ee; fail_ee += !ee; rej_ee += er; open_ee += !er && !ee;
    // the vertex near an edge or a corner of the face, or anywhere
    P v = x0;
    if (kind == 2 || kind == 4 || kind == 6) {
      const double s = U(-0.2, 1.2), t = (gen() & 1 ? 0.0 : 1.0 - s) + tiny * Nm();
      v = Add(Add(Add(y0, f, s), Add(y2, y0, -1), t), R(scale), tiny);
    }
    p[0] = i % 97 == 0 ? p[0] : F(Add(v, o));
    const int4 tr = make_int4(1, 2, 3, 0);
    const bool vf = VfSigns(0, tr, false, p[0], p[2], p[3], p[4], num);
    const bool vr = VfReject(p[0], p[2], p[3], p[4]);
    if (vf && vr) { printf("VF rejected but passes, kind %d case %ld\n", kind, i); return 1; }
    pass_vf += vf; fail_vf += !vf; rej_vf += vr; open_vf += !vr && !vf;
  }
  printf("EE pass %ld fail %ld rejected %ld open %ld; VF pass %ld fail %ld rejected %ld open %ld\n",
         pass_ee, fail_ee, rej_ee, open_ee, pass_vf, fail_vf, rej_vf, open_vf);
  // (half of the kinds graze on purpose, and scales below 1e-7 are under the error's floor)
  return rej_ee > 0.7 * fail_ee && rej_vf > 0.7 * fail_vf && pass_ee > n / 50 && pass_vf > n / 50 ? 0 : 2;
}
"""


def test_rejected_items_never_pass_the_full_test(tmp_path):
    (tmp_path / "main.cpp").write_text(DRIVER)
    exe = tmp_path / "reject"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{CSRC}", str(tmp_path / "main.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe), "4000000"], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
