"""The quantisers' scale and quotients without a division (csrc/quotient.hip.h), compiled for the host, against IEEE division."""
import os
import subprocess
import textwrap

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llmmm_amd", "csrc")

PROGRAM = textwrap.dedent("""
    #include "quotient.hip.h"
    #include <cmath>
    #include <cstdint>
    #include <cstdio>
    #include <cstring>
    using namespace llmmm;
    static float    flt(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
    static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
    // rounded to three mantissa bits, to even: the e4m3 code of 2^-6 and above, up to the clamp
    static uint32_t code(float f) { const uint32_t u = bits(f); return (u + 0x7FFFF + ((u >> 20) & 1)) >> 20; }
    static float    estimate(float s, int ulps) { return flt(bits(1.0f / s) + ulps); }

    int main()
    {
      // scales: every mantissa at both ends of the range that is claimed and between, zero
      const int exponents[] = {-90, -89, -60, -1, 0, 8, 9, 100, 120, 126, 127};
      for (int e : exponents)
        for (uint32_t m = 0; m < 1u << 23; ++m) {
          const float a = flt((uint32_t)(e + 127) << 23 | m);
          if (bits(scale_of_amax(a)) != bits(a / 448.0f)) return printf("amax %a\\n", a), 1;
        }
      if (bits(scale_of_amax(0.0f)) != 0) return 2;

      // reciprocals: every mantissa, from the rounded one and its neighbours; where the result is not the rounded one, every quotient
      int off = 0, misrounded = 0;
      for (uint32_t m = 0; m < 1u << 23; ++m) {
        const float s = flt(127u << 23 | m);
        for (int ulps = -1; ulps <= 1; ++ulps) {
          const float y = refined_reciprocal(s, estimate(s, ulps));
          if (bits(y) == bits(1.0f / s)) continue;
          ++off;
          for (uint32_t k = 0; k < 1u << 23; ++k) {
            const float v = flt(127u << 23 | k), q = rounded_quotient(v, s, y);
            if (bits(q) == bits(v / s)) continue;
            ++misrounded;
            if (code(q) != code(v / s)) return printf("%a / %a\\n", v, s), 3;
          }
        }
      }
      if (off != 33 || misrounded != 3) return printf("%d reciprocals, %d quotients\\n", off, misrounded), 4;

      // quotients: values on and next to the boundaries of the 3-bit mantissa, scales over the range, both signs, zeros, NaN
      uint64_t st = 88172645463325252ull;
      for (int i = 0; i < 20000000; ++i) {
        st ^= st << 13, st ^= st >> 7, st ^= st << 17;
        const int   e    = (int)(st % 161) - 69;  // of the scale: -69 .. 91
        const float s    = flt((uint32_t)(e + 127) << 23 | (uint32_t)(st >> 8 & 0x7FFFFF));
        const int   qe   = (int)(st >> 31 & 31) % 19 - 10;  // of the quotient: -10 .. 8
        const float near = ldexpf(1.0f + (float)(2 * (st >> 36 & 7) + 1) / 16.0f, qe);
        float       v    = (st >> 40 & 3) ? (float)((double)near * (double)s) : flt((uint32_t)(qe + e + 127) << 23 | (uint32_t)(st >> 41));
        if (st >> 40 & 3) v = flt(bits(v) + (uint32_t)(st >> 44 & 7) - 3);
        if (st >> 63) v = -v;
        const float y = refined_reciprocal(s, estimate(s, (int)(st >> 48) % 3 - 1)), q = rounded_quotient(v, s, y);
        if (bits(q) != bits(v / s)) return printf("%a / %a = %a, %a\\n", v, s, v / s, q), 5;
        // a value too small for a code (below 2^-10 of the scale) keeps its sign and stays there
        const float t = flt(bits(v) & 0x80000000u | (uint32_t)(st >> 13) % (uint32_t)(e - 11 + 127) << 23 | (uint32_t)(st >> 20 & 0x7FFFFF));
        const float z = rounded_quotient(t, s, y);
        if (std::signbit(z) != std::signbit(t) || !(fabsf(z) <= 0x1p-10f)) return printf("%a / %a = %a\\n", t, s, z), 6;
      }
      const float y = refined_reciprocal(3.0f, estimate(3.0f, 0));
      if (bits(rounded_quotient(-0.0f, 3.0f, y)) != 0x80000000u || bits(rounded_quotient(0.0f, 3.0f, y)) != 0 || !std::isnan(rounded_quotient(NAN, 3.0f, y))) return 7;
      return 0;
    }
""")


def test_against_division(tmp_path):
    (tmp_path / "q.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "q")
    res = subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-Xarch_host", "-mfma", "-ffp-contract=off", "-std=c++17", "-Wno-unused-command-line-argument",
                          "-I", CSRC, "-o", exe, str(tmp_path / "q.cpp")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    res = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0, (res.returncode, res.stdout)
