"""Jumping ahead in the RANLUX stream (csrc/ranlux_jump.h) against advancing it step by step,
on the CPU: the chunk lengths of the seed table from the smallest mesh to the largest (1 to
171 advances of 202 steps), from fresh and from later states, to the bit."""
import os
import subprocess


HERE = os.path.dirname(os.path.abspath(__file__))
CODE = r"""
#include <cstdio>
#include <cstring>
#include "ranlux_jump.h"
int main() {
  const unsigned long seeds[] = {0, 1, 2, 5001, 4101, 2147483647ul, 4294967295ul};
  const unsigned advances[] = {1, 2, 3, 16, 17, 27, 43, 128, 171};
  long bad = 0, n = 0;
  for (unsigned long s : seeds)
    for (unsigned adv : advances) {
      Ranlxd1 serial, jumped;
      serial.seed(s);
      const rlx::Num jump = rlx::step_power(202ull * adv);
      rlx::Num X = rlx::from_state(serial);
      for (int chunk = 0; chunk < 40; chunk++) {
        for (unsigned a = 0; a < adv; a++) serial.advance();
        rlx::to_state(X = rlx::mul(X, jump), jumped);
        bad += memcmp(serial.y, jumped.y, sizeof serial.y) != 0 || serial.carry != jumped.carry;
        n++;
      }
      // and on from a state that the generator itself has reached
      X = rlx::mul(rlx::from_state(serial), jump);
      for (unsigned a = 0; a < adv; a++) serial.advance();
      rlx::to_state(X, jumped);
      bad += memcmp(serial.y, jumped.y, sizeof serial.y) != 0 || serial.carry != jumped.carry;
      n++;
    }
  printf("%ld of %ld states differ\n", bad, n);
  return bad || n != 7 * 9 * 41;
}
"""


def test_jumped_states_equal_serial_ones(tmp_path):
    (tmp_path / "t.cpp").write_text(CODE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(HERE, "..", "mg-picola-public_amd", "csrc"), "-o", str(tmp_path / "t"),
                    str(tmp_path / "t.cpp")], check=True)
    p = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout
