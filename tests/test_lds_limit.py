"""The record of which devices took a kernel's dynamic LDS limit
(libcmol_amd/csrc/hip/lds_limit.h), compiled for the host: every device is
asked once, a refusal is reported and asked again."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "lds_limit.h"
#include <cstdio>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main()
{
    LdsLimit l, other;
    int asked = 0;
    bool accept = false;
    auto set = [&] { asked++; return accept; };
    CHECK(!l.raise(0, set) && asked == 1);   // refused: reported,
    CHECK(!l.raise(0, set) && asked == 2);   // and asked again
    accept = true;
    CHECK(l.raise(0, set) && asked == 3);
    CHECK(l.raise(0, set) && asked == 3);    // device 0 took it
    accept = false;
    CHECK(!l.raise(1, set) && asked == 4);   // device 1 is another matter
    CHECK(l.raise(0, set) && asked == 4);
    accept = true;
    CHECK(l.raise(63, set) && l.raise(63, set) && asked == 5);
    CHECK(l.raise(64, set) && l.raise(64, set) && asked == 7);   // past the record
    CHECK(l.raise(-1, set) && l.raise(-1, set) && asked == 9);   // unknown
    CHECK(other.raise(0, set) && asked == 10);                   // another kernel
    return 0;
}
"""


def test_every_device_is_asked_once_and_refusals_again(tmp_path):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text(SOURCE)
    inc = os.path.join(ROOT, "libcmol_amd", "csrc", "hip")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", inc, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout

