"""Index arithmetic of the kernels at the ends of the ranges that a context accepts
(2^20 functions in a molecule), compiled for the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ENG = os.path.join(ROOT, "planck-refactored_amd", "csrc", "engine")


def _run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include "eri_common.h"\nint main() {\n%s\nreturn 0; }\n' % body)
    # the undefined-behaviour sanitizer ends the program on an integer overflow
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-w",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + ENG, str(src), "-o", str(exe)], check=True)
    return [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]


def test_matrix_elements(tmp_path):
    cases = [(0, 1, 0), (46340, 46341, 46340), (46341, 46342, 7), (65535, 65536, 65535), (65536, 70000, 69999),
             ((1 << 20) - 1, 1 << 20, (1 << 20) - 1)]
    got = _run(tmp_path, "".join('std::printf("%%zu\\n", pk::elem(%d, %d, %d));\n' % c for c in cases))
    assert got == [r * nb + c for r, nb, c in cases]


def test_ket_positions_at_the_end_of_a_full_list(tmp_path):
    """A wave looks two groups ahead: past the end of the list by up to the turns of
    four waves of eight groups of 21 kets."""
    end = (1 << 31) - 1
    cases = [(0, 0, 1), (5, 3, 9), (5, 3, 8), (end - 1, 0, end), (end - 1, 20, end), (end + 2 * 4 * 8 * 21, 20, end)]
    got = _run(tmp_path, "".join('std::printf("%%u\\n", pk::ket_pos(%du, %du, %du));\n' % c for c in cases))
    assert got == [min(g + s, e - 1) for g, s, e in cases]
