"""The path tracer's scheduling arithmetic (csrc/pt_schedule.h), compiled for the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cloudrendering-vulkan_amd", "csrc")


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    """Values of C++ expressions over the header, as Python integers."""
    d = tmp_path_factory.mktemp("schedule")

    def run(*exprs, before=""):
        src, exe = d / "s.cpp", d / "s"
        body = "".join(f'    printf("%lld\\n", (long long)({e}));\n' for e in exprs)
        src.write_text(f'#include <cstdio>\n#include "pt_schedule.h"\nusing namespace cr;\n{before}\nint main()\n{{\n{body}}}\n')
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
        return [int(v) for v in subprocess.run([str(exe)], capture_output=True, check=True, timeout=60).stdout.split()]

    return run


def test_workgroups(evaluate):
    cases = [(1, 1024, 1), (256, 1024, 1), (257, 1024, 2), (0, 1024, 1), (1 << 20, 1024, 1024), (1 << 20, 0, 1),
             # any number of items: as many as the chip holds
             (0xFFFFFFFF, 1024, 1024), (0xFFFFFFFFFFFFFFFF, 1024, 1024)]
    got = evaluate(*(f"pt_blocks({n}ull, {r})" for n, r, _ in cases))
    assert got == [w for _, _, w in cases]


def test_chunks(evaluate):
    lanes = 1024 * 256
    cases = [(1920 * 1080, 32, 4, 16, 16), (1920 * 1080, 8, 4, 16, 15), (256 * 256, 8, 4, 16, 1), (256 * 256, 256, 8, 4, 4),
             (1, 1, 8, 4, 1), (1 << 28, 0xFFFFFFFF, 8, 4, 4)]
    got = evaluate(*(f"pt_chunk({px}, {n}u, {lanes}, {per}, {most})" for px, n, per, most, _ in cases))
    assert got == [w for *_, w in cases]


def test_sample_room(evaluate):
    # a device with room for `free` samples; the attempts made are counted
    before = """
static int tries;
static long long room(unsigned long long want, unsigned long long least, unsigned long long had, unsigned long long free)
{
    tries = 0;
    return (long long)pt_sample_room(want, least, had, [&](uint64_t n) { tries++; return n <= free; });
}
"""
    cases = [((1000, 20, 0, 5000), 1000), ((1000, 20, 0, 1000), 1000), ((1000, 20, 0, 600), 500), ((1000, 20, 0, 30), 20),
             ((1000, 20, 0, 20), 20), ((1000, 20, 0, 19), 0), ((1000, 1000, 0, 999), 0),
             # what was held before is tried once it is the next smaller size
             ((1000, 20, 700, 700), 700), ((1000, 20, 700, 400), 350), ((1000, 20, 300, 300), 300), ((1000, 20, 300, 499), 300),
             ((1, 1, 0, 0), 0), ((1 << 28, 2, 0, 0), 0)]
    got = evaluate(*(f"room({w}u, {l}u, {h}u, {f}u)" for (w, l, h, f), _ in cases), before=before)
    assert got == [v for _, v in cases]
