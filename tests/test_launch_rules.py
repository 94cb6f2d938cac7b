"""The rules that choose a kernel's form by the number of block parts (zeno_amd/csrc/launch_rules.h, plain
C++): what the autotuner found is what is launched, for any number of parts."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r"""
#include <cstdio>
#include "launch_rules.h"
int main() {
    long parts, n;
    int flip, move, update, wave;
    while (std::scanf("%ld %ld %d %d %d %d", &parts, &n, &flip, &move, &update, &wave) == 6)
        std::printf("%d %d %d\n", zmpm::g2p_move_threads(parts, n, flip != 0, move),
                    zmpm::g2p_update_threads(parts, n, flip != 0, update), (int)zmpm::p2g_one_wave(parts, n, wave));
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("rules")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "zeno_amd", "csrc"),
                    str(d / "main.cpp"), "-o", str(d / "rules")], check=True, capture_output=True, text=True)

    def ask(queries):
        text = "".join("%d %d %d %d %d %d\n" % q for q in queries)
        out = subprocess.run([str(d / "rules")], input=text, check=True, capture_output=True, text=True).stdout
        return [tuple(int(w) for w in line.split()) for line in out.splitlines()]

    return ask


PARTS = (1, 180, 512, 513, 1535, 1536, 16384, 80000)


def test_the_tuned_choice_is_launched(rules):
    cases = [(p, p * k, flip, move, update, wave) for p in PARTS for k in (10, 60, 400) for flip in (0, 1)
             for move in (64, 256) for update in (64, 256) for wave in (0, 1)]
    assert rules(cases) == [(c[3], c[4], c[5]) for c in cases]


def test_untuned_sizes_exist(rules):
    """Sizes that the launches know: 512 threads only for the update of the APIC transfer."""
    cases = [(p, p * k, flip, 0, 0, -1) for p in PARTS for k in (10, 60, 400) for flip in (0, 1)]
    for c, (move, update, wave) in zip(cases, rules(cases)):
        assert move in (64, 256) and update in ((64, 256) if c[2] else (64, 256, 512)) and wave in (0, 1)
        assert c[0] >= 1536 or (move, wave) == (256, 0)


def test_one_wave_p2g_only_for_small_blocks(rules):
    """Blocks of 60 particles on average, many of more than 64, are faster without it."""
    assert [r[2] for r in rules([(77514, 77514 * k, 0, 0, 0, -1) for k in (20, 48, 49, 60)])] == [1, 1, 0, 0]
    assert [r[2] for r in rules([(32767, 32767 * k, 0, 0, 0, -1) for k in (36, 37)])] == [1, 0]
    assert [r[2] for r in rules([(p, p * 20, 0, 0, 0, -1) for p in (16383, 16384)])] == [0, 1]
