"""K-split rules of the Gram products (csrc/gram_rules.hpp), on the CPU.

U^T U, U^T X of two blocks and the FP32 product run different kernels at the
same size, so what was measured on one does not decide for another.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rsdft_develop_amd", "csrc")
SAME, PAIR, F32 = 0, 1, 2


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("rules") / "gram_rules")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, os.path.join(HERE, "gram_rules.cpp"),
                    "-o", exe], check=True)

    def ask(*lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
        assert r.returncode == 0
        return [[int(v) for v in a.split()] for a in r.stdout.splitlines()]

    return ask


@pytest.mark.parametrize("nb", [20, 96, 97, 128, 129, 160, 192, 193, 480])
def test_tuned_splits_stay_with_the_kernel_that_was_timed(rules, nb):
    N = 72 ** 3
    default = [c[0] for c in rules(*[f"chunk {N} {nb} {f}" for f in (SAME, PAIR, F32)])]
    tuned = [c[0] for c in rules(f"tune {N} {nb} 0 4567", *[f"chunk {N} {nb} {f}" for f in (SAME, PAIR, F32)])]
    own_pair, = rules(f"own {nb} {PAIR}")[0]
    assert tuned == [0, 4567, default[F32] if own_pair else 4567]
    # another grid or band count, and a second tuning
    other = rules(f"tune {N} {nb} 0 4567", f"chunk {N + 1} {nb} {SAME}", f"chunk {N} {nb + 1} {PAIR}")
    assert other == rules(f"chunk {N + 1} {nb} {SAME}", f"chunk {N} {nb + 1} {PAIR}")
    assert rules(f"tune {N} {nb} 0 4567", f"tune {N} {nb} 999 0", f"chunk {N} {nb} {SAME}",
                 f"chunk {N} {nb} {PAIR}") == [[999], [0]]


@pytest.mark.parametrize("nb", [20, 77, 112, 160, 192])
@pytest.mark.parametrize("form", [SAME, PAIR])
def test_the_untuned_split_is_always_a_candidate(rules, nb, form):
    for N in (36 ** 3, 72 ** 3):
        (d,), first = rules(f"chunk {N} {nb} {form}", f"cand {N} {nb} {form}")
        again, = rules(f"tune {N} {nb} 0 0", f"cand {N} {nb} {form}")
        assert d in first and again == first and len(set(first)) == len(first)
