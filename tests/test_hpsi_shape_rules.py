"""Launch-shape rules of the H psi kernels (csrc/hpsi_shape.hpp), on the CPU.

The rules are host code without a HIP call; tests/hpsi_shape_rules.cpp puts
them behind a line protocol.  A shape is what the launch code takes: it has
to fit the kernel it is for.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rsdft_develop_amd", "csrc")
FIELDS = ("ry", "ty", "zlen", "chunk", "bt", "rx", "psplit", "fits")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("rules") / "hpsi_shape_rules")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "hpsi_shape_rules.cpp"), "-o", exe], check=True)

    def ask(lines, raw=False):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, f"exit {r.returncode} after {len(r.stdout.splitlines())} of {len(lines)} answers"
        rows = [list(map(int, a.split())) for a in r.stdout.splitlines()]
        return rows if raw else [dict(zip(FIELDS, a)) for a in rows]

    return ask


def _resolve(n, md=6, size=8, nb=64, nonlocal_=1, analytic=1, nseg=2000, max_chunk=0, **shape):
    s = {k: shape.get(k, 0) for k in FIELDS[:-1]}
    return (f"resolve {n[0]} {n[1]} {n[2]} {md} {size} {nb} {nonlocal_} {analytic} {nseg} "
            f"{s['ry']} {s['ty']} {s['zlen']} {s['chunk']} {s['bt']} {s['rx']} {s['psplit']} {max_chunk}")


@pytest.mark.parametrize("size", [8, 4])
def test_derived_shapes_fit_ordinary_grids(rules, size):
    """Rows of 16 to 128 points with every finite-difference order whose halo
    four elements a thread cover."""
    grids = [(n1, n2, n3) for n1 in range(16, 129, 7) for n2 in (9, 24, 45, 108) for n3 in (3, 36, 99)]
    ask = [(n, md, nb) for n in grids for md in (1, 4, 6, 8) for nb in (1, 37, 480)]
    for (n, md, nb), sh in zip(ask, rules([_resolve(n, md=md, size=size, nb=nb) for n, md, nb in ask])):
        assert sh["fits"] and 1 <= sh["zlen"] <= n[2] and 1 <= sh["chunk"] <= nb, (n, md, nb, sh)


def test_rows_too_long_for_whole_ones_go_in_parts(rules):
    """FP64 rows above 170 points (md 6): three whole rows no longer stage
    their halo in 512 threads, so every such row is split, odd ones too."""
    ask = [((n1, n2, 20), md, ry) for n1 in (171, 172, 180, 192, 255, 256, 320, 511, 512) for n2 in (5, 24, 36)
           for md in (6, 7) for ry in (0, 1, 2)]
    for (n, md, ry), sh in zip(ask, rules([_resolve(n, md=md, ry=ry) for n, md, ry in ask])):
        assert sh["fits"] and sh["ry"] == 2 and n[0] * sh["ty"] // 2 > 512, (n, md, ry, sh)


@pytest.mark.parametrize("n,md,size", [((171, 24, 24), 6, 4), ((192, 25, 24), 5, 4), ((129, 24, 24), 8, 8),
                                       ((513, 8, 8), 6, 8)])
def test_rows_that_no_kernel_takes_have_no_tile(rules, n, md, size):
    sh, = rules([_resolve(n, md=md, size=size)])
    assert sh["ty"] == 0 and not sh["fits"]


@pytest.mark.parametrize("n,size,ty,rx", [
    ((72, 72, 72), 4, 10, 1), ((72, 72, 72), 4, 14, 1),  # no divisor of n2: not for the pair kernel
    ((72, 72, 72), 4, 12, 2), ((72, 72, 72), 4, 9, 2),   # divisors: the pair kernel, 9 with one row a thread
    ((75, 38, 70), 4, 12, 1),                            # odd rows
    ((108, 108, 108), 8, 4, 1), ((108, 108, 108), 8, 8, 1), ((144, 144, 144), 8, 3, 1),  # beside rows in parts
    ((36, 36, 36), 8, 18, 1), ((36, 36, 36), 8, 9, 1),
])
def test_tile_rows_that_a_caller_sets_are_used(rules, n, size, ty, rx):
    """With ry and rx left to the rules; a second answer with all three set
    is the same."""
    for nb in (2, 160):
        sh, = rules([_resolve(n, size=size, ty=ty, nb=nb)])
        assert (sh["ty"], sh["rx"], sh["fits"]) == (ty, rx, 1), sh
        again, = rules([_resolve(n, size=size, ty=ty, nb=nb, ry=sh["ry"], rx=sh["rx"])])
        assert again == sh


def test_tile_rows_that_fit_no_kernel_are_replaced(rules):
    for size in (8, 4):
        sh, derived = rules([_resolve((72, 72, 72), size=size, ty=97), _resolve((72, 72, 72), size=size)])
        assert sh == derived and sh["fits"]


SHAPE = ("ry", "ty", "zlen", "chunk", "bt", "order", "rx", "proj", "plds", "psplit")


def _search(rules, n, size, nb, analytic=1, ry=0, rx=0, psplit=0, chunk=0, ty=0, cold=0):
    row, = rules([f"search {n[0]} {n[1]} {n[2]} 6 {size} {nb} 1 {analytic} 2000 {ry} {rx} {psplit} {chunk} {ty} {cold}"], raw=True)
    shapes = [dict(zip(SHAPE, row[1 + 10 * k:11 + 10 * k])) for k in range(row[0] + 1)]
    return shapes[0], shapes[1:]


@pytest.mark.parametrize("n,size", [((36, 36, 36), 4), ((72, 72, 72), 4), ((72, 72, 72), 8), ((108, 108, 108), 8),
                                    ((75, 38, 70), 4), ((75, 38, 70), 8)])
def test_autotuner_times_every_value_once(rules, n, size):
    """One and two rows a thread, one and two points a thread where the pair
    kernel fits, all piece counts; no shape twice but the derived one, which
    is the first."""
    best, timed = _search(rules, n, size, 40)
    derived, = rules([_resolve(n, size=size, nb=40)])
    assert all(timed[0][k] == derived[k] for k in FIELDS[:-1]) and best == timed[0]
    again = [t for t in timed[1:] if t != timed[0]]
    assert len(again) == len(timed) - 2 and len({tuple(t.values()) for t in again}) == len(again)
    pair = size == 4 and n[0] % 2 == 0
    assert {(t["rx"], t["ry"]) for t in timed} == {(x, y) for x in ((1, 2) if pair else (1,)) for y in (1, 2)}
    assert {t["psplit"] for t in timed} == {1, 2, 4, 8}
    assert {t["bt"] for t in timed} == {4, 8, 16, 20, 32} and {t["proj"] for t in timed} == {0, 1, 2}


@pytest.mark.parametrize("want", [dict(rx=1), dict(rx=1, ry=1), dict(rx=2, ry=1), dict(psplit=1), dict(psplit=8, rx=1),
                                  dict(chunk=20)])
def test_autotuner_finds_what_is_fast(rules, want):
    best, _ = _search(rules, (72, 72, 72), 4, 160, **want)
    assert all(best[k] == v for k, v in want.items()), best


@pytest.mark.parametrize("n,nb", [((72, 72, 72), 160), ((108, 108, 108), 480), ((144, 144, 144), 1100)])
@pytest.mark.parametrize("limit", [1, 10, 37, 5000])
@pytest.mark.parametrize("analytic", [0, 1])
def test_z_runs_and_apply_waves_suit_the_chunk_a_scratch_holds(rules, n, nb, limit, analytic):
    """A caller's scratch bounds the bands of a chunk: the shape is the one
    for chunks of that many bands, in chunks of equal size."""
    free, sh = rules([_resolve(n, nb=nb, analytic=analytic), _resolve(n, nb=nb, analytic=analytic, max_chunk=limit)])
    assert sh["chunk"] <= limit and -(-nb // sh["chunk"]) == -(-nb // min(limit, free["chunk"]))
    same, = rules([_resolve(n, nb=nb, analytic=analytic, chunk=sh["chunk"])])
    assert sh == same
    given, = rules([_resolve(n, nb=nb, analytic=analytic, chunk=7, zlen=5, bt=8, max_chunk=limit)])
    assert (given["zlen"], given["bt"], given["chunk"] <= min(7, limit)) == (5, 8, True)


@pytest.mark.parametrize("n,rows", [
    ((72, 18, 72), 1), ((80, 17, 40), 1), ((84, 16, 84), 1), ((78, 27, 60), 1),  # two full rows pad too much
    ((84, 25, 60), 2), ((74, 25, 60), 2),                                        # ... and one row's halo spills
    ((144, 9, 72), 1), ((108, 22, 72), 1), ((72, 9, 72), 1),                     # parts would pad too much
    ((96, 23, 60), "parts"), ((108, 13, 72), "parts"), ((108, 108, 108), "parts"), ((144, 144, 144), "parts"),
    ((72, 72, 72), 2), ((75, 38, 70), 2), ((99, 99, 99), 1),                     # little padding; odd rows
])
def test_rows_a_thread_where_tiles_pad(rules, n, rows):
    """FP64, each choice being the faster one where they were measured."""
    sh, = rules([_resolve(n, nb=300)])
    parts = n[0] * sh["ty"] // sh["ry"] > 512
    assert sh["fits"] and ("parts" if parts else sh["ry"]) == rows, sh


@pytest.mark.parametrize("n,size", [((72, 72, 72), 8), ((72, 72, 72), 4), ((108, 108, 108), 8)])
def test_a_slow_first_timing_does_not_decide(rules, n, size):
    """The derived shape is the fastest; its first timing, on an idle GPU, is not."""
    derived, = rules([_resolve(n, size=size, nb=160)])
    best, timed = _search(rules, n, size, 160, cold=1, **{k: derived[k] for k in ("ry", "rx", "psplit", "chunk", "ty")})
    assert best == timed[0]


@pytest.mark.parametrize("n,size", [((72, 72, 72), 8), ((36, 36, 36), 4)])
def test_timings_that_are_low_once_do_not_move_the_shape(rules, n, size):
    """Every third timing comes out a little low: a candidate has to win again."""
    derived, = rules([_resolve(n, size=size, nb=160)])
    best, timed = _search(rules, n, size, 160, cold=3, **{k: derived[k] for k in ("ry", "rx", "psplit", "chunk", "ty")})
    assert best == timed[0]
