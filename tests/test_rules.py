"""Which form a call takes (redzone_amd/csrc/rz_rules.hpp), through a small host
program: over whole ranges of sizes, without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "rules_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", exe, os.path.join(ROOT, "tests", "native", "rules_host.cpp")],
                   check=True)

    def run(questions):
        text = "\n".join(" ".join(str(x) for x in q) for q in questions)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=60).stdout.split("\n")
        assert len(out) == len(questions) + 1
        return out[:-1]

    return run


def test_partition_marks_read_the_removals_a_bounded_number_of_times(ask):
    """Marks by ranges read all removals once per range: never more than 24 of
    them, up to the largest list."""
    sizes = [1 << b for b in range(10, 31)] + [(1 << 29) + 1, 3 << 28, (1 << 31) - 1]
    qs = [("part", n, max(1, int(n / f))) for n in sizes for f in (1.01, 1.5, 2, 3.9, 4, 4.1, 11.9, 12, 12.1, 100)]
    kinds = set()
    for q, a in zip(qs, ask(qs)):
        kinds.add(a.split()[0])
        assert not a.startswith("ranges") or int(a.split()[1]) <= 24, (q, a)
        if q[1] > 1 << 29:
            assert a == "atomic", (q, a)
    assert kinds == {"atomic", "ranges", "buckets"}


def test_partition_marks_at_the_edges(ask):
    assert ask([("part", 1 << 29, 1 << 27), ("part", (1 << 29) + 1, 1 << 27), ("part", 3 << 20, 1 << 19),
                ("part", (3 << 20) + 1, 1 << 19), ("part", 12 << 15, 1 << 15), ("part", (12 << 15) + 1, 1 << 15),
                ("part", 12 * ((1 << 19) - 1), (1 << 19) - 1), ("part", 1 << 28, (1 << 19) - 1),
                ("part", 1 << 28, 1 << 19)]) == \
        ["buckets", "atomic", "ranges 12", "buckets", "ranges 3", "atomic", "ranges 24", "atomic", "buckets"]


def test_dense_lists_that_windows_would_read_too_often(ask):
    """The dense form writes through windows up to half a GiB of head (1 GiB of
    16-byte items) and in denser lists above; sparse lists of several GiB never do."""
    assert ask([("dense", 4, 1 << 27, 1 << 26), ("dense", 4, 1 << 28, 1 << 27), ("dense", 4, 1 << 28, 1 << 26),
                ("dense", 4, (1 << 31) - 1, 1 << 24), ("dense", 4, (1 << 31) - 1, 9 << 27), ("dense", 8, 1 << 26, 1 << 24),
                ("dense", 8, 1 << 29, 1 << 24), ("dense", 8, 1 << 29, 1 << 28), ("dense", 16, 1 << 26, 1 << 24),
                ("dense", 16, 1 << 30, 1 << 24), ("dense", 16, 1 << 30, 3 << 28), ("dense", 16, 1 << 30, (3 << 28) - 1),
                ("dense", 16, 1 << 28, 3 << 26)]) == \
        ["windows", "windows", "stores 12", "stores 12", "windows", "windows", "stores 9", "stores 11", "windows",
         "stores 9", "windows", "stores 9", "windows"]
    for esz in (4, 8, 16):
        sizes = [int(2 ** (b / 4)) for b in range(60, 125)]
        qs = [("dense", esz, n, int(n * f)) for n in sizes for f in (.001, .01, .1, .3, .34, .5, .9)]
        for (_, e, n, k), a in zip(qs, ask(qs)):
            if n * e > 1 << 33 and 10 * k <= n:
                assert a.startswith("stores"), (e, n, k)
            if (n - k) * e <= 1 << 29:
                assert a == "windows", (e, n, k)


def test_dense_shapes_count_every_kernels_lds(ask):
    """A shape is refused before anything is launched where one of its kernels does
    not fit: with 64 KiB a workgroup, every shape that writes whole windows.  All
    installed and candidate shapes fit 160 KiB."""
    small = [("lds", e, 256, 4, s, (1 << 17).bit_length() - 1 - {4: 2, 8: 3, 16: 4}[e]) for e in (4, 8, 16) for s in (0, 1)]
    assert [int(a) > 65536 for a in ask(small)] == [True, False, True, False, True, True]
    full = [("lds", e, wg, it, s, 17 - {4: 2, 8: 3, 16: 4}[e]) for e, wg, it in
            ((4, 1024, 8), (8, 1024, 8), (16, 1024, 4), (16, 512, 8), (4, 512, 8)) for s in (0, 1)]
    assert all(int(a) <= 163840 for a in ask(full))
    assert int(ask([("lds", 16, 1024, 8, 0, 13)])[0]) > 163840  # refused, as it was
    assert ask([("lds", 4, 256, 4, 0, 10), ("lds", 4, 256, 4, 0, 15)]) == ["59392", "135168"]


def test_gather_forms(ask):
    """Two passes for fewer than an eighth kept and in the band of 4-byte lists, never
    from 2^22 kept items on."""
    M = 1000000
    assert ask([("gather", 4, 8 * 1000, 1000), ("gather", 4, 8 * 1000 + 1, 1000), ("gather", 4, 4 * M, 3500000 - 1),
                ("gather", 4, 4 * M, 3500000), ("gather", 8, 4 * M, 3500000), ("gather", 4, 22 * M, 3 * M),
                ("gather", 4, 22 * M + 1, 3 * M), ("gather", 4, 10 * M, 1 << 22), ("gather", 4, 10 * M, (1 << 22) - 1),
                ("gather", 16, 1 << 26, 1 << 22), ("gather", 8, 1 << 23, 1 << 22), ("gather", 4, 1 << 28, 1 << 26),
                ("gather", 4, (1 << 28) - 1, 1 << 26), ("gather", 4, 1 << 28, (3 << 23) - 1)]) == \
        ["one 0", "two", "one 0", "two", "one 0", "two", "one 0", "one 0", "two", "one 32", "one 0", "one 16", "one 0",
         "one 0"]


def test_installed_shapes_are_the_tuners():
    """Every shape of the installed table is one that the tuner times, so tuning a
    context again can find it."""
    import redzone_amd as rz

    plain = {c.as_tuple() for c in rz.Context.candidates()}
    batch = {c.as_tuple() for c in rz.Context.candidates(batch=True)}
    for line in open(os.path.join(ROOT, "redzone_amd", "tuned_gfx950.txt")):
        words = line.split()
        if words and words[0] == "plain":
            assert tuple(map(int, words[3:])) in plain, line
        elif words and words[0] == "batch":
            assert tuple(map(int, words[1:])) in batch, line
