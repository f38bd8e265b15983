"""The launch-shape rules (fhe-mamba_amd/csrc/launch_rules.hpp) over all shapes
they accept, on the CPU: every choice is a shape the kernel takes, and none
leaves wave slots to wavefronts without work or idle."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "fhe-mamba_amd", "csrc")
LDS = 160 * 1024  # a gfx950 compute unit's, and the most a workgroup may take
CUS = 256


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("rules") / "launch_rules_driver")
    subprocess.run([cxx, "-std=c++17", "-O1", "-I" + CSRC,
                    os.path.join(HERE, "launch_rules_driver.cpp"), "-o", exe], check=True,
                   capture_output=True)

    def ask(op, shapes):
        text = "\n".join(" ".join([op, *map(str, s)]) for s in shapes)
        out = subprocess.run([exe], input=text, capture_output=True, check=True, text=True).stdout
        rows = [tuple(map(int, line.split())) for line in out.splitlines()]
        assert len(rows) == len(shapes)
        return rows
    return ask


def lines_per_wave(s1):
    return 2 if s1 == 7 else 1


def test_middle_kernel_waves(rules):
    """Four waves at least (the kernel's unit) and no more than its launch
    bounds; LDS that fits; no form half of whose waves have no line; and, where
    a launch is more than a round of workgroups, none that keeps fewer waves on
    a compute unit than another."""
    shapes = [(s1, tiles, nsrc, ndst, LDS) for s1 in (7, 8, 9)
              for tiles in (64, 512, 768, 1024, 2048, 4096, 16384) for nsrc in range(1, 17)
              for ndst in (1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 24, 31, 45, 60)]
    for (s1, tiles, nsrc, ndst, _), (nw, *lds) in zip(shapes, rules("mid", shapes)):
        forms = {4: lds[0], 8: lds[1]}
        if s1 == 9:
            forms[16] = lds[2]
        per_simd = {7: 6, 8: 7, 9: 4}[s1]
        groups = {w: min(LDS // b, 4 * per_simd // w) for w, b in forms.items()}
        what = (s1, tiles, nsrc, ndst, nw)
        assert nw in forms and groups[nw] >= 1, what
        assert nw == 4 or max(nsrc, ndst) > nw // 2 * lines_per_wave(s1), what
        if max(nsrc, ndst) > 4 * lines_per_wave(s1) and tiles > CUS * groups[8]:
            assert nw * groups[nw] == max(w * g for w, g in groups.items()), what


def test_middle_kernel_waves_as_measured(rules):
    """Both sides of each line the rule's comment gives figures for."""
    want = {(9, 8192, 1, 1): 4, (8, 16384, 1, 1): 4, (7, 8192, 2, 2): 4,
            (9, 1024, 5, 15): 4, (9, 2048, 8, 16): 8, (9, 2048, 15, 30): 16,
            (8, 4096, 4, 16): 4, (8, 2048, 15, 30): 8, (7, 8192, 8, 24): 4,
            (8, 15360, 8, 24): 8, (8, 512, 8, 24): 8}
    got = rules("mid", [(*s, LDS) for s in want])
    assert {s: r[0] for s, r in zip(want, got)} == want


def test_middle_kernel_waves_with_little_lds(rules):
    """A 64 KB workgroup limit: whatever fits at four waves is launched at a
    form that fits."""
    shapes = [(s1, tiles, nsrc, ndst, 65536) for s1 in (7, 8, 9) for tiles in (64, 4096)
              for nsrc in range(1, 17) for ndst in (4, 16, 45)]
    for (s1, _, nsrc, ndst, _), (nw, *lds) in zip(shapes, rules("mid", shapes)):
        if lds[0] <= 65536:
            assert lds[{4: 0, 8: 1, 16: 2}[nw]] <= 65536, (s1, nsrc, ndst, nw)


def test_digits_finished_in_moddown(rules):
    """One and two digits always, more only above 5 MiB of digits, as measured."""
    want = {(1, 2, 1 << 13, 1): 1, (2, 3, 1 << 13, 1): 1, (3, 4, 1 << 13, 1): 0,
            (4, 5, 1 << 13, 1): 0, (4, 5, 1 << 14, 2): 0, (4, 5, 1 << 15, 1): 0,
            (3, 32, 1 << 13, 1): 1, (3, 20, 1 << 15, 1): 1, (4, 5, 1 << 13, 32): 1,
            (3, 32, 1 << 16, 1): 1, (4, 53, 1 << 17, 32): 1}
    got = rules("digits", [(*s, 0) for s in want])
    assert {s: r[0] for s, r in zip(want, got)} == want


def test_rescale_route(rules):
    """The column kernel but for batches of 128-row columns whose intermediate
    is over 32 MiB; its waves no more than the lines fill, 16 for up to 512 tiles
    below 512 rows, as measured."""
    shapes = [(s1, tiles, l, 0, 0) for s1 in (7, 8, 9)
              for tiles in (64, 128, 512, 768, 1024, 1280, 2048, 4096, 16384)
              for l in (1, 2, 4, 8, 9, 12, 16, 17, 19, 29, 44, 63)]
    for (s1, tiles, l, _, _), (columns, nw) in zip(shapes, rules("rescale", shapes)):
        what = (s1, tiles, l, columns, nw)
        assert columns == (s1 > 7 or tiles <= 1024 or tiles * l <= 32 * 1024), what
        assert nw in (2, 4, 8, 16) and (nw == 2 or l > nw // 2 * lines_per_wave(s1)), what
        assert nw < 16 or (tiles <= 512 and s1 < 9), what
    want = {(7, 4096, 1): 2, (9, 4096, 1): 2, (8, 8192, 4): 4, (8, 512, 29): 16,
            (7, 128, 44): 16, (9, 512, 44): 8,
            (8, 768, 29): 8, (7, 1024, 44): 8, (7, 1280, 19): 4, (8, 8192, 44): 8}
    got = rules("rescale", [(*s, 0, 0) for s in want])
    assert {s: r[1] for s, r in zip(want, got)} == want
