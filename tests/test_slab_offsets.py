"""The bound on the slab copies of the beam projectors: whatever it accepts has 32-bit byte offsets below 2^31, it
accepts eight planes of ordinary volumes, and a thin volume with planes of 13000 x 13000 gets fewer.  The kernel's
offsets are formed here in exact integers; in 32 bits eight of the thin volume's planes wrapped."""
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tigre_amd", "csrc")


@pytest.fixture(scope="module")
def fits(tmp_path_factory):
    d = tmp_path_factory.mktemp("slab")
    src = d / "fits.cpp"
    src.write_text('#include <cstdio>\n#include "%s/common.hpp"\nint main() {\n    int p, r, z, a;\n'
                   '    while (std::scanf("%%d %%d %%d %%d", &p, &r, &z, &a) == 4)\n'
                   '        std::printf("%%d\\n", (int)tigre::slab_offsets_fit(p, r, z, a));\n}\n' % CSRC)
    exe = d / "fits"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.path.join(rocm, "bin", "hipcc"), "-std=c++17", "-x", "hip", "--cuda-host-only", str(src), "-o", str(exe)],
                   check=True, capture_output=True)

    def ask(cases):
        text = "\n".join("%d %d %d %d" % c for c in cases)
        out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.split()
        return [v == "1" for v in out]
    return ask


def _last_byte(planes, rows, stage_rows, columns, stage_columns):
    """Past the last byte of the last lane's 16: plane planes - 1, row rows - 1, the box's last four columns."""
    return 4 * (((planes - 1) * stage_rows + rows - 1) * stage_columns + columns)


def test_ordinary_volumes_keep_eight_planes(fits):
    cases = [(8 + tap, rows, n + 2, (n + 3 & ~3) + 8) for n in (64, 512, 1024, 2048, 7000) for tap in (0, 1) for rows in (8, 100)]
    assert all(fits(cases))


def test_thin_volume(fits):
    stage_rows, stage_columns = 13002, 13008
    assert _last_byte(8, 8, stage_rows, 24, stage_columns) > 1 << 32  # wraps in 32 bits
    assert fits([(8, 8, stage_rows, stage_columns), (4, 8, stage_rows, stage_columns), (3, 8, stage_rows, stage_columns),
                 (1, 8, stage_rows, stage_columns)]) == [False, True, True, True]


def test_accepted_offsets_are_below_two_gib(fits):
    rng = random.Random(4)
    cases = []
    for _ in range(2000):
        stage_rows, stage_columns = rng.randint(3, 40000), 4 * rng.randint(3, 10000)
        columns = 4 * rng.randint(1, min(200, stage_columns // 4))
        cases.append((rng.randint(1, 9), min(rng.randint(1, 200), stage_rows), stage_rows, columns, stage_columns))
    got = fits([c[:3] + c[4:] for c in cases])
    assert any(got) and not all(got)
    for c, ok in zip(cases, got):
        last = _last_byte(*c)
        assert last <= 1 << 31 or not ok, c
        # and nothing that fits by a whole row is refused
        assert ok or last + 4 * c[4] > 1 << 31, c
