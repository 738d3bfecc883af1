"""How the resident TDSE kernels cover a grid (tdse_plan.h, compiled here for the host): every point in one window, halos
that hold the steps between two loads, chunks that a scan reaches over, and where one cover ends and the next begins."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = """
#include <cstdio>
#include "tdse_plan.h"
int main()
{
    int nx, reach;
    while (std::scanf("%d %d", &nx, &reach) == 2) {
        TdseResident r{}, o{};
        const bool a = plan_resident(nx, reach, r), b = plan_one(nx, reach, o);
        for (int k = 0; k < 2; k++) {
            const TdseResident &R = k ? o : r;
            std::printf("%d %d %d %d %d %d %d ", k ? b : a, R.chunk, R.waves, R.windows, R.steps, R.stride, R.halo);
        }
        std::printf("\\n");
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "plan")
    subprocess.run([gxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "mma_amd", "csrc"),
                    str(d / "main.cpp"), "-o", exe], check=True)

    def get(cases):
        text = "\n".join("%d %d" % c for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        rows = np.array([[int(v) for v in line.split()] for line in out.splitlines()]).reshape(len(cases), 2, 7)
        keys = ("ok", "chunk", "waves", "windows", "steps", "stride", "halo")
        return [[dict(zip(keys, r)) for r in pair] for pair in rows]

    return get


# reach: 151 points at dx 0.1, dt 0.25; the table builder takes 320 at most
REACHES = [1, 20, 96, 139, 151, 192, 193, 256, 257, 320]


def test_every_point_in_one_window(plans):
    rng = np.random.default_rng(5)
    sizes = sorted({3, 61, 1009, 1010, 4081, 4082, 6121, 8177, 8178, 12265, 12266, 16353, 16354, 131072, 1000001}
                   | {int(v) for v in np.exp(rng.uniform(np.log(3), np.log(3e5), 60))})
    cases = [(n, r) for n in sizes for r in REACHES]
    for (nx, reach), (batch, one) in zip(cases, plans(cases)):
        for p, most_waves in ((batch, 8), (one, 4)):
            what = (nx, reach, p)
            assert p["ok"] and p["chunk"] in (16, 24, 32) and 1 <= p["waves"] <= most_waves, what
            lead = p["chunk"] - 1  # a grid starts up to so many points into its first lane
            chunks = -(-(nx + lead) // p["chunk"])
            lanes = 64 * p["waves"]
            assert reach <= 16 * p["chunk"], what  # a scan looks over a row of 16 lanes and the row before
            assert 1 <= p["steps"] <= 16, what
            if p["windows"] == 1:
                assert lanes >= chunks, what
                continue
            stride, halo, n = p["stride"], p["halo"], p["windows"]
            assert lanes == 64 * most_waves and stride >= 1, what
            assert halo * p["chunk"] >= p["steps"] * (reach + 2), what
            assert stride + 2 * halo <= lanes, what  # what a window owns is halo chunks from its ends
            assert (n - 1) * stride + lanes >= chunks > (n - 2) * stride + lanes, what
            # the windows' own chunks, as place_lane deals them
            edges = [0] + [w * stride + halo for w in range(1, n)] + [chunks]
            assert all(a < b for a, b in zip(edges, edges[1:])), what
        assert one["windows"] <= 64 or one["steps"] == 1, (nx, reach, one)


def test_where_the_covers_change(plans):
    # a window of C points a lane has ceil((nx + C - 1) / 64 C) waves, 8 at most
    expect = {1009: (16, 1, 1), 8177: (16, 8, 1), 8178: (24, 6, 1), 12265: (24, 8, 1), 12266: (32, 7, 1),
              16353: (32, 8, 1), 16354: (24, 8, 2)}
    cases = [(n, 151) for n in expect]
    for (nx, _), (p, _) in zip(cases, plans(cases)):
        assert (p["chunk"], p["waves"], p["windows"]) == expect[nx], (nx, p)
    # one window ends at 16353 points for every reach that 32 points a lane serve
    for reach in REACHES:
        a, b = plans([(16353, reach), (16354, reach)])
        assert a[0]["windows"] == 1 and b[0]["windows"] > 1


def test_grids_beyond_32_bit_offsets_are_left_to_the_streaming_kernels(plans):
    last = (1 << 27) - (1 << 16)
    for (batch, one), ok in zip(plans([(last, 151), (last + 1, 151), ((1 << 31) - 64, 151)]), (1, 0, 0)):
        assert batch["ok"] == one["ok"] == ok
        assert ok or batch["chunk"] == one["chunk"] == 0
