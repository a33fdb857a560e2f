"""Host check of the threads that share an upload's host copy
(cujpegxl_amd/csrc/copy_team.h), as a small program built from the header:
every piece of a job is copied once, whatever the pauses between the releases;
helpers of an open job without a released piece do not occupy processors; a job
closed early ends."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <time.h>

#include <atomic>
#include <cstdio>
#include <memory>

#include "copy_team.h"

namespace {

double cpu_ms() {
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return t.tv_sec * 1e3 + t.tv_nsec * 1e-6;
}

void pause_us(int us) {
    if (us > 0) {
        std::this_thread::sleep_for(std::chrono::microseconds(us));
    }
}

std::atomic<unsigned> copies[4096];

// A job of `groups` groups of 8 pieces (the last one shorter by `less`), two
// groups ahead of the one being finished released at a time.
bool job(cjx::CopyTeam& team, unsigned groups, unsigned less, int pause) {
    const unsigned pieces{groups * 8 - less};
    for (unsigned i{0}; i < pieces; ++i) {
        copies[i] = 0;
    }
    team.open(pieces, 8, [](std::uint32_t i) { copies[i].fetch_add(1); }, true);
    bool ok{true};
    for (unsigned g{0}; g < groups; ++g) {
        pause_us(pause);
        const unsigned upto{(g + 2) * 8};
        team.release(upto < pieces ? upto : pieces);
        team.finish_group(g);
        for (unsigned i{g * 8}; i < g * 8 + 8 && i < pieces; ++i) {
            ok = ok && copies[i] == 1;
        }
    }
    team.close();
    return ok;
}

}  // namespace

int main() {
    auto team{std::make_unique<cjx::CopyTeam>(3u)};
    bool ok{true};
    for (int n{0}; n < 300; ++n) {
        // Releases at once, within and past the helpers' polling.
        ok = job(*team, 1 + n % 9, n % 8, n % 3 == 0 ? 0 : (n % 3 == 1 ? 30 : 600)) && ok;
    }
    std::printf("copied_once %d\n", ok ? 1 : 0);
    // Nothing released for 300 ms.
    const double before{cpu_ms()};
    team->open(64, 8, [](std::uint32_t) {}, true);
    pause_us(300000);
    std::printf("idle_cpu_ms %.3f\n", cpu_ms() - before);
    team->close();
    ok = job(*team, 5, 0, 0);
    // Closed with a released group left, and with nothing released.
    team->open(64, 8, [](std::uint32_t) {}, true);
    team->release(8);
    pause_us(2000);
    team->close();
    ok = job(*team, 3, 1, 600) && ok;
    std::printf("after_close %d\n", ok ? 1 : 0);
    team.reset();
    std::printf("done 1\n");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_pieces_idle_helpers_and_early_close(tmp_path):
    src, exe = tmp_path / "team.cc", tmp_path / "team"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{ROOT / 'cujpegxl_amd' / 'csrc'}", str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=100).stdout
    values = dict(line.split() for line in out.splitlines())
    assert values["copied_once"] == values["after_close"] == values["done"] == "1"
    # Three helpers that poll throughout take 900 ms, one alone 300; asleep
    # after their 0.2 ms of polling they take about 0.6 ms together.
    assert float(values["idle_cpu_ms"]) < 30.0, out
