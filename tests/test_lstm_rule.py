"""CPU check of how many blocks the BiLSTM recurrences split a sequence over (kokoro-rust_amd/csrc/kk_lstm.h).

The blocks of a sequence wait for each other, so every choice must make progress with four launches
starting their blocks at once, whatever order the device takes them in.  A model of the device (XCDs of
32 CUs, blocks to XCDs in turn, in order within a launch, a group ends once all of its blocks are
resident) runs the rule's choices over batch and device sizes under the worst order -- every launch
stops one block short of completing a group while another can start a block -- and under random ones.
The same model must find the stall of choices that the rule refuses."""
import os
import random
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kokoro-rust_amd", "csrc")
ITEMS = [1, 2, 4, 5, 6, 8, 9, 12, 16, 17, 24, 32, 33, 64]
CUS = [32, 64, 128, 256]  # a whole device and its partitions: 1, 2, 4 or 8 XCDs

PRINT = r"""
#include <cstdio>
#include <initializer_list>
#include "kk_lstm.h"
int main() {
    for (int n_cu : {CUS})
        for (int nb : {ITEMS})
            for (long longest : {500L, 1024L})
                for (int sel : {-1, 0, 1})
                    std::printf("%d %d %ld %d %d\n", n_cu, nb, longest, sel, kk::lstm_parts(nb, longest, n_cu, sel));
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("lstm_rule")
    src = d / "rule.cpp"
    src.write_text(PRINT.replace("CUS", ",".join(map(str, CUS))).replace("ITEMS", ",".join(map(str, ITEMS))))
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(d / "rule")], check=True)
    out = subprocess.run([str(d / "rule")], check=True, capture_output=True, text=True).stdout
    return {tuple(map(int, l.split()[:4])): int(l.split()[4]) for l in out.splitlines()}


def stalls(parts, nb, n_cu, launches, rng=None):
    """True if `launches` launches of the same size can end up waiting on each other for good."""
    xcds = max(1, n_cu // 32)
    free = [(2 if parts >= 8 else 1) * n_cu // xcds] * xcds
    groups = min(2 * nb, 64)
    if parts == 2:
        groups = 2 * nb
    # per launch and XCD: the groups of its blocks, in order (blocks past the last group end at once)
    todo = [[[] for _ in range(xcds)] for _ in range(launches)]
    for q in todo:
        for b in range((groups + 7) // 8 * 8 * parts):
            g = b // (8 * parts) * 8 + b % 8
            if g < groups:
                q[b % xcds].append(g)
    held = [dict() for _ in range(launches)]  # group -> its resident blocks
    while any(any(q) for q in todo):
        can = [(l, x) for l in range(launches) for x in range(xcds) if todo[l][x] and free[x] > 0]
        if not can:  # only now do the complete groups end (the worst time for everybody else)
            done = [(l, g) for l in range(launches) for g, n in held[l].items() if n == parts]
            if not done:
                return True
            for l, g in done:
                # (a group's blocks lie on one XCD when the number of XCDs divides 8)
                for p in range(parts):
                    free[(g // 8 * 8 * parts + g % 8 + 8 * p) % xcds] += 1
                del held[l][g]
            continue
        if rng:
            l, x = rng.choice(can)
        else:  # the blocks that complete no group first
            l, x = min(can, key=lambda c: held[c[0]].get(todo[c[0]][c[1]][0], 0) + 1 == parts)
        g = todo[l][x].pop(0)
        free[x] -= 1
        held[l][g] = held[l].get(g, 0) + 1
    return any(n < parts for h in held for n in h.values())


def test_every_choice_makes_progress(rule):
    seen = set()
    for (n_cu, nb, longest, sel), parts in rule.items():
        if (parts, nb, n_cu) not in seen:
            seen.add((parts, nb, n_cu))
            launches = 4 if n_cu > 32 else 3  # (the pairs, the last choice, fill 32 CUs with four)
            for rng in (None, random.Random(1), random.Random(2)):
                assert not stalls(parts, nb, n_cu, launches, rng), (n_cu, nb, longest, sel, parts)
    assert {p for p, _, _ in seen} == {2, 4, 8, 16}
    # the model finds the stalls of what is refused: 32 CUs (one XCD as a device), and a fifth launch
    assert rule[32, 5, 500, -1] == 2 and stalls(16, 5, 32, 1) and stalls(8, 8, 32, 2)
    assert rule[64, 8, 1024, 1] == 2 and stalls(4, 4, 64, 4)
    assert stalls(16, 8, 256, 5)


def test_choices_on_256_cus(rule):
    for nb in ITEMS:
        short = 16 if nb <= 8 else 8 if nb <= 16 else 4 if nb <= 32 else 2
        assert rule[256, nb, 500, -1] == short
        assert rule[256, nb, 1024, -1] == rule[256, nb, 500, 1] == max(short, 4)
        assert rule[256, nb, 1024, 0] == 2


def test_registers_leave_the_blocks_per_cu(tmp_path):
    """The kernels of 8 and 16 parts hold two blocks of 512 threads per CU: 4 waves on each SIMD."""
    cmd = [os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang",
           "-target-feature", "-Xclang", "-packed-fp32-ops", "-fhip-fp32-correctly-rounded-divide-sqrt", "-I", CSRC,
           "--cuda-device-only", "-c", os.path.join(CSRC, "kk_upstream.hip"), "-o", str(tmp_path / "u.o"),
           "-Rpass-analysis=kernel-resource-usage"]
    log = subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=300).stderr
    found = {}
    for part in log.split("Function Name: ")[1:]:
        m = re.match(r"\S*lstm_split_kernelILi(\d+)E", part)
        if m:
            found[int(m[1])] = (int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", part)[1]),
                                int(re.search(r"VGPRs Spill: (\d+)", part)[1]))
    assert set(found) == {4, 8, 16}, log[:2000]
    for p, (waves, spill) in found.items():
        assert waves >= (4 if p >= 8 else 2) and spill == 0, (p, waves, spill)
