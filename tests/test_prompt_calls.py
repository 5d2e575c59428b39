"""What a prompt call launches, over a made-up HIP runtime (host_calls.cpp): no
GPU. A prompt's key segments follow from the sequence and the device alone -
alone, beside others, captured, through the entry point without allocation -
and cost a call no more workgroups and partials than segments that give each
compute unit one workgroup do."""
import os
import subprocess

import pytest

import janas_amd
from janas_amd.build import LIB, ROOT

CLANG = "/opt/rocm/llvm/bin/clang++"
F16, I8, I16 = janas_amd.KV_F16, janas_amd.KV_I8, janas_amd.KV_I16
CUS = 256


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """run(lines) -> the program's answer lines, split."""
    janas_amd.lib()
    exe = tmp_path_factory.mktemp("host") / "host_calls"
    libdir = os.path.dirname(LIB)
    subprocess.run([CLANG, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-Wno-unused-result",
                    os.path.join(ROOT, "tests", "host_calls.cpp"), "-o", str(exe), "-L", libdir,
                    "-ljanas_attn", f"-Wl,-rpath,{libdir}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)

    def run(lines):
        p = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True,
                           text=True, timeout=60)
        assert p.returncode == 0, p.stderr
        return [line.split() for line in p.stdout.splitlines()]
    return run


class Call:
    """An answer to a call line."""

    def __init__(self, words):
        self.rc, self.allocs, self.frees, self.refused, self.waits = (int(x) for x in words[:5])
        self.launches = []
        for w in words[5:]:
            what, wg, parts, halves, seqs = w.split(":")
            self.launches.append((what, int(wg), parts == "1", int(halves),
                                  [int(x) for x in seqs.split(",")]))

    def prompts(self):
        """(halves, segments, partials) of each prompt launch's sequences"""
        return [(h, s, parts) for what, _, parts, h, segs in self.launches if what == "prefill"
                for s in segs]

    def workgroups(self):
        return sum(wg for what, wg, *_ in self.launches if what == "prefill")


def exact(geom, kv):
    return 0 if kv == F16 or geom[2] > 256 else 2 if kv == I16 else 1


def fill(host, geom, kv, window, n, pos0):
    """(halves, segments) that give each compute unit a workgroup: the two-halves
    kernel where the other's row blocks and segments leave units idle, at least 6
    tiles a segment (12 of the halves'), at most 16."""
    h, n_kv, hd = geom
    words = host([f"new {h} {n_kv} {hd} {window} 256",
                  f"first {kv} {exact(geom, kv)} {n} {pos0}"])[1]
    blocks, tile = [int(words[0]), int(words[2])], [int(words[1]), int(words[3])]
    last = pos0 + n - 1

    def segments(hv):
        wg = n_kv * blocks[hv]
        if wg >= CUS:
            return 1
        lo = last + 1 - window if window and last + 1 > window else 0
        tiles = last // tile[hv] - lo // tile[hv] + 1
        return min(-(-CUS // wg), max(1, tiles // (12 if hv else 6)), 16)
    halves = int(words[4]) if kv == F16 else 0
    hv = int(halves and n_kv * blocks[0] * segments(0) < CUS)
    return hv, segments(hv), n_kv * blocks[hv]


# prompts of more than one round of workgroups, of like length in a window
WINDOWED = [((16, 2, 256), I16, 1024, 3001, 0), ((16, 2, 256), F16, 700, 3001, 0),
            ((8, 2, 256), I8, 400, 4333, 900)]


@pytest.mark.parametrize("geom,kv,window,n,pos0", WINDOWED)
def test_prompts_that_fill_the_device_use_no_partials(host, geom, kv, window, n, pos0):
    """Row blocks that fill the device are not cut: nothing of the instance
    beside an integer cache's exact copy."""
    hv, most, blocks = fill(host, geom, kv, window, n, pos0)
    assert blocks >= CUS and most == 1
    h, n_kv, hd = geom
    for m in (1, 3):
        got = Call(host([f"new {h} {n_kv} {hd} {window} 8192",
                         f"call dev {kv} 0 0" + f" {n} {pos0}" * m])[1])
        assert got.rc == 0
        assert got.prompts() == [(hv, 1, False)] * m
        assert got.workgroups() == m * blocks
