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
            ((8, 2, 256), I8, 400, 4333, 900), ((32, 8, 128), F16, 512, 4432, 4000)]


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


# short prompts, chunks, and prompts of less than a round of workgroups
PROMPTS = [((32, 8, 128), F16, 0, 80, 1024), ((12, 4, 64), F16, 1024, 1000, 0),
           ((16, 2, 256), F16, 0, 300, 256), ((32, 8, 128), I8, 0, 150, 512),
           ((32, 4, 128), I8, 0, 300, 512), ((16, 2, 256), I16, 0, 200, 0),
           ((32, 8, 128), I8, 0, 80, 1000), ((16, 2, 256), I16, 0, 300, 8000),
           ((12, 4, 64), F16, 0, 1147, 0), ((12, 4, 64), I16, 0, 900, 300),
           ((32, 8, 128), F16, 0, 512, 2048), ((16, 2, 512), F16, 0, 99, 7452),
           ((16, 2, 512), I16, 1024, 399, 972), ((32, 8, 128), F16, 0, 1432, 0),
           ((12, 4, 64), F16, 1024, 3500, 0), ((32, 8, 128), F16, 512, 1432, 4000)] + WINDOWED


@pytest.mark.parametrize("geom,kv,window,n,pos0", PROMPTS)
def test_segments_follow_the_sequence_and_stay_few(host, geom, kv, window, n, pos0):
    """The kernel that fills the device, and no more segments than fill it: in a
    call alone, in one of 2 to 40 prompts, beside a longer one, through the entry
    point without allocation (where a copy and partials fit it), after calls that
    grew the instance, and captured - always the same."""
    hv, most, blocks = fill(host, geom, kv, window, n, pos0)
    h, n_kv, hd = geom
    new = f"new {h} {n_kv} {hd} {window} 256"
    one = f" {n} {pos0}"
    lines = [new, f"call dev {kv} 0 0{one}", f"call noalloc {kv} 0 0{one}",
             f"call dev {kv} 0 0 4000 3000{one}", f"call dev {kv} 0 1{one}"]
    alone, noalloc, beside, captured = (Call(w) for w in host(lines)[1:])
    assert alone.rc == 0
    (got,) = alone.prompts()
    assert got[0] == hv and 1 <= got[1] <= most and got[2] == (got[1] > 1)
    assert alone.workgroups() == blocks * got[1]
    assert noalloc.rc in (0, janas_amd.ERANGE)
    if noalloc.rc == 0:
        assert noalloc.prompts() == [got]
    assert got[:2] in [x[:2] for x in beside.prompts()]
    assert captured.rc == 0 and captured.refused == 0
    assert captured.prompts() == [got]
    for m in (2, 3, 8, 16, 40):
        many = Call(host([new, f"call dev {kv} 0 0" + one * m])[1])
        assert many.prompts() == [got] * m
        assert many.workgroups() == m * blocks * got[1]


@pytest.mark.parametrize("geom,kv,window,n,pos0", [c for c in PROMPTS if c[1] == F16])
def test_prompts_without_segments_leave_the_instance_alone(host, geom, kv, window, n, pos0):
    """An f16 prompt that segments cannot make fill the device any better uses no
    memory of the instance: nothing is allocated at its first call, a captured
    one holds none that a later call could free, and after work of the instance
    on another stream it neither waits for it nor is refused under capture."""
    _, most, _ = fill(host, geom, kv, window, n, pos0)
    if most > 1:
        pytest.skip("a prompt that takes segments")
    h, n_kv, hd = geom
    one = f" {n} {pos0}"
    # (a decode of 300 positions leaves partials on stream 0)
    for captured in (0, 1):
        new, decode, call = host([f"new {h} {n_kv} {hd} {window} 256", f"call dev {kv} 0 0 1 299",
                                  f"call dev {kv} 1 {captured}{one}"])
        got = Call(call)
        assert got.rc == 0
        assert (got.allocs, got.frees, got.refused, got.waits) == (0, 0, 0, 0)
        assert all(not parts for _, _, parts, _, _ in got.launches)


@pytest.mark.parametrize("geom,n_ctx", [((32, 8, 128), 256), ((12, 4, 64), 600),
                                        ((16, 2, 512), 32768), ((8, 8, 8), 0)])
def test_an_instance_holds_a_blocks_partials(host, geom, n_ctx):
    """What janas_attn_part_bytes says from the creation on (at least a chunk's),
    in one allocation for the pairs and one for the values."""
    h, n_kv, hd = geom
    rows, allocs = (int(x) for x in host([f"new {h} {n_kv} {hd} 0 {n_ctx}"])[0])
    assert rows * (hd + 2) * 4 == janas_amd.part_bytes(h, n_kv, hd, max(n_ctx, 1))
    assert allocs == 2


def test_the_merge_alone_finds_partials(host):
    """janas_attn_run_dev_kernels: 1 and 3 leave partials, 2 merges them; after a
    call of one chunk, whose split kernel wrote the outputs, 2 makes them first."""
    calls = ["dev", "kernels2", "kernels2", "kernels3", "kernels2", "split", "kernels1", "kernels2",
             "dev", "noalloc", "kernels2"]
    want = ["split", "split merge", "merge", "split merge", "merge", "split", "split", "merge",
            "split", "split", "split merge"]
    got = host(["new 32 8 128 0 256"] + [f"call {c} {F16} 0 0 1 99" for c in calls])[1:]
    assert [" ".join(x[0] for x in Call(w).launches) for w in got] == want
    # of two chunks every call leaves them
    got = host(["new 32 8 128 0 512", f"call dev {F16} 0 0 1 299", f"call kernels2 {F16} 0 0 1 299"])
    assert [" ".join(x[0] for x in Call(w).launches) for w in got[1:]] == ["split merge", "merge"]
