"""janas_attn_run_dev_noalloc: the same results as janas_attn_run_dev,
bit for bit, with its partials in the device's fixed array - two calls in
a row (a long decode, then a smaller block and a prompt chunk whose key
segments need partials), and a call needing more than the array is refused
with JANAS_ATTN_ERANGE."""
import numpy as np
import pytest
import torch

import janas_amd
from attn_helpers import TOL_F16_ABS, TOL_FLOAT_ABS, abs_err, threads, within
from cases import normal
from janas_amd import Attention
from oracle import orc

pytestmark = pytest.mark.gpu

NOALLOC_BYTES = 64 << 20


def dev(x, device):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


def both(a, kv, seqs, gate_mode, noalloc_outs):
    """run_dev into the seqs' outs, then run_dev_noalloc into noalloc_outs
    (same inputs)."""
    a.run_dev(kv, seqs, gate_mode=gate_mode)
    seqs2 = [dict(s, out=o) for s, o in zip(seqs, noalloc_outs)]
    a.run_dev(kv, seqs2, gate_mode=gate_mode, path="noalloc")
    torch.cuda.synchronize()


def test_noalloc_equals_run_dev_twice(gpu):
    # call 1: config 4's decode (16 / 2 / 256, 32k positions, gated)
    h, kvh, hd, L = 16, 2, 256, 32768
    k = dev(normal(101, kvh * L * hd).reshape(kvh, L, hd).astype(np.float16), gpu)
    v = dev(normal(103, kvh * L * hd).reshape(kvh, L, hd).astype(np.float16), gpu)
    q = dev(normal(107, h * hd).reshape(1, h, hd), gpu)
    g = dev(normal(109, h * hd).reshape(1, h, hd), gpu)
    out, out2 = torch.empty_like(q), torch.full_like(q, float("nan"))
    with Attention(h, kvh, hd, L) as a:
        a.set_scale(1.0 / 16.0)
        both(a, janas_amd.KV_F16, [dict(k=k, v=v, q=q, out=out, gate=g, cap=L,
                                        n=1, pos0=L - 1)],
             janas_amd.GATE_ELEM, [out2])
    assert torch.equal(out, out2)
    # call 2, smaller: a 16-token block (split path) and a 512-token chunk
    # of a prompt at 4096 (prefill path, split into key segments) over an
    # int8 cache, 32 / 8 / 128
    h, kvh, hd, L = 32, 8, 128, 4608
    k8 = np.clip(np.rint(normal(111, kvh * L * hd) * 30), -127, 127).astype(np.int8)
    v8 = np.clip(np.rint(normal(113, kvh * L * hd) * 30), -127, 127).astype(np.int8)
    ks = (0.01 + 0.01 * np.abs(normal(117, kvh * L))).astype(np.float32)
    vs = (0.01 + 0.01 * np.abs(normal(119, kvh * L))).astype(np.float32)
    kd, vd = dev(k8.reshape(kvh, L, hd), gpu), dev(v8.reshape(kvh, L, hd), gpu)
    ksd, vsd = dev(ks.reshape(kvh, L), gpu), dev(vs.reshape(kvh, L), gpu)
    qa = dev(normal(121, 16 * h * hd).reshape(16, h, hd), gpu)
    qb = dev(normal(123, 512 * h * hd).reshape(512, h, hd), gpu)
    oa, ob = torch.empty_like(qa), torch.empty_like(qb)
    oa2, ob2 = torch.full_like(qa, float("nan")), torch.full_like(qb, float("nan"))
    with Attention(h, kvh, hd, L) as a:
        both(a, janas_amd.KV_I8,
             [dict(k=kd, v=vd, ks=ksd, vs=vsd, q=qa, out=oa, cap=L, n=16, pos0=3000),
              dict(k=kd, v=vd, ks=ksd, vs=vsd, q=qb, out=ob, cap=L, n=512, pos0=4096)],
             janas_amd.GATE_NONE, [oa2, ob2])
    assert torch.equal(oa, oa2)
    assert torch.equal(ob, ob2)


@pytest.mark.parametrize("L,fits", [(16128, True), (16384, False), (65536, False)])
def test_noalloc_refuses_more_than_the_array(gpu, L, fits):
    """The array's capacity for the split path's partials: a row of m, l and
    hd values takes (hd + 2) x 4 bytes, a launch n_kv x chunks x n x group
    rows (the m, l pairs padded to 256 bytes). A 64-token block over 8 KV
    heads of 128 (32 query heads) at positions L - 64 .. L - 1 takes 2048
    rows a chunk: 63 chunks (L = 16128: 67,092,480 bytes) fit in the
    67,108,864, 64 chunks (L = 16384: 68,157,440) do not and are refused
    with ERANGE, as is 64k. The block that fits equals janas_attn_run_dev's
    result bit for bit."""
    h, kvh, hd = 32, 8, 128
    k = torch.zeros((kvh, L, hd), dtype=torch.float16, device=gpu)
    q = dev(normal(161, 64 * h * hd).reshape(64, h, hd), gpu)
    out = torch.full_like(q, float("nan"))
    chunks = (L + 255) // 256
    rows = kvh * chunks * 64 * (h // kvh)
    need = (rows * 2 * 4 + 255) // 256 * 256 + rows * hd * 4
    assert (need <= NOALLOC_BYTES) == fits
    seq = dict(k=k, v=k, q=q, out=out, cap=L, n=64, pos0=L - 64)
    with Attention(h, kvh, hd, L) as a:
        if not fits:
            with pytest.raises(janas_amd.AttnError) as e:
                a.run_dev(janas_amd.KV_F16, [seq], path="noalloc")
            assert e.value.code == janas_amd.ERANGE
            return
        a.run_dev(janas_amd.KV_F16, [seq], path="noalloc")
        want = torch.full_like(q, float("nan"))
        a.run_dev(janas_amd.KV_F16, [dict(seq, out=want)])
        torch.cuda.synchronize()
    assert torch.equal(out, want)


# (heads, KV heads, hd, n, pos0, window, ring, with last[]): prompts whose
# segments (or kernel) follow the estimate: two rounds of workgroups a window
# holds alike, a second round that was nearly empty, a prefix too short for 6
# tiles a segment, one round and a bit of a causal prompt, the two-halves kernel
RESPLIT = [(12, 4, 64, 1000, 0, 1024, False, False), (16, 2, 256, 300, 1000, 0, False, True),
           (32, 8, 128, 80, 1000, 0, False, False), (32, 8, 128, 1432, 0, 0, False, False),
           (12, 4, 64, 117, 2082, 300, True, False), (6, 3, 200, 251, 700, 0, False, True),
           # past whole rounds of row blocks, those split: a window's ramp, a ring
           # (a last block of few rows), spans that end past their blocks' tokens
           (16, 2, 256, 3001, 0, 700, False, False), (8, 2, 256, 4333, 900, 400, True, False),
           (32, 2, 512, 1201, 50, 512, False, True)]


@pytest.mark.parametrize("kv", [janas_amd.KV_F16, janas_amd.KV_I8, janas_amd.KV_I16])
@pytest.mark.parametrize("case", range(len(RESPLIT)))
def test_prompt_splits(gpu, kv, case):
    """A prompt alone, through the entry point without allocation, beside
    another one, and recorded into a graph by an instance whose partials are too
    few (it then splits less): the first three the same bits, all of them the
    restatement's outputs, gated, with its Q8_K blocks those of its output."""
    h, kvh, hd, n, pos0, window, ring, spans = RESPLIT[case]
    cap = (window + n + 512) // 256 * 256 if ring else pos0 + n + 3
    f32 = [normal(1000 + case + i, kvh * cap * hd).reshape(kvh, cap, hd) for i in (0, 7)]
    scales = [None, None]
    if kv == janas_amd.KV_F16:
        cache = [x.astype(np.float16) for x in f32]
    else:
        top = 127 if kv == janas_amd.KV_I8 else 32767
        scales = [(np.abs(x).max(axis=2) / top).astype(np.float32) for x in f32]
        cache = [np.rint(x / z[..., None]).astype(np.int8 if top == 127 else np.int16)
                 for x, z in zip(f32, scales)]
    q = normal(1020 + case, n * h * hd).reshape(n, h, hd)
    g = normal(1030 + case, n * h * hd).reshape(n, h, hd)
    last = None
    if spans:
        last = np.minimum(pos0 + np.arange(n) // 3 * 3 + 2, pos0 + n - 1).astype(np.uint32)
    d = dict(k=dev(cache[0], gpu), v=dev(cache[1], gpu), q=dev(q, gpu), gate=dev(g, gpu),
             cap=cap, n=n, pos0=pos0)
    if scales[0] is not None:
        d.update(ks=dev(scales[0], gpu), vs=dev(scales[1], gpu))
    if spans:
        d.update(last=dev(last.view(np.int32), gpu), last_max=int(last.max()))
    nb = h * hd // 256 if h * hd % 256 == 0 else 0

    def seq():
        s = dict(d, out=torch.full(d["q"].shape, float("nan"), device=gpu))
        if nb:
            s["out_q8k"] = torch.zeros((n, nb, 628), dtype=torch.uint8, device=gpu)
        return s
    alone, fixed, beside, other, graphed = (seq() for _ in range(5))
    st = torch.cuda.Stream()

    def instance(n_ctx):
        a = Attention(h, kvh, hd, n_ctx, 1, janas_amd.FLOAT)
        a.set_window(window)
        a.set_ring(ring)
        return a
    with instance(cap) as a, instance(256) as small:
        gate = janas_amd.GATE_ELEM
        a.run_dev(kv, [alone], gate)
        a.run_dev(kv, [fixed], gate, path="noalloc")
        a.run_dev(kv, [dict(other, n=70, last=None), beside], gate)
        # (the plain split has no segments here; an integer cache's copy allocates)
        captured = case == 0 and kv == janas_amd.KV_F16
        if captured:
            call = small.prepare(kv, [graphed], gate, stream=st.cuda_stream)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=st):
                call()
            for _ in range(3):
                graphed["out"].zero_()
                torch.cuda.synchronize()
                with torch.cuda.stream(st):
                    graph.replay()
                torch.cuda.synchronize()
                assert float((graphed["out"] - alone["out"]).abs().max()) <= TOL_F16_ABS
        torch.cuda.synchronize()
    assert torch.equal(alone["out"], fixed["out"])
    assert torch.equal(alone["out"], beside["out"])
    ref = orc.run(q.astype(np.float32), cache[0], cache[1], scales[0], scales[1], n_head=h,
                  n_kv=kvh, hd=hd, pos0=pos0, kv=kv, window=window, ring=ring, last=last,
                  threads=threads(), block=64)
    orc.gate(ref, g)
    bar = TOL_F16_ABS if kv == janas_amd.KV_F16 or hd > 256 else TOL_FLOAT_ABS
    assert within(abs_err(alone["out"].cpu().numpy(), ref), bar, "vs oracle")
    if nb:
        want = orc.q8k_quantize(alone["out"].cpu().numpy().reshape(n, h * hd))
        assert alone["out_q8k"].cpu().numpy().tobytes() == want.tobytes()


def test_noalloc_prompts_that_pass_the_array_together(gpu):
    """Prompts whose segments' partials fit the array one by one and not
    together split less there, and still run: outputs within the f16 bar of
    janas_attn_run_dev's."""
    h, kvh, hd, n, L = 12, 4, 64, 1000, 1000
    k = dev(normal(171, kvh * L * hd).reshape(kvh, L, hd).astype(np.float16), gpu)
    q = dev(normal(173, n * h * hd).reshape(n, h, hd), gpu)
    outs = [[torch.full_like(q, float("nan")) for _ in range(12)] for _ in range(2)]
    with Attention(h, kvh, hd, L) as a:
        for path, out in zip(("auto", "noalloc"), outs):
            a.run_dev(janas_amd.KV_F16, [dict(k=k, v=k, q=q, out=o, cap=L, n=n, pos0=0)
                                         for o in out], path=path)
        torch.cuda.synchronize()
    for x, y in zip(*outs):
        assert float((x - y).abs().max()) <= TOL_F16_ABS


def test_noalloc_under_graph_capture(gpu):
    """The entry point's reason: code under HIP graph capture. A decode
    step (f16, gated) and a 16-token block over an int8 cache, captured
    into one graph through janas_attn_run_dev_noalloc and replayed three
    times - with eager work in between that overwrites the device's
    partials array - each replay equal bit for bit to the eager result."""
    h, kvh, hd, L = 16, 2, 256, 4096
    k = dev(normal(131, kvh * L * hd).reshape(kvh, L, hd).astype(np.float16), gpu)
    v = dev(normal(133, kvh * L * hd).reshape(kvh, L, hd).astype(np.float16), gpu)
    q = dev(normal(137, h * hd).reshape(1, h, hd), gpu)
    g = dev(normal(139, h * hd).reshape(1, h, hd), gpu)
    k8 = np.clip(np.rint(normal(141, kvh * L * hd) * 30), -127, 127).astype(np.int8)
    v8 = np.clip(np.rint(normal(143, kvh * L * hd) * 30), -127, 127).astype(np.int8)
    ks = dev((0.01 + 0.01 * np.abs(normal(147, kvh * L))).astype(np.float32).reshape(kvh, L), gpu)
    vs = dev((0.01 + 0.01 * np.abs(normal(149, kvh * L))).astype(np.float32).reshape(kvh, L), gpu)
    kd, vd = dev(k8.reshape(kvh, L, hd), gpu), dev(v8.reshape(kvh, L, hd), gpu)
    qb = dev(normal(151, 16 * h * hd).reshape(16, h, hd), gpu)
    qo = dev(normal(153, 16 * h * hd).reshape(16, h, hd), gpu)
    want_a, want_b = torch.empty_like(q), torch.empty_like(qb)
    out_a, out_b = torch.empty_like(q), torch.empty_like(qb)
    scratch_out = torch.empty_like(qb)
    s = torch.cuda.Stream()
    with Attention(h, kvh, hd, L) as a:
        def calls(oa, ob, path):
            return [a.prepare(janas_amd.KV_F16, [dict(k=k, v=v, q=q, out=oa, gate=g, cap=L,
                                                      n=1, pos0=L - 1)],
                              gate_mode=janas_amd.GATE_ELEM, stream=s.cuda_stream,
                              path=path),
                    a.prepare(janas_amd.KV_I8, [dict(k=kd, v=vd, ks=ks, vs=vs, q=qb, out=ob,
                                                     cap=L, n=16, pos0=L - 16)],
                              stream=s.cuda_stream, path=path)]
        with torch.cuda.stream(s):
            for f in calls(want_a, want_b, "auto"):
                f()
            captured = calls(out_a, out_b, "noalloc")
            for f in captured:   # once outside the capture
                f()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            for f in captured:
                f()
        torch.cuda.synchronize()
        other = a.prepare(janas_amd.KV_I8, [dict(k=kd, v=vd, ks=ks, vs=vs, q=qo,
                                                 out=scratch_out, cap=L, n=16, pos0=1000)],
                          stream=s.cuda_stream, path="noalloc")
        for _ in range(3):
            out_a.zero_()
            out_b.zero_()
            with torch.cuda.stream(s):
                other()          # eager: overwrites the partials array
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out_a, want_a)
            assert torch.equal(out_b, want_b)
        assert a.status() == 0
