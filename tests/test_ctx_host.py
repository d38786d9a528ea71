"""A context's own memory over calls that share it (greedy steps, batches of more and more logits rows): what each call reads
and writes is allocated, and everything is freed once."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_context_memory_is_live_and_freed_once(tmp_path):
    """gw_forward.c on the CPU (tests/ctx_host.c); whatever else it links against returns 0"""
    def run(*cmd):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    obj, stubs, exe = str(tmp_path / "h.o"), str(tmp_path / "stubs.c"), str(tmp_path / "h")
    csrc = os.path.join(ROOT, "gwenedeg_amd", "csrc")
    run("gcc", "-O1", "-g", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I", csrc, "-I", os.path.join(ROOT, "include"),
        "-I", "/opt/rocm/include", "-c", os.path.join(ROOT, "tests", "ctx_host.c"), "-o", obj)
    names = [line.split()[-1] for line in run("nm", "-u", obj).splitlines()]
    with open(stubs, "w") as f:
        f.writelines(f"int {n}() {{ return 0; }}\n" for n in names if n.startswith(("gw_", "hip", "rq_")))
    run("gcc", "-w", obj, stubs, "-lm", "-o", exe)
    assert run(exe) == "ok\n"


@pytest.mark.gpu
@pytest.mark.parametrize("shape", ["tiny", "tiny_kq"])
def test_greedy_after_a_larger_batch_on_one_context(synth_models, shape):
    """greedy steps, a batch of more selected rows than before, greedy steps again, on one context: the tokens and the logits of
    a context that runs nothing else"""
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import gwenedeg_amd as gw
    m = gw.Model(synth_models(shape), ctx_len=512)
    ids = np.random.default_rng(4).integers(0, m.vocab, 9).astype(np.int32)

    def alone(n):  # (n greedy tokens behind ids, step by step on contexts of their own)
        c, s, got = m.ctx(max_batch=16), m.seq(512), []
        lg = c.prefill(s, ids)
        for _ in range(n):
            tok = int(np.argmax(lg))
            got.append(tok)
            lg = c.decode(s, tok)
        return got + [int(np.argmax(lg))]
    want = alone(12)
    c, s = m.ctx(max_batch=16), m.seq(512)
    assert int(np.argmax(c.prefill(s, ids))) == want[0]
    assert [int(t) for t in c.decode_greedy(s, want[0], 6)] == want[1:7]
    for rows in (2, 9):
        o = m.seq(512)
        one = m.ctx(max_batch=16).prefill(m.seq(512), ids[:rows], mode=gw.RQ_LOGITS_ALL)
        got = c.prefill(o, ids[:rows], mode=gw.RQ_LOGITS_ALL)
        assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
        n = len(s) - len(ids)
        assert [int(t) for t in c.decode_greedy(s, want[n], 3)] == want[n + 1:n + 4]
