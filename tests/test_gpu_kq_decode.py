"""The one-row K-quant matmuls with their producers in front (k_gemvk), through whole decode steps: against the oracle and
against the rows of a prompt pass, which other kernels compute, bit for bit."""
import numpy as np
import pytest

from gwenedeg_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gw():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import gwenedeg_amd
    return gwenedeg_amd


def _bits_equal(a, b):
    return np.array_equal(np.ascontiguousarray(a, np.float32).view(np.uint32), np.ascontiguousarray(b, np.float32).view(np.uint32))


# 2: K from one super-block to ten (units per row that divide a block's 512 threads and that do not), Q4_K, Q5_K and Q6_K in
# each place, rows that leave a block's last run short, positions on both sides of 1,024 (the combine in front of wo, then a
# launch of its own); 3: a classifier of more rows per block than LDS holds terms for (60,000 rows of 4,096 over 256 blocks:
# 235 rows, in runs), tied to the Q4_K, Q5_K or Q6_K embedding
@pytest.mark.parametrize("over", [
    dict(), dict(dim=256, hidden=768, n_heads=2, vocab=1001), dict(dim=768, hidden=2560, n_heads=6, vocab=515, type_down=12),
    dict(type_default=13, dim=1280, hidden=256, vocab=777, type_down=13),
    dict(type_default=14, type_v=12, dim=768, hidden=1792, n_heads=4, n_kv_heads=1, type_out=13),
    *[dict(type_default=t, type_v=t, type_down=t, tied=1, dim=4096, hidden=256, n_layers=1, n_heads=2, vocab=60000) for t in (12, 13, 14)]])
def test_kq_decode_equals_oracle_and_prompt_rows(gw, tmp_path, over):
    from oracle import oracle as orc
    path = synth.write_gguf(str(tmp_path / "m.gguf"), "tiny_kq", seed=5, **over)
    m = gw.Model(path, ctx_len=1280)
    om = orc.Model(path, cap=64)
    ids = np.random.default_rng(6).integers(0, m.vocab, 4).astype(np.int32)
    c = m.ctx(max_batch=8)
    s, so = m.seq(1280), om.seq()
    for t in ids:
        lg, ref = c.decode(s, int(t)), so.forward(int(t))
        assert _bits_equal(lg, ref), f"{over}: max diff {np.abs(lg - ref).max()}"
    s.fill_synthetic(1279, 3)
    for n in (255, 256, 1023, 1024, 1277):
        s.truncate(n)
        one = [c.decode(s, int(ids[0])), c.decode(s, int(ids[1]))]
        s.truncate(n)
        rows = c.prefill(s, ids[:2], mode=gw.RQ_LOGITS_ALL)
        assert _bits_equal(one[0], rows[0]) and _bits_equal(one[1], rows[1]), f"{over}: position {n}"
        s.fill_synthetic(1279, 3)


# the hidden row of a fused one-row pass (its final rmsnorm as a launch of its own, then the classifier on its codes) beside those
# of a prompt pass
@pytest.mark.parametrize("shape", ["tiny_kq", "tiny_q5k"])
def test_kq_hidden_rows_equal_prompt_rows(gw, synth_models, shape):
    m = gw.Model(synth_models(shape), ctx_len=64)
    c, a, b = m.ctx(max_batch=8), m.seq(64), m.seq(64)
    ids = np.random.default_rng(7).integers(0, m.vocab, 5).astype(np.int32)
    rows, hid = c.prefill_hidden(a, ids, mode=gw.RQ_LOGITS_ALL)
    for i, t in enumerate(ids):
        lg, h = c.decode_hidden(b, int(t))
        assert _bits_equal(lg, rows[i]) and _bits_equal(h, hid[i]), i
