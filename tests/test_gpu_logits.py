"""The logits' way to the host: by a kernel up to 8 MB (float4s and a rest), by a copy above."""
import numpy as np
import pytest

from gwenedeg_amd import synth

pytestmark = pytest.mark.gpu


# 8,193 columns: 255 rows are 8,356,860 bytes, 256 rows 8,389,632 (past 8 MB); 1 and 2 rows leave 1 and 2 floats past the float4s
def test_logits_rows_equal_single_rows(tmp_path):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import gwenedeg_amd as gw
    m = gw.Model(synth.write_gguf(str(tmp_path / "m.gguf"), "tiny", seed=2, vocab=8193), ctx_len=1024)
    ids = np.random.default_rng(1).integers(0, m.vocab, 256).astype(np.int32)
    c1, c = m.ctx(max_batch=1), m.ctx(max_batch=256)
    s = m.seq(1024)
    one = np.stack([c1.decode(s, int(t)).copy() for t in ids])
    for n in (1, 2, 3, 255, 256):
        s.truncate(0)
        assert np.array_equal(c.prefill(s, ids[:n], mode=gw.RQ_LOGITS_ALL).view(np.uint32), one[:n].view(np.uint32)), n
