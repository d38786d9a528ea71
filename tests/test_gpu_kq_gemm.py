"""The LDS-copied K-quant GEMMs (k_gemm_kql, k_gemm_kqt) against the oracle bit for bit, at the edges of their tiles, stages
and dispatch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import gwenedeg_amd as gw
    return torch, gw


# 12 Q4_K, 13 Q5_K, 14 Q6_K. k_gemm_kqt: above 32 rows, one to several stages (K / 256), row and column remainders of its
# 32 x 32 tiles; 6 .. 32 rows once its tiles are more than one per CU (8,193 weight rows); Q5_K from 9 rows. k_gemm_kql (Q4_K):
# 64 x 128 blocks that fill the CUs (25,700 weight rows, 33 rows; 1 row past a block: 25,601 at 65 and, with three stages, 9,601
# at 129; 12,801 at 129 leave two fifths of a round empty: k_gemm_kqt). 131,100-row Q6_K at 33 rows keeps k_gemm_kq (4 blocks
# per CU)
@pytest.mark.parametrize("typ,N,K,M", [
    (12, 31, 256, 33), (12, 33, 512, 64), (12, 200, 2560, 65), (12, 1000, 768, 97),
    (13, 33, 256, 33), (13, 200, 1024, 9), (13, 70, 512, 32), (13, 129, 768, 70),
    (14, 1, 256, 33), (14, 33, 512, 40), (14, 200, 2560, 65), (14, 130, 9728, 36),
    (12, 8193, 256, 6), (12, 8193, 512, 32), (13, 8193, 256, 7), (14, 8193, 256, 6), (14, 8200, 512, 31),
    (12, 25700, 256, 33), (12, 25601, 512, 65), (12, 12801, 768, 129), (12, 9601, 768, 129),
    (14, 131100, 256, 33)])
def test_lds_copied_kq_gemm_bitexact(dev, typ, N, K, M):
    torch, gw = dev
    from oracle import oracle as orc
    from gwenedeg_amd import synth
    rng = np.random.default_rng(typ * 1000 + N + M)
    sl = synth.synth_library()
    rb = sl.gw_synth_row_bytes(typ, K)
    base = np.zeros((min(N, 300), rb), np.uint8)  # (300 distinct rows, repeated shifted by one per repetition)
    w = rng.normal(0, 0.02, size=(len(base), K)).astype(np.float32)
    for r in range(len(base)):
        sl.gw_synth_encode_row(typ, base[r].ctypes.data, w[r].ctypes.data, K)
    idx = (np.arange(N) + np.arange(N) // len(base)) % len(base)
    xq, xs = orc.quantize(rng.normal(0, 1, size=(M, K)).astype(np.float32))
    xq[0, :64] = 127           # the largest group sums
    xq[M - 1, :32], xs[M - 1, 0] = 0, 0.0
    ref = orc.kq_matmul(typ, base, xq, xs, len(base), K)[:, idx]
    buf = torch.from_numpy(base[idx].reshape(-1)).cuda()
    out = torch.full((M + 1, N), 7.0, dtype=torch.float32, device="cuda")
    XQ, XS = torch.from_numpy(xq).cuda(), torch.from_numpy(xs).cuda()
    assert gw.lib.gw_kq_matmul(out.data_ptr(), typ, buf.data_ptr(), N, K, XQ.data_ptr(), XS.data_ptr(), M, None) == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.array_equal(got[:M].view(np.uint32), ref.view(np.uint32)), f"max diff {np.abs(got[:M] - ref).max()}"
    assert (got[M] == 7.0).all()


# q, k and v of a layer in one launch (9 .. 32 rows: k_gemm_kq32_3, above: k_gemm_kqt_3): each pair of types they take, and
# those they leave to launches of their own (Q6_K q / k beside Q4_K v); k and v of one tile and of several
@pytest.mark.parametrize("typ,typ_v", [(12, 14), (12, 12), (14, 14), (14, 12)])
@pytest.mark.parametrize("rows,heads,kv", [(9, 2, 1), (32, 6, 2), (17, 16, 8), (33, 2, 1), (65, 16, 8)])
def test_kq_qkv_launch_equals_oracle(dev, tmp_path, typ, typ_v, rows, heads, kv):
    _, gw = dev
    from oracle import oracle as orc
    from gwenedeg_amd import synth
    path = synth.write_gguf(str(tmp_path / "m.gguf"), "tiny_kq", seed=8, type_default=typ, type_v=typ_v, dim=768, n_heads=heads,
                            n_kv_heads=kv)
    m, so = gw.Model(path, ctx_len=80), orc.Model(path, cap=80).seq()
    ids = np.random.default_rng(rows).integers(0, m.vocab, rows).astype(np.int32)
    ref = np.stack([so.forward(int(t)) for t in ids])
    got = m.ctx(max_batch=80).prefill(m.seq(80), ids, mode=gw.RQ_LOGITS_ALL)
    assert np.array_equal(np.ascontiguousarray(got, np.float32).view(np.uint32), ref.astype(np.float32).view(np.uint32)), \
        f"max diff {np.abs(got - ref).max()}"


# w1 and w3 in one launch of k_gemm_kql (33 rows: 100 blocks of 128 weight rows each, 200 of the 256 CUs) and of k_gemm_kqt (80
# each), w2 of 50 and of 40 super-blocks
@pytest.mark.parametrize("hidden", [12800, 10240])
def test_kq_ffn_launch_equals_oracle(dev, tmp_path, hidden):
    _, gw = dev
    from oracle import oracle as orc
    from gwenedeg_amd import synth
    path = synth.write_gguf(str(tmp_path / "m.gguf"), "tiny_kq", seed=9, dim=256, hidden=hidden, n_heads=2, n_kv_heads=1, n_layers=1)
    m, so = gw.Model(path, ctx_len=64), orc.Model(path, cap=64).seq()
    ids = np.random.default_rng(hidden).integers(0, m.vocab, 33).astype(np.int32)
    ref = np.stack([so.forward(int(t)) for t in ids])
    got = m.ctx(max_batch=64).prefill(m.seq(64), ids, mode=gw.RQ_LOGITS_ALL)
    assert np.array_equal(np.ascontiguousarray(got, np.float32).view(np.uint32), ref.astype(np.float32).view(np.uint32)), \
        f"max diff {np.abs(got - ref).max()}"
