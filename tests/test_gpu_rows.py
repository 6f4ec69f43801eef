"""Bit parity of the row-parallel products and prompts with the CPU oracle.

Several activation rows share one pass over the weights (q4_0_gemm, a bit-exact
prompt, a batch's steps and prompts).  Every row must be the oracle's
forward_core for that row alone, bit for bit: the row products run the same FMA
chains on the f32 matrix cores, and the rest of a block is the same arithmetic.
"""
import struct

import numpy as np
import pytest

from conftest import GNORM_MODEL, write_genomic_norm_model

pytestmark = pytest.mark.gpu

TINY = dict(n_embd=128, n_head=4, n_head_kv=2, n_blocks=2, ffn=256, vocab_size=1000, eps=1e-6,
            rope_base=1e4, arch_family=1, qkv_bias=1, tied_embeddings=0)
HD64 = dict(TINY, n_embd=256, ffn=544)
HD128 = dict(TINY, n_embd=384, n_head=3, n_head_kv=1, ffn=512, n_blocks=1)
LONG = dict(TINY, n_embd=128, n_head=2, n_head_kv=1, ffn=128, n_blocks=1, vocab_size=300)
NAN_TOKEN = 42


@pytest.fixture(scope="module")
def hip():
    import gaje_hip
    if gaje_hip.ops.device_count() < 1:
        pytest.fail("no HIP device visible")
    return gaje_hip


@pytest.fixture(scope="module")
def O():
    from oracle import oracle
    return oracle


def _same(a, b):
    """Equal bits, any NaN equal to any NaN."""
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    nan = np.isnan(a) & np.isnan(b)
    return a.shape == b.shape and bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | nan))


def _blocks(rng, n, k):
    nb = k // 32
    w = np.zeros((n, nb, 20), np.uint8)
    s = (0.01 + 0.04 * rng.random((n, nb))).astype(np.float16)
    w[..., 0:2] = s.view(np.uint8).reshape(n, nb, 2)
    w[..., 2:4] = (-7.5 * s).astype(np.float16).view(np.uint8).reshape(n, nb, 2)
    w[..., 4:] = rng.integers(0, 256, (n, nb, 16), np.uint8)
    return w.reshape(-1)


# rows below, at and past the 4-, 8-, 16- and 32-row tiles; last groups of 1, 2, 3 and 4
# blocks; one weight row; long sums; then products large enough for the 16 x 32 tiles,
# for the 32 x 64, of wide matrices at and past 16 rows, and of two rows on either side
# of the lines to two matvecs
@pytest.mark.parametrize("m,n,k", [(2, 1, 32), (3, 37, 96), (4, 8, 128), (5, 200, 160), (8, 33, 576), (9, 64, 896),
                                   (16, 65, 1536), (17, 31, 64), (31, 40, 224), (33, 129, 1152), (4, 24, 8960),
                                   (7, 40, 5888), (64, 16, 4864), (17, 4200, 64), (16, 5153, 1152),
                                   (33, 2600, 224), (66, 1310, 576), (100, 1000, 32), (70, 24608, 96), (65, 24610, 160),
                                   (16, 73794, 32), (17, 73794, 32), (2, 49152, 64), (2, 49153, 64), (2, 24577, 672),
                                   (2, 20481, 2816), (2, 20481, 2848), (3, 20481, 2848)])
def test_row_products_match_the_oracle(hip, O, m, n, k):
    rng = np.random.default_rng(m * 1000003 + n * 1009 + k)
    blocks, X = _blocks(rng, n, k), rng.standard_normal((m, k)).astype(np.float32)
    X[m - 1, :k // 2] *= np.float32(1e-38)     # no effect on bits: the row's flush hides subnormal sums
    if m > 2:
        X[1, k - 1], X[2, 0] = np.inf, np.nan  # stay in their own rows
    bias = rng.standard_normal(max(n - 3, 1)).astype(np.float32)
    ops = hip.ops
    Y = ops.DeviceBuffer(m * n * 4)
    ops.q4_0_gemm(ops.q4_0_upload(blocks, n, k), ops.DeviceBuffer.from_array(X), Y, m, n, k,
                  ops.DeviceBuffer.from_array(bias), bias.size)
    ops.synchronize()
    got = Y.read(np.float32, m * n).reshape(m, n)
    L = O.GenomicLinear(blocks, b"", None, n, k, bias, 4)
    for r in range(m):
        assert _same(got[r], L.forward_core(X[r])), f"row {r}"


def test_row_products_past_one_launch(hip, O):
    """More tiles than one launch holds (1048575 of 32 rows x 64): 33.6M activation rows, of
    which those at the ends and about the line are compared."""
    from gaje_hip._lib import check, lib
    line, n, k = 1048575 * 32, 64, 32
    m = line + 65
    rng = np.random.default_rng(3)
    blocks = _blocks(rng, n, k)
    ops = hip.ops
    X, Y = ops.DeviceBuffer(m * k * 4), ops.DeviceBuffer(m * n * 4)
    parts = {r0: rng.standard_normal((c, k)).astype(np.float32) for r0, c in ((0, 5), (line - 33, 70), (m - 20, 20))}
    for r0, x in parts.items():
        X.write(x, r0 * k * 4)
    ops.q4_0_gemm(ops.q4_0_upload(blocks, n, k), X, Y, m, n, k)
    ops.synchronize()
    L = O.GenomicLinear(blocks, b"", None, n, k, np.zeros(0, np.float32), 4)
    for r0, x in parts.items():
        got = np.empty((len(x), n), np.float32)
        check(lib().gaje_hip_memcpy_d2h(got.ctypes.data, Y.ptr + r0 * n * 4, got.nbytes))
        for r in range(len(x)):
            assert _same(got[r], L.forward_core(x[r])), f"row {r0 + r}"


def _write(hip, tmp_models, name, cfg):
    if cfg is GNORM_MODEL:
        return write_genomic_norm_model(str(tmp_models), seed=17)
    p = tmp_models / f"rows_{name}.flat"
    if not p.exists():
        hip.synth.write_flat(str(p), seed=61, **cfg)
    return str(p)


def _with_nan_token(path, out, n_embd):
    from oracle.flat import FlatFile
    ff, data = FlatFile(path), bytearray(open(path, "rb").read())
    off = ff.weights_offset + ff.tensors["token_embd"]["dna_off"] + NAN_TOKEN * n_embd * 4
    data[off:off + 4] = struct.pack("<f", float("nan"))
    open(out, "wb").write(bytes(data))
    return str(out)


def _oracle(O, path, kwta):
    r = O.load_genomic(path)
    r.set_k_wta_ratio(kwta)
    r.clear_cache_core()
    return r


# prompts of two tokens, of a few tiles, and of more rows than one pass takes, on an
# empty cache and after it; `long`'s second prompt has contexts past what the rows'
# attention holds in LDS; then numbers of rows and contexts on either side of the lines
# between that attention (whole tiles, ragged ones, on a cache) and one row at a time
@pytest.mark.parametrize("name,cfg,kwta,lengths", [("tiny", TINY, 0.0, [2, 33, 1]), ("tiny", TINY, 0.5, [19]),
                                                   ("hd64", HD64, 0.0, [65, 3]), ("hd128", HD128, 0.0, [130]),
                                                   ("gnorm", GNORM_MODEL, 0.0, [17]), ("tiny", TINY, 0.0, [2060]),
                                                   ("long", LONG, 0.0, [2490, 20]),
                                                   ("hd64", HD64, 0.0, [63, 1, 64, 64]), ("hd64", HD64, 0.0, [64, 127]),
                                                   ("hd64", HD64, 0.0, [128, 128, 192, 191]),
                                                   ("hd128", HD128, 0.0, [171, 170, 175, 186])])
def test_prompt_rows_match_the_oracle(hip, O, tmp_models, name, cfg, kwta, lengths):
    p = _write(hip, tmp_models, name, cfg)
    g, r = hip.load_genomic_auto(p), _oracle(O, p, kwta)
    g.set_k_wta_ratio(kwta)
    rng = np.random.default_rng(sum(lengths))
    for n in lengths:
        ids = rng.integers(0, cfg["vocab_size"], n).astype(np.uint32)
        got = g.prefill(ids, want_logits=True)
        for t in ids:
            want = r.forward_core(int(t))
        assert _same(got, want), f"prompt of {n}"
    assert g.cache_len() == sum(lengths)
    assert _same(g.forward(7), r.forward_core(7))
    g.close()


def test_prompt_rows_stop_at_a_guard(hip, O, tmp_models):
    p = _with_nan_token(_write(hip, tmp_models, "tiny", TINY), tmp_models / "rows_nan.flat", TINY["n_embd"])
    g, r = hip.load_genomic_auto(p), _oracle(O, p, 0.0)
    g.set_k_wta_ratio(0.0)
    ids = [5, 6, 7, 8, NAN_TOKEN, 9, 10]
    with pytest.raises(ValueError, match="Input x is NaN"):
        g.prefill(ids)
    assert g.cache_len() == 4
    for t in ids[:4]:
        r.forward_core(t)
    assert _same(g.forward(11), r.forward_core(11))
    g.close()


def test_batch_rows_with_gaps_and_a_guard(hip, O, tmp_models):
    """Skipped steps inside a prompt, a sequence that never runs, and one that a
    guard halts in the middle of its prompt while the others go on."""
    p = _with_nan_token(_write(hip, tmp_models, "tiny", TINY), tmp_models / "rows_nan.flat", TINY["n_embd"])
    g = hip.load_genomic_auto(p)
    g.set_k_wta_ratio(0.0)
    X = hip.BATCH_INACTIVE
    for nan_at in (None, 2):
        ids = np.array([[1, 2, X, 3, 4, 5], [9, 8, 7, 6, 5, 4], [X] * 6, [X, 11, 12, X, 13, 14]], np.uint32)
        if nan_at is not None:
            ids[1, nan_at] = NAN_TOKEN
        b = hip.GenomicBatch(g, 4, 64)
        logits, status, rc = b.feed(ids, want_logits=True, status=True)
        assert (rc == 0) == (nan_at is None)
        for s in (0, 1, 3):
            r = _oracle(O, p, 0.0)
            toks = [int(t) for t in ids[s] if t != X]
            if s == 1 and nan_at is not None:
                assert status[1] == 1 and b.cache_len(1) == nan_at
                continue
            assert status[s] == 0 and b.cache_len(s) == len(toks)
            for t in toks:
                want = r.forward_core(t)
            assert _same(logits[s], want), f"sequence {s}"
        assert b.cache_len(2) == 0
        b.close()
    g.close()


def test_batch_rows_past_the_tiled_attention(hip, O, tmp_models):
    """Two sequences in one pass, one with contexts past what the tiled attention holds
    in LDS (one row at a time, each in its own cache); then a prompt of whole tiles for
    the short one while the long one is idle."""
    p = _write(hip, tmp_models, "long", LONG)
    g = hip.load_genomic_auto(p)
    g.set_k_wta_ratio(0.0)
    X, rng = hip.BATCH_INACTIVE, np.random.default_rng(12)
    b, r = hip.GenomicBatch(g, 2, 2800), [_oracle(O, p, 0.0) for _ in range(2)]
    for lengths in ((2490, 3), (20, 17), (0, 257)):
        n = max(lengths)
        ids = np.full((2, n), X, np.uint32)
        for s, k in enumerate(lengths):
            ids[s, n - k:] = rng.integers(0, LONG["vocab_size"], k)
        logits = b.feed(ids, want_logits=True)
        for s, k in enumerate(lengths):
            for t in ids[s, n - k:]:
                want = r[s].forward_core(int(t))
            assert k == 0 or _same(logits[s], want), (lengths, s)
    assert (b.cache_len(0), b.cache_len(1)) == (2510, 277)
    b.close()
    g.close()


def _subnormal_weights_model(hip, O, tmp_models, values):
    """One block whose attention weights are subnormal wherever the values are not zero:
    token 7 scores about 95 below token 9 (the query is a bias in the slowest RoPE pair,
    the keys read elements 32.. of the normed embedding), token 9's values are zero and
    token 7's about 1e36 (a huge norm weight on elements ..31, which only the values
    read), or all zero without `values`."""
    from oracle.flat import FlatFile
    base = _write(hip, tmp_models, "hd64_1", dict(HD64, n_blocks=1))
    ff, data = FlatFile(base), bytearray(open(base, "rb").read())

    def view(name, dtype, what="dna"):
        e = ff.tensors[name]
        return np.frombuffer(data, dtype, e[what + "_len"] // np.dtype(dtype).itemsize, ff.weights_offset + e[what + "_off"])
    emb = view("token_embd", np.float32).reshape(-1, 256)
    norm, bias = view("blk.0.attn_norm", np.float32), view("blk.0.attn_qkv", np.float32, "bias")
    qkv = view("blk.0.attn_qkv", np.uint8).reshape(512, 8, 20)  # rows: 4 x 64 queries, 2 x 64 keys, 2 x 64 values
    emb[9, :32] = 0
    norm[:32], norm[32:] = 1e37 if values else 0, 1
    qkv[:256], qkv[256:384, 0], qkv[384:, 1:] = 0, 0, 0
    bias[:] = 0
    x = emb[[7, 9]] / np.sqrt((emb[[7, 9]].astype(np.float64) ** 2).mean(1, keepdims=True))
    for h in range(4):
        k = x @ O.q4_0_dequant(qkv[256 + 64 * (h // 2) + 31].reshape(-1).copy()).astype(np.float64)
        bias[64 * h + 31] = -95 * 8 / (k[0] - k[1])
    out = str(tmp_models / f"rows_subnormal_{int(values)}.flat")
    open(out, "wb").write(bytes(data))
    return out


def test_prompt_attention_keeps_subnormal_weights(hip, O, tmp_models):
    ids = np.full(130, 9, np.uint32)
    ids[[3, 40, 77, 100]] = 7
    want = []
    for values in (True, False):
        r = _oracle(O, _subnormal_weights_model(hip, O, tmp_models, values), 0.0)
        for t in ids:
            last = r.forward_core(int(t))
        want.append(last)
    assert np.mean(want[0] != want[1]) > 0.9  # what the subnormal weights carry reaches the logits
    g = hip.load_genomic_auto(_subnormal_weights_model(hip, O, tmp_models, True))
    g.set_k_wta_ratio(0.0)
    assert _same(g.prefill(ids, want_logits=True), want[0])
    g.close()
