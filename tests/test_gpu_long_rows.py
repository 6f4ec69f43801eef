"""Bit parity of the long-row Q4_0 matvec (rows of more than 18 packed groups, of more
than 12 in matrices of 1056 rows and more, at most eight per compute unit) with the CPU
oracle: a row's chains run as batons handed from lane to lane, fma by fma in the
reference's order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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


# the shortest rows it serves and the longest before them (12, 13, 18 and 19 groups; the
# last of 1 and 4 blocks), one and several tiles of phases, one and two rows per wave,
# ragged numbers of rows
@pytest.mark.parametrize("n,k", [(3, 2304), (3, 2336), (1055, 1568), (1056, 1568), (1057, 1536), (1024, 2432),
                                 (1, 1568), (5, 1664), (33, 1760), (1023, 2080), (1025, 2048), (2047, 1632), (7, 4096),
                                 (1030, 4128), (64, 8960), (1026, 8960)])
def test_long_rows_match_the_oracle(hip, O, n, k):
    rng = np.random.default_rng(n * 10007 + k)
    nb = k // 32
    w = np.zeros((n, nb, 20), np.uint8)
    s = (0.01 + 0.04 * rng.random((n, nb))).astype(np.float16)
    w[..., 0:2] = s.view(np.uint8).reshape(n, nb, 2)
    w[..., 2:4] = (-7.5 * s).astype(np.float16).view(np.uint8).reshape(n, nb, 2)
    w[..., 4:] = rng.integers(0, 256, (n, nb, 16), np.uint8)
    x = rng.standard_normal(k).astype(np.float32)
    bias = rng.standard_normal(max(n - 2, 1)).astype(np.float32)
    ops = hip.ops
    y = ops.DeviceBuffer(n * 4)
    ops.q4_0_gemv(ops.q4_0_upload(w.reshape(-1), n, k), ops.DeviceBuffer.from_array(x), y, n, k,
                  ops.DeviceBuffer.from_array(bias), bias.size)
    ops.synchronize()
    want = O.GenomicLinear(w.reshape(-1), b"", None, n, k, bias, 4).forward_core(x)
    assert np.array_equal(y.read(np.float32, n).view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("kwta", [0.0, 0.5])
def test_long_rows_in_a_decode_step(hip, O, tmp_models, kwta):
    """The down product (residual, from the SwiGLU's chain-major copy) and, with
    1664 hidden values, the attention output."""
    for name, cfg in (("ffn", dict(n_embd=128, n_head=4, n_head_kv=2, ffn=1696)),
                      ("embd", dict(n_embd=1664, n_head=26, n_head_kv=2, ffn=1568))):
        p = str(tmp_models / f"long_{name}.flat")
        hip.synth.write_flat(p, n_blocks=2, vocab_size=300, eps=1e-6, rope_base=1e4, arch_family=1, qkv_bias=1,
                             tied_embeddings=0, seed=5, **cfg)
        g, r = hip.load_genomic_auto(p), O.load_genomic(p)
        g.set_k_wta_ratio(kwta)
        r.set_k_wta_ratio(kwta)
        for i, t in enumerate([3, 141, 59]):
            a, b = g.forward(t, i == 0), r.forward_core(t, i == 0)
            assert np.array_equal(a.view(np.uint32), np.asarray(b, np.float32).view(np.uint32)), (name, i)
        g.close()


# odd numbers of blocks, partial workgroups, a table per row and block or the shared
# one, tables of only the first rows, and rows that leave LDS for one wave a workgroup; then
# both sides of the lines to a lane per chain (more rows than a round takes, short rows,
# a second round) and to the walk (three rounds)
@pytest.mark.parametrize("n,k,own", [(10240, 640, 10240), (10243, 640, 10243), (10243, 640, 5000), (24580, 672, 24580),
                                     (10250, 96, 10250), (10240, 96, 7), (10240, 896, -1), (10253, 928, -1),
                                     (6144, 3712, 6144), (6145, 3712, 6145), (3073, 8960, 3073),
                                     (9, 96, 9), (6, 32, 3), (21, 928, 21), (13, 928, -1), (7, 6016, 7), (10, 8960, 5),
                                     (5, 8992, -1)])
def test_lut4_rows_match_the_oracle(hip, O, n, k, own):
    codes, lut = hip.synth.lut4_tensor(41, f"long.{n}.{k}", n, k)
    lut = lut[:16 if own < 0 else own * (k // 32) * 16].copy()
    x, b = hip.synth.normal(42, f"x.{k}", k), hip.synth.normal(43, f"b.{n}", n)
    ops = hip.ops
    y = ops.DeviceBuffer(n * 4)
    dev = ops.DeviceBuffer.from_array
    ops.lut4_gemv(dev(codes), dev(lut), lut.size, dev(x), y, n, k, bias=dev(b), bias_len=n)
    ops.synchronize()
    want = O.GenomicLinear(codes, b"", lut, n, k, b, 4).forward_core(x)
    assert np.array_equal(y.read(np.float32, n).view(np.uint32), np.asarray(want, np.float32).view(np.uint32))
