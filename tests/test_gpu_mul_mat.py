"""GPU parity of activation quantization, integer block dots, GEMV and the MFMA GEMM against
the CPU oracle (and, where it has been built, the reference's own CPU backend)."""
import numpy as np
import pytest

import orc

pytestmark = pytest.mark.gpu

TYPES = list(orc.WEIGHT_TYPES.items())


def _weights(rng, t, N, K, kind="oracle"):
    Wf = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    return orc.quantize_mt("ref" if (kind == "ref" and orc.ref is not None) else "oracle", t, Wf)


def _to_dev(dev, a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("K", [32, 256, 4096, 14336])
@pytest.mark.parametrize("dist", ["normal", "uniform", "special"])
def test_quantize_q8_1_bit_exact(dev, K, dist):
    import mi355
    rng = np.random.default_rng(7 + K)
    nrows = 5
    if dist == "normal":
        x = rng.standard_normal((nrows, K)).astype(np.float32)
    elif dist == "uniform":
        x = rng.uniform(-1, 1, (nrows, K)).astype(np.float32)
    else:
        x = rng.standard_normal((nrows, K)).astype(np.float32)
        x[0, :32] = 0.0                      # all-zero block: d = 0, q = 0, s = 0
        x[1, :32] = 0.0
        x[1, 5] = -3.25                      # single -amax: that level is exactly -127
        x[2, :32] = np.concatenate([[127.0], np.arange(31) - 15 + 0.5])   # d = 1: x*id lands on .5 ties (away from zero)
        x[3, :32] = 1e-30                    # tiny but non-zero scale
        x[4, :32] = 65504.0 * 100            # d overflows fp16 -> inf in the d field
    got = mi355.quantize_q8_1(_to_dev(dev, x)).cpu().numpy()
    want = orc.quantize("oracle", orc.Q8_1, x)
    assert np.array_equal(got, want)
    if orc.ref is not None:
        assert np.array_equal(got, orc.quantize("ref", orc.Q8_1, x))


@pytest.mark.parametrize("seed", [0, 1])
def test_quantize_q8_1_every_scale(dev, seed):
    """block maxima of every magnitude whose reciprocal scale is finite: the quotients by correction step agree with IEEE division on both sides of the range (2^-90 .. 2^90)
    they are used in, and levels that land on halves round away from zero"""
    import mi355
    rng = np.random.default_rng(seed)
    amax = np.ldexp(rng.uniform(1, 2, (64, 246)), np.arange(-118, 128)).astype(np.float32)      # one per block
    x = (rng.uniform(-1, 1, (64, 246, 32)) * amax[..., None]).astype(np.float32)
    ties = (rng.integers(-127, 127, (64, 246, 32)) + 0.5).astype(np.float32) * (amax / np.float32(127))[..., None]
    x = np.where(rng.random(x.shape) < 0.5, x, ties)
    x[..., 7] = np.where(rng.random(amax.shape) < 0.5, amax, -amax)
    x = np.clip(x, -amax[..., None], amax[..., None]).reshape(64, 246 * 32)
    got = mi355.quantize_q8_1(_to_dev(dev, x)).cpu().numpy()
    assert np.array_equal(got, orc.quantize("oracle", orc.Q8_1, x))


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("K", [256, 2048, 4096])
def test_weight_layout_round_trip(dev, name, t, K):
    """scatter (upload) then gather (read-back) returns the reference's bytes, also for partial ranges"""
    import torch
    import mi355
    rng = np.random.default_rng(11)
    N = 9
    raw = rng.integers(0, 256, (N, orc.row_bytes(t, K)), dtype=np.uint8)
    d_raw = _to_dev(dev, raw)
    d_dev = mi355.upload_weights(t, d_raw)
    back = mi355.download_weights(t, d_dev).cpu().numpy()
    assert np.array_equal(back, raw)
    # partial range, not block aligned
    lib = mi355.load()
    total = raw.size
    off, size = 37, total - 101
    part = torch.zeros(size, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_weights_gather(None, t, d_dev.data_ptr(), part.data_ptr(), K, N, off, size))
    torch.cuda.synchronize()
    assert np.array_equal(part.cpu().numpy(), raw.reshape(-1)[off:off + size])
    d2 = torch.zeros_like(d_dev)
    mi355.check(lib.mi355_weights_scatter(None, t, d_raw.reshape(-1)[:off].contiguous().data_ptr(), d2.data_ptr(), K, N, 0, off))
    mi355.check(lib.mi355_weights_scatter(None, t, d_raw.reshape(-1)[off:].contiguous().data_ptr(), d2.data_ptr(), K, N, off, total - off))
    torch.cuda.synchronize()
    assert torch.equal(d2, d_dev)


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("K", [2048, 4096, 14336])
def test_block_dots_bit_exact(dev, name, t, K):
    import mi355
    rng = np.random.default_rng(3)
    N = 33
    Wq = _weights(rng, t, N, K)
    x = rng.standard_normal((1, K)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    got = mi355.block_dots(t, Wd, _to_dev(dev, x)[0]).cpu().numpy()
    want = orc.block_dots(t, Wq, orc.quantize("oracle", orc.Q8_1, x)[0], K)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("N,K", [(4096, 4096), (1024, 14336), (257, 2048), (16, 256)])
@pytest.mark.parametrize("B", [1, 2, 3, 5, 8])
def test_gemv_matches_oracle(dev, name, t, N, K, B):
    import mi355
    rng = np.random.default_rng(N + K + B)
    Nt = min(N, 512)     # the oracle is scalar C: check a slice of rows exactly, all rows through the reference below
    Wq = _weights(rng, t, N, K, "ref")
    x = rng.standard_normal((B, K)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    got = mi355.mul_mat(t, Wd, _to_dev(dev, x)).cpu().numpy()
    want = orc.mul_mat("q8_1", t, Wq[:Nt], x)
    # same integer dots, f32 vs f64 scale algebra: only summation-order noise remains
    assert orc.nmse(got[:, :Nt], want) < 1e-9
    cpu = orc.mul_mat("ref", t, Wq, x) if orc.ref is not None else orc.mul_mat("cpu", t, Wq[:Nt], x)
    assert orc.nmse(got[:, :cpu.shape[1]], cpu) <= 5e-4      # tests/test-backend-ops.cpp:1916


@pytest.mark.parametrize("K", [256, 4096, 14336])
@pytest.mark.parametrize("dist", ["normal", "special"])
def test_quantize_q8k_bit_exact(dev, K, dist):
    """levels and scale equal block_q8_K of the reference; the sub-block sums are its bsums pairwise"""
    import mi355
    rng = np.random.default_rng(11 + K)
    nrows = 6
    x = rng.standard_normal((nrows, K)).astype(np.float32)
    if dist == "special":
        x[0, :256] = 0.0                       # all-zero super-block: d = 0, levels 0
        x[1, :256] = 0.0
        x[1, 77] = 2.5                         # single +amax: its level is exactly -127 and d is negative
        x[2, 3] = 9.0
        x[2, 200] = -9.0                       # equal magnitudes: the first one decides the sign of the scale
        x[3, :256] = -1e-30
        x[4, :256] = 0.0
        x[4, 0] = -127.0                       # scale exactly 1: the values below are exact .5 ties (round half to even)
        x[4, 1:202] = np.arange(-100, 101) + 0.5
    got = mi355.quantize_act_q8k(_to_dev(dev, x)).cpu().numpy()
    nsb = K // 256
    q = got[:nrows * K].view(np.int8).reshape(nrows, nsb, 256)
    d = got[nrows * K:nrows * K + nrows * nsb * 4].view(np.float32).reshape(nrows, nsb)
    off = (nrows * K + nrows * nsb * 4 + 15) // 16 * 16
    bs = got[off:off + nrows * nsb * 32].view(np.float16).reshape(nrows, nsb, 16).astype(np.int64)
    for kind in ["oracle"] + (["ref"] if orc.ref is not None else []):
        want = orc.quantize(kind, orc.Q8_K, x).reshape(nrows, nsb, 292)
        wd = np.ascontiguousarray(want[:, :, :4]).view(np.float32).reshape(nrows, nsb)
        wq = want[:, :, 4:260].view(np.int8)
        assert np.array_equal(d.view(np.uint32), wd.view(np.uint32))
        assert np.array_equal(q, wq)
        sums = wq.astype(np.int64).reshape(nrows, nsb, 8, 32).sum(axis=3)
        assert np.array_equal(64 * bs[:, :, 8:] + bs[:, :, :8], sums)
        assert bs[:, :, :8].min() >= 0 and bs[:, :, :8].max() <= 63


@pytest.mark.parametrize("seed", [0, 1])
def test_quantize_q8k_every_scale(dev, seed):
    """block maxima of every magnitude whose reciprocal scale is finite, the largest value of either sign at any place and several times over: both quotients and the choice
    of the first largest element agree with the host on both sides of the range (2^-90 .. 2^90) the correction steps are used in"""
    import mi355
    rng = np.random.default_rng(seed)
    nsb, nrows = 236, 24
    amax = np.ldexp(rng.uniform(1, 2, (nrows, nsb)), np.arange(-118, 118)).astype(np.float32)
    x = (rng.uniform(-1, 1, (nrows, nsb, 256)) * amax[..., None]).astype(np.float32)
    for _ in range(3):   # up to three elements of the largest magnitude
        at, sign = rng.integers(0, 256, (nrows, nsb, 1)), rng.choice([-1, 1], (nrows, nsb, 1)).astype(np.float32)
        np.put_along_axis(x, at, sign * amax[..., None], axis=2)
    x = x.reshape(nrows, nsb * 256)
    K = nsb * 256
    got = mi355.quantize_act_q8k(_to_dev(dev, x)).cpu().numpy()
    want = orc.quantize("oracle", orc.Q8_K, x).reshape(nrows, nsb, 292)
    assert np.array_equal(got[nrows * K:nrows * K + nrows * nsb * 4].view(np.uint32).reshape(nrows, nsb), np.ascontiguousarray(want[:, :, :4]).view(np.uint32).reshape(nrows, nsb))
    assert np.array_equal(got[:nrows * K].view(np.int8).reshape(nrows, nsb, 256), want[:, :, 4:260].view(np.int8))


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("N,K,B", [(512, 4096, 64), (384, 2048, 512), (130, 1024, 33), (4096, 4096, 9), (128, 14336, 100)])
def test_mmq_matches_oracle(dev, name, t, N, K, B):
    import mi355
    rng = np.random.default_rng(N * 3 + K + B)
    Wq = _weights(rng, t, N, K, "ref")
    x = rng.standard_normal((B, K)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    got = mi355.mul_mat(t, Wd, _to_dev(dev, x)).cpu().numpy()
    Nt, Bt = min(N, 64), min(B, 24)
    skinny = B <= 32 and K % 256 == 0 and (t != orc.Q6_K or K % 2048 == 0)   # up to 32 activation rows: the weight-streaming kernel, Q8_1 activations
    if B > 8 and not skinny and (t in (orc.Q4_K, orc.Q5_K) or (t == orc.Q6_K and K % 2048 == 0) or
                                 (t == orc.IQ4_XS and B >= 256 and K % 512 == 0)):   # Q6_K / IQ4_XS rows are 16-byte aligned only then
        # K-quants take the activation format of the CPU path (one scale per 256): integer sums are the
        # CPU's own (ggml-cpu-quants.c:6817-6848, 8262-8283), only the f32 summation order differs
        want = orc.mul_mat("cpu", t, Wq[:Nt], x[:Bt])
    else:
        want = orc.mul_mat("q8_1", t, Wq[:Nt], x[:Bt])
    assert orc.nmse(got[:Bt, :Nt], want) < 1e-11      # exact block dots, f32 sums over at most 448 blocks (an f16 block minimum would leave 1e-7)
    if orc.ref is not None:
        cpu = orc.mul_mat("ref", t, Wq, x)
        assert orc.nmse(got, cpu) <= 5e-4


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("N,K,B", [(100, 256, 5), (257, 1024, 8), (4096, 4096, 13), (1024, 14336, 17), (64, 3584, 24), (333, 2048, 32), (4096, 4096, 1),
                                   (77, 6144, 9)])
@pytest.mark.parametrize("split", [False, True])
def test_skinny_matches_oracle(dev, name, t, N, K, B, split):
    """the weight-streaming matrix-core kernel for a few activation rows: ragged row and batch counts, K that does not divide
    evenly over the four waves, with and without slices along K, with a residual"""
    import mi355
    if t == orc.Q6_K and K % 2048 != 0:
        pytest.skip("Q6_K rows are 16-byte aligned only when K is a multiple of 2048")
    if t == orc.IQ4_XS and K % 512 != 0:
        pytest.skip("IQ4_XS rows (136 bytes per super-block) are 16-byte aligned only when K is a multiple of 512")
    rng = np.random.default_rng(N * 5 + K + B)
    Wq = _weights(rng, t, N, K, "ref")
    x = rng.standard_normal((B, K)).astype(np.float32)
    res = rng.standard_normal((B, N)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    got = mi355.mul_mat_skinny(t, Wd, _to_dev(dev, x), split=split).cpu().numpy()
    got_res = mi355.mul_mat_skinny(t, Wd, _to_dev(dev, x), residual=_to_dev(dev, res), split=split).cpu().numpy()
    assert np.array_equal(got_res, got + res)
    Nt, Bt = min(N, 64), min(B, 24)
    want = orc.mul_mat("q8_1", t, Wq[:Nt], x[:Bt])
    assert orc.nmse(got[:Bt, :Nt], want) < 1e-9      # exact integer dots; f32 against f64 scale algebra
    if orc.ref is not None:
        assert orc.nmse(got, orc.mul_mat("ref", t, Wq, x)) <= 5e-4      # tests/test-backend-ops.cpp:1916


@pytest.mark.parametrize("N,K,B", [(100, 256, 33), (257, 1024, 64), (4096, 4096, 50), (1024, 14336, 100), (64, 3584, 128), (333, 2048, 96), (77, 6144, 65),
                                   (130, 512, 20), (4096, 4096, 128), (512, 4096, 40)])
@pytest.mark.parametrize("split", [False, True])
def test_mid_matches_oracle(dev, N, K, B, split):
    """the weight-streaming matrix-core kernel for 33..128 activation rows on Q4_K (sub-block scales folded into two int8 operand
    planes): the CPU path's integer sums (ggml-cpu-quants.c:6817-6848) - ragged row and batch counts, both activation halves, K that
    does not divide evenly over the four waves, with and without slices along K, with a residual"""
    import mi355
    t = orc.Q4_K
    rng = np.random.default_rng(N * 5 + K + B)
    Wq = _weights(rng, t, N, K, "ref")
    x = rng.standard_normal((B, K)).astype(np.float32)
    res = rng.standard_normal((B, N)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    got = mi355.mul_mat_mid(t, Wd, _to_dev(dev, x), split=split).cpu().numpy()
    got_res = mi355.mul_mat_mid(t, Wd, _to_dev(dev, x), residual=_to_dev(dev, res), split=split).cpu().numpy()
    assert np.array_equal(got_res, got + res)
    Nt = min(N, 48)
    assert orc.nmse(got[:, :Nt], orc.mul_mat("cpu", t, Wq[:Nt], x)) < 1e-9          # every activation row, the first weight rows
    assert orc.nmse(got[B - 9:, N - 40:], orc.mul_mat("cpu", t, Wq[N - 40:], x[B - 9:])) < 1e-9
    if orc.ref is not None:
        assert orc.nmse(got, orc.mul_mat("ref", t, Wq, x)) <= 5e-4      # tests/test-backend-ops.cpp:1916
    if B > 32:   # mi355_mul_mat takes this kernel for 33..128 rows
        assert np.array_equal(mi355.mul_mat(t, Wd, _to_dev(dev, x), split=split).cpu().numpy(), got)


@pytest.mark.parametrize("N,K,B,split", [(4096, 4096, 128, True), (4096, 14336, 64, True), (2048, 1024, 100, True), (4096, 4096, 128, False), (8192, 2048, 50, True)])
def test_mid_norm_equals_product_then_norm(dev, N, K, B, split):
    """the 33..128-row product (+ residual) -> RMS_NORM -> MUL(weight) -> tile image as one call: the bits of the product followed by
    the norm launch, in the row, in the normalised row and in the image"""
    import torch
    import mi355
    lib = mi355.load()
    t = orc.Q4_K
    rng = np.random.default_rng(N + K + B)
    xd = _to_dev(dev, rng.standard_normal((B, K)).astype(np.float32))
    act = mi355.quantize_act_q8k_tiled(xd)
    Wd = mi355.upload_weights(t, _to_dev(dev, _weights(rng, t, N, K, "ref")))
    res = _to_dev(dev, rng.standard_normal((B, N)).astype(np.float32))
    nw = _to_dev(dev, rng.standard_normal(N).astype(np.float32))
    want_x = mi355.mul_mat_mid(t, Wd, xd, residual=res, split=split)
    want_y = torch.empty((B, N), dtype=torch.float32, device=dev)
    want_img = torch.zeros(lib.mi355_act_q8k_tiled_bytes(N, B), dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_rms_norm_mul_quant_q8k_tiled(None, want_x.data_ptr(), N, nw.data_ptr(), want_y.data_ptr(), N, want_img.data_ptr(), N, B, 1e-5))
    got_x = torch.empty((B, N), dtype=torch.float32, device=dev)
    got_y = torch.empty((B, N), dtype=torch.float32, device=dev)
    got_img = torch.zeros_like(want_img)
    nws = lib.mi355_mul_mat_mid_ws_bytes(N, K, B) if split else 0
    ws = torch.empty(max(nws, 16), dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_mul_mat_mid_norm(None, t, Wd.data_ptr(), act.data_ptr(), got_x.data_ptr(), res.data_ptr(), N, K, B, N, ws.data_ptr() if nws else None, nws,
                                           nw.data_ptr(), 1e-5, got_y.data_ptr(), N, got_img.data_ptr()))
    torch.cuda.synchronize()
    assert np.array_equal(got_x.cpu().numpy(), want_x.cpu().numpy())
    assert np.array_equal(got_y.cpu().numpy(), want_y.cpu().numpy())
    assert np.array_equal(got_img.cpu().numpy(), want_img.cpu().numpy())


@pytest.mark.parametrize("Ns,K,B", [((4096, 1024, 1024), 4096, 128), ((14336, 14336), 4096, 64), ((100, 257, 64), 2048, 100), ((2048, 512), 1024, 40)])
@pytest.mark.parametrize("split", [False, True])
def test_mid_multi_equals_single_launches(dev, Ns, K, B, split):
    """up to three Q4_K matrices on one activation in one launch of the 33..128-row kernel: without slices every matrix has the bits of
    its own launch; with slices (chosen for the launch as a whole) the same integer sums in another f32 order; residuals per matrix"""
    import mi355
    t = orc.Q4_K
    rng = np.random.default_rng(sum(Ns) + K + B)
    x = rng.standard_normal((B, K)).astype(np.float32)
    Wq = [_weights(rng, t, N, K, "ref") for N in Ns]
    Wd = [mi355.upload_weights(t, _to_dev(dev, W)) for W in Wq]
    res = [_to_dev(dev, rng.standard_normal((B, N)).astype(np.float32)) if i != 1 else None for i, N in enumerate(Ns)]
    xd = _to_dev(dev, x)
    alone = [mi355.mul_mat_mid(t, W, xd, split=False).cpu().numpy() for W in Wd]
    multi = [o.cpu().numpy() for o in mi355.mul_mat_mid_multi(t, Wd, xd, split=split)]
    with_res = [o.cpu().numpy() for o in mi355.mul_mat_mid_multi(t, Wd, xd, residuals=res, split=split)]
    for i, N in enumerate(Ns):
        if not split:
            assert np.array_equal(multi[i], alone[i])
        assert orc.nmse(multi[i], alone[i]) < 1e-12
        assert np.array_equal(with_res[i], multi[i] + res[i].cpu().numpy() if res[i] is not None else multi[i])
        Nt = min(N, 40)
        assert orc.nmse(multi[i][:, :Nt], orc.mul_mat("cpu", t, Wq[i][:Nt], x)) < 1e-9
        assert orc.nmse(multi[i][B - 5:, N - 7:], orc.mul_mat("cpu", t, Wq[i][N - 7:], x[B - 5:])) < 1e-9


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("N,K", [(14336, 4096), (4096, 14336)])
def test_mmq_llama8b_ffn_shapes(dev, name, t, N, K):
    """the FFN products of an 8B llama (gate/up 14336 x 4096, down 4096 x 14336) at batch 64 and 512, whole: every output against
    the reference CPU backend (NMSE <= 5e-4, tests/test-backend-ops.cpp:1916), a 64 x 24 corner and the last rows/columns against
    the oracle's integer arithmetic; the K-quants additionally through their tile images"""
    import mi355
    rng = np.random.default_rng(N + K + t)
    Wq = _weights(rng, t, N, K, "ref")
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    kq = t in (orc.Q4_K, orc.Q5_K, orc.Q6_K, orc.IQ4_XS)
    tiles = mi355.kq_unpack_tiles(t, Wd) if kq else None
    for B in (64, 512):
        x = rng.standard_normal((B, K)).astype(np.float32)
        xd = _to_dev(dev, x)
        got = mi355.mul_mat(t, Wd, xd).cpu().numpy()
        # K-quants (IQ4_XS from 256 rows on) compute in the CPU path's Q8_K format, the others in Q8_1
        kind = "cpu" if (kq and (t != orc.IQ4_XS or B >= 256)) else "q8_1"
        corner = orc.mul_mat(kind, t, Wq[:64], x[:24])
        edge = orc.mul_mat(kind, t, Wq[N - 9:], x[B - 3:])
        assert orc.nmse(got[:24, :64], corner) < 1e-11      # exact block dots, f32 sums over at most 448 blocks
        assert orc.nmse(got[B - 3:, N - 9:], edge) < 1e-11
        want = orc.mul_mat_all(t, Wq, x)
        assert orc.nmse(got, want) <= 5e-4
        if kq:
            act = mi355.quantize_act_q8k_tiled(xd)
            wide = mi355.mul_mat_q8k_tiled(t, tiles, act, N, K, B).cpu().numpy()
            assert orc.nmse(wide, want) <= 5e-4
            if kind == "cpu":
                assert orc.nmse(wide[:24, :64], corner) < 1e-9
                assert orc.nmse(wide[B - 3:, N - 9:], edge) < 1e-9
                assert orc.nmse(wide, got) < 1e-12      # same integer sums in both tile kernels
            else:
                assert orc.nmse(wide[:24, :64], orc.mul_mat("cpu", t, Wq[:64], x[:24])) < 1e-9


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t in (orc.Q4_K, orc.Q6_K)])
@pytest.mark.parametrize("N,K,B", [(256, 4096, 64), (130, 1024, 33)])
def test_mmq_q8_1_path_for_k_quants(dev, name, t, N, K, B):
    """the per-32-block tile kernel stays reachable for K-quants through mi355_mul_mat_q"""
    import mi355
    import torch
    rng = np.random.default_rng(N + K + B)
    Wq = _weights(rng, t, N, K)
    x = rng.standard_normal((B, K)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    act = mi355.quantize_act(_to_dev(dev, x))
    dst = torch.empty((B, N), dtype=torch.float32, device=dev)
    mi355.check(mi355.load().mi355_mul_mat_q(None, t, Wd.data_ptr(), act.data_ptr(), dst.data_ptr(), N, K, B, N))
    torch.cuda.synchronize()
    assert orc.nmse(dst.cpu().numpy()[:24, :64], orc.mul_mat("q8_1", t, Wq[:64], x[:24])) < 1e-11


@pytest.mark.parametrize("name,t", TYPES)
def test_unaligned_rows_fallback(dev, name, t):
    """a matrix at an odd address (byte-load kernel), with rows that are no 16-byte multiples, and the same rows at an even one"""
    import torch
    import mi355
    rng = np.random.default_rng(5)
    be = orc.BLOCK[t][0]
    K = be * 3
    for B in (1, 12, 40):
        Wq = _weights(rng, t, 19, K)
        x = rng.standard_normal((B, K)).astype(np.float32)
        Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
        odd = torch.empty(Wd.numel() + 17, dtype=torch.uint8, device=dev)
        odd = odd[1 + (-odd.data_ptr()) % 2:][:Wd.numel()].reshape(Wd.shape)
        odd.copy_(Wd)
        assert odd.data_ptr() % 2 == 1
        got = mi355.mul_mat(t, odd, _to_dev(dev, x)).cpu().numpy()
        assert orc.nmse(got, orc.mul_mat("q8_1", t, Wq, x)) < 1e-11      # f32 products of f32 weights and activations
        got = mi355.mul_mat(t, Wd, _to_dev(dev, x)).cpu().numpy()
        # Q4_K and Q5_K rows are always 16-byte aligned, so B > 32 takes the super-block tile kernels and the CPU's activation format
        # (5..32 rows: the weight-streaming kernel with Q8_1 activations)
        want = orc.mul_mat("cpu" if (t in (orc.Q4_K, orc.Q5_K) and B > 32) else "q8_1", t, Wq, x)
        assert orc.nmse(got, want) < 1e-11


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t not in (orc.Q4_K, orc.Q5_K)])   # those two are 16-byte aligned at any K
@pytest.mark.parametrize("blocks", [1, 7, 9, 43, 47])
def test_ragged_rows(dev, name, t, blocks):
    """rows that start at any even address and whose length is no whole number of the kernels' K steps: GEMV, weight-streaming and tile
    kernels, with and without slices along K, against exact integer block dots (f32 sums: NMSE of some 1e-14)"""
    import mi355
    rng = np.random.default_rng(blocks)
    K = orc.BLOCK[t][0] * blocks
    N = 150
    Wq = _weights(rng, t, N, K)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    for B in (1, 3, 4, 8, 9, 32, 33, 130):
        x = rng.standard_normal((B, K)).astype(np.float32)
        want = orc.mul_mat("q8_1", t, Wq, x)
        for split in (False, True):
            got = mi355.mul_mat(t, Wd, _to_dev(dev, x), split=split).cpu().numpy()
            assert orc.nmse(got, want) < 1e-11, (B, split)


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("K", [1280, 2048])
def test_ragged_last_column_tile(dev, name, t, K):
    """batches whose last 128-column tile holds 1, 64, 65 and 128 columns (up to 64 it runs with half the columns per wave): every column
    against the same arithmetic on the CPU; integer sums are exact, f32 sums over at most 64 blocks leave an NMSE of some 1e-14"""
    import mi355
    rng = np.random.default_rng(K)
    N = 130
    Wq = _weights(rng, t, N, K)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    x = rng.standard_normal((384, K)).astype(np.float32)
    for B in (129, 192, 193, 256, 257, 320, 321):
        aligned = K % 2048 == 0 or t in (orc.Q4_K, orc.Q5_K)
        q8k = (t in (orc.Q4_K, orc.Q5_K, orc.Q6_K) or (t == orc.IQ4_XS and B >= 256)) and aligned
        want = orc.mul_mat("cpu" if q8k else "q8_1", t, Wq, x[:B])
        for split in (False, True):
            got = mi355.mul_mat(t, Wd, _to_dev(dev, x[:B]), split=split).cpu().numpy()
            assert orc.nmse(got, want) < 1e-11, (B, split)


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t in (orc.Q4_K, orc.Q5_K, orc.Q6_K, orc.IQ4_XS)])
@pytest.mark.parametrize("nsb", [1, 2, 3, 4, 5, 8, 16])
def test_q8k_tile_stages_and_rows(dev, name, t, nsb):
    """the super-block tile kernel walks K in pairs of super-blocks with the last one or two apart, on tiles of 64 rows (few of them) or
    128, with half or all of the columns per wave: integer sums are exact, f32 sums over at most 16 super-blocks leave an NMSE of some
    1e-14.  The large matrix repeats 65 rows, so every output has an equal among the checked ones."""
    import torch
    import mi355
    K = 256 * nsb
    if (t == orc.Q6_K and K % 2048) or (t == orc.IQ4_XS and K % 512):
        pytest.skip("rows of no multiple of 16 bytes do not run here")
    rng = np.random.default_rng(nsb)
    Wq = _weights(rng, t, 65, K)
    x = rng.standard_normal((100, K)).astype(np.float32)
    want = orc.mul_mat("cpu", t, Wq, x)
    for reps, N in ((2, 130), (260, 65 * 260)):
        Wd = mi355.upload_weights(t, _to_dev(dev, np.tile(Wq, (reps, 1))))
        for B in (1, 33, 64, 65, 100):
            act = mi355.quantize_act_q8k(_to_dev(dev, x[:B]))
            got = torch.empty((B, N), dtype=torch.float32, device=dev)
            mi355.check(mi355.load().mi355_mul_mat_q8k(None, t, Wd.data_ptr(), act.data_ptr(), got.data_ptr(), N, K, B, N))
            torch.cuda.synchronize()
            first = got[:, :65].cpu().numpy()
            assert orc.nmse(first, want[:B]) < 1e-11, (N, B)
            assert torch.equal(got.view(B, reps, 65), got[:, None, :65].expand(B, reps, 65)), (N, B)


KQ_TYPES = [(n, t) for n, t in TYPES if t in (orc.Q4_K, orc.Q6_K)]
TILED_TYPES = [(n, t) for n, t in TYPES if t in (orc.Q4_K, orc.Q5_K, orc.Q6_K, orc.IQ4_XS)]   # types with tile images for the wide-tile GEMM


def _tile_off(row, k, K):
    """byte offset of element (row, k) in a tile image (16 rows x 64 elements per 1 KiB tile, chunk c of row r at c ^ ((r >> 2) & 3))"""
    r, c = row & 15, (k >> 4) & 3
    return ((row >> 4) * (K >> 6) + (k >> 6)) * 1024 + r * 64 + ((c ^ ((r >> 2) & 3)) << 4) + (k & 15)


def _slabs_written(ws, N, B):
    """how many [B][N] slabs a product has left in a workspace that was NaN before"""
    import torch
    return int((~torch.isnan(ws)).sum().item()) / (N * B)


@pytest.mark.parametrize("t,N,K,B,slabs", [(orc.Q4_0, 4096, 2048, 900, 2), (orc.Q6_K, 4096, 2048, 900, 2), (orc.Q4_0, 2688, 2048, 1000, 3), (orc.Q4_0, 4096, 2048, 130, 4),
                                           (orc.Q4_0, 4096, 4096, 300, 5), (orc.Q4_0, 1028, 2048, 256, 8), (orc.Q6_K, 4096, 11008, 140, 8), (orc.Q4_0, 768, 8192, 70, 16),
                                           (orc.Q6_K, 1024, 14336, 200, 16)])
def test_slab_sums_by_four_and_by_one(dev, t, N, K, B, slabs):
    """products cut along K into two, three, four and more slabs (counted), summed into dst rows that allow 16-byte stores and into rows one float apart from that (small ones by one
    element per lane either way): the same bits, nothing between the rows is touched, and the values are the oracle's for these operands"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(N + K + B)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((N, K)) * 0.05).astype(np.float32))
    x = rng.standard_normal((B, K)).astype(np.float32)
    Wd, act = mi355.upload_weights(t, _to_dev(dev, Wq)), mi355.quantize_act(_to_dev(dev, x))
    wide, odd = torch.full((B, N + 4), 7.0, device=dev), torch.full((B, N + 5), 7.0, device=dev)
    for dst in (wide, odd):
        ws = torch.full((20 * N * B,), float("nan"), device=dev)
        mi355.check(lib.mi355_mul_mat_q_ws(None, t, Wd.data_ptr(), act.data_ptr(), dst.data_ptr(), N, K, B, dst.stride(0), ws.data_ptr(), ws.numel() * 4))
        assert _slabs_written(ws, N, B) == slabs
    assert torch.equal(wide[:, :N], odd[:, :N]) and bool((wide[:, N:] == 7.0).all()) and bool((odd[:, N:] == 7.0).all())
    got = wide.cpu().numpy()
    assert orc.nmse(got[:24, :64], orc.mul_mat("q8_1", t, Wq[:64], x[:24])) < 1e-11
    assert orc.nmse(got[B - 3:, N - 9:N], orc.mul_mat("q8_1", t, Wq[N - 9:], x[B - 3:])) < 1e-11


@pytest.mark.parametrize("t,N,K,B,slabs", [(orc.Q4_K, 4096, 4096, 300, 2), (orc.Q4_K, 3072, 2048, 300, 3), (orc.Q4_K, 1024, 2048, 65, 4), (orc.Q5_K, 3072, 8192, 130, 5),
                                           (orc.Q4_K, 1536, 4096, 300, 6), (orc.Q6_K, 1024, 14336, 200, 8)])
@pytest.mark.parametrize("add", [False, True])
def test_slab_sums_of_tile_products(dev, t, N, K, B, slabs, add):
    """the same for the products of tile images, with a residual that is dst itself and without"""
    import torch
    import mi355
    lib = mi355.load()
    assert lib.mi355_mul_mat_q8k_tiled_ws_bytes(N, K, B) == slabs * N * B * 4
    rng = np.random.default_rng(N + K + B)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((N, K)) * 0.05).astype(np.float32))
    x, res = (rng.standard_normal(shape).astype(np.float32) for shape in ((B, K), (B, N)))
    tiles = mi355.kq_unpack_tiles(t, mi355.upload_weights(t, _to_dev(dev, Wq)))
    act = mi355.quantize_act_q8k_tiled(_to_dev(dev, x))
    got = []
    for pad in (4, 5):
        dst = torch.full((B, N + pad), 7.0, device=dev)
        dst[:, :N] = _to_dev(dev, res)
        ws = torch.full((slabs * N * B,), float("nan"), device=dev)
        mi355.check(lib.mi355_mul_mat_q8k_tiled(None, t, tiles.data_ptr(), act.data_ptr(), dst.data_ptr(), dst.data_ptr() if add else None, N, K, B, dst.stride(0), ws.data_ptr(),
                                                ws.numel() * 4))
        assert _slabs_written(ws, N, B) == slabs and bool((dst[:, N:] == 7.0).all())
        got.append(dst[:, :N].cpu().numpy())
    assert np.array_equal(*got)
    for b, n in ((slice(0, 24), slice(0, 64)), (slice(B - 3, B), slice(N - 9, N))):
        assert orc.nmse(got[0][b, n], orc.mul_mat("cpu", t, Wq[n], x[b]) + (res[b, n] if add else 0)) < 1e-9


@pytest.mark.parametrize("K,B", [(256, 5), (4096, 33), (14336, 130)])
def test_quantize_q8k_tiled_bit_exact(dev, K, B):
    """the tile-image form holds the same levels, scales and sub-block sums as block_q8_K of the reference"""
    import mi355
    rng = np.random.default_rng(23 + K)
    x = rng.standard_normal((B, K)).astype(np.float32)
    x[0, :256] = 0.0
    got = mi355.quantize_act_q8k_tiled(_to_dev(dev, x)).cpu().numpy()
    nsb, b16 = K // 256, (B + 15) // 16 * 16
    cb_pad = ((b16 // 16) + 15) // 16 * 16
    rows, ks = np.meshgrid(np.arange(B), np.arange(K), indexing="ij")
    q = got[_tile_off(rows, ks, K)].view(np.int8).reshape(B, nsb, 256)
    aux = got[b16 * K:]
    want = orc.quantize("oracle", orc.Q8_K, x).reshape(B, nsb, 292)
    wd = np.ascontiguousarray(want[:, :, :4]).view(np.float32).reshape(B, nsb)
    wq = want[:, :, 4:260].view(np.int8)
    assert np.array_equal(q, wq)
    sums = wq.astype(np.int64).reshape(B, nsb, 8, 32).sum(axis=3)
    for b in range(B):
        for sb in range(nsb):
            e = aux[(sb * cb_pad + b // 16) * 576:][:576]
            d = e[:64].view(np.float32)[b % 16]
            bs = e[64:].view(np.float16).reshape(16, 16)[b % 16].astype(np.int64)
            assert d.view(np.uint32) == wd[b, sb].view(np.uint32)
            assert np.array_equal(64 * bs[8:] + bs[:8], sums[b, sb])
    if orc.ref is not None:
        assert np.array_equal(want, orc.quantize("ref", orc.Q8_K, x).reshape(B, nsb, 292))


@pytest.mark.parametrize("name,t", TILED_TYPES)
@pytest.mark.parametrize("N,K,B", [(512, 4096, 64), (384, 2048, 512), (130, 2048, 33), (128, 14336, 100), (200, 2048, 77), (1000, 6144, 300),
                                   (200, 2048, 250), (1000, 6144, 450), (4096, 4096, 512)])     # 193+ rows: 256-row column tiles where the last is over half full
@pytest.mark.parametrize("split", [False, True])
def test_mmq_tiled_matches_oracle(dev, name, t, N, K, B, split):
    """the wide-tile K-quant GEMM on tile images: the CPU's own integer sums (ggml-cpu-quants.c:6817-6848, 8262-8283), ragged row and
    batch counts, with and without slices along K, with a residual; against the oracle, ggml-cpu and the 64 x 128 tile kernel"""
    import torch
    import mi355
    rng = np.random.default_rng(N * 7 + K + B)
    Wq = _weights(rng, t, N, K, "ref")
    x = rng.standard_normal((B, K)).astype(np.float32)
    res = rng.standard_normal((B, N)).astype(np.float32)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    tiles = mi355.kq_unpack_tiles(t, Wd)
    act = mi355.quantize_act_q8k_tiled(_to_dev(dev, x))
    got = mi355.mul_mat_q8k_tiled(t, tiles, act, N, K, B, split=split).cpu().numpy()
    got_res = mi355.mul_mat_q8k_tiled(t, tiles, act, N, K, B, residual=_to_dev(dev, res), split=split).cpu().numpy()
    assert np.array_equal(got_res, got + res)
    if B > 192 and not split:   # the 128 x 256 tile kernel holds the bits of the 128 x 128 one (which a 128-row batch takes)
        a128 = mi355.quantize_act_q8k_tiled(_to_dev(dev, x[B - 128:]))
        assert np.array_equal(got[B - 128:], mi355.mul_mat_q8k_tiled(t, tiles, a128, N, K, 128, split=False).cpu().numpy())
    Nt, Bt = min(N, 64), min(B, 24)
    assert orc.nmse(got[:Bt, :Nt], orc.mul_mat("cpu", t, Wq[:Nt], x[:Bt])) < 1e-9
    # the last rows and columns (partial tiles)
    assert orc.nmse(got[B - 5:, N - 7:], orc.mul_mat("cpu", t, Wq[N - 7:], x[B - 5:])) < 1e-9
    if True:   # the 64 x 128 tile kernel that unpacks the packed rows itself
        old = torch.empty((B, N), dtype=torch.float32, device=dev)
        a2 = mi355.quantize_act_q8k(_to_dev(dev, x))
        mi355.check(mi355.load().mi355_mul_mat_q8k(None, t, Wd.data_ptr(), a2.data_ptr(), old.data_ptr(), N, K, B, N))
        torch.cuda.synchronize()
        assert orc.nmse(got, old.cpu().numpy()) < 1e-12      # same integer sums, f32 summation order only
    if orc.ref is not None:
        assert orc.nmse(got, orc.mul_mat("ref", t, Wq, x)) <= 5e-4      # tests/test-backend-ops.cpp:1916


@pytest.mark.parametrize("name,t", KQ_TYPES)
def test_fused_producers_write_tile_images(dev, name, t):
    """RMS_NORM+MUL and SiLU*up with the tile-image activation output equal the separate quantization of their f32 result"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(3)
    B, K = 37, 4096
    x = _to_dev(dev, rng.standard_normal((B, K)).astype(np.float32))
    w = _to_dev(dev, rng.standard_normal(K).astype(np.float32))
    nbytes = lib.mi355_act_q8k_tiled_bytes(K, B)
    y = torch.empty((B, K), dtype=torch.float32, device=dev)
    a1 = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_rms_norm_mul_quant_q8k_tiled(None, x.data_ptr(), K, w.data_ptr(), y.data_ptr(), K, a1.data_ptr(), K, B, 1e-5))
    a2 = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_quantize_act_q8k_tiled(None, y.data_ptr(), a2.data_ptr(), K, B, K))
    torch.cuda.synchronize()
    rows, ks = np.meshgrid(np.arange(B), np.arange(K), indexing="ij")
    sel = _tile_off(rows, ks, K)
    assert np.array_equal(a1.cpu().numpy()[sel], a2.cpu().numpy()[sel])
    b16 = (B + 15) // 16 * 16
    n1, n2 = a1.cpu().numpy()[b16 * K:], a2.cpu().numpy()[b16 * K:]
    cb_pad = ((b16 // 16) + 15) // 16 * 16
    for sb in range(K // 256):
        for cb in range(b16 // 16):
            nrow = min(16, B - cb * 16)
            e1, e2 = n1[(sb * cb_pad + cb) * 576:][:576], n2[(sb * cb_pad + cb) * 576:][:576]
            assert np.array_equal(e1[:4 * nrow], e2[:4 * nrow]) and np.array_equal(e1[64:64 + 32 * nrow], e2[64:64 + 32 * nrow])
    g = _to_dev(dev, rng.standard_normal((B, K)).astype(np.float32))
    u = _to_dev(dev, rng.standard_normal((B, K)).astype(np.float32))
    a3 = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_swiglu_quant_q8k_tiled(None, g.data_ptr(), u.data_ptr(), K, y.data_ptr(), K, a3.data_ptr(), K, B))
    a4 = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_quantize_act_q8k_tiled(None, y.data_ptr(), a4.data_ptr(), K, B, K))
    torch.cuda.synchronize()
    assert np.array_equal(a3.cpu().numpy()[sel], a4.cpu().numpy()[sel])


@pytest.mark.parametrize("types,Ns,K,B", [((orc.Q4_K, orc.Q4_K, orc.Q6_K), (4096, 1024, 1024), 4096, 512),   # Q, K, V of the Q4_K_M mix
                                          ((orc.Q6_K, orc.Q5_K, orc.Q4_K), (1000, 8300, 130), 2048, 300),    # ragged rows and batch
                                          ((orc.Q6_K, orc.Q4_K), (14336, 14336), 4096, 512),                  # 896 tiles
                                          ((orc.Q6_K, orc.Q6_K), (520, 130), 2048, 200),                       # Q6_K only: the form without a min term
                                          ((orc.IQ4_XS, orc.IQ4_XS, orc.Q5_K), (1024, 260, 512), 2048, 300),  # Q, K, V of an IQ4_XS file
                                          ((orc.IQ4_XS, orc.Q6_K), (520, 130), 2048, 200)])                    # both without minima
def test_mmq_tiled_mixed_types(dev, types, Ns, K, B):
    """matrices of different K-quant types in one launch of the wide-tile GEMM: every matrix equals its own launch bit for bit, with
    and without a residual, and the oracle's integer arithmetic at the corners"""
    import mi355
    rng = np.random.default_rng(sum(Ns) + K + B + sum(types))
    x = rng.standard_normal((B, K)).astype(np.float32)
    act = mi355.quantize_act_q8k_tiled(_to_dev(dev, x))
    Wq = [_weights(rng, t, N, K, "ref") for t, N in zip(types, Ns)]
    tiles = [mi355.kq_unpack_tiles(t, mi355.upload_weights(t, _to_dev(dev, W))) for t, W in zip(types, Wq)]
    res = [_to_dev(dev, rng.standard_normal((B, N)).astype(np.float32)) if i != 1 else None for i, N in enumerate(Ns)]
    alone = [mi355.mul_mat_q8k_tiled(t, tl, act, N, K, B, split=False).cpu().numpy() for t, tl, N in zip(types, tiles, Ns)]
    mixed = [o.cpu().numpy() for o in mi355.mul_mat_q8k_tiled_multi(list(types), tiles, act, list(Ns), K, B)]
    with_res = [o.cpu().numpy() for o in mi355.mul_mat_q8k_tiled_multi(list(types), tiles, act, list(Ns), K, B, residuals=res)]
    for i, (t, N) in enumerate(zip(types, Ns)):
        assert np.array_equal(mixed[i], alone[i])
        assert np.array_equal(with_res[i], mixed[i] + res[i].cpu().numpy() if res[i] is not None else mixed[i])
        Nt, Bt = min(N, 40), min(B, 16)
        assert orc.nmse(mixed[i][:Bt, :Nt], orc.mul_mat("cpu", t, Wq[i][:Nt], x[:Bt])) < 1e-9
        assert orc.nmse(mixed[i][B - 5:, N - 7:], orc.mul_mat("cpu", t, Wq[i][N - 7:], x[B - 5:])) < 1e-9


@pytest.mark.parametrize("name,t", TILED_TYPES)
@pytest.mark.parametrize("N,K,B,split", [(4096, 4096, 512, True),       # wo of an 8B llama: cut along K, the sum launch carries the norm
                                         (4096, 14336, 512, True),      # ffn_down
                                         (2048, 2048, 300, True),       # ragged batch
                                         (4096, 4096, 512, False),      # no workspace: uncut, the norm is its own launch
                                         (4096, 2048, 2048, True),      # enough tiles: uncut
                                         (8192, 2048, 200, True)])      # rows longer than the fused form takes
def test_mmq_tiled_norm_equals_product_then_norm(dev, name, t, N, K, B, split):
    """MUL_MAT (+ residual) -> RMS_NORM -> MUL(weight) -> tile image as one call: the bits of the product followed by the norm launch,
    in the row, in the normalised row and in every byte of the image that the norm launch writes"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(N + K + B + t)
    x = rng.standard_normal((B, K)).astype(np.float32)
    act = mi355.quantize_act_q8k_tiled(_to_dev(dev, x))
    tiles = mi355.kq_unpack_tiles(t, mi355.upload_weights(t, _to_dev(dev, _weights(rng, t, N, K, "ref"))))
    res = _to_dev(dev, rng.standard_normal((B, N)).astype(np.float32))
    nw = _to_dev(dev, rng.standard_normal(N).astype(np.float32))
    for residual in (res, None):
        want_x = mi355.mul_mat_q8k_tiled(t, tiles, act, N, K, B, residual=residual, split=split)
        want_y = torch.empty((B, N), dtype=torch.float32, device=dev)
        want_img = torch.zeros(lib.mi355_act_q8k_tiled_bytes(N, B), dtype=torch.uint8, device=dev)
        mi355.check(lib.mi355_rms_norm_mul_quant_q8k_tiled(None, want_x.data_ptr(), N, nw.data_ptr(), want_y.data_ptr(), N, want_img.data_ptr(), N, B, 1e-5))
        got_x, got_y, got_img = mi355.mul_mat_q8k_tiled_norm(t, tiles, act, N, K, B, nw, 1e-5, residual=residual, split=split)
        torch.cuda.synchronize()
        assert np.array_equal(got_x.cpu().numpy(), want_x.cpu().numpy())
        assert np.array_equal(got_y.cpu().numpy(), want_y.cpu().numpy())
        assert np.array_equal(got_img.cpu().numpy(), want_img.cpu().numpy())     # both start from zeros: bytes neither writes agree too
    # in place: the residual is the destination (what the ggml graph allocator hands out for MUL_MAT -> ADD)
    dst = res.clone()
    got_x, got_y, got_img = mi355.mul_mat_q8k_tiled_norm(t, tiles, act, N, K, B, nw, 1e-5, residual=dst, split=split, dst=dst)
    want_x = mi355.mul_mat_q8k_tiled(t, tiles, act, N, K, B, residual=res, split=split)
    torch.cuda.synchronize()
    assert np.array_equal(got_x.cpu().numpy(), want_x.cpu().numpy())


@pytest.mark.parametrize("name,t", TILED_TYPES)
@pytest.mark.parametrize("Ns,K,B", [((14336, 14336), 4096, 512),       # gate + up of an 8B llama: 896 tiles
                                    ((4096, 1024, 1024), 4096, 512),    # Q, K, V: 192 tiles in one round
                                    ((8200, 8300, 130), 2048, 300),     # ragged rows and batch
                                    ((1000,), 6144, 300)])              # one matrix: cut along K like the single-matrix entry point
def test_mmq_tiled_multi(dev, name, t, Ns, K, B):
    """several matrices in one launch of the wide-tile GEMM: every matrix equals its own launch bit for bit, with and without
    residual (also in place), and the oracle's integer arithmetic at the corners"""
    import torch
    import mi355
    rng = np.random.default_rng(sum(Ns) + K + B + t)
    x = rng.standard_normal((B, K)).astype(np.float32)
    act = mi355.quantize_act_q8k_tiled(_to_dev(dev, x))
    Wq = [_weights(rng, t, N, K, "ref") for N in Ns]
    tiles = [mi355.kq_unpack_tiles(t, mi355.upload_weights(t, _to_dev(dev, W))) for W in Wq]
    res = [_to_dev(dev, rng.standard_normal((B, N)).astype(np.float32)) if i != 1 else None for i, N in enumerate(Ns)]
    alone = [mi355.mul_mat_q8k_tiled(t, tl, act, N, K, B, split=len(Ns) == 1).cpu().numpy() for tl, N in zip(tiles, Ns)]
    multi = [o.cpu().numpy() for o in mi355.mul_mat_q8k_tiled_multi(t, tiles, act, list(Ns), K, B)]
    dsts = [torch.empty((B, N + 8 * i), dtype=torch.float32, device=dev)[:, :N] for i, N in enumerate(Ns)]    # a row stride per matrix
    for i, N in enumerate(Ns):
        if res[i] is not None:
            dsts[i].copy_(res[i])     # residual in place: dst is its own residual
    inplace = mi355.mul_mat_q8k_tiled_multi(t, tiles, act, list(Ns), K, B, dsts=dsts, residuals=[d if r is not None else None for d, r in zip(dsts, res)])
    for i, N in enumerate(Ns):
        assert np.array_equal(multi[i], alone[i])
        want = multi[i] + res[i].cpu().numpy() if res[i] is not None else multi[i]
        assert np.array_equal(inplace[i].cpu().numpy(), want)
        Nt, Bt = min(N, 40), min(B, 16)
        assert orc.nmse(multi[i][:Bt, :Nt], orc.mul_mat("cpu", t, Wq[i][:Nt], x[:Bt])) < 1e-9
        assert orc.nmse(multi[i][B - 5:, N - 7:], orc.mul_mat("cpu", t, Wq[i][N - 7:], x[B - 5:])) < 1e-9


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t in (orc.Q4_0, orc.Q5_1, orc.Q8_0, orc.Q6_K)])
@pytest.mark.parametrize("K,B", [(512, 33), (2048, 65), (1024, 300)])
def test_mul_mat_q_multi(dev, name, t, K, B):
    """up to three matrices in one launch of the per-block tile kernel, ragged row counts, a residual that is the destination, with and
    without slices along K: the product of each matrix alone plus the residual (f32 sums in another order: NMSE of some 1e-14)"""
    import ctypes as C
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(K + B)
    Ns = [300, 64, 129]
    Ws = [mi355.upload_weights(t, _to_dev(dev, _weights(rng, t, N, K))) for N in Ns]
    act = mi355.quantize_act(_to_dev(dev, rng.standard_normal((B, K)).astype(np.float32)))
    res = [_to_dev(dev, rng.standard_normal((B, N)).astype(np.float32)) for N in Ns]
    want = []
    for W, r, N in zip(Ws, res, Ns):
        d = torch.empty((B, N), dtype=torch.float32, device=dev)
        mi355.check(lib.mi355_mul_mat_q(None, t, W.data_ptr(), act.data_ptr(), d.data_ptr(), N, K, B, N))
        want.append((d.double() + r.double()).cpu().numpy())
    need = lib.mi355_mul_mat_q_multi_ws_bytes(3, (C.c_int64 * 3)(*Ns), K, B)
    for nws in {0, int(need)}:
        ws = torch.empty(max(nws, 16), dtype=torch.uint8, device=dev)
        dst = [r.clone() for r in res]
        arr = (mi355.GemvMat * 3)()
        for i in range(3):
            arr[i].type, arr[i].W, arr[i].N, arr[i].dst, arr[i].dst_stride, arr[i].residual = t, Ws[i].data_ptr(), Ns[i], dst[i].data_ptr(), Ns[i], dst[i].data_ptr()
        mi355.check(lib.mi355_mul_mat_q_multi(None, t, 3, arr, act.data_ptr(), K, B, ws.data_ptr() if nws else None, nws))
        torch.cuda.synchronize()
        for d, w in zip(dst, want):
            assert orc.nmse(d.cpu().numpy(), w) < 1e-11, nws


@pytest.mark.parametrize("name,t", [("q4_0", orc.Q4_0), ("q8_0", orc.Q8_0)])
@pytest.mark.parametrize("K", [(1 << 24) + 96, (1 << 25) + 128])
def test_batches_over_very_long_rows(dev, name, t, K):
    """rows on both sides of what the tile kernel's 32-bit offsets reach, as a batch and through experts: integer weights and activations with
    scales of 1, exact block dots; f32 sums of 2^20 blocks whose magnitude grows with the square root leave some 2^-24 * 2^10 of the result"""
    import torch
    import mi355
    lib = mi355.load()
    N, B, lim = 3, 33, (7 if t == orc.Q4_0 else 127)
    g = torch.Generator(device=dev).manual_seed(1)
    W = torch.randint(-lim, lim + 1, (N, K), device=dev, generator=g, dtype=torch.int32).float()
    W[:, ::32] = -8 if t == orc.Q4_0 else 127
    x = torch.randint(-127, 128, (B, K), device=dev, generator=g, dtype=torch.int32).float()
    # (the first of 32 sets the scale.  Its sign is random: terms of one sign and size are all rounded the same way once a lane's f32 sum is 2^13 times larger)
    x[:, ::32] = 127 * torch.sign(x[:, 1::32] + 0.5)
    Wd = mi355.upload_weights(t, mi355.quantize_weights(t, W))
    act = mi355.quantize_act(x)
    want = torch.zeros((B, N), dtype=torch.float64, device=dev)
    for k in range(0, K, 1 << 22):
        want += x[:, k:k + (1 << 22)].double() @ W[:, k:k + (1 << 22)].double().T.contiguous()
    del x, W
    got = torch.full((B, N), float("nan"), device=dev)
    mi355.check(lib.mi355_mul_mat_q(None, t, Wd.data_ptr(), act.data_ptr(), got.data_ptr(), N, K, B, N))
    torch.cuda.synchronize()
    assert orc.nmse(got.cpu().numpy(), want.cpu().numpy()) < 1e-7
    assert lib.mi355_mul_mat_id_q_supported(t, Wd.data_ptr(), 1, K, N) == 1      # three experts of one row
    ids = torch.tensor([[b % 3, (b + 1) % 3] for b in range(B)], dtype=torch.int32, device=dev)
    got = torch.full((B, 2, 1), float("nan"), device=dev)
    route = torch.empty(int(lib.mi355_mul_mat_id_q8k_route_bytes(N, 2, B)), dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_mul_mat_id_q(None, t, Wd.data_ptr(), act.data_ptr(), ids.data_ptr(), 2, got.data_ptr(), 1, K, N, 2, 1, B, route.data_ptr(), route.numel()))
    torch.cuda.synchronize()
    assert orc.nmse(got[..., 0].cpu().numpy(), want.gather(1, ids.long()).cpu().numpy()) < 1e-7


@pytest.mark.parametrize("name,t,nb,rows,B", [("q6_K", orc.Q6_K, 1280000, 18, 3), ("iq4_xs", orc.IQ4_XS, 1974000, 18, 1), ("q4_K", orc.Q4_K, 1866240, 18, 2),   # 16 rows: more than 4 GiB
                                              ("q4_K", orc.Q4_K, 420000, 4, 41), ("q6_K", orc.Q6_K, 420000, 4, 41)])                                           # activations: more than 4 GiB
def test_super_block_tiles_beyond_32_bit_offsets(dev, name, t, nb, rows, B):
    """mi355_mul_mat_q8k, its form on planes and its routed form where sixteen weight rows or the activation rows pass 4 GiB: all zeros but a few
    super-blocks, against the oracle's product of those alone (f32 sums over six super-blocks: NMSE 1e-14)"""
    import torch
    import mi355
    lib = mi355.load()
    K = nb * 256
    at = [0, 1, 5, nb // 2 + 1, nb - 2, nb - 1]
    rng = np.random.default_rng(t)
    Wq = _weights(rng, t, rows, 256 * len(at))
    part = mi355.upload_weights(t, _to_dev(dev, Wq))
    W = torch.zeros(rows, nb * mi355.BLOCK[t][1], dtype=torch.uint8, device=dev)
    o = o_big = 0
    for size in {orc.Q6_K: (128, 64, 16, 2), orc.IQ4_XS: (128, 8), orc.Q4_K: (144,)}[t]:      # the pieces of a row in device layout
        for j, a in enumerate(at):
            W[:, o_big + a * size:o_big + (a + 1) * size] = part[:, o + j * size:o + (j + 1) * size]
        o, o_big = o + len(at) * size, o_big + nb * size
    xs = rng.standard_normal((B, 256 * len(at))).astype(np.float32)
    x = torch.zeros(B, K, device=dev)
    for j, a in enumerate(at):
        x[:, a * 256:(a + 1) * 256] = _to_dev(dev, xs[:, j * 256:(j + 1) * 256])
    act = mi355.quantize_act_q8k(x)
    del x
    want = orc.mul_mat("cpu", t, Wq, xs)
    res = _to_dev(dev, rng.standard_normal((B, rows)).astype(np.float32))
    dst = torch.empty(B, rows, device=dev)
    mi355.check(lib.mi355_mul_mat_q8k(None, t, W.data_ptr(), act.data_ptr(), dst.data_ptr(), rows, K, B, rows))
    assert orc.nmse(dst.cpu().numpy(), want) < 1e-11
    need = int(lib.mi355_mul_mat_q8k_ws_bytes(rows, K, B))
    ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_mul_mat_q8k_ws(None, t, W.data_ptr(), act.data_ptr(), dst.data_ptr(), res.data_ptr(), rows, K, B, rows, ws.data_ptr(), need))
    assert orc.nmse(dst.cpu().numpy(), want + res.cpu().numpy()) < 1e-11
    if rows * K < 1 << 32:
        planes = torch.empty(int(lib.mi355_kq_planes_bytes(rows, K)), dtype=torch.uint8, device=dev)
        mi355.check(lib.mi355_kq_unpack_planes(None, t, W.data_ptr(), planes.data_ptr(), rows, K))
        mi355.check(lib.mi355_mul_mat_q8k_planes_ws(None, t, planes.data_ptr(), act.data_ptr(), dst.data_ptr(), res.data_ptr(), rows, K, B, rows, ws.data_ptr(), need))
        assert orc.nmse(dst.cpu().numpy(), want + res.cpu().numpy()) < 1e-11
        del planes
    N = rows // 2                                          # the same rows as two experts
    ids = torch.tensor([[b % 2, 1 - b % 2, 0] for b in range(B)], dtype=torch.int32, device=dev)
    route = torch.empty(int(lib.mi355_mul_mat_id_q8k_route_bytes(2, 2, B)), dtype=torch.uint8, device=dev)
    dst = torch.empty(B, 2, N, device=dev)
    mi355.check(lib.mi355_mul_mat_id_q8k(None, t, W.data_ptr(), act.data_ptr(), ids.data_ptr(), 3, dst.data_ptr(), N, K, 2, 2, 1, B, route.data_ptr(), route.numel()))
    routed = np.stack([np.stack([want[b, e * N:(e + 1) * N] for e in (b % 2, 1 - b % 2)]) for b in range(B)])
    assert orc.nmse(dst.cpu().numpy(), routed) < 1e-11


@pytest.mark.parametrize("name,t,bound", [("q8_0", orc.Q8_0, 1.04e-7), ("iq4_nl", orc.IQ4_NL, 1.04e-7), ("iq4_xs", orc.IQ4_XS, 1.04e-7), ("q4_0", orc.Q4_0, 1.04e-7),
                                          ("q5_0", orc.Q5_0, 1.04e-7)])
def test_tile_kernel_sums_against_f64(dev, name, t, bound):
    """the error of the tile kernel's f32 sums over 32 blocks (2-norm, 2 M sums; their own scatter is 0.05 %): block sums converted and multiplied by both scales at
    once leave 1.030e-7; rounded once more, 1.055e-7 where levels have eight bits"""
    import torch
    import mi355
    rng = np.random.default_rng(1)
    N, K, B = 4096, 1024, 512
    Wq = _weights(rng, t, N, K)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    act = mi355.quantize_act(_to_dev(dev, rng.standard_normal((B, K)).astype(np.float32)))
    a = act[:B * K].view(torch.int8).reshape(B, K // 32, 32).double() * act[B * K:B * K + B * K // 4].view(torch.float32).reshape(B, K // 32, 2)[..., :1].double()
    want = a.reshape(B, K) @ _to_dev(dev, orc.dequantize("oracle", t, Wq, K)).double().T.contiguous()
    got = torch.empty((B, N), dtype=torch.float32, device=dev)
    mi355.check(mi355.load().mi355_mul_mat_q(None, t, Wd.data_ptr(), act.data_ptr(), got.data_ptr(), N, K, B, N))
    torch.cuda.synchronize()
    assert float((got.double() - want).norm() / want.norm()) < bound


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t in (orc.Q8_0, orc.IQ4_NL, orc.IQ4_XS)])
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 6, 8, 9, 13, 16, 17, 21])
def test_tile_kernel_last_stage(dev, name, t, blocks):
    """one to six stages of four blocks whose last holds one to four, where the last stage, or the last two, are summed on their own; alone and
    through experts (one column tile, and a second one of a few columns); exact block dots, f32 sums"""
    import torch
    import mi355
    rng = np.random.default_rng(blocks)
    K, N = (32 if t != orc.IQ4_XS else 256) * blocks, 130
    Wq = _weights(rng, t, 2 * N, K)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    for B in (33, 65, 130):
        x = rng.standard_normal((B, K)).astype(np.float32)
        want = orc.mul_mat("q8_1", t, Wq, x)
        act = mi355.quantize_act(_to_dev(dev, x))
        for split in (False, True):
            need = int(mi355.load().mi355_mul_mat_q_ws_bytes(2 * N, K, B)) if split else 0
            ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
            got = torch.full((B, 2 * N), float("nan"), device=dev)
            mi355.check(mi355.load().mi355_mul_mat_q_ws(None, t, Wd.data_ptr(), act.data_ptr(), got.data_ptr(), 2 * N, K, B, 2 * N, ws.data_ptr(), need))
            torch.cuda.synchronize()
            assert orc.nmse(got.cpu().numpy(), want) < 1e-11, (B, split)
        ids = torch.arange(B, dtype=torch.int32, device=dev).reshape(B, 1) % 31 // 30          # expert 1: every 31st row
        route = torch.empty(int(mi355.load().mi355_mul_mat_id_q8k_route_bytes(2, 1, B)), dtype=torch.uint8, device=dev)
        got = torch.full((B, N), float("nan"), device=dev)
        mi355.check(mi355.load().mi355_mul_mat_id_q(None, t, Wd.data_ptr(), act.data_ptr(), ids.data_ptr(), 1, got.data_ptr(), N, K, 2, 1, 1, B, route.data_ptr(), route.numel()))
        torch.cuda.synchronize()
        pick = ids.cpu().numpy().astype(bool)
        assert orc.nmse(got.cpu().numpy(), np.where(pick, want[:, N:], want[:, :N])) < 1e-11, B


@pytest.mark.parametrize("name,t", TYPES)
@pytest.mark.parametrize("B", [40, 130])
def test_tile_kernel_infinite_scales(dev, name, t, B):
    """a weight block whose f16 scale is infinite gives plus or minus infinity by the sign of the block's sum, in its row alone; with and without
    slices along K, through experts, and beside NaN activation rows, which stay NaN"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(B)
    be, bb = orc.BLOCK[t]
    K, N = 2048, 150
    Wf = (np.abs(rng.standard_normal((N, K))) * 0.02 + 0.002).astype(np.float32)      # one sign: the groups of a super-block agree
    Wq = orc.quantize("oracle", t, Wf)
    x = (np.abs(rng.standard_normal((B, K))) + 0.1).astype(np.float32) * np.where(np.arange(B) % 3 == 0, -1, 1)[:, None].astype(np.float32)
    at = 208 if t == orc.Q6_K else 0                                                     # where a block's f16 scale lies
    clean = orc.mul_mat("q8_1", t, Wq, x)
    bad = Wq.copy()
    want = clean.copy()
    for row, block, bits in ((3, 0, 0x7C00), (70, K // be // 2, 0xFC00), (149, K // be - 1, 0x7C00)):
        d = bad[row].reshape(K // be, bb)[block, at:at + 2].view(np.uint16)
        sign = (-1.0 if d[0] & 0x8000 else 1.0) * (-1.0 if bits & 0x8000 else 1.0)      # the levels carry the sign of the scale they were made for
        d[0] = bits
        want[:, row] = np.where(np.arange(B) % 3 == 0, -1, 1) * sign * np.inf
    Wd = mi355.upload_weights(t, _to_dev(dev, bad))
    for spoiled in (False, True):
        act = mi355.quantize_act(_to_dev(dev, x))
        if spoiled:                                                                      # activation row 5: a NaN scale
            act[B * K:B * K + B * K // 4].view(torch.float32).reshape(B, K // 32, 2)[5, 7, 0] = float("nan")
            want[5] = np.nan
        results = []
        for split in (False, True):
            need = int(lib.mi355_mul_mat_q_ws_bytes(N, K, B)) if split else 0
            ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
            got = torch.full((B, N), 1.0, device=dev)
            m = (mi355.GemvMat * 1)()
            m[0].type, m[0].W, m[0].N, m[0].dst, m[0].dst_stride, m[0].residual = t, Wd.data_ptr(), N, got.data_ptr(), N, got.data_ptr()
            mi355.check(lib.mi355_mul_mat_q_multi(None, t, 1, m, act.data_ptr(), K, B, ws.data_ptr() if need else None, need))
            torch.cuda.synchronize()
            results.append(got.cpu().numpy() - 1.0)
        if lib.mi355_mul_mat_id_q_supported(t, Wd.data_ptr(), N, K, 1):
            ids = torch.zeros((B, 1), dtype=torch.int32, device=dev)
            route = torch.empty(int(lib.mi355_mul_mat_id_q8k_route_bytes(1, 1, B)), dtype=torch.uint8, device=dev)
            got = torch.full((B, N), 1.0, device=dev)
            mi355.check(lib.mi355_mul_mat_id_q(None, t, Wd.data_ptr(), act.data_ptr(), ids.data_ptr(), 1, got.data_ptr(), N, K, 1, 1, 1, B, route.data_ptr(), route.numel()))
            torch.cuda.synchronize()
            results.append(got.cpu().numpy())
        for got in results:
            finite = np.isfinite(want)
            assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
            assert orc.nmse(got[finite], want[finite]) < 1e-11


@pytest.mark.parametrize("name,t", TYPES)
def test_few_rows_in_one_launch(dev, name, t):
    """one to three activation rows quantized inside the product launch: the bytes of a quantization launch and a product launch, at the
    edges of a group's rows (8 and 16), of one and two rows per wave (2048), of a pass over K (4096 elements) and with padded rows of x"""
    import torch
    import mi355
    lib = mi355.load()
    be = mi355.BLOCK[t][0]
    gen = torch.Generator(device=dev).manual_seed(t)
    shapes = [(1, be, 1), (7, 3 * be, 3), (9, 4096, 2), (2047, 2048, 2), (2049, 1024 + be, 3), (4096, 4096, 3), (4095, 4096 + be, 1), (33, 8192, 1), (14336, 4096, 1)]
    for N, K, B in shapes:
        raw = np.random.default_rng(N + K).standard_normal((min(N, 64), K)).astype(np.float32) * 0.02
        Wq = np.resize(orc.quantize("oracle", t, raw), (N, orc.row_bytes(t, K)))
        W = mi355.upload_weights(t, _to_dev(dev, Wq))
        wide = torch.randn(B, K + 8, device=dev, generator=gen)
        wide[0, :be] = 0.0
        if B > 1:
            wide[1, K - 3] = float("inf")
        x = wide[:, :K]
        assert lib.mi355_mul_mat_vec_f32_supported(t, W.data_ptr(), N, K, B), (N, K, B)
        act = torch.empty(int(lib.mi355_act_bytes(K, B)), dtype=torch.uint8, device=dev)
        want = torch.empty(B, N, device=dev)
        mi355.check(lib.mi355_quantize_act(None, x.data_ptr(), act.data_ptr(), K, B, x.stride(0)))
        mi355.check(lib.mi355_mul_mat_vec_q(None, t, W.data_ptr(), act.data_ptr(), want.data_ptr(), N, K, B, N))
        guard = torch.full((B, N + 3), 7.0, device=dev)
        mi355.check(lib.mi355_mul_mat_vec_f32(None, t, W.data_ptr(), x.data_ptr(), guard.data_ptr(), N, K, B, x.stride(0), N + 3))
        torch.cuda.synchronize()
        assert torch.equal(guard[:, :N].contiguous().view(torch.int32), want.view(torch.int32)), (N, K, B)
        assert (guard[:, N:] == 7.0).all()
        assert torch.equal(mi355.mul_mat(t, W, x).view(torch.int32), want.view(torch.int32)), (N, K, B)
    assert not lib.mi355_mul_mat_vec_f32_supported(t, W.data_ptr(), 4096, 4096, 4)      # more rows, longer rows, many groups: two launches
    assert not lib.mi355_mul_mat_vec_f32_supported(t, W.data_ptr(), 4096, 14336, 1)
    assert not lib.mi355_mul_mat_vec_f32_supported(t, W.data_ptr() + 1, 4096, 4096, 1)
    with pytest.raises(mi355.Mi355Error, match="aligned"):
        mi355.check(lib.mi355_mul_mat_vec_f32(None, t, W.data_ptr(), x.data_ptr() + 4, guard.data_ptr(), N, K, 1, K, N))


@pytest.mark.parametrize("name,t", [("q4_0", orc.Q4_0), ("q6_K", orc.Q6_K)])
@pytest.mark.parametrize("B,offset", [(1, 0), (2, 0), (3, 0), (1, 1024), (3, 68), (1, -512), (40, 0)])
def test_dst_over_x(dev, name, t, B, offset):
    """a dst that overlaps x (in place, `offset` floats behind or before it) gives the bits of the same call on apart buffers, with a workspace
    and on the library's own scratch; rows of dst between rows of x share nothing with them; a workspace at an odd address is refused"""
    import torch
    import mi355
    lib = mi355.load()
    N = K = 2048
    W = mi355.upload_weights(t, _to_dev(dev, _weights(np.random.default_rng(B), t, N, K)))
    x = torch.randn(B, K, device=dev, generator=torch.Generator(device=dev).manual_seed(B))
    want = mi355.mul_mat(t, W, x, split=False)
    need = int(lib.mi355_mul_mat_ws_bytes(K, B))
    ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
    for static in (False, True):
        buf = torch.zeros(B * K + 4096, device=dev)
        xv = buf[2048:2048 + B * K].reshape(B, K)
        xv.copy_(x)
        dst = buf[2048 + offset:2048 + offset + B * N].reshape(B, N)
        if static:
            mi355.mul_mat_static(t, W, xv, dst)
        else:
            mi355.check(lib.mi355_mul_mat(None, t, W.data_ptr(), xv.data_ptr(), dst.data_ptr(), N, K, B, K, N, ws.data_ptr(), need))
        torch.cuda.synchronize()
        assert torch.equal(dst, want) or (static and orc.nmse(dst.cpu().numpy(), want.cpu().numpy()) < 1e-12)   # the scratch has room for slices
    if B > 3:
        return
    with pytest.raises(mi355.Mi355Error, match="overlap"):
        mi355.check(lib.mi355_mul_mat_vec_f32(None, t, W.data_ptr(), xv.data_ptr(), dst.data_ptr(), N, K, B, K, N))
    with pytest.raises(mi355.Mi355Error, match="aligned"):
        mi355.check(lib.mi355_mul_mat(None, t, W.data_ptr(), x.data_ptr(), want.data_ptr(), N, K, B, K, N, ws.data_ptr() + 4, need))
    both = torch.zeros(B, K + N, device=dev)
    both[:, :K] = x
    before = lib.mi355_launch_count()
    mi355.check(lib.mi355_mul_mat(None, t, W.data_ptr(), both.data_ptr(), both[:, K:].data_ptr(), N, K, B, K + N, K + N, ws.data_ptr(), need))
    assert lib.mi355_launch_count() - before == 1
    assert torch.equal(both[:, K:], want)


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t in (orc.Q4_K, orc.Q5_K, orc.Q6_K, orc.IQ4_XS)])
@pytest.mark.parametrize("N", [129, 130, 131, 132])
def test_slices_of_any_number_of_rows(dev, name, t, N):
    """a product cut along K whose slabs pad their rows to 16 bytes: integer sums are exact, f32 sums over 16 super-blocks leave an NMSE
    of some 1e-14; with a residual, and without touching what lies behind a row of dst"""
    import torch
    import mi355
    lib = mi355.load()
    K, B = 4096, 37
    rng = np.random.default_rng(N)
    Wq = _weights(rng, t, N, K)
    W = mi355.upload_weights(t, _to_dev(dev, Wq))
    x = rng.standard_normal((B, K)).astype(np.float32)
    res = rng.standard_normal((B, N + 5)).astype(np.float32)
    act = mi355.quantize_act_q8k(_to_dev(dev, x))
    need = int(lib.mi355_mul_mat_q8k_ws_bytes(N, K, B))
    assert need > 0
    ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)     # NaNs where nothing is written
    dst = torch.full((B, N + 5), 7.0, device=dev)
    r = _to_dev(dev, res)
    mi355.check(lib.mi355_mul_mat_q8k_ws(None, t, W.data_ptr(), act.data_ptr(), dst.data_ptr(), r.data_ptr(), N, K, B, N + 5, ws.data_ptr(), need))
    torch.cuda.synchronize()
    want = orc.mul_mat("cpu", t, Wq, x)
    assert orc.nmse(dst[:, :N].cpu().numpy(), want + res[:, :N]) < 1e-11
    assert (dst[:, N:] == 7.0).all()


@pytest.mark.parametrize("N,K,B,cut", [(1895, 1280, 606, False), (7263, 1024, 125, False), (2505, 2304, 68, True), (2026, 1792, 210, True), (1896, 1280, 606, True)])
def test_short_rows_are_cut_only_where_the_sum_pays(dev, N, K, B, cut):
    """few super-blocks per row and a number of rows that is no multiple of 4: one launch where the cut's sum costs more than it saves"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(N)
    Wq = np.resize(_weights(rng, orc.Q5_K, 80, K), (N, orc.row_bytes(orc.Q5_K, K)))      # the rows repeat every 80
    x = rng.standard_normal((B, K)).astype(np.float32)
    W, xd = mi355.upload_weights(orc.Q5_K, _to_dev(dev, Wq)), _to_dev(dev, x)
    assert (int(lib.mi355_mul_mat_q8k_ws_bytes(N, K, B)) > 0) == cut
    before = lib.mi355_launch_count()
    got = mi355.mul_mat(orc.Q5_K, W, xd)
    assert lib.mi355_launch_count() - before == (3 if cut else 2)
    got = got.cpu().numpy()
    for rows in (slice(0, 3), slice(B - 3, B)):
        want = orc.mul_mat("cpu", orc.Q5_K, Wq[:80], x[rows])
        assert orc.nmse(got[rows], np.tile(want, (1, N // 80 + 1))[:, :N]) < 1e-11


@pytest.mark.parametrize("name,t", [(n, t) for n, t in TYPES if t not in (orc.Q4_K, orc.Q5_K)])
@pytest.mark.parametrize("N,K,B", [(130, 5376, 65), (130, 1280, 40), (130, 4352, 130)])
def test_tile_kernel_many_slices(dev, name, t, N, K, B):
    """up to sixteen slices of a few stages each, the last one shorter, and as many as the workspace holds: integer sums are exact, f32 sums
    over at most 168 blocks leave an NMSE of some 1e-14"""
    import torch
    import mi355
    lib = mi355.load()
    rng = np.random.default_rng(N + K)
    Wq = _weights(rng, t, N, K)
    Wd = mi355.upload_weights(t, _to_dev(dev, Wq))
    x = rng.standard_normal((B, K)).astype(np.float32)
    act = mi355.quantize_act(_to_dev(dev, x))
    want = orc.mul_mat("q8_1", t, Wq, x)
    need = int(lib.mi355_mul_mat_q_ws_bytes(N, K, B))
    assert need >= 8 * N * B * 4 or K < 2048
    for room in (need, need // 2, 2 * N * B * 4, 0):
        ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)      # NaNs where nothing is written
        got = torch.full((B, N), float("nan"), device=dev)
        mi355.check(lib.mi355_mul_mat_q_ws(None, t, Wd.data_ptr(), act.data_ptr(), got.data_ptr(), N, K, B, N, ws.data_ptr(), room))
        torch.cuda.synchronize()
        assert orc.nmse(got.cpu().numpy(), want) < 1e-11, room
        assert (ws[room:] == 255).all()


def test_products_of_many_tiles_are_not_cut(dev):
    """per-block tiles: from 600 tiles on the chip is busy without slices along K"""
    import mi355
    lib = mi355.load()
    for N, K, B, cut in ((28743, 6400, 326, False), (20630, 5888, 481, False), (38400, 8192, 256, False), (18629, 7168, 415, True), (1115, 11776, 184, True)):
        assert (int(lib.mi355_mul_mat_q_ws_bytes(N, K, B)) > 0) == cut, (N, K, B)


def test_a_short_last_slice_costs_no_round():
    """per-block tiles: the fewest slices stay where only the groups of a short last slice exceed what the compute units hold at once"""
    import mi355
    lib = mi355.load()
    for N, K, B, slices in ((2813, 2080, 287, 4), (4755, 2176, 144, 4), (5309, 3392, 231, 6), (10772, 4640, 65, 6), (2477, 4096, 626, 5), (12317, 4096, 54, 5),
                            (2537, 13792, 527, 9)):
        assert int(lib.mi355_mul_mat_q_ws_bytes(N, K, B)) == slices * N * B * 4, (N, K, B)


@pytest.mark.parametrize("name,t", list(orc.WEIGHT_TYPES.items()))
@pytest.mark.parametrize("N,K", [(1, 256), (9, 4096 + 256), (2047, 1024), (2049, 2048), (33, 14336), (1030, 16384 + 512), (17, 32768), (8200, 4096)])
def test_one_row_launch_has_the_bits_of_the_multi_matrix_one(dev, name, t, N, K):
    """one row against one matrix (a wave per weight row, several steps of it in flight): the sums of the launch that walks it step by step, residual in place"""
    import torch
    import mi355
    from mi355 import llama_graph as lg
    lib = mi355.load()
    if t in orc.WEIGHT_TYPES.values() and (K // 256) % 8 and name in ("q6_K", "iq4_xs"):
        K = K // 2048 * 2048 or 2048      # rows of whole 16 bytes, as the launch of several matrices reads them
    if name not in ("q4_K", "q5_K", "q6_K", "iq4_xs"):
        K += 64                           # a last step of one or two blocks
    gen = torch.Generator(device=dev).manual_seed(N + K)
    W = mi355.upload_weights(t, lg.random_quantized(t, N, K, torch.device(dev), gen))
    x = torch.randn(1, K, device=dev, generator=gen)
    act = mi355.quantize_act(x)
    res = torch.randn(N, device=dev, generator=gen)
    for with_res in (False, True):
        outs = [res.clone() for _ in range(3)]
        arr = (mi355.GemvMat * 2)()
        for i, o in enumerate(outs[:2]):
            arr[i].type, arr[i].W, arr[i].N, arr[i].dst, arr[i].dst_stride, arr[i].residual = t, W.data_ptr(), N, o.data_ptr(), N, o.data_ptr() if with_res else None
        mi355.check(lib.mi355_mul_mat_vec_q_multi(None, 2, arr, act.data_ptr(), K, 1))
        arr[0].dst, arr[0].residual = outs[2].data_ptr(), outs[2].data_ptr() if with_res else None
        mi355.check(lib.mi355_mul_mat_vec_q_multi(None, 1, arr, act.data_ptr(), K, 1))
        assert bool(torch.isfinite(outs[2]).all()) and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
