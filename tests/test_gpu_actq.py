"""GPU parity of the activation fake-quant forward kernels against the CPU oracle: codes, scales and bf16 values bit-exact
for the plain and RMSNorm sources; the SiLU source carries expf and is compared through its own activation bits."""
import numpy as np
import pytest

import oracle as O
from gpu_util import F, I, L64, NULL, bits_equal, call, close_16, dev, host, outliers, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('M,K,qmax', [(5, 896, 7), (3, 2048, 7), (2, 8192, 7), (4, 128, 3), (3, 768, 127), (9, 1152, 7), (6, 1920, 7), (301, 1024, 7),
                                      (5, 2176, 7)])
def test_actq_fwd(M, K, qmax):
    """rows of at most 2048 values take the wave-per-row kernel when the outputs are 16-byte (values) and 4-byte (codes) aligned,
    the workgroup-per-row kernel otherwise: both against the oracle"""
    import ctypes
    rng = np.random.default_rng(K + qmax)
    x = outliers(rng, (M, K)); x[0] = 0
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        ry, rs, rc = O.actq_fwd(src, clip=0.9, qmax=qmax, bf16=bf)
        srcd = dev(src)
        for shift in (0, 1):                                            # shift: outputs moved off their 16- / 4-byte alignment
            y = dev(np.zeros(M * K + 8, np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros(M * K // 2 + 8, np.uint8))
            yp = ctypes.c_void_p(y.data_ptr() + 8 * shift); cp = ctypes.c_void_p(c.data_ptr() + 2 * shift)
            call('camx_actq_fwd', ptr(srcd), I(int(bf)), yp, ptr(s), cp if qmax <= 7 else NULL, I(K), F(0.9), I(qmax), I(M))
            assert bits_equal(host(s), rs) and bits_equal(host(y, np.uint16)[4 * shift:4 * shift + M * K].reshape(M, K), ry)
            if qmax <= 7: assert bits_equal(host(c)[2 * shift:2 * shift + M * K // 2].reshape(M, K // 2), rc)


@pytest.mark.parametrize('K', [1024, 2304])
@pytest.mark.parametrize('qmax,clip', [(127, 0.51), (127, 0.4), (511, 1.0), (2047, 0.55), (2047, 0.45), (32767, 1.0), (7, 0.02), (7, 1e-3)])
def test_actq_fwd_large_quotients(K, qmax, clip):
    """row maxima of 249 to 32767 scales: either side of the limits up to which a lane may round u * rcp(s)"""
    rng = np.random.default_rng(K + qmax)
    M = 64
    x = outliers(rng, (M, K))
    x[1] = 0; x[1, ::128] = np.arange(K // 128) + 1                        # (chunks of one value each: equal quotients, half-integers among them)
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        ry, rs, rc = O.actq_fwd(src, clip=clip, qmax=qmax, bf16=bf)
        y = dev(np.zeros((M, K), np.uint16)); s = dev(np.zeros(M, np.float32))
        call('camx_actq_fwd', ptr(dev(src)), I(int(bf)), ptr(y), ptr(s), NULL, I(K), F(clip), I(qmax), I(M))
        assert bits_equal(host(s), rs) and bits_equal(host(y, np.uint16), ry)


@pytest.mark.parametrize('M,d,nab', [(6, 896, 8), (5, 1024, 16), (3, 2048, 5), (2, 4096, 2), (130, 1024, 14), (4, 128, 1), (3, 8192, 3), (7, 768, 0),
                                     (9, 512, 6), (5, 256, 16), (300, 640, 3), (4, 1152, 9)])
def test_block_entry_fwd(M, d, nab):
    """rows of at most 1024 values: one wave per row, every round count; longer rows: a workgroup per row. The projections run one
    per wave (rows w, w + W, ... of wab): counts that are not multiples of four, rows that keep bf16(h) in registers and longer ones"""
    rng = np.random.default_rng(11 + d + nab)
    x = outliers(rng, (M, d)); nw = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32); wab = O.f2bf(rng.standard_normal((nab, d)) * 0.05)
    ry, rs, rc, rab, rstd = O.block_entry_fwd(x, nw, wab if nab else None, 1e-6)
    y = dev(np.zeros((M, d), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, d // 2), np.uint8))
    ab = dev(np.zeros((M, max(nab, 1)), np.uint16)); rstd_d = dev(np.zeros(M, np.float32))
    call('camx_block_entry_fwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(wab)) if nab else NULL, I(nab), F(1e-6), ptr(y), ptr(s), ptr(c),
         ptr(ab) if nab else NULL, ptr(rstd_d), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(rstd_d), rstd) and bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    if nab: assert bits_equal(host(ab, np.uint16), rab)


@pytest.mark.parametrize('M,Fh', [(5, 768), (2100, 1024), (2050, 1920), (2049, 2176), (4099, 128), (5, 2304), (303, 2048)])
def test_silu_mul_actq_fwd(M, Fh):
    rng = np.random.default_rng(12 + M)
    gu = O.f2bf(outliers(rng, (M, 2 * Fh)))
    gu[M - 1, :10] = O.f2bf(np.array([256., -256., 255., -255., 2.0 ** -24, -2.0 ** -24, 2.0 ** -25, -2.0 ** -25, 1e4, -1e-30], np.float32))      # the edges of the small table
    y = dev(np.zeros((M, Fh), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, Fh // 2), np.uint8))
    gud = dev(gu)
    call('camx_silu_mul_actq_fwd', ptr(gud), I(2 * Fh), I(Fh), ptr(y), ptr(s), ptr(c), F(1.0), I(7), I(M))
    # the activation is the table's (the oracle's bits), then the exact stages on it
    act = dev(np.zeros((M, Fh), np.uint16))
    call('camx_silu_mul_bf16', ptr(gud), ptr(act), I(Fh), L64(M * Fh))
    assert bits_equal(host(act, np.uint16), O.silu_mul_bf16(gu))
    ry, rs, rc = O.actq_fwd(host(act, np.uint16), bf16=True)
    assert bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    fy, fs, fc = O.silu_mul_actq_fwd(gu)
    assert bits_equal(host(s), fs) and bits_equal(host(c), fc) and bits_equal(host(y, np.uint16), fy)


# ---- backward ----------------------------------------------------------------------------------------------------------------

@pytest.mark.parametrize('M,K,qmax', [(5, 896, 7), (3, 2048, 7), (2, 8192, 7), (4, 128, 3), (3, 768, 127), (300, 1024, 7), (7, 5120, 7), (9, 1152, 7), (6, 1920, 7),
                                      (5, 1536, 15), (4, 4096, 7), (4, 6144, 7), (3, 7168, 7)])
def test_actq_bwd(M, K, qmax):
    rng = np.random.default_rng(100 + K + qmax)
    x = outliers(rng, (M, K)); x[0] = 0
    if M > 2: x[2, :] = 0; x[2, 7] = 3.0                                   # rotates to a constant row: every element ties for the max
    g = O.f2bf(rng.standard_normal((M, K)).astype(np.float32))
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        want = O.actq_bwd(src, g, clip=0.9, qmax=qmax, bf16=bf)
        dx = dev(np.zeros((M, K), np.uint16 if bf else np.float32))
        call('camx_actq_bwd', ptr(dev(src)), I(int(bf)), ptr(dev(g)), ptr(dx), I(K), F(0.9), I(qmax), I(M))
        assert bits_equal(host(dx, np.uint16) if bf else host(dx), want)


@pytest.mark.parametrize('K', [1024, 2048, 2560])
def test_actq_bwd_quotients_at_the_exponent_limits(K):
    """u / s where the quotient, the scale or their ratio leaves the range in which the kernel divides by a refined reciprocal:
    rows scaled to 1e-30 and 1e30, a row of 1e-12 with one chunk at 1e20 (quotients near 1e-32), a row whose values span
    1e-38 .. 1e38, inf and NaN entries, and a clip of 1e-20 (quotients near 1e21): the IEEE quotient in every case"""
    rng = np.random.default_rng(500 + K)
    M = 8
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0] *= 1e-30; x[1] *= 1e30
    x[2] *= 1e-12; x[2, 128:256] *= 1e32
    x[3] *= (10.0 ** rng.uniform(-38, 38, K)).astype(np.float32)
    x[4, 5] = np.inf; x[5, 130] = np.nan
    x[6] *= 1e-12; x[6, :128] = 0; x[6, 300] = 1e25
    x[7] = 0; x[7, 128:256] = 1e-30 * rng.standard_normal(128)
    g = O.f2bf(rng.standard_normal((M, K)).astype(np.float32))
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        for clip in (1.0, 1e-20):
            want = O.actq_bwd(src, g, clip=clip, qmax=7, bf16=bf)
            dx = dev(np.zeros((M, K), np.uint16 if bf else np.float32))
            call('camx_actq_bwd', ptr(dev(src)), I(int(bf)), ptr(dev(g)), ptr(dx), I(K), F(clip), I(7), I(M))
            got = host(dx, np.uint16) if bf else host(dx)
            nan_w = np.isnan(O.bf2f(want)) if bf else np.isnan(want); nan_g = np.isnan(O.bf2f(got)) if bf else np.isnan(got)
            assert np.array_equal(nan_w, nan_g) and bits_equal(np.where(nan_w, 0, got), np.where(nan_w, 0, want))


@pytest.mark.parametrize('M,d,nab', [(6, 896, 14), (5, 1024, 0), (9, 256, 2), (130, 896, 16), (7, 1024, 16), (3, 128, 4), (171, 896, 8), (12, 640, 6), (9, 384, 0),
                                     (10, 256, 14), (6, 128, 16), (5, 512, 10), (6, 768, 16)])
def test_block_entry_bwd(M, d, nab):
    """every round count of the wave-per-row kernel; row 1 has one value in the row's last chunk and one in chunk 1 with the same
    |h|: their chunks rotate to constants, so 256 elements tie for the row's maximum across rounds that not all lanes take part in"""
    rng = np.random.default_rng(200 + d + nab)
    x = outliers(rng, (M, d)); nw = (0.5 + rng.random(d)).astype(np.float32)
    if d >= 384 and M > 1:
        last = d - 128 + 5
        nw[last] = nw[128 + 7]; x[1] = 0; x[1, 128 + 7] = 3.0; x[1, last] = -3.0
    wab = O.f2bf((rng.standard_normal((max(nab, 2), d)) / 30).astype(np.float32))[:nab]
    dy = O.f2bf(rng.standard_normal((M, d)).astype(np.float32)); dab = O.f2bf(rng.standard_normal((M, max(nab, 1))).astype(np.float32))[:, :nab]
    rstd = O.block_entry_fwd(x, nw, wab if nab else None, 1e-6)[4]
    want = O.block_entry_bwd(x, nw, rstd, wab if nab else None, dy, dab if nab else None)
    dx = dev(np.zeros((M, d), np.float32))
    call('camx_block_entry_bwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(rstd)), ptr(dev(wab)) if nab else NULL, I(nab), ptr(dev(dy)),
         ptr(dev(np.ascontiguousarray(dab))) if nab else NULL, ptr(dx), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(dx), want)


@pytest.mark.parametrize('M,Fh,ld', [(24, 768, 1536), (12, 2048, 4608), (9, 256, 512), (1100, 256, 520), (2300, 1024, 2048), (4099, 128, 256),
                                      (24, 768, 1540), (1030, 2304, 4608), (7, 2304, 4612), (1500, 640, 1284)])
def test_silu_mul_actq_bwd(M, Fh, ld):
    """the recomputed activation is the table's (the oracle's bits); the sigmoid of silu's derivative comes from a table of the correctly
    rounded expf, the oracle's from the C library's (within an ulp of it): one bf16 step at most. Row widths and strides that take
    the wave-per-row form (tables in LDS, gates at their edges in the last row) and the workgroup-per-row form (longer or unaligned rows)"""
    rng = np.random.default_rng(300 + Fh)
    base = O.f2bf((rng.standard_normal((M, ld)) * 2).astype(np.float32))
    base[0, :8] = O.f2bf(np.array([30., -30., 0., -0.0, 1e-3, -88., 88., 3.], np.float32))
    base[M - 1, :10] = O.f2bf(np.array([256., -256., 255., -255., 2.0 ** -24, -2.0 ** -24, 2.0 ** -25, -2.0 ** -25, 1e4, -1e-30], np.float32))    # the edges of the small tables
    g = O.f2bf(rng.standard_normal((M, Fh)).astype(np.float32))
    bd = dev(base)
    dgu = dev(np.zeros((M, 2 * Fh), np.uint16))
    call('camx_silu_mul_actq_bwd', ptr(bd), I(ld), I(Fh), ptr(dev(g)), ptr(dgu), F(1.0), I(7), I(M))
    gu = np.ascontiguousarray(base[:, :2 * Fh])
    act = dev(np.zeros((M, Fh), np.uint16))
    call('camx_silu_mul_bf16', ptr(dev(gu)), ptr(act), I(Fh), L64(M * Fh))
    assert bits_equal(host(act, np.uint16), O.silu_mul_bf16(gu))
    want = O.silu_mul_actq_bwd(gu, g)
    got = host(dgu, np.uint16)
    assert close_16(got, want, 'bf16')
    assert (got == want).mean() > 0.99
    assert bits_equal(got, O.silu_mul_actq_bwd(gu, g, table=True))        # bit for bit against the table's own definition (every gate here is finite)


@pytest.mark.parametrize('Fh', [128, 1152, 1920, 2048, 2304])
def test_silu_mul_actq_zero_gates(Fh):
    """zeros of both signs are inside the small tables: rows of nothing else, half zeros, one zero among eight gates, zeros beside gates
    outside the tables, and zero multipliers; row widths that leave lanes of a wave without a chunk. Forward and backward bit for bit"""
    rng = np.random.default_rng(40 + Fh)
    M = 9
    gate = (rng.standard_normal((M, Fh)) * 2).astype(np.float32); up = rng.standard_normal((M, Fh)).astype(np.float32)
    gate[0] = 0.0; gate[1] = -0.0; gate[2] = np.where(rng.random(Fh) < 0.5, 0.0, gate[2]); gate[3, 3::8] = -0.0
    gate[4, ::8] = 0.0; gate[4, 1::16] = 300.0; gate[4, 2::32] = -2.0 ** -26; gate[5, ::8] = 2.0 ** -24; gate[5, 1::8] = -0.0; gate[6] = 0.0; gate[6, 9] = 1e-30
    up[7] = 0.0; up[8, ::2] = -0.0
    gu = O.f2bf(np.concatenate([gate, up], axis=1)); g = O.f2bf(rng.standard_normal((M, Fh)).astype(np.float32))
    y = dev(np.zeros((M, Fh), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, Fh // 2), np.uint8)); dgu = dev(np.zeros((M, 2 * Fh), np.uint16))
    call('camx_silu_mul_actq_fwd', ptr(dev(gu)), I(2 * Fh), I(Fh), ptr(y), ptr(s), ptr(c), F(1.0), I(7), I(M))
    fy, fs, fc = O.silu_mul_actq_fwd(gu)
    assert bits_equal(host(s), fs) and bits_equal(host(c), fc) and bits_equal(host(y, np.uint16), fy)
    call('camx_silu_mul_actq_bwd', ptr(dev(gu)), I(2 * Fh), I(Fh), ptr(dev(g)), ptr(dgu), F(1.0), I(7), I(M))
    assert bits_equal(host(dgu, np.uint16), O.silu_mul_actq_bwd(gu, g, table=True))


@pytest.mark.parametrize('M,Fh', [(6, 1024), (1200, 256), (5, 2304)])
def test_silu_mul_actq_gates_of_every_magnitude(M, Fh):
    """gates and multipliers over the whole bf16 exponent range (most gates outside the small tables the wave-per-row kernels hold in
    LDS), +-inf gates, a NaN gate and a NaN multiplier: the forward bit for bit, the backward within a bf16 step, NaN for NaN"""
    from test_gpu_value_sweeps import values
    rng = np.random.default_rng(900 + M)
    with np.errstate(all='ignore'):
        gu = O.f2bf(values(rng, (M, 2 * Fh), emin=-130.0, emax=120.0))
        gu[1, :Fh] = O.f2bf(values(rng, Fh, emin=-30.0, emax=12.0))
        gu[2, 5] = 0x7f80; gu[2, 6] = 0xff80; gu[3, 9] = 0x7fc1; gu[4, Fh + 3] = 0xffc0
        g = O.f2bf(rng.standard_normal((M, Fh)).astype(np.float32))
        fy, fs, fc = O.silu_mul_actq_fwd(gu)
        want = O.silu_mul_actq_bwd(gu, g)
    gud = dev(gu)
    y = dev(np.zeros((M, Fh), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, Fh // 2), np.uint8))
    call('camx_silu_mul_actq_fwd', ptr(gud), I(2 * Fh), I(Fh), ptr(y), ptr(s), ptr(c), F(1.0), I(7), I(M))
    nan_s = np.isnan(fs)
    assert np.array_equal(np.isnan(host(s)), nan_s) and bits_equal(host(s)[~nan_s], fs[~nan_s])
    assert bits_equal(host(y, np.uint16)[~nan_s], fy[~nan_s]) and bits_equal(host(c)[~nan_s], fc[~nan_s])
    dgu = dev(np.zeros((M, 2 * Fh), np.uint16))
    call('camx_silu_mul_actq_bwd', ptr(gud), I(2 * Fh), I(Fh), ptr(dev(g)), ptr(dgu), F(1.0), I(7), I(M))
    got = host(dgu, np.uint16)
    nan_w = np.isnan(O.bf2f(want)); nan_g = np.isnan(O.bf2f(got))
    assert np.array_equal(nan_w, nan_g)
    assert close_16(np.where(nan_w, 0, got).astype(np.uint16), np.where(nan_w, 0, want).astype(np.uint16), 'bf16')


def test_actq_autograd_wrappers():
    """caminus_amd.train.actq end to end: values, codes, scales and every gradient equal the C entry points' results"""
    import torch
    from caminus_amd.train import actq as A
    rng = np.random.default_rng(7)
    M, K = 33, 1024
    x = outliers(rng, (M, K)); gy = rng.standard_normal((M, K)).astype(np.float32)
    for bf in (False, True):
        xt = torch.from_numpy(x).to('cuda:0'); xt = (xt.bfloat16() if bf else xt).requires_grad_()
        src = host(xt.detach().view(torch.int16), np.uint16) if bf else x
        y, c, s = A.actq_codes(xt.view(3, 11, K), 4, 0.9)
        ry, rs, rc = O.actq_fwd(src, clip=0.9, qmax=7, bf16=bf)
        assert y.shape == (3, 11, K) and bits_equal(host(y.view(torch.int16), np.uint16).reshape(M, K), ry) and bits_equal(host(s), rs) and bits_equal(host(c), rc)
        gt = torch.from_numpy(gy).to('cuda:0').view(3, 11, K)
        y.backward(gt)
        want = O.actq_bwd(src, O.f2bf(gy), clip=0.9, qmax=7, bf16=bf)
        assert xt.grad.dtype == xt.dtype
        assert bits_equal(host(xt.grad.view(torch.int16), np.uint16) if bf else host(xt.grad), want)
        x2 = xt.detach().clone().requires_grad_()
        A.actq(x2, 4, 0.9).backward(gt.view(M, K))
        assert torch.equal(x2.grad, xt.grad)
        assert torch.equal(A.scales(xt.detach(), 4, 0.9), s) and torch.equal(A.codes(xt.detach(), 4, 0.9)[0], c)
    # block entry
    d, nab = 896, 14
    xb = outliers(rng, (M, d)); nw = (0.5 + rng.random(d)).astype(np.float32); wab = O.f2bf((rng.standard_normal((nab, d)) / 30).astype(np.float32))
    dy = rng.standard_normal((M, d)).astype(np.float32); dab = rng.standard_normal((M, nab)).astype(np.float32)
    xt = torch.from_numpy(xb).to('cuda:0').requires_grad_(); nwt = torch.from_numpy(nw).to('cuda:0'); wt = dev(wab).view(torch.bfloat16)
    y, c, s, ab = A.block_entry(xt, nwt, wt, 1e-6)
    ry, rs, rc, rab, rstd = O.block_entry_fwd(xb, nw, wab, 1e-6)
    assert bits_equal(host(y.view(torch.int16), np.uint16), ry) and bits_equal(host(ab.view(torch.int16), np.uint16), rab) and bits_equal(host(c), rc)
    torch.autograd.backward([y, ab], [torch.from_numpy(dy).to('cuda:0'), torch.from_numpy(dab).to('cuda:0')])
    assert bits_equal(host(xt.grad), O.block_entry_bwd(xb, nw, rstd, wab, O.f2bf(dy), O.f2bf(dab)))
    # silu-mul: gradient has gu's shape and dtype, strided input accepted
    base = torch.randn(M, 4608, device='cuda:0').bfloat16()
    gu = base[:, 256:256 + 2048].detach().requires_grad_()
    yq, cq, sq = A.silu_mul_actq(gu)
    yq.backward(torch.randn(M, 1024, device='cuda:0').bfloat16())
    assert gu.grad.shape == (M, 2048) and gu.grad.dtype == torch.bfloat16 and torch.isfinite(gu.grad.float()).all()


@pytest.mark.parametrize('M,d,nab', [(1, 1024, 16), (2, 384, 14), (3, 256, 2), (5, 128, 4), (4, 768, 12), (1023, 1024, 10)])
def test_block_entry_rows_shared_by_a_workgroup(M, d, nab):
    """four rows share the projections: row counts around multiples of four, projection counts around the waves' four, every round
    count; a row of zeros, one with an infinity and one of subnormals (their products and sums round like fmaf)"""
    rng = np.random.default_rng(77 + M + d)
    x = outliers(rng, (M, d)); nw = (0.5 + rng.random(d)).astype(np.float32); wab = O.f2bf(rng.standard_normal((nab, d)) * 0.05)
    if M > 1: x[1] = 0
    if M > 2: x[2, 3] = np.inf
    if M > 3: x[3] *= 1e-38
    ry, rs, rc, rab, rstd = O.block_entry_fwd(x, nw, wab, 1e-6)
    y = dev(np.zeros((M, d), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, d // 2), np.uint8))
    ab = dev(np.full((M + 4, nab), 0x1234, np.uint16)); rstd_d = dev(np.zeros(M, np.float32))
    call('camx_block_entry_fwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(wab)), I(nab), F(1e-6), ptr(y), ptr(s), ptr(c), ptr(ab), ptr(rstd_d), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(rstd_d), rstd) and bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    assert bits_equal(host(ab, np.uint16)[:M], rab) and (host(ab, np.uint16)[M:] == 0x1234).all()
    x[2 % M] = 1.0                                                             # (finite rows for the backward)
    rstd = O.block_entry_fwd(x, nw, wab, 1e-6)[4]
    dy = O.f2bf(rng.standard_normal((M, d)).astype(np.float32)); dab = O.f2bf(rng.standard_normal((M, nab)).astype(np.float32))
    dx = dev(np.full((M + 4, d), 7.0, np.float32))
    call('camx_block_entry_bwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(rstd)), ptr(dev(wab)), I(nab), ptr(dev(dy)), ptr(dev(dab)), ptr(dx), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(dx)[:M], O.block_entry_bwd(x, nw, rstd, wab, dy, dab)) and (host(dx)[M:] == 7.0).all()


@pytest.mark.parametrize('M,d,nab', [(5, 384, 4), (2, 128, 16), (4, 896, 10), (3, 512, 2), (3, 1152, 3)])
def test_block_entry_infinite_rstd(M, d, nab):
    """eps = 0 and rows whose squares underflow: rstd is infinite, the projections of the row's own elements are +inf or NaN as the signs
    have it, and rows that end inside a round of 256 add nothing for the padding behind them"""
    rng = np.random.default_rng(d + nab)
    x = (1e-30 * (0.5 + rng.random((M, d)))).astype(np.float32); x[1] *= np.where(rng.random(d) < 0.5, -1, 1)
    nw = (0.5 + rng.random(d)).astype(np.float32); wab = O.f2bf((0.01 + rng.random((nab, d))).astype(np.float32))
    ry, rs, rc, rab, rstd = O.block_entry_fwd(x, nw, wab, 0.0)
    assert np.isinf(rstd).all() and np.isinf(O.bf2f(rab)[0]).all() and np.isnan(O.bf2f(rab)[1]).all()
    y = dev(np.zeros((M, d), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, d // 2), np.uint8))
    ab = dev(np.zeros((M, nab), np.uint16)); rstd_d = dev(np.zeros(M, np.float32))
    call('camx_block_entry_fwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(wab)), I(nab), F(0.0), ptr(y), ptr(s), ptr(c), ptr(ab), ptr(rstd_d), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(rstd_d), rstd) and bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    assert bits_equal(host(ab, np.uint16), rab)


@pytest.mark.parametrize('K', [128, 512, 640, 1024, 1536, 1664, 2048, 2176, 3072, 3200, 4096])
@pytest.mark.parametrize('streams', [False, True])
def test_actq_rounds_and_waves_of_a_row(K, streams):
    """every number of rounds of 512 values and of waves a row, whole and with a partial last round, below and from the batch size on
    whose outputs pass by the caches: rows with a NaN, an infinity, nothing but zeros, negative zeros, one value per chunk whose quotients
    are half-integers (3.5 = 7 / (14 / 7)), and a row whose maximum is everywhere"""
    rng = np.random.default_rng(700 + K)
    M = (1 << 20) // K + 3 if streams else 7
    x = outliers(rng, (M, K))
    x[0, K // 2] = np.nan; x[1, K - 1] = np.inf; x[2] = 0; x[3, :] = -0.0; x[3, 64] = 0.5
    x[4] = 0; x[4, 0::128] = 14.0 * 0.5 ** (np.arange(K // 128) % 4)
    x[5] = 0; x[5, ::128] = 3.0
    g = O.f2bf(rng.standard_normal((M, K)).astype(np.float32)); g[6, :4] = 0x8000
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        srcd = dev(src)
        ry, rs, rc = O.actq_fwd(src, bf16=bf)
        y = dev(np.zeros((M, K), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, K // 2), np.uint8))
        call('camx_actq_fwd', ptr(srcd), I(int(bf)), ptr(y), ptr(s), ptr(c), I(K), F(1.0), I(7), I(M))
        assert bits_equal(host(s), rs) and bits_equal(host(y, np.uint16), ry) and bits_equal(host(c), rc)
        want = O.actq_bwd(src, g, bf16=bf)
        dx = dev(np.zeros((M, K), np.uint16 if bf else np.float32))
        call('camx_actq_bwd', ptr(srcd), I(int(bf)), ptr(dev(g)), ptr(dx), I(K), F(1.0), I(7), I(M))
        assert bits_equal(host(dx, np.uint16) if bf else host(dx), want)


@pytest.mark.parametrize('M,d,nab,eps', [(4097, 1024, 16, 1e-6), (4111, 384, 10, 0.0), (4096, 128, 9, 1e-6), (8193, 640, 6, 0.0), (8207, 512, 8, 1e-6), (4100, 896, 13, 0.0)])
def test_block_entry_fwd_sixteen_rows_a_workgroup(M, d, nab, eps):
    """batches whose projections are shared by sixteen rows: last workgroups of 1, 15, 0, 1, 15 and 4 rows, every number of rounds, and rows of
    zeros (with eps = 0 an infinite rstd), an infinity and a NaN beside ordinary ones"""
    rng = np.random.default_rng(900 + d + nab)
    x = outliers(rng, (M, d)); x[M - 2] = 0; x[5] = 0; x[17, 3] = np.inf; x[40, d - 1] = np.nan
    nw = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32); wab = O.f2bf(rng.standard_normal((nab, d)) * 0.05)
    with np.errstate(all='ignore'): ry, rs, rc, rab, rstd = O.block_entry_fwd(x, nw, wab, eps)
    y = dev(np.zeros((M, d), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, d // 2), np.uint8))
    ab = dev(np.zeros((M, nab), np.uint16)); rstd_d = dev(np.zeros(M, np.float32))
    call('camx_block_entry_fwd', ptr(dev(x)), ptr(dev(nw)), ptr(dev(wab)), I(nab), F(eps), ptr(y), ptr(s), ptr(c), ptr(ab), ptr(rstd_d), I(d), F(1.0), I(7), I(M))
    assert bits_equal(host(rstd_d), rstd) and bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    assert bits_equal(host(ab, np.uint16), rab)


@pytest.mark.parametrize('K', [128, 640, 2048])
def test_actq_signs_of_zeros(K):
    """rows whose chunks begin with -0: the sign of a zero result comes through the rotation of the wave-per-row kernels (all zeros of one
    sign, of either at random, pairs that cancel behind a -0, and ordinary rows beside them), in x and in the gradient"""
    rng = np.random.default_rng(K)
    M = 24
    x = outliers(rng, (M, K))
    x[0] = -0.0; x[1] = 0.0
    x[2] = np.where(rng.random(K) < 0.5, -0.0, 0.0); x[3, ::128] = -0.0; x[3, 1::128] = 0.0
    x[4] = np.where(np.arange(K) % 2, 0.0, -0.0)
    x[5] = -0.0; x[5, 64::128] = 3.0; x[5, 65::128] = -3.0; x[5, 96::128] = 3.0; x[5, 97::128] = 3.0
    x[6, :128] = -0.0
    g = rng.standard_normal((M, K)).astype(np.float32); g[7] = -0.0; g[8] = np.where(np.arange(K) % 3, 0.0, -0.0); g[9, ::128] = -0.0; g[9, 1::128] = -0.0; g[0] = -0.0
    g = O.f2bf(g)
    for bf in (False, True):
        src = O.f2bf(x) if bf else x
        ry, rs, rc = O.actq_fwd(src, clip=1.0, qmax=7, bf16=bf)
        y = dev(np.zeros((M, K), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, K // 2), np.uint8))
        call('camx_actq_fwd', ptr(dev(src)), I(int(bf)), ptr(y), ptr(s), ptr(c), I(K), F(1.0), I(7), I(M))
        assert bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
        dx = dev(np.zeros((M, K), np.uint16 if bf else np.float32))
        call('camx_actq_bwd', ptr(dev(src)), I(int(bf)), ptr(dev(g)), ptr(dx), I(K), F(1.0), I(7), I(M))
        assert bits_equal(host(dx, np.uint16) if bf else host(dx), O.actq_bwd(src, g, clip=1.0, qmax=7, bf16=bf))


def test_block_entry_gradient_of_one_output():
    """an output nothing depends on has a zero gradient: y alone, ab alone"""
    import torch
    from caminus_amd.train import actq as A
    rng = np.random.default_rng(8)
    M, d, nab = 9, 256, 4
    x = outliers(rng, (M, d)); nw = (0.5 + rng.random(d)).astype(np.float32); wab = O.f2bf((rng.standard_normal((nab, d)) / 30).astype(np.float32))
    dy = O.f2bf(rng.standard_normal((M, d)).astype(np.float32)); dab = O.f2bf(rng.standard_normal((M, nab)).astype(np.float32))
    rstd = O.block_entry_fwd(x, nw, wab, 1e-6)[4]
    for use_y in (True, False):
        xt = torch.from_numpy(x).to('cuda:0').requires_grad_()
        y, c, s, ab = A.block_entry(xt, torch.from_numpy(nw).to('cuda:0'), dev(wab).view(torch.bfloat16), 1e-6)
        if use_y: y.backward(dev(dy).view(torch.bfloat16))
        else: ab.backward(dev(dab).view(torch.bfloat16))
        assert bits_equal(host(xt.grad), O.block_entry_bwd(x, nw, rstd, wab, dy if use_y else np.zeros_like(dy), np.zeros_like(dab) if use_y else dab))


@pytest.mark.parametrize('bf', [False, True])
def test_actq_fwd_and_bwd_four_million_values(bf):
    """enough values that the forward's division-free rounding meets its fallback thousands of times"""
    rng = np.random.default_rng(5150)
    M, K = 2048, 2048
    x = (rng.standard_normal((M, K)) * np.exp(rng.standard_normal((M, 1)))).astype(np.float32)
    g = O.f2bf(rng.standard_normal((M, K)).astype(np.float32))
    src = O.f2bf(x) if bf else x
    ry, rs, rc = O.actq_fwd(src, clip=0.95, qmax=7, bf16=bf)
    y = dev(np.zeros((M, K), np.uint16)); s = dev(np.zeros(M, np.float32)); c = dev(np.zeros((M, K // 2), np.uint8))
    xd = dev(src)
    call('camx_actq_fwd', ptr(xd), I(int(bf)), ptr(y), ptr(s), ptr(c), I(K), F(0.95), I(7), I(M))
    assert bits_equal(host(s), rs) and bits_equal(host(c), rc) and bits_equal(host(y, np.uint16), ry)
    dx = dev(np.zeros((M, K), np.uint16 if bf else np.float32))
    call('camx_actq_bwd', ptr(xd), I(int(bf)), ptr(dev(g)), ptr(dx), I(K), F(0.95), I(7), I(M))
    assert bits_equal(host(dx, np.uint16) if bf else host(dx), O.actq_bwd(src, g, clip=0.95, qmax=7, bf16=bf))


@pytest.mark.parametrize('M', [511, 513, 1023, 1025])
@pytest.mark.parametrize('K', [2176, 3072, 3200, 4096])
def test_actq_two_waves_of_a_row(M, K):
    """rows of 2049 to 4096 values on both sides of the batch sizes that give them two waves (512 and 1024), plain and SiLU-fused, forward and backward,
    odd row counts: a NaN or an infinity in one wave's chunks only (chunks 0 .. 3 and 4 .. 7 of every 8 are the first and the second wave's), zeros,
    maxima in either half. Bit for bit against the same rows in batches that a workgroup a row takes, and the ordinary rows against the oracle"""
    import torch
    rng = np.random.default_rng(K + M)
    x = outliers(rng, (M, K)); g = O.f2bf(rng.standard_normal((M, K)).astype(np.float32))
    gate = (rng.standard_normal((M, K)) * 2).astype(np.float32); gate[rng.random((M, K)) < 1e-3] *= 200
    for a in (x, gate):
        a[0, 5] = np.nan; a[1, 5 * 128 + 3] = np.nan; a[2, 3] = np.inf; a[3, 6 * 128] = -np.inf; a[M - 1, K - 1] = np.nan; a[M - 2, 0] = np.inf
        a[4] = 0; a[5] = -0.0; a[6] = 0; a[6, 7] = 3.0; a[7] = 0; a[7, 4 * 128 + 7] = 3.0; a[8, 128:256] *= 100; a[9, 4 * 128:5 * 128] *= 100
    gu = O.f2bf(np.concatenate([gate, x], axis=1))
    plain = [4, 5, 6, 7, 8, 9, 10, M // 2, M - 3]                 # rows without a NaN or an infinity
    gd, n = dev(g), 255

    def equal(a, b):
        nan = torch.isnan(a) & torch.isnan(b)
        return bool(((a.view(torch.int16) == b.view(torch.int16)) if a.dtype == torch.bfloat16 else (a.view(torch.int32) == b.view(torch.int32))).logical_or(nan).all())

    def buffers(dt, width): return [torch.full((M + 1, width), 5.0, device='cuda', dtype=dt) for _ in range(2)]

    def both(run):                                                # the whole batch, then 255 rows at a time
        run(0, 0, M)
        for lo in range(0, M, n): run(1, lo, min(n, M - lo))
        torch.cuda.synchronize()

    for form in ('f32', 'bf16', 'silu'):
        src = dev(x) if form == 'f32' else dev(O.f2bf(x)).view(torch.bfloat16) if form == 'bf16' else dev(gu).view(torch.bfloat16)
        y, s = buffers(torch.bfloat16, K), [torch.full((M + 1,), 5.0, device='cuda') for _ in range(2)]
        c = [torch.full((M + 1, K // 2), 5, device='cuda', dtype=torch.uint8) for _ in range(2)]
        d = buffers(torch.float32 if form == 'f32' else torch.bfloat16, 2 * K if form == 'silu' else K)

        def forward(i, lo, m):
            a = (ptr(y[i][lo:]), ptr(s[i][lo:]), ptr(c[i][lo:]))
            if form == 'silu': call('camx_silu_mul_actq_fwd', ptr(src[lo:]), I(2 * K), I(K), *a, F(1.0), I(7), I(m))
            else: call('camx_actq_fwd', ptr(src[lo:]), I(int(form == 'bf16')), *a, I(K), F(1.0), I(7), I(m))

        def backward(i, lo, m):
            if form == 'silu': call('camx_silu_mul_actq_bwd', ptr(src[lo:]), I(2 * K), I(K), ptr(gd[lo:]), ptr(d[i][lo:]), F(1.0), I(7), I(m))
            else: call('camx_actq_bwd', ptr(src[lo:]), I(int(form == 'bf16')), ptr(gd[lo:]), ptr(d[i][lo:]), I(K), F(1.0), I(7), I(m))
        both(forward); both(backward)
        for a, b in (y, [t.view(M + 1, 1) for t in s], d): assert equal(a, b), form
        assert torch.equal(c[0], c[1]), form
        for t in (y[0], s[0], c[0], d[0]): assert bool((t[M] == 5).all()), form
        rows = np.array(plain)
        if form == 'silu': (ry, rs, rc), want = O.silu_mul_actq_fwd(gu[rows]), O.silu_mul_actq_bwd(gu[rows], g[rows], table=True)
        else:
            a = O.f2bf(x[rows]) if form == 'bf16' else x[rows]
            (ry, rs, rc), want = O.actq_fwd(a, bf16=form == 'bf16'), O.actq_bwd(a, g[rows], bf16=form == 'bf16')
        got = host(d[0][:M].view(torch.int16), np.uint16) if d[0].dtype == torch.bfloat16 else host(d[0][:M])
        assert bits_equal(host(y[0][:M].view(torch.int16), np.uint16)[rows], ry) and bits_equal(host(s[0])[rows], rs) and bits_equal(host(c[0])[rows], rc), form
        assert bits_equal(got[rows], want), form


@pytest.mark.parametrize('M,d,nab,eps', [(8177, 1024, 16, 1e-6), (8191, 384, 10, 0.0), (4096, 896, 5, 1e-6), (12284, 640, 13, 0.0), (8192, 512, 8, 1e-6), (8190, 128, 13, 0.0)])
def test_block_entry_fwd_sixteen_rows_from_a_full_chip(M, d, nab, eps):
    """batches just below whole multiples of 4096 rows, which sixteen rows a workgroup take: last workgroups of 1, 15, 16, 12, 16 and 14 rows"""
    test_block_entry_fwd_sixteen_rows_a_workgroup(M, d, nab, eps)
