"""GPU parity of the elementwise / small row kernels against the CPU oracle: exact where no transcendental is involved,
1e-5 relative (fp32) / one 16-bit ulp otherwise."""
import numpy as np
import pytest

import oracle as O
from gpu_util import F, I, L64, NULL, bits_equal, call, close_16, close_fp32, dev, host, outliers, ptr

pytestmark = pytest.mark.gpu
EXTREMES = np.array([30, -30, 0, -0.0, 1e-3, -88, 88, 5], np.float32)


@pytest.mark.parametrize('n', [8 * 768, 1001, 7])
def test_swiglu(n):
    rng = np.random.default_rng(n)
    g = outliers(rng, n); u = outliers(rng, n); g[:min(8, n)] = EXTREMES[:min(8, n)]
    y16 = dev(np.zeros(n, np.uint16)); y32 = dev(np.zeros(n, np.float32)); gd, ud = dev(g), dev(u)
    call('camx_q3p_swiglu', ptr(gd), ptr(ud), ptr(y16), I(n))
    call('camx_gg_silu_mul', ptr(gd), ptr(ud), ptr(y32), I(n))
    assert close_16(host(y16, np.uint16), O.swiglu16(g, u), 'f16')
    assert close_fp32(host(y32), O.silu_mul_f32(g, u))


@pytest.mark.parametrize('R,H', [(4, 17408), (3, 7), (256, 17408), (1100, 4096)])
def test_silu_mul_bf16(R, H):
    """bf16(silu g) comes from the table of the correctly rounded value at every size (in device memory for small inputs, in LDS
    from 2^22 values on): bit-equal to the oracle, NaN (canonical) and infinities included"""
    rng = np.random.default_rng(H)
    gu = O.f2bf(outliers(rng, (R, 2 * H)) * np.float32(2))
    gu[0, :6] = [0x7fc0, 0xffc1, 0x7f80, 0xff80, 0x0000, 0x8000]; gu[0, H:H + 6] = [0x3f80, 0x3f80, 0x0000, 0x3f80, 0x7f80, 0x7fa5]
    act = dev(np.zeros((R, H), np.uint16))
    call('camx_silu_mul_bf16', ptr(dev(gu)), ptr(act), I(H), L64(R * H))
    want = O.silu_mul_bf16(gu); got = host(act, np.uint16)
    assert np.array_equal(got, want)


def test_gate_mul():
    rng = np.random.default_rng(1004)
    T, H, D = 16, 24, 256
    a = outliers(rng, (T * H, D)); qg = outliers(rng, (T * H, 2 * D)); qg[0, D:D + 8] = EXTREMES
    ad, gd = dev(a), dev(qg)
    y = dev(np.zeros_like(a)); y16 = dev(np.zeros(a.shape, np.uint16))
    call('camx_gate_mul', ptr(ad), ptr(gd), ptr(y), L64(a.size), I(D), I(2 * D), I(D), I(0))
    call('camx_gate_mul', ptr(ad), ptr(gd), ptr(y16), L64(a.size), I(D), I(2 * D), I(D), I(1))
    assert close_fp32(host(y), O.gate_mul(a, qg, D, 2 * D, D))
    assert close_16(host(y16, np.uint16), O.gate_mul(a, qg, D, 2 * D, D, f16=True), 'f16')
    abf, gbf = O.f2bf(a), O.f2bf(qg)
    ybf = dev(np.zeros(a.shape, np.uint16))
    call('camx_gate_mul', ptr(dev(abf)), ptr(dev(gbf)), ptr(ybf), L64(a.size), I(D), I(2 * D), I(D), I(2))
    assert close_16(host(ybf, np.uint16), O.f2bf(O.gate_mul(O.bf2f(abf), O.bf2f(gbf), D, 2 * D, D)), 'bf16')


@pytest.mark.parametrize('T,C', [(16, 10240), (1, 64), (2, 100), (5, 256), (37, 512), (3, 6), (520, 8192), (130, 8200)])
def test_gdn_conv(T, C):
    rng = np.random.default_rng(C)
    ldx = C + 4
    x = outliers(rng, (T, ldx)); w = rng.standard_normal((C, 4)).astype(np.float32); st = rng.standard_normal((C, 3)).astype(np.float32)
    ref_y, ref_st = O.gdn_conv(x, w, st, ldx=ldx)
    xd, wd, sd = dev(x), dev(w), dev(st); y = dev(np.zeros((T, C), np.float32))
    call('camx_pf_gdn_conv', ptr(xd), ptr(wd), ptr(sd), ptr(y), I(C), I(T), I(ldx), I(C), I(0))
    call('camx_pf_conv_state', ptr(xd), ptr(sd), I(C), I(T), I(ldx), I(0))
    assert close_fp32(host(y), ref_y) and bits_equal(host(sd), ref_st)


@pytest.mark.parametrize('T,heads,K', [(16, 32, 128), (16, 48, 128), (3, 5, 256), (2, 3, 96), (1030, 32, 128), (683, 48, 128), (2049, 32, 128), (1401, 48, 128)])
def test_gdn_l2(T, heads, K):
    rng = np.random.default_rng(K + heads)
    ldx = heads * K + 64
    x = outliers(rng, (T, ldx))
    y = dev(np.zeros((T * heads, K), np.float32))
    call('camx_pf_gdn_l2', ptr(dev(x)), ptr(y), I(heads), I(K), I(ldx), F(np.float32(1e-6 / K)), I(T), I(0))
    ref = O.gdn_l2(x, T, heads, K, 1e-6, ldx=ldx)
    assert bits_equal(host(y), ref)
    if K == 128:                                                       # bf16 in / out (a prefill chunk's form)
        xb = O.f2bf(x); yb = dev(np.zeros((T * heads, K), np.uint16))
        call('camx_pf_gdn_l2', ptr(dev(xb)), ptr(yb), I(heads), I(K), I(ldx), F(np.float32(1e-6 / K)), I(T), I(1))
        assert bits_equal(host(yb, np.uint16), O.f2bf(O.gdn_l2(O.bf2f(xb), T, heads, K, 1e-6, ldx=ldx)))


def test_core_and_fuse():
    rng = np.random.default_rng(5)
    T, D, V = 9, 896, 50
    emb = rng.standard_normal((V, D)).astype(np.float32); tok = rng.integers(0, V, T).astype(np.int32)
    out = dev(np.zeros((T, D), np.float32))
    call('camx_embedding_f32', ptr(dev(tok)), ptr(dev(emb)), ptr(out), I(D), I(T))
    assert bits_equal(host(out), O.embedding_f32(tok, emb))
    x = outliers(rng, (T, D))
    m = O.f2bf(outliers(rng, (T, D))); y = O.f2bf(outliers(rng, (T, D)))
    o = dev(np.zeros((T, D), np.float32))
    call('camx_residual3', ptr(dev(x)), ptr(dev(m)), ptr(dev(y)), ptr(o), L64(T * D))
    assert bits_equal(host(o), O.residual3(x, m, y))
    o1 = dev(np.zeros(T * D - 3, np.float32))                          # a length that is no multiple of four: the element-wise form
    call('camx_residual3', ptr(dev(x)), ptr(dev(m)), ptr(dev(y)), ptr(o1), L64(T * D - 3))
    assert bits_equal(host(o1), O.residual3(x, m, y).reshape(-1)[:T * D - 3])
    x[0, :6] = [np.nan, np.inf, -np.inf, 1e-40, -np.nan, 3.3895314e38]
    c = dev(np.zeros((T, D), np.uint16))
    call('camx_cast_bf16', ptr(dev(x)), ptr(c), L64(T * D))
    assert bits_equal(host(c, np.uint16), O.f2bf(x))
    c1 = dev(np.zeros(T * D - 5, np.uint16))
    call('camx_cast_bf16', ptr(dev(x)), ptr(c1), L64(T * D - 5))
    assert bits_equal(host(c1, np.uint16), O.f2bf(x).reshape(-1)[:T * D - 5])
    dst = rng.integers(0, 65536, (T, 64)).astype(np.uint16); dd = dev(dst)
    call('camx_copy_cols_bf16', ptr(dev(m)), I(D), I(5), ptr(dd), I(64), I(3), I(40), L64(T))
    assert bits_equal(host(dd, np.uint16), O.copy_cols_bf16(m, 5, dst, 3, 40))
    dd2 = dev(dst)                                                     # offsets and width in whole 16-byte units
    call('camx_copy_cols_bf16', ptr(dev(m)), I(D), I(8), ptr(dd2), I(64), I(16), I(40), L64(T))
    assert bits_equal(host(dd2, np.uint16), O.copy_cols_bf16(m, 8, dst, 16, 40))
    whole = rng.integers(0, 65536, (517, 64)).astype(np.uint16); dd3 = dev(np.zeros((517, 64), np.uint16))     # whole contiguous rows: the flat copy
    call('camx_copy_cols_bf16', ptr(dev(whole)), I(64), I(0), ptr(dd3), I(64), I(0), I(64), L64(517))
    assert bits_equal(host(dd3, np.uint16), whole)
    ys = O.f2bf(outliers(rng, (4, D))); pos = np.array([-1, 0, 3, -1, 2, 1, -1, -1, 0], np.int32)
    x2 = outliers(rng, (T, D))
    for has in (True, False):
        o2 = dev(np.zeros((T, D), np.float32))
        call('camx_residual_slices_fwd', ptr(dev(x2)), ptr(dev(m)), ptr(dev(y)), ptr(dev(ys)) if has else NULL, ptr(dev(pos)) if has else NULL,
             ptr(o2), I(D), L64(T * D // 4))
        assert bits_equal(host(o2), O.residual_slices_fwd(x2, m, y, ys if has else None, pos if has else None))


@pytest.mark.parametrize('T,D', [(9, 896), (300, 2048), (7, 892), (33, 100), (5, 8)])
def test_residual_slices_widths(T, D):
    """several row widths and counts, forward and backward, with and without slices, non-finite and subnormal values"""
    rng = np.random.default_rng(60 + D)
    nys = 4
    x = outliers(rng, (T, D)); m = O.f2bf(outliers(rng, (T, D))); mlp = O.f2bf(outliers(rng, (T, D))); ys = O.f2bf(outliers(rng, (nys, D)))
    pos = rng.integers(-1, nys, T).astype(np.int32); pos[rng.random(T) < 0.5] = -1
    taken = pos[pos >= 0]; pos[pos >= 0] = np.where(np.arange(len(taken)) < nys, rng.permutation(nys)[np.arange(len(taken)) % nys], -1)   # each slice at most once
    seen = set()
    for r in range(T):
        if pos[r] >= 0 and int(pos[r]) in seen: pos[r] = -1
        elif pos[r] >= 0: seen.add(int(pos[r]))
    x[0, :4] = [np.nan, np.inf, -0.0, 1e-40]
    for has in (True, False):
        o = dev(np.zeros((T, D), np.float32))
        call('camx_residual_slices_fwd', ptr(dev(x)), ptr(dev(m)), ptr(dev(mlp)), ptr(dev(ys)) if has else NULL, ptr(dev(pos)) if has else NULL, ptr(o), I(D), L64(T * D // 4))
        want = O.residual_slices_fwd(x, m, mlp, ys if has else None, pos if has else None)
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(host(o)), nan) and bits_equal(np.where(nan, 0, host(o)), np.where(nan, 0, want))
    rdm, rdmlp, rdys = O.residual_slices_bwd(x, pos, nys)
    dm = dev(np.zeros((T, D), np.uint16)); dmlp = dev(np.zeros((T, D), np.uint16)); dys = dev(np.zeros((nys, D), np.uint16))
    call('camx_residual_slices_bwd', ptr(dev(x)), ptr(dev(pos)), ptr(dm), ptr(dmlp), ptr(dys), I(D), L64(T * D // 4))
    used = sorted(seen)
    assert bits_equal(host(dm, np.uint16), rdm) and bits_equal(host(dmlp, np.uint16), rdmlp) and bits_equal(host(dys, np.uint16)[used], rdys[used])


def test_residual_slices_bwd_and_autograd():
    """the backward kernel against the oracle, and the autograd wrapper end to end against torch's own graph of the same sum"""
    import torch
    from caminus_amd.train.fuse import residual_slices
    rng = np.random.default_rng(6)
    T, D, nys = 11, 896, 5
    dout = outliers(rng, (T, D)); dout[0, :3] = [np.nan, np.inf, 3.3895314e38]
    pos = np.array([-1, 0, 3, -1, 2, 1, -1, -1, 4, -1, -1], np.int32)
    rdm, rdmlp, rdys = O.residual_slices_bwd(dout, pos, nys)
    dm = dev(np.zeros((T, D), np.uint16)); dmlp = dev(np.zeros((T, D), np.uint16)); dys = dev(np.zeros((nys, D), np.uint16))
    call('camx_residual_slices_bwd', ptr(dev(dout)), ptr(dev(pos)), ptr(dm), ptr(dmlp), ptr(dys), I(D), L64(T * D // 4))
    assert bits_equal(host(dm, np.uint16), rdm) and bits_equal(host(dmlp, np.uint16), rdmlp) and bits_equal(host(dys, np.uint16), rdys)
    x = torch.randn(T, D, device='cuda:0', requires_grad=True)
    m = torch.randn(T, D, device='cuda:0').bfloat16().requires_grad_(); mlp = torch.randn(T, D, device='cuda:0').bfloat16().requires_grad_()
    ys = torch.randn(nys, D, device='cuda:0').bfloat16().requires_grad_(); pd = torch.from_numpy(pos).to('cuda:0')
    out = residual_slices(x, m, mlp, ys, pd)
    gsel = torch.zeros(T, D, device='cuda:0'); sel = pd >= 0
    gsel[sel] = ys.detach().float()[pd[sel].long()]
    want = ((x.detach() + m.detach().float()) + mlp.detach().float()) + gsel
    assert torch.equal(out.detach(), want)
    go = torch.randn(T, D, device='cuda:0')
    out.backward(go)
    assert torch.equal(x.grad, go) and torch.equal(m.grad, go.bfloat16()) and torch.equal(mlp.grad, go.bfloat16())
    assert torch.equal(ys.grad[pd[sel].long()], go[sel].bfloat16())


def test_cast_bf16_every_upper_half_with_edge_lower_halves():
    """fp32 -> bf16 over every sign / exponent / top-mantissa pattern combined with the lower halves where rounding decides
    (ties, one off a tie, all ones), NaN payloads and denormals included: 0x7fc0 for every NaN, nearest-even elsewhere"""
    hi = np.arange(65536, dtype=np.uint32) << 16
    lows = np.array([0x0000, 0x0001, 0x7fff, 0x8000, 0x8001, 0xffff, 0x4000, 0xc000, 0x8000 - 2, 0x1234, 0xfedc, 0x8002], np.uint32)
    x = (hi[:, None] | lows[None, :]).reshape(-1).view(np.float32)
    c = dev(np.zeros(x.size, np.uint16))
    call('camx_cast_bf16', ptr(dev(x)), ptr(c), L64(x.size))
    assert bits_equal(host(c, np.uint16), O.f2bf(x))
    c1 = dev(np.zeros(x.size - 1, np.uint16))                             # the element-wise form
    call('camx_cast_bf16', ptr(dev(x)), ptr(c1), L64(x.size - 1))
    assert bits_equal(host(c1, np.uint16), O.f2bf(x)[:-1])


@pytest.mark.parametrize('C,T', [(10240, 16), (96, 5), (300, 1)])
def test_op_gdn_conv_lazy_commit(C, T):
    """OP_GDN_CONV: two passes with every commit count; the state after the commit and the next pass's xprev bit for bit, the outputs
    within the FP class (silu) and equal to the chunk kernel's on the same state"""
    from gpu_util import close_fp32
    rng = np.random.default_rng(C + T)
    w = rng.standard_normal((C, 4)).astype(np.float32); st0 = rng.standard_normal((C, 3)).astype(np.float32)
    x1 = outliers(rng, (T, C)); x2 = outliers(rng, (T, C)); junk = rng.standard_normal((T, C)).astype(np.float32)
    wd = dev(w)
    for m in sorted({0, 1, T // 2, T}):
        std = dev(st0); xp = dev(junk); y = dev(np.zeros((T, C), np.float32))
        call('camx_op_gdn_conv', ptr(wd), ptr(std), ptr(dev(x1)), ptr(dev(np.array([0, 0, 0, 0], np.int32))), ptr(y), ptr(xp), I(C), I(T))
        ry1, rst1, rxp1 = O.op_gdn_conv(w, st0, x1, 0, junk)
        assert bits_equal(host(std), rst1) and bits_equal(host(xp), rxp1) and close_fp32(host(y), ry1)
        y2 = dev(np.zeros((T, C), np.float32))
        call('camx_op_gdn_conv', ptr(wd), ptr(std), ptr(dev(x2)), ptr(dev(np.array([7, m, 0, 0], np.int32))), ptr(y2), ptr(xp), I(C), I(T))
        ry2, rst2, rxp2 = O.op_gdn_conv(w, rst1, x2, m, rxp1)
        assert bits_equal(host(std), rst2) and bits_equal(host(xp), rxp2) and close_fp32(host(y2), ry2)
        yc = dev(np.zeros((T, C), np.float32))                      # the chunk kernel from the committed state: the same bits
        call('camx_pf_gdn_conv', ptr(dev(x2)), ptr(wd), ptr(std), ptr(yc), I(C), I(T), I(C), I(C), I(0))
        assert bits_equal(host(yc), host(y2))


def _same(a, b):
    import torch
    return bool(((a == b) | (torch.isnan(a) & torch.isnan(b))).all())


@pytest.mark.parametrize('T', [128, 129, 131, 257, 2047, 2048, 2049, 2053])
@pytest.mark.parametrize('bf16', [0, 1])
def test_gdn_conv_tokens_do_not_depend_on_the_chunk(T, bf16):
    """the chunk kernel (from 2^20 values, more tokens a wave from 2^24 fp32 or 3 x 2^21 bf16) against the same tokens in pieces of 64, which the kernel of one value a
    thread takes, its state advanced by camx_pf_conv_state; the committing entry's y and state against both; chunks that end inside a
    wave's tokens and inside a workgroup; values beyond the exponential's short form, infinities and a NaN; nothing behind the last row"""
    import torch
    C, ldx, ldy = 8192, 8200, 8208
    g = torch.Generator(device='cuda'); g.manual_seed(T)
    x = torch.randn(T, ldx, generator=g, device='cuda')
    x[::7, 5::11] *= 300; x[T // 2, 17] = float('inf'); x[3, 40] = float('nan'); x[T - 1, 8191] = -float('inf'); x[5, :16] = 0
    w = torch.randn(C, 4, generator=g, device='cuda'); st0 = torch.randn(C, 3, generator=g, device='cuda')
    dt = torch.bfloat16 if bf16 else torch.float32
    x = x.to(dt)
    parts, st = torch.empty(T, ldy, device='cuda', dtype=dt), st0.clone()
    for lo in range(0, T, 64):
        m = min(64, T - lo)
        call('camx_pf_gdn_conv', ptr(x[lo:]), ptr(w), ptr(st), ptr(parts[lo:]), I(C), I(m), I(ldx), I(ldy), I(bf16))
        call('camx_pf_conv_state', ptr(x[lo:]), ptr(st), I(C), I(m), I(ldx), I(bf16))
    for entry in ('camx_pf_gdn_conv', 'camx_pf_gdn_conv_commit'):
        y, st1 = torch.full((T + 1, ldy), 7.0, device='cuda', dtype=dt), st0.clone()
        call(entry, ptr(x), ptr(w), ptr(st1), ptr(y), I(C), I(T), I(ldx), I(ldy), I(bf16))
        torch.cuda.synchronize()
        assert _same(y[:T, :C], parts[:, :C]) and bool((y[T] == 7).all()) and bool((y[:, C:] == 7).all())
        assert _same(st1, st if entry.endswith('commit') else st0)
    y, qk, qk2 = torch.empty(T, C, device='cuda', dtype=dt), torch.empty(T * 16, 128, device='cuda', dtype=dt), torch.empty(T * 16, 128, device='cuda', dtype=dt)
    call('camx_gdn_conv_l2', ptr(x), ptr(w), ptr(st0), ptr(y), ptr(qk), I(C), I(T), I(ldx), I(C), I(16), F(1e-8), I(bf16))
    call('camx_pf_gdn_l2', ptr(y), ptr(qk2), I(16), I(128), I(C), F(1e-8), I(T), I(bf16))
    torch.cuda.synchronize()
    assert _same(y, parts[:, :C]) and _same(qk, qk2)


@pytest.mark.parametrize('T,C,bf16', [(16 * 65535 + 5, 8, 1), (16 * 65535 + 21, 4, 0), (32 * 65535, 8, 0), (32 * 65535 + 77, 128, 1)])
def test_gdn_conv_past_65535_groups_of_tokens(T, C, bf16):
    """more token groups than a grid has workgroups in y (eight tokens a wave, then the one-value kernel): the same rows in slices through that kernel"""
    import torch
    g = torch.Generator(device='cuda'); g.manual_seed(C)
    dt = torch.bfloat16 if bf16 else torch.float32
    x = torch.randn(T, C, generator=g, device='cuda').to(dt); w = torch.randn(C, 4, generator=g, device='cuda'); st0 = torch.randn(C, 3, generator=g, device='cuda')
    want, st, n = torch.empty_like(x), st0.clone(), (1 << 20) // C - 1
    for lo in range(0, T, n):
        m = min(n, T - lo)
        call('camx_pf_gdn_conv', ptr(x[lo:]), ptr(w), ptr(st), ptr(want[lo:]), I(C), I(m), I(C), I(C), I(bf16))
        call('camx_pf_conv_state', ptr(x[lo:]), ptr(st), I(C), I(m), I(C), I(bf16))
    y, st1 = torch.full_like(x, 7.0), st0.clone()
    call('camx_pf_gdn_conv_commit', ptr(x), ptr(w), ptr(st1), ptr(y), I(C), I(T), I(C), I(C), I(bf16))
    torch.cuda.synchronize()
    assert _same(y, want) and _same(st1, st)
    if C % 128 == 0:
        y.fill_(7.0); qk, qk2 = torch.empty(T, 128, device='cuda', dtype=dt), torch.empty(T, 128, device='cuda', dtype=dt)
        call('camx_gdn_conv_l2', ptr(x), ptr(w), ptr(st0), ptr(y), ptr(qk), I(C), I(T), I(C), I(C), I(1), F(1e-8), I(bf16))
        call('camx_pf_gdn_l2', ptr(want), ptr(qk2), I(1), I(128), I(C), F(1e-8), I(T), I(bf16))
        torch.cuda.synchronize()
        assert _same(y, want) and _same(qk, qk2)


@pytest.mark.parametrize('T,C', [(1, 64), (2, 8192), (3, 64), (130, 8200), (200, 6000)])
def test_gdn_conv_commit_is_the_two_launches(T, C):
    """chunks shorter than the state, below the chunk kernel's size, and channels it does not take"""
    import torch
    g = torch.Generator(device='cuda'); g.manual_seed(T)
    x = torch.randn(T, C, generator=g, device='cuda'); w = torch.randn(C, 4, generator=g, device='cuda'); a = torch.randn(C, 3, generator=g, device='cuda'); b = a.clone()
    ya, yb = torch.empty(T, C, device='cuda'), torch.empty(T, C, device='cuda')
    call('camx_pf_gdn_conv', ptr(x), ptr(w), ptr(a), ptr(ya), I(C), I(T), I(C), I(C), I(0)); call('camx_pf_conv_state', ptr(x), ptr(a), I(C), I(T), I(C), I(0))
    call('camx_pf_gdn_conv_commit', ptr(x), ptr(w), ptr(b), ptr(yb), I(C), I(T), I(C), I(C), I(0))
    torch.cuda.synchronize()
    assert torch.equal(ya, yb) and torch.equal(a, b)


@pytest.mark.parametrize('entry', ['gdn', 'ple'])
@pytest.mark.parametrize('part', range(4))
def test_silu_of_every_finite_value(entry, part):
    """a token's bits do not depend on the batch it came in: the convolutions' chunk kernels (their own division up to 80) against the kernels
    for small batches (the IEEE division), the last tap alone, over all finite fp32 inputs, 2^28 at a time"""
    import torch
    T, C = 32768, 8192
    w = torch.zeros(C, 4, device='cuda'); w[:, 3] = 1.0; st = torch.zeros(C, 3, device='cuda'); w16 = w.half()

    def conv(x, y, n):
        if entry == 'gdn': call('camx_pf_gdn_conv', ptr(x), ptr(w), ptr(st), ptr(y), I(C), I(n), I(C), I(C), I(0))
        else: call('camx_pf_ple_conv', ptr(x), NULL, NULL, ptr(w16), ptr(st), ptr(y), NULL, NULL, I(C), I(n), I(C), I(1))
    for k in range(4 * part, 4 * part + 4):
        first = (k << 28) - (1 << 31)
        bits = torch.arange(1 << 28, dtype=torch.int32, device='cuda') + first
        bits[(bits & 0x7f800000) == 0x7f800000] = 0
        x = bits.view(torch.float32).view(T, C)
        y, z = torch.empty_like(x), torch.empty_like(x)
        conv(x, y, T)
        for lo in range(0, T, 127): conv(x[lo:], z[lo:], min(127, T - lo))          # (127 x 8192 values: below every chunk kernel's batch)
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int32), z.view(torch.int32)), k
