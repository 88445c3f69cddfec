"""Workloads of the fused per-layer row kernels, each through the entry points that a user's program calls: the decode tape (TapeOps),
the prefill wrappers (prefill.*, Module('camx')) and the training functions with their backward passes (train.*).

Sizes are those of the repository's benchmark and tests: the qwen3moe-class decode token and prefill chunk (hidden 2048, 32 / 4 heads of
128, 8 experts of 768), the dense 27B-class chunk (hidden 5120, 64 / 8 heads of 128, MLP 17408), the hybrid line (hidden 5120, 24 / 4
heads of 256, convolution over 10240 channels, 48 value heads of 128), the hyper-connection glue (4 streams of 2560) and the trainer's
rows (1024 / 2048 values); the token counts run from one to a chunk of 4096, and to a batch of 32768 rows in training.
"""
import math

import numpy as np
import torch

DEV = 'cuda:0'
F32, F64, F16, BF16, I32, U8 = torch.float32, torch.float64, torch.float16, torch.bfloat16, torch.int32, torch.uint8
EPS = 1e-6


def listed():
    return [
        # one generated token of the qwen3moe-class model: the row ops of a layer, latency only
        {'name': 'decode_token', 'kind': 'moe_tape', 'tokens': 1, 'pos': 1234, 'q8': False},
        # a speculative verify pass of 16 tokens: the row ops of a linear and of a full-attention layer of the hybrid line
        {'name': 'verify_batch', 'kind': 'hybrid_tape', 'tokens': 16, 'pos': 40000},
        # continuous batching: 256 sequences take one token each: embedding gather + norm, rotary into the paged Q8 cache, add + norm
        {'name': 'batched_decode', 'kind': 'paged', 'seqs': 256, 'q8': True},
        # a prefill chunk of the dense line, bf16 activations (the benchmark's step)
        {'name': 'dense_prefill', 'kind': 'dense', 'tokens': 4096, 'pos': 0},
        # the last, ragged chunk of a prompt of the dense line
        {'name': 'dense_prefill_tail', 'kind': 'dense', 'tokens': 777, 'pos': 8192},
        # a prefill chunk of the qwen3moe line: Q8 cache, expert feed scattered to the router's columns
        {'name': 'moe_prefill', 'kind': 'moe', 'tokens': 2048, 'pos': 2048, 'q8': True},
        # a linear-attention layer of the hybrid line over a ragged chunk: convolution, L2 norm, gates, gated norm
        {'name': 'hybrid_linear', 'kind': 'gdn', 'tokens': 3001, 'bf16': False},
        # a full-attention layer of the same line with the Q8 cache: QK-norm + rotary, Hadamard, append, and the cache read back for a chunk at depth
        {'name': 'hybrid_attention', 'kind': 'attn', 'tokens': 2048, 'pos': 14336},
        # the hyper-connection glue and the per-layer-embedding block of a chunk (the shape the reference publishes times for)
        {'name': 'hyper_connections', 'kind': 'hyper', 'tokens': 2048},
        # activation fake-quant of a training batch, forward and backward
        {'name': 'train_actq', 'kind': 'actq', 'rows': 32768, 'width': 2048, 'bf16': True},
        # the MLP's fused SiLU-multiply + fake-quant, forward and backward
        {'name': 'train_mlp', 'kind': 'mlp', 'rows': 16384, 'width': 2048},
        # a training block's entry (RMSNorm + fake-quant + gate projections) and its fused residual, forward and backward
        {'name': 'train_block', 'kind': 'block', 'rows': 32768, 'width': 1024, 'proj': 16},
    ]


def _size(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['moe_tape', 'hybrid_tape', 'paged', 'dense', 'moe', 'gdn', 'attn', 'hyper', 'actq', 'mlp', 'block'])
    if kind == 'moe_tape': return {'kind': kind, 'tokens': _size(rng, 1, 16), 'pos': rng.randrange(4000), 'q8': rng.random() < 0.5}
    if kind == 'hybrid_tape': return {'kind': kind, 'tokens': _size(rng, 1, 32), 'pos': rng.randrange(40000)}
    if kind == 'paged': return {'kind': kind, 'seqs': _size(rng, 1, 1024), 'q8': rng.random() < 0.7}
    if kind == 'dense': return {'kind': kind, 'tokens': _size(rng, 64, 4096), 'pos': rng.randrange(30000)}
    if kind == 'moe': return {'kind': kind, 'tokens': _size(rng, 64, 4096), 'pos': rng.randrange(8192), 'q8': rng.random() < 0.6}
    if kind == 'gdn': return {'kind': kind, 'tokens': _size(rng, 64, 4096), 'bf16': rng.random() < 0.5}
    if kind == 'attn': return {'kind': kind, 'tokens': _size(rng, 64, 2048), 'pos': rng.randrange(14336)}
    if kind == 'hyper': return {'kind': kind, 'tokens': _size(rng, 64, 2048)}
    width = 128 * rng.randint(4, 32)
    if kind == 'actq': return {'kind': kind, 'rows': _size(rng, 4096, min(32768, (1 << 25) // width)), 'width': width, 'bf16': rng.random() < 0.6}
    if kind == 'mlp': return {'kind': kind, 'rows': _size(rng, 4096, min(16384, (1 << 25) // width)), 'width': width}
    return {'kind': kind, 'rows': _size(rng, 4096, 32768), 'width': 128 * rng.randint(4, 8), 'proj': 2 * rng.randint(0, 8)}


# ---- inputs --------------------------------------------------------------------------------------------------------------------------------
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=F32):
        return torch.randn(shape, generator=self.g, device=DEV).to(dtype)

    def acts(self, *shape, dtype=F32):
        """activations: N(0, 1) with one value in a thousand fifty times as large"""
        x = torch.randn(shape, generator=self.g, device=DEV)
        x = torch.where(torch.rand(shape, generator=self.g, device=DEV) < 1e-3, x * 50, x)
        return x.to(dtype)

    def gamma(self, n):
        return 1 + 0.1 * torch.randn(n, generator=self.g, device=DEV)

    def rand(self, *shape):
        return torch.rand(shape, generator=self.g, device=DEV)

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device=DEV, dtype=I32)


def _new(*shape, dtype=F32):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _par(g, base, yarn):
    from caminus_amd import rope
    tail = [float(np.float32(base) ** np.float32(-2.0 / 128)), EPS]
    if yarn: tail += [float(v) for v in rope.yarn_table(128, base, 4.0, 32768)]
    return torch.cat([g.gamma(128), g.gamma(128), torch.tensor(tail, device=DEV)])


def _q4k_table(g, vocab, N):
    tab = torch.randint(0, 256, (vocab, N // 256, 144), generator=g.g, device=DEV, dtype=U8)
    tab[:, :, :4] = (g.rand(vocab, N // 256, 2) * 9e-3 + 1e-3).to(F16).view(U8).view(vocab, N // 256, 4)
    return tab


def prepare(case, seed):
    g = _Gen(seed)
    return _PREPARE[case['kind']](case, g)


def run(state):
    return _RUN[state['kind']](state)


def exact(case, seed):
    return _EXACT[case['kind']](case, prepare(case, seed))


def work(case):
    return {'bytes': float(_BYTES[case['kind']](case)), 'flops': 0}


def tolerance(case):
    # the trainer's outputs are bits that the repository's oracle fixes (every sum has one order, silu and the sigmoid are tables)
    if case['kind'] in ('actq', 'mlp', 'block'): return 'exact'
    # behind cosf / sinf / expf: two libraries differ in the last place of fp32, which flips about one fp16 / bf16 rounding or int8 code in a
    # thousand; one flipped value is off by one step of its type (2^-10 of itself in fp16, 2^-7 in bf16)
    if case['kind'] == 'dense' or case.get('bf16'): return {'rel': 4e-4, 'max': 9e-3, 'differ': 2e-3}
    return {'rel': 1e-4, 'max': 2.5e-3, 'differ': 2e-3}


# ---- 64-bit statements -----------------------------------------------------------------------------------------------------------------------
def _rms(x, w, eps=EPS):
    x = x.to(F64)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.to(F64)


def _angles(pos, freq):
    """position x frequency as the statement has it: a single-precision product of single-precision factors"""
    return (pos.to(F32)[:, None] * freq.to(F32)[None, :]).to(F64)


def _freqs(ts, n):
    return torch.pow(torch.tensor(float(np.float32(ts)), dtype=F64, device=DEV), torch.arange(n, device=DEV, dtype=F64)).to(F32)


def _rotate(y, pos, freq, nrot, ms=1.0):
    """NeoX rotary of the first nrot values of y [T, heads, D]"""
    th = _angles(pos, freq)
    c, s = (th.cos() * ms)[:, None, :], (th.sin() * ms)[:, None, :]
    a, b = y[..., :nrot // 2], y[..., nrot // 2:nrot]
    return torch.cat([a * c - b * s, a * s + b * c, y[..., nrot:]], -1)


def _hadamard_matrix(n):
    h = torch.ones(1, 1, dtype=F64, device=DEV)
    while h.shape[0] < n: h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _hadamard(x, n):
    return ((x.reshape(-1, n) @ _hadamard_matrix(n)) / math.sqrt(n)).reshape(x.shape)


def _silu(x):
    return x * torch.sigmoid(x)


def _own_rope(qkv, nh, nkv, par, pos, yarn, q8):
    T = qkv.shape[0]
    x = qkv.to(F64).view(T, nh + 2 * nkv, 128)
    freq, ms = (par[258:322], float(par[322])) if yarn else (_freqs(float(par[256]), 64), 1.0)
    q, k = (_rotate(_rms(x[:, :nh], par[:128]), pos, freq, 128, ms), _rotate(_rms(x[:, nh:nh + nkv], par[128:256]), pos, freq, 128, ms))
    if q8: q = _hadamard(q.to(F16).to(F64), 128)
    return q, k, x[:, nh + nkv:]


def _q4k_rows(tab, toks):
    b = tab[toks.long()]
    n, nb = b.shape[:2]
    d, dmin = b[..., 0:2].contiguous().view(F16).to(F64), b[..., 2:4].contiguous().view(F16).to(F64)
    sc, qs = b[..., 4:16].to(torch.int64), b[..., 16:].to(torch.int64).view(n, nb, 4, 32)
    scale = torch.cat([sc[..., :4] & 63, (sc[..., 8:12] & 15) | ((sc[..., :4] >> 6) << 4)], -1)
    low = torch.cat([sc[..., 4:8] & 63, (sc[..., 8:12] >> 4) | ((sc[..., 4:8] >> 6) << 4)], -1)
    q = torch.stack([qs & 15, qs >> 4], 3).view(n, nb, 8, 32)
    return (d * scale)[..., None].mul(q).sub((dmin * low)[..., None]).view(n, nb * 256)


HSCALE = 0.08837890625        # bf16(1 / sqrt(128))


def _bf(x):
    return x.to(F32).to(BF16).to(F64)


def _turn(x):
    return _bf((x.reshape(-1, 128) @ _hadamard_matrix(128)) * HSCALE).reshape(x.shape)


def _fake_quant(src):
    u = _turn(_bf(src))
    amax = u.abs().amax(-1, keepdim=True)
    s = (amax / 7).clamp_min(1e-8)
    return u, amax, s, (u / s).round().clamp(-8, 7)


def _fake_quant_grad(src, gy):
    u, amax, s, _ = _fake_quant(src)
    t = u / s
    r = t.round()
    q, inside, tie = r.clamp(-8, 7), (r > -8) & (r < 7), u.abs() == amax
    dlds = (gy * torch.where(inside, q - t, q)).sum(-1, keepdim=True)
    coef = torch.where(amax / 7 >= 1e-8, dlds / 7 / tie.sum(-1, keepdim=True), torch.zeros_like(dlds))
    d = gy * inside + torch.where(tie, u.sign() * coef, torch.zeros_like(u))
    return _turn(_bf(d))


# ---- the qwen3moe-class decode token: the layer's row ops through the tape --------------------------------------------------------------------
MH, MNH, MNKV, MEXP, MFF = 2048, 32, 4, 8, 768
THETA6 = float(np.float32(1e6) ** np.float32(-2.0 / 128))


def _moe_tape_prepare(case, g):
    from caminus_amd.engine import k3
    T, rows = case['tokens'], 4096
    st = dict(kind='moe_tape', x=g.acts(T, MH), d=g.acts(T, MEXP, MH), w=g.rand(T, MEXP), nw=g.gamma(MH), h=_new(T, MH), h16=_new(T, MH, dtype=F16),
              q=g.acts(T, MNH, 128), k=g.acts(T, MNKV, 128), v=g.acts(T, MNKV * 128), qn=g.gamma(128), kn=g.gamma(128),
              pos=torch.tensor([case['pos']], dtype=I32, device=DEV), qo=_new(T, MNH, 128), err=_new(1, dtype=I32), o=g.acts(T, MH), nw2=g.gamma(MH),
              h2=_new(T, MH), h216=_new(T, MH, dtype=F16), gate=g.acts(T, MEXP, MFF), up=g.acts(T, MEXP, MFF), y16=_new(T, MEXP, MFF, dtype=F16), q8=case['q8'])
    st['cache'] = _new(rows, 2 * (MNKV * 128 // 32) * 34, dtype=U8) if case['q8'] else _new(rows, 2 * MNKV * 128, dtype=F16)
    st['ops'] = k3.TapeOps(T=T, kv_error=st['err'])
    st['T'] = T
    return st


def _moe_tape_run(s):
    t = s['ops']
    t.own_add_rms16(s['x'], s['nw'], s['h'], s['h16'], EPS, d=s['d'], slots=MEXP, w=s['w'], tokens=s['T'])
    t.qk_nr_kv(s['q'], 128, MNH, s['k'], 128, s['v'], MNKV, 128, s['qn'], s['kn'], s['pos'], s['qo'], s['cache'], 128, THETA6, EPS, q8=s['q8'])
    t.own_add_rms16(s['x'], s['nw2'], s['h2'], s['h216'], EPS, d=s['o'], slots=1, tokens=s['T'])
    t.own_swiglu16(s['gate'], s['up'], s['y16'])
    return [s['x'], s['h'], s['h16'], s['qo'], s['cache'], s['h2'], s['h216'], s['y16'], s['err']]


def _moe_tape_exact(case, s):
    pos = s['pos'][0] + torch.arange(s['T'], device=DEV)
    x1 = s['x'].to(F64) + (s['w'].to(F64)[..., None] * s['d'].to(F64)).sum(1)
    x2 = x1 + s['o'].to(F64)
    freq = _freqs(THETA6, 64)
    h, h2 = _rms(x1, s['nw']), _rms(x2, s['nw2'])
    cache = None
    if not case['q8']:
        cache = s['cache'].to(F64)
        cache[pos, :MNKV * 128] = _rotate(_rms(s['k'], s['kn']), pos, freq, 128).view(s['T'], -1)
        cache[pos, MNKV * 128:] = s['v'].to(F64)
    return [x2, h, h, _rotate(_rms(s['q'], s['qn']), pos, freq, 128), cache, h2, h2, _silu(s['gate'].to(F64)) * s['up'].to(F64), None]


def _moe_tape_bytes(c):
    kv = 2 * (MNKV * 128 // 32) * 34 if c['q8'] else 4 * MNKV * 128
    return c['tokens'] * (MH * 4 * (2 + MEXP + 1) + MH * 12 + (2 * MNH + 2 * MNKV) * 512 + kv + MEXP * MFF * 10) + 2 * MH * 4


# ---- the hybrid line's verify pass ---------------------------------------------------------------------------------------------------------------
HH, HC_, HHEADS, HV, HNH, HNKV, HD = 5120, 10240, 32, 48, 24, 4, 256
THETA7 = float(np.float32(1e7) ** np.float32(-2.0 / 64))


def _hybrid_tape_prepare(case, g):
    from caminus_amd.engine import k3
    T, M = case['tokens'], HNKV * HD
    st = dict(kind='hybrid_tape', T=T, x=g.acts(T, HH), d=g.acts(T, HH), nw=g.gamma(HH), h=_new(T, HH), h16=_new(T, HH, dtype=F16),
              cx=g.acts(T, HC_), cw=g.normal(HC_, 4), state=g.normal(HC_, 3), cy=_new(T, HC_), xprev=_new(T, HC_), qk=_new(T * HHEADS, 128),
              al=g.normal(T, HV), be=g.normal(T, HV), dt=g.normal(HV), a=g.normal(HV), gates=_new(T, 2 * HV),
              o=g.acts(T, HV, 128), gw=g.gamma(128), z=g.normal(T, HV, 128), y16=_new(T, HV, 128, dtype=F16),
              q=g.acts(T, HNH, 2 * HD), k=g.acts(T, M), v=g.acts(T, M), qn=g.gamma(HD), kn=g.gamma(HD), qo=_new(T, HNH, HD),
              pos=torch.tensor([case['pos']], dtype=I32, device=DEV), err=_new(1, dtype=I32), cache=_new(40960, 2 * (M // 32) * 34, dtype=U8),
              att=g.acts(T, HNH, HD), att16=_new(T, HNH, HD, dtype=F16))
    st['ops'] = k3.TapeOps(T=T, kv_q8_dense=True, kv_error=st['err'], q35=True)
    st['ops'].params = _new(4, dtype=I32)
    return st


def _hybrid_tape_run(s):
    t = s['ops']
    t.own_add_rms16(s['x'], s['nw'], s['h'], s['h16'], EPS, d=s['d'], slots=1, tokens=s['T'])
    t.gdn_conv_l2_gates(s['cx'], s['cw'], s['state'], s['cy'], s['xprev'], s['qk'], HHEADS, 128, EPS, s['al'], s['be'], s['dt'], s['a'], s['gates'])
    t.gdn_norm16(s['o'], s['gw'], s['z'], s['y16'], HV, 128, EPS)
    t.qk_nr_q8(s['q'], 2 * HD, HNH, s['k'], s['v'], HNKV, s['qn'], s['kn'], s['pos'], s['qo'], s['cache'], 64, THETA7, EPS)
    t.hadamard_gate_mul16(s['att'], 64, s['q'], 2 * HD, HD, s['att16'], HD)
    return [s['x'], s['h'], s['h16'], s['cy'], s['xprev'], s['qk'], s['gates'], s['y16'], s['qo'], s['cache'], s['att'], s['att16'], s['err']]


def _conv(x, w, state):
    """y [T, C] = silu of the causal 4-tap convolution of [state | x]"""
    w, xs = w.to(F64), torch.cat([state.to(F64).T, x.to(F64)], 0)
    T = x.shape[0]
    return _silu(sum(xs[i:i + T] * w[:, i] for i in range(4)))


def _hybrid_tape_exact(case, s):
    T = s['T']
    pos = s['pos'][0] + torch.arange(T, device=DEV)
    x1 = s['x'].to(F64) + s['d'].to(F64)
    h = _rms(x1, s['nw'])
    y = _conv(s['cx'], s['cw'], s['state'])
    gates = torch.cat([torch.nn.functional.softplus((s['al'] + s['dt']).to(F64)) * s['a'].to(F64), torch.sigmoid(s['be'].to(F64))], -1)
    gn = _rms(s['o'], s['gw']) * _silu(s['z'].to(F64))
    q = _hadamard(_rotate(_rms(s['q'][..., :HD], s['qn']), pos, _freqs(THETA7, 32), 64), 256)
    att = _hadamard(s['att'].to(F64), 64)
    l2 = y[:, :HHEADS * 128].reshape(T * HHEADS, 128)
    return [x1, h, h, y, s['cx'].to(F64), l2 * torch.rsqrt(l2.square().sum(-1, keepdim=True) + EPS), gates, gn, q, None, att,
            att * torch.sigmoid(s['q'][..., HD:].to(F64)), None]


def _hybrid_tape_bytes(c):
    return c['tokens'] * (HH * 18 + HC_ * 12 + HHEADS * 512 + HV * 16 + HV * 128 * 10 + (HNH * 2 + HNKV * 2) * HD * 4 + 2176 + HNH * HD * 14) + HC_ * 28 + HH * 4


# ---- continuous batching: gather + norm + q8_1, rotary into a paged cache, add + norm + q8_1 -----------------------------------------------------
VOCAB, PAGE, PAGES = 151936, 256, 1024


def _paged_prepare(case, g):
    from caminus_amd.device.hip import Module
    n = case['seqs']
    ldq = (MNH + 2 * MNKV) * 128
    at = torch.randperm(PAGE * PAGES, generator=g.g, device=DEV)[:n].to(I32)      # every sequence at a row of its own
    st = dict(kind='paged', n=n, tab=_q4k_table(g, VOCAB, MH), toks=g.ints(VOCAB, n), x=_new(n, MH), xbf=_new(n, MH, dtype=BF16), nw=g.gamma(MH),
              q81=_new(n, MH // 32, 36, dtype=U8), qkv=g.acts(n, ldq), ldq=ldq, par=_par(g, 1e6, False), pos=(at % PAGE + 2 * PAGE).contiguous(),
              q16=_new(n, MNH, 128, dtype=F16), err=_new(1, dtype=I32), d=g.acts(n, MH), nw2=g.gamma(MH), h16=_new(n, MH, dtype=F16), q82=_new(n, MH // 32, 36, dtype=U8),
              q8=int(case['q8']), m=Module('camx'))
    st['pt'] = torch.zeros(n, 8, dtype=I32, device=DEV)
    st['pt'][:, 2] = at // PAGE
    row = 2 * (MNKV * 128 // 32) * 34
    st['cache'] = _new(PAGE * PAGES, row, dtype=U8) if case['q8'] else _new(PAGE * PAGES, 2 * MNKV * 128, dtype=F16)
    return st


def _paged_run(s):
    from ctypes import c_float as F, c_int as I, c_long as L, c_void_p as P
    m, n, one = s['m'], s['n'], (1,)
    m.camx_emb_gather_add_rms(one, one, s['tab'], L(MH // 256 * 144), I(VOCAB), s['toks'], s['x'], s['xbf'], P(None), s['nw'], F(EPS), P(None), P(None), s['q81'],
                              I(MH), I(n), I(0))
    m.camx_qk_rope_paged(one, one, s['qkv'], I(s['ldq']), I(MNH), I(MNKV), s['par'], s['pos'], s['q16'], s['cache'], s['err'], s['pt'], I(8), I(PAGE), I(PAGES),
                         I(n), I(0), I(s['q8']))
    m.camx_add_rms_q8_1(one, one, s['x'], s['d'], P(None), I(1), s['nw2'], F(EPS), P(None), s['h16'], s['q82'], I(MH), I(n))
    return [s['x'], s['xbf'], s['q81'], s['q16'], s['cache'], s['h16'], s['q82'], s['err']]


def _paged_exact(case, s):
    emb = _q4k_rows(s['tab'], s['toks'])
    q, k, v = _own_rope(s['qkv'], MNH, MNKV, s['par'], s['pos'], False, case['q8'])
    cache = None
    if not case['q8']:
        cache = s['cache'].to(F64)
        at = s['pt'][:, 2].long() * PAGE + s['pos'].long() % PAGE
        cache[at] = torch.cat([k.reshape(s['n'], -1), v.reshape(s['n'], -1)], -1)
    x = emb + s['d'].to(F64)
    return [x, emb, None, q, cache, _rms(x, s['nw2']), None, None]


def _paged_bytes(c):
    kv = 1088 if c['q8'] else 2048
    return c['seqs'] * (1152 + MH * 6 + 2304 + 5120 * 4 + MNH * 256 + kv + MH * 12 + MH * 2 + 2304) + 2 * MH * 4


# ---- the dense line's prefill chunk, bf16 activations ---------------------------------------------------------------------------------------------
DH, DNH, DNKV, DFF = 5120, 64, 8, 17408


def _dense_prepare(case, g):
    from caminus_amd.device.hip import Module
    from caminus_amd.prefill import mmq
    T = case['tokens']
    ldq = (DNH + 2 * DNKV) * 128
    return dict(kind='dense', T=T, pos=case['pos'], ldq=ldq, x=g.acts(T, DH), d=g.acts(T, DH, dtype=BF16), nw=g.gamma(DH), hbf=_new(T, DH, dtype=BF16),
                qkv=g.acts(T, ldq, dtype=BF16), par=_par(g, 1e6, True), q16=_new(T, DNH, 128, dtype=F16), cache=_new(case['pos'] + T, 2 * DNKV * 128, dtype=F16),
                gu=g.acts(T, 2 * DFF, dtype=BF16), y=_new(mmq.y_bytes(DFF, T), dtype=U8), m=Module('camx'), mmq=mmq.MMQ(DEV))


def _dense_run(s):
    from ctypes import c_float as F, c_int as I, c_void_p as P
    m, T, one = s['m'], s['T'], (1,)
    m.camx_add_rms_bf16(one, one, s['x'], s['d'], s['nw'], F(EPS), P(None), s['hbf'], I(DH), I(T))
    m.camx_qk_rope_bf16(one, one, s['qkv'], I(s['ldq']), I(DNH), I(DNKV), s['par'], I(s['pos']), s['q16'], s['cache'], I(T), I(1))
    s['mmq'].swiglu_quantize(s['gu'], DFF, T, s['y'], 1)
    return [s['x'], s['hbf'], s['q16'], s['cache'], s['y']]


def _dense_exact(case, s):
    x = s['x'].to(F64) + s['d'].to(F64)
    pos = case['pos'] + torch.arange(s['T'], device=DEV)
    q, k, v = _own_rope(s['qkv'], DNH, DNKV, s['par'], pos, True, False)
    cache = s['cache'].to(F64)
    cache[case['pos']:] = torch.cat([k.reshape(s['T'], -1), v.reshape(s['T'], -1)], -1)
    return [x, _rms(x, s['nw']), q, cache, None]


def _dense_bytes(c):
    return c['tokens'] * (DH * 12 + 80 * 128 * 4 + DFF * 4 + DFF // 128 * 144) + DH * 4


# ---- the qwen3moe line's prefill chunk ----------------------------------------------------------------------------------------------------------------
def _moe_prepare(case, g):
    from caminus_amd.prefill import mmq, q3m_ops
    T = case['tokens']
    ldq = (MNH + 2 * MNKV) * 128
    st = dict(kind='moe', T=T, pos=case['pos'], ldq=ldq, x=g.acts(T, MH), d=g.acts(T, MEXP, MH), w=g.rand(T, MEXP), nw=g.gamma(MH), h=_new(T, MH), h16=_new(T, MH, dtype=F16),
              qkv=g.acts(T, ldq), par=_par(g, 1e6, False), q16=_new(T, MNH, 128, dtype=F16), err=_new(1, dtype=I32), gate=g.acts(T * MEXP * MFF), up=g.acts(T * MEXP * MFF),
              y16=_new(T * MEXP * MFF, dtype=F16), y=_new(mmq.y_bytes(MH, T * MEXP), dtype=U8), yd=_new(mmq.y_bytes(MH, T), dtype=U8),
              ops=q3m_ops.Ops(DEV, q8=case['q8']), mmq=mmq.MMQ(DEV), q8=case['q8'])
    st['cache'] = _new(case['pos'] + T, 1088, dtype=U8) if case['q8'] else _new(case['pos'] + T, 2 * MNKV * 128, dtype=F16)
    # the columns as the router's sort gives them: grouped by expert, a group's tokens in order; 128 experts, 8 of them a token
    pick = g.rand(T, 128).topk(MEXP, dim=1).indices.reshape(-1)
    order = torch.argsort(pick, stable=True)
    st['ids'] = torch.empty(T * MEXP, dtype=I32, device=DEV)
    st['ids'][order] = torch.arange(T * MEXP, dtype=I32, device=DEV)
    return st


def _moe_run(s):
    o, T = s['ops'], s['T']
    o.add_rms16(s['x'], s['nw'], EPS, s['h16'], T, MH, d=s['d'], w=s['w'], S=MEXP, h=s['h'])
    o.qk_rope(s['qkv'], s['ldq'], MNH, MNKV, s['par'], s['pos'], s['q16'], s['cache'], T, err=s['err'] if s['q8'] else None)
    s['mmq'].quantize(s['h'], MH, T, s['yd'], 1)
    s['mmq'].quantize_scatter(s['h'], MH, T, s['ids'], MEXP, s['y'], 1)
    o.swiglu(s['gate'], s['up'], s['y16'], T * MEXP * MFF)
    return [s['x'], s['h'], s['h16'], s['q16'], s['cache'], s['yd'], s['y'], s['y16'], s['err']]


def _moe_exact(case, s):
    x = s['x'].to(F64) + (s['w'].to(F64)[..., None] * s['d'].to(F64)).sum(1)
    h = _rms(x, s['nw'])
    pos = case['pos'] + torch.arange(s['T'], device=DEV)
    q, k, v = _own_rope(s['qkv'], MNH, MNKV, s['par'], pos, False, case['q8'])
    cache = None
    if not case['q8']:
        cache = s['cache'].to(F64)
        cache[case['pos']:] = torch.cat([k.reshape(s['T'], -1), v.reshape(s['T'], -1)], -1)
    return [x, h, h, q, cache, None, None, _silu(s['gate'].to(F64)) * s['up'].to(F64), None]


def _moe_bytes(c):
    blocks = MH // 128 * 144
    return c['tokens'] * (MH * 4 * (2 + MEXP + 1) + MH * 2 + 5120 * 4 + MNH * 256 + (1088 if c['q8'] else 2048) + MH * 8 + blocks * (1 + MEXP) + MEXP * MFF * 10) + MH * 4


# ---- a linear-attention layer of the hybrid line over a chunk -------------------------------------------------------------------------------------------
def _gdn_prepare(case, g):
    from caminus_amd.device.hip import Module
    from caminus_amd.prefill import gdn, glue, q35_ops
    T = case['tokens']
    dt = BF16 if case['bf16'] else F32
    return dict(kind='gdn', T=T, bf16=case['bf16'], x=g.acts(T, HC_, dtype=dt), w=g.normal(HC_, 4), state=g.normal(HC_, 3), y=_new(T, HC_, dtype=dt), qk=_new(T * HHEADS, 128, dtype=dt),
                al=g.normal(T, HV), be=g.normal(T, HV), dt=g.normal(HV), a=g.normal(HV), gates=_new(T, 2 * HV), o=g.acts(T, HV, 128), gw=g.gamma(128), z=g.normal(T, HV, 128),
                y16=_new(T, HV, 128, dtype=F16), glue=glue.Glue(DEV, 'prefill_glue_q35d'), gdn=gdn.Gdn(DEV, 'prefill_gdn_q35'), ops=q35_ops.Ops(DEV), m=Module('camx'))


def _gdn_run(s):
    T = s['T']
    if s['bf16']:
        from ctypes import c_float as F, c_int as I
        one = (1,)
        s['m'].camx_gdn_conv_l2(one, one, s['x'], s['w'], s['state'], s['y'], s['qk'], I(HC_), I(T), I(HC_), I(HC_), I(HHEADS), F(EPS / 128), I(1))
        s['m'].camx_pf_conv_state(one, one, s['x'], s['state'], I(HC_), I(T), I(HC_), I(1))
    else:
        s['glue'].gdn_conv(s['x'], s['w'], s['state'], s['y'], HC_, T)
        s['gdn'].l2(s['y'], s['qk'], T, HHEADS, EPS, ldx=HC_)
    s['gdn'].gates(s['al'], s['be'], s['dt'], s['a'], s['gates'], T, HV)
    s['ops'].gdn_norm16(s['o'], s['gw'], s['z'], s['y16'], T, HV, 128, EPS)
    return [s['y'], s['state'], s['qk'], s['gates'], s['y16']]


def _gdn_exact(case, s):
    T = s['T']
    y = _conv(s['x'], s['w'], s['state'])
    state = torch.cat([s['state'].to(F64).T, s['x'].to(F64)], 0)[-3:].T
    l2 = (_bf(y) if case['bf16'] else y)[:, :HHEADS * 128].reshape(T * HHEADS, 128)
    gates = torch.cat([torch.nn.functional.softplus((s['al'] + s['dt']).to(F64)) * s['a'].to(F64), torch.sigmoid(s['be'].to(F64))], -1)
    return [y, state, l2 * torch.rsqrt(l2.square().sum(-1, keepdim=True) + EPS), gates, _rms(s['o'], s['gw']) * _silu(s['z'].to(F64))]


def _gdn_bytes(c):
    e = 2 if c['bf16'] else 4
    return c['tokens'] * (HC_ * 2 * e + HHEADS * 128 * e * (1 if c['bf16'] else 2) + HV * 16 + HV * 128 * 10) + HC_ * 40


# ---- a full-attention layer of the hybrid line over a chunk, Q8 cache -----------------------------------------------------------------------------------
def _attn_prepare(case, g):
    from caminus_amd.device import kv_codec
    from caminus_amd.prefill import attn, q35_ops
    T, M = case['tokens'], HNKV * HD
    rows = case['pos'] + T
    row = 2 * (M // 32) * 34
    cache = torch.randint(0, 256, (rows, row // 34, 34), generator=g.g, device=DEV, dtype=U8)          # earlier positions, as an encoder leaves them
    cache[:, :, :2] = (g.rand(rows, row // 34, 1) * 9e-3 + 1e-3).to(F16).view(U8).view(rows, row // 34, 2)
    return dict(kind='attn', T=T, pos=case['pos'], M=M, q=g.acts(T, HNH, 2 * HD), k=g.acts(T, HNKV, HD), v=g.acts(T, M), qn=g.gamma(HD), kn=g.gamma(HD), qo=_new(T, HNH, HD),
                ko=_new(T, HNKV, HD), cache=cache.view(rows, row), err=_new(1, dtype=I32), kd=_new(rows, M, dtype=F16), vd=_new(rows, M, dtype=F16), att=g.acts(T, HNH, HD),
                y16=_new(T, HNH, HD, dtype=F16), attn=attn.Attn(DEV, name='prefill_attn_q35d'), ops=q35_ops.Ops(DEV), codec=kv_codec.Q8KVCodec(DEV))


def _attn_run(s):
    T, a, M = s['T'], s['attn'], s['M']
    a.qk_nr(s['k'], HD, HNKV, HD, s['kn'], 64, THETA7, EPS, s['pos'], s['ko'], T)
    a.hadamard(s['ko'], 256, T * HNKV)
    a.hadamard(s['v'], 64, T * M // 64)
    s['codec'].append(s['ko'], M, s['v'], M, M, s['cache'], s['pos'], T, s['err'])
    a.qk_nr(s['q'], 2 * HD, HNH, HD, s['qn'], 64, THETA7, EPS, s['pos'], s['qo'], T)
    a.hadamard(s['qo'], 256, T * HNH)
    s['codec'].read(s['cache'], M, s['kd'], M, s['vd'], M, 0, s['pos'] + T, s['err'])
    a.hadamard(s['att'], 64, T * HNH * HD // 64)
    s['ops'].gate_mul16(s['att'], s['q'], s['y16'], T * HNH * HD, HD, 2 * HD, HD)
    return [s['ko'], s['v'], s['cache'], s['qo'], s['kd'], s['vd'], s['att'], s['y16'], s['err']]


def _attn_exact(case, s):
    pos = case['pos'] + torch.arange(s['T'], device=DEV)
    fr = _freqs(THETA7, 32)
    k = _hadamard(_rotate(_rms(s['k'], s['kn']), pos, fr, 64), 256)
    q = _hadamard(_rotate(_rms(s['q'][..., :HD], s['qn']), pos, fr, 64), 256)
    att = _hadamard(s['att'].to(F64), 64)
    return [k, _hadamard(s['v'].to(F64), 64), None, q, None, None, att, att * torch.sigmoid(s['q'][..., HD:].to(F64)), None]


def _attn_bytes(c):
    T, M = c['tokens'], HNKV * HD
    return T * (M * 4 * 4 + M * 8 + 2176 + HNH * HD * 4 * 4 + HNH * HD * 18) + (c['pos'] + T) * (2176 + 4 * M)


# ---- hyper-connection glue and the per-layer-embedding block ----------------------------------------------------------------------------------------------
YH, YD, YDIL = 4, 2560, 3


def _hyper_prepare(case, g):
    from caminus_amd.prefill import glue
    T = case['tokens']
    C = YH * YD
    return dict(kind='hyper', T=T, b=g.acts(T, YD), inj=g.normal(T, YH), res=g.acts(T, YH, YD), w=g.gamma(C), xnbf=_new(T, YH, YD, dtype=BF16), scale=_new(T, YH),
                gmean=g.acts(T, YH, YD), mean=_new(T, YD), kn=g.normal(T, YH, YD), val=g.normal(T, YD), gated=_new(T, YH, YD), gate=_new(T, YH),
                cw=(g.normal(C, 4) * 0.5).to(F16), hist=g.normal(C, 3 * YDIL), y=_new(T, C), glue=glue.Glue(DEV))


def _hyper_run(s):
    gl, T = s['glue'], s['T']
    gl.hc_post_rms(s['b'], s['inj'], s['res'], s['w'], T, YH, EPS, xnbf=s['xnbf'], scale=s['scale'])
    gl.hc_mean(s['res'], s['gmean'], s['mean'], T, YH, scale=s['scale'], w=s['w'])
    gl.ple_gate(s['kn'], s['res'], s['val'], s['gated'], s['gate'], T, YH, qscale=s['scale'], qw=s['w'])
    gl.ple_conv(s['gated'], s['cw'], s['hist'], YH * YD, T, dil=YDIL, y=s['y'])
    return [s['res'], s['xnbf'], s['scale'], s['mean'], s['gated'], s['gate'], s['y'], s['hist']]


def _hyper_exact(case, s):
    T, C = s['T'], YH * YD
    res = s['res'].to(F64) + s['b'].to(F64)[:, None] * 2 * torch.sigmoid(s['inj'].to(F64) * 0.25)[..., None]
    scale = torch.rsqrt(res.square().mean(-1) + EPS)
    xn = res * scale[..., None] * s['w'].to(F64).view(YH, YD)
    mean = 0.25 * (xn * torch.sigmoid(s['gmean'].to(F64))).sum(1)
    dot = (s['kn'].to(F64) * xn).sum(-1) / math.sqrt(YD)
    gate = torch.sigmoid(dot.sign() * dot.abs().clamp_min(1e-6).sqrt())
    gated = s['val'].to(F64)[:, None] * gate[..., None]
    xs = torch.cat([s['hist'].to(F64).T, gated.view(T, C)], 0)
    y = _silu(sum(xs[YDIL * i:YDIL * i + T] * s['cw'].to(F64)[:, i] for i in range(4)))
    return [res, xn, scale, mean, gated, gate, y, xs[-3 * YDIL:].T]


def _hyper_bytes(c):
    C = YH * YD
    return c['tokens'] * (YD * 4 + C * 10 + C * 8 + YD * 4 + C * 12 + YD * 4 + C * 8 + YH * 12) + C * 80


# ---- training: fake-quant forward and backward ---------------------------------------------------------------------------------------------------------------
def _actq_prepare(case, g):
    dt = BF16 if case['bf16'] else F32
    return dict(kind='actq', x=g.acts(case['rows'], case['width'], dtype=dt).requires_grad_(), gy=g.normal(case['rows'], case['width'], dtype=BF16))


def _actq_run(s):
    from caminus_amd.train import actq
    y = actq.actq(s['x'])
    (dx,) = torch.autograd.grad(y, s['x'], s['gy'])
    return [y.detach(), dx]


def _actq_exact(case, s):
    src = s['x'].detach().to(F64)
    _, _, sc, q = _fake_quant(src)
    return [q * sc, _fake_quant_grad(src, s['gy'].to(F64))]


def _actq_bytes(c):
    e = 2 if c['bf16'] else 4
    return c['rows'] * c['width'] * (e + 2 + e + 2 + e)


def _mlp_prepare(case, g):
    return dict(kind='mlp', gu=g.acts(case['rows'], 2 * case['width'], dtype=BF16).requires_grad_(), gy=g.normal(case['rows'], case['width'], dtype=BF16))


def _mlp_run(s):
    from caminus_amd.train import actq
    y, codes, scales = actq.silu_mul_actq(s['gu'])
    (dgu,) = torch.autograd.grad(y, s['gu'], s['gy'])
    return [y.detach(), codes, scales, dgu]


def _mlp_exact(case, s):
    gate, up = s['gu'].detach().to(F64).chunk(2, -1)
    sl = _bf(_silu(gate))
    act = _bf(sl * up)
    _, _, sc, q = _fake_quant(act)
    dact = _fake_quant_grad(act, s['gy'].to(F64))
    sig = torch.sigmoid(gate)
    return [q * sc, None, sc[:, 0], torch.cat([_bf(dact * up) * sig * (1 + gate * (1 - sig)), dact * sl], -1)]


def _mlp_bytes(c):
    return c['rows'] * c['width'] * (4 + 2.5 + 4 + 2 + 4) + c['rows'] * 4


def _block_prepare(case, g):
    M, d, nab = case['rows'], case['width'], case['proj']
    slices = max(1, M // 8)
    pos = torch.full((M,), -1, dtype=I32, device=DEV)
    pos[torch.randperm(M, generator=g.g, device=DEV)[:slices]] = torch.arange(slices, dtype=I32, device=DEV)
    return dict(kind='block', x=g.acts(M, d).requires_grad_(), nw=g.rand(d) + 0.5, wab=(g.normal(nab, d) / 30).to(BF16) if nab else None,
                gy=g.normal(M, d, dtype=BF16), gab=g.normal(M, nab, dtype=BF16) if nab else None, m=g.acts(M, d, dtype=BF16).requires_grad_(),
                mlp=g.acts(M, d, dtype=BF16).requires_grad_(), ys=g.acts(slices, d, dtype=BF16).requires_grad_(), pos=pos, go=g.normal(M, d))


def _block_run(s):
    from caminus_amd.train import actq, fuse
    y, codes, scales, ab = actq.block_entry(s['x'], s['nw'], s['wab'], EPS)
    out = fuse.residual_slices(s['x'], s['m'], s['mlp'], s['ys'], s['pos'])
    outs, grads = ([y, ab, out], [s['gy'], s['gab'], s['go']]) if s['wab'] is not None else ([y, out], [s['gy'], s['go']])
    dx, dm, dmlp, dys = torch.autograd.grad(outs, [s['x'], s['m'], s['mlp'], s['ys']], grads)
    return [y.detach(), codes, scales, ab.detach(), out.detach(), dx, dm, dmlp, dys]


def _block_exact(case, s):
    x, nw = s['x'].detach().to(F64), s['nw'].to(F64)
    rstd = torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    h = x * rstd * nw
    _, _, sc, q = _fake_quant(h)
    dh = _fake_quant_grad(h, s['gy'].to(F64))
    ab = None
    if s['wab'] is not None:
        w, gab, half = s['wab'].to(F64), s['gab'].to(F64), s['wab'].shape[0] // 2
        ab = _bf(h) @ w.T
        dh = dh + _bf(gab[:, :half] @ w[:half]) + _bf(gab[:, half:] @ w[half:])
    go, pos = s['go'].to(F64), s['pos'].long()
    out = x + s['m'].detach().to(F64) + s['mlp'].detach().to(F64)
    at = pos >= 0
    out[at] += s['ys'].detach().to(F64)[pos[at]]
    dys = torch.zeros(s['ys'].shape, dtype=F64, device=DEV)
    dys[pos[at]] = go[at]
    dx = rstd * (dh * nw - x * rstd * (dh * nw * x * rstd).mean(-1, keepdim=True)) + go
    return [q * sc, None, sc[:, 0], ab, out, dx, go, go, dys]


def _block_bytes(c):
    M, d, n = c['rows'], c['width'], c['proj']
    # entry forward and backward, residual forward and backward, and the sum of the two gradients of x
    return M * (d * 6.5 + n * 2 + 8 + d * 10 + n * 2 + 4 + d * 12 + d / 4 + d * 8 + d / 4 + d * 12)


_NAMES = ('moe_tape', 'hybrid_tape', 'paged', 'dense', 'moe', 'gdn', 'attn', 'hyper', 'actq', 'mlp', 'block')
_PREPARE, _RUN, _EXACT, _BYTES = ({k: globals()[f'_{k}_{what}'] for k in _NAMES} for what in ('prepare', 'run', 'exact', 'bytes'))
