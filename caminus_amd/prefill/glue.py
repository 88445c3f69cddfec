"""Launch wrappers of the prefill glue row kernels this library provides: rms_mul, the hyper-connection glue (hc_post_rms,
hc_post, hc_mean), the GDN short convolution, the per-layer-embedding gate and dilated conv, add_sum and the bf16 operand
copies (the reference's python/caminus/prefill/glue.py:116-185, 212-265, 303-313; same arguments, checks and refusals).
The router, the thin matrix-vector products and the GEMM glue of that class belong to other kernels and are not here."""
import ctypes

import torch

from ..device.bufcheck import LaunchCheck
from ..device import hip
from ..device.hip import Module

GLUE_MODULES = {'prefill_glue': 2560, 'prefill_glue_q35': 2048, 'prefill_glue_q35d': 5120}     # module -> row length
F32, BF16, I32 = torch.float32, torch.bfloat16, torch.int32
TPAD = 128                                   # token rows of a bf16 GEMM operand are padded to whole tiles of 128


def tpad(T):
    return -(-int(T) // TPAD) * TPAD

_check = LaunchCheck('prefill_ops')


class Glue:
    module, D = 'prefill_glue', 2560

    def __init__(self, device, module='prefill_glue'):
        self.dev = torch.device(device)
        if module not in GLUE_MODULES:
            raise ValueError(f'Glue: module {module!r} ({sorted(GLUE_MODULES)})')
        self.module, self.D = module, GLUE_MODULES[module]
        with torch.cuda.device(self.dev):
            self.m = Module(module)

    def _go(self, fn, n, *args, threads=256):
        with torch.cuda.device(self.dev):
            getattr(self.m, fn)((-(-int(n) // threads),), (threads,), *args)

    @staticmethod
    def _nul(t):
        return t if t is not None else ctypes.c_void_p(0)

    def rms_mul(self, x, w, y, R, eps, ybf=None, scale=None):
        """y[r] = rms_norm(x[r]) * w[r % wr] for R rows of D values (w [wr, D], wr divides R). Outputs, each optional (at
        least one): y fp32 (y is x allowed), ybf its bf16 copy, scale [R] the row's 1 / sqrt(mean(x^2) + eps)"""
        K = self.D; R = int(R); wr = w.numel() // K
        if R < 1 or wr < 1 or w.numel() != wr * K or R % wr:
            raise ValueError(f'rms_mul: R {R}, w {w.numel()} (rows of {K})')
        if y is None and ybf is None and scale is None:
            raise ValueError('rms_mul: no output')
        _check(self.dev, 'rms_mul', dict(x=(x, F32, R * K), w=(w, F32, wr * K), y=(y, F32, R * K), ybf=(ybf, BF16, R * K), scale=(scale, F32, R)),
               ('y', 'ybf', 'scale'), same_ok=[('y', 'x')], opt=('y', 'ybf', 'scale'))
        with torch.cuda.device(self.dev):
            self.m.pf_rms_mul((R,), (256,), x, w, self._nul(y), self._nul(ybf), self._nul(scale), ctypes.c_int(R), ctypes.c_int(wr), ctypes.c_float(eps))

    def hc_post_rms(self, block, inj, res, w, T, HC, eps, rs=0.25, xn=None, xnbf=None, scale=None):
        """res[t, h] += block[t] * 2 sigmoid(inj[t, h] * rs) in place, then the norm of every (token, stream) row with w[h]:
        xn fp32 [T, HC, D], xnbf its bf16 copy, scale [T * HC], each optional"""
        T, HC, D = int(T), int(HC), self.D
        _check(self.dev, 'hc_post_rms', dict(block=(block, F32, T * D), inj=(inj, F32, T * HC), res=(res, F32, T * HC * D), w=(w, F32, HC * D),
                                             xn=(xn, F32, T * HC * D), xnbf=(xnbf, BF16, T * HC * D), scale=(scale, F32, T * HC)),
               ('res', 'xn', 'xnbf', 'scale'), opt=('xn', 'xnbf', 'scale'))
        with torch.cuda.device(self.dev):
            self.m.pf_hc_post_rms((T * HC,), (256,), block, inj, res, w, self._nul(xn), self._nul(xnbf), self._nul(scale), ctypes.c_int(T),
                                  ctypes.c_int(HC), ctypes.c_float(rs), ctypes.c_float(eps))

    def hc_post(self, block, inj, res, T, HC, D=None, rs=0.25):
        """res[t, h, i] += block[t, i] * 2 sigmoid(inj[t, h] * rs)"""
        T, HC, D = int(T), int(HC), self.D if D is None else int(D)
        _check(self.dev, 'hc_post', dict(block=(block, F32, T * D), inj=(inj, F32, T * HC), res=(res, F32, T * HC * D)), ('res',))
        self._go('pf_hc_post', T * D, block, inj, res, ctypes.c_int(T), ctypes.c_int(HC), ctypes.c_int(D), ctypes.c_float(rs))

    def hc_mean(self, xn, gate, out, T, HC, D=None, rs=0.25, scale=None, w=None):
        """out[t, i] = rs * sum_h xn[t, h, i] * sigmoid(gate[t, h, i]); xn given [T, HC, D], or (scale and w given) the
        residual whose norm is recomputed as (res * scale[t, h]) * w[h]"""
        T, HC, D = int(T), int(HC), self.D if D is None else int(D)
        if (scale is None) != (w is None):
            raise ValueError('hc_mean: scale and w go together')
        _check(self.dev, 'hc_mean', dict(xn=(xn, F32, T * HC * D), gate=(gate, F32, T * HC * D), out=(out, F32, T * D), scale=(scale, F32, T * HC),
                                         w=(w, F32, HC * D)), ('out',), opt=('scale', 'w'))
        self._go('pf_hc_mean', T * D, xn, self._nul(scale), self._nul(w), gate, out, ctypes.c_int(T), ctypes.c_int(HC), ctypes.c_int(D), ctypes.c_float(rs))

    def gdn_conv(self, x, w, state, y, C, T, ldx=None, ldy=None):
        """y[t, c] = silu(conv4([state | x][t .. t + 3], w[c])) for T tokens, then state = the last 3 inputs.
        x / y [T, C] (row strides ldx / ldy); y must not overlap x"""
        C, T = int(C), int(T); ldx = C if ldx is None else int(ldx); ldy = C if ldy is None else int(ldy)
        if T < 1 or C < 1 or ldx < C or ldy < C:
            raise ValueError(f'gdn_conv: C {C} T {T} ldx {ldx} ldy {ldy}')
        _check(self.dev, 'gdn_conv', dict(x=(x, F32, (T - 1) * ldx + C), w=(w, F32, C * 4), state=(state, F32, C * 3), y=(y, F32, (T - 1) * ldy + C)),
               ('y', 'state'))
        I = ctypes.c_int
        if hip.RECORD is None:
            self._go('pf_gdn_conv_commit', T * C, x, w, state, y, I(C), I(T), I(ldx), I(ldy))
        else:                                     # a recorder sees the reference's two launches
            self._go('pf_gdn_conv', T * C, x, w, state, y, I(C), I(T), I(ldx), I(ldy))
            self._go('pf_conv_state', C, x, state, I(C), I(T), I(ldx))

    def ple_gate(self, kn, qn, val, gated, gate, T, HC, D=None, ldv=None, qscale=None, qw=None):
        """per token and stream: gate = sigmoid(sgn(s) sqrt(max(|s|, 1e-6))), s = kn . qn / sqrt(D); gated = val * gate.
        kn / gated [T, HC, D] (gated may be kn itself), val [T, D] at row stride ldv, gate [T, HC]; qn [T, HC, D] given, or with
        qscale [T * HC] and qw [HC, D] the residual whose norm is recomputed"""
        T, HC, D = int(T), int(HC), self.D if D is None else int(D)
        ldv = D if ldv is None else int(ldv)
        if HC > 8:
            raise ValueError(f'ple_gate: HC {HC} > 8')
        if (qscale is None) != (qw is None):
            raise ValueError('ple_gate: qscale and qw go together')
        bufs = dict(kn=(kn, F32, T * HC * D), qn=(qn, F32, T * HC * D), gated=(gated, F32, T * HC * D), qscale=(qscale, F32, T * HC), qw=(qw, F32, HC * D),
                    val=(val, F32, (T - 1) * ldv + D), gate=(gate, F32, T * HC))
        _check(self.dev, 'ple_gate', bufs, ('gated', 'gate'), same_ok=[('gated', 'kn')], opt=('qscale', 'qw'))
        with torch.cuda.device(self.dev):
            self.m.pf_ple_gate((T,), (256,), kn, qn, self._nul(qscale), self._nul(qw), val, ctypes.c_int(ldv), gated, gate, ctypes.c_int(HC), ctypes.c_int(D))

    def ple_conv(self, x, w_f16, hist, C, T, dil=3, y=None, a=None, res=None, xscale=None, xw=None, D=None):
        """conv[t, c] = silu of the dilated 4-tap causal conv over [hist | x] with fp16 weights [C, 4] (float16, or the same
        bytes as uint8); x [T, C] given, or with xscale [T * C / D] and xw [C] the pre-norm rows. y receives conv; res / a:
        res += a + conv. Afterwards hist holds the last 3 dil inputs. Neither y nor res may overlap x."""
        C, T, dil = int(C), int(T), int(dil)
        D = self.D if D is None else int(D)
        if 3 * dil > 32 or T < 1 or C % D:
            raise ValueError(f'ple_conv: dil {dil} (history <= 32), T {T}, C {C} (rows of {D})')
        if y is None and res is None:
            raise ValueError('ple_conv: neither y nor res')
        if (res is None) != (a is None):
            raise ValueError('ple_conv: res and a go together')
        if (xscale is None) != (xw is None):
            raise ValueError('ple_conv: xscale and xw go together')
        wspec = (w_f16, torch.uint8, C * 8) if getattr(w_f16, 'dtype', None) == torch.uint8 else (w_f16, torch.float16, C * 4)
        bufs = dict(x=(x, F32, T * C), xscale=(xscale, F32, T * (C // D)), xw=(xw, F32, C), w=wspec, hist=(hist, F32, C * 3 * dil), y=(y, F32, T * C),
                    a=(a, F32, T * C), res=(res, F32, T * C))
        _check(self.dev, 'ple_conv', bufs, ('hist', 'y', 'res'), opt=('xscale', 'xw', 'y', 'a', 'res'))
        n, tail = self._nul, (ctypes.c_int(C), ctypes.c_int(T), ctypes.c_int(D), ctypes.c_int(dil))
        if hip.RECORD is None:
            self._go('pf_ple_conv_commit', T * C, x, n(xscale), n(xw), w_f16, hist, n(y), n(a), n(res), *tail)
        else:                                     # a recorder sees the reference's two launches
            self._go('pf_ple_conv', T * C, x, n(xscale), n(xw), w_f16, hist, n(y), n(a), n(res), *tail)
            self._go('pf_ple_hist', C, x, n(xscale), n(xw), hist, *tail)

    def add_sum(self, a, b, y, n):
        """y += a + b (y may be a or b exactly)"""
        n = int(n)
        _check(self.dev, 'add_sum', dict(a=(a, F32, n), b=(b, F32, n), y=(y, F32, n)), ('y',), same_ok=[('y', 'a'), ('y', 'b')])
        self._go('pf_add_sum', n, a, b, y, ctypes.c_long(n))

    def silu_bf16(self, x, y, T, K, rs, ldx=None):
        """y [tpad(T), K] bf16 = bf16(silu(fma(rs, x, 0))) for the T rows of x (row stride ldx), zero rows up to tpad(T)"""
        T, K = int(T), int(K)
        ldx = K if ldx is None else int(ldx)
        _check(self.dev, 'silu_bf16', dict(x=(x, F32, (T - 1) * ldx + K), y=(y, BF16, tpad(T) * K)), ('y',))
        self._go('pf_silu_bf16', tpad(T) * K, x, ctypes.c_int(ldx), y, ctypes.c_int(T), ctypes.c_int(tpad(T)), ctypes.c_int(K), ctypes.c_float(rs))

    def to_bf16(self, x, y, T, K, ldx=None):
        """y [tpad(T), K] bf16 = bf16(x) for the T rows of x, zero rows up to tpad(T)"""
        T, K = int(T), int(K)
        ldx = K if ldx is None else int(ldx)
        _check(self.dev, 'to_bf16', dict(x=(x, F32, (T - 1) * ldx + K), y=(y, BF16, tpad(T) * K)), ('y',))
        self._go('pf_to_bf16', tpad(T) * K, x, ctypes.c_int(ldx), y, ctypes.c_int(T), ctypes.c_int(tpad(T)), ctypes.c_int(K))
