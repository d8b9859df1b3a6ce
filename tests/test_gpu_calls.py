"""The binding's native calls and the same calls through ctypes: the same results, bit for bit."""
from __future__ import annotations

import pytest
import torch

import mbrt
from gpu_util import say
from mbrt import _abi, _calls

pytestmark = pytest.mark.gpu


def _cases():
    g = torch.Generator(device="cuda").manual_seed(3)
    f = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    b = lambda *s: f(*s).to(torch.bfloat16)  # noqa: E731
    e = lambda t: torch.empty_like(t)  # noqa: E731
    x, r, gamma, wide = f(33, 96), f(33, 96), f(96), b(7, 64)
    cos, sin = (torch.from_numpy(t).to("cuda") for t in mbrt.rotary_tables(19, 64))
    qkv = b(2, 19, 3 * 4 * 64)
    q, k, v = qkv.view(2, 19, 3, 4, 64).unbind(2)
    hn = lambda t: t.permute(0, 2, 1, 3).contiguous()  # noqa: E731
    gate, win, spec = b(2, 19, 4), mbrt.hann_window(), f(1, 1025, 6, 2)
    sig, n = f(2, 3001), mbrt.stft_num_frames(3001, 441)
    chunk = (f(2, 100), f(100).abs(), f(2, 41), f(41))

    def of(name, make):  # the call's outputs from fresh buffers, so that each side starts alike
        return name, make

    return [
        of("fill", lambda: (o := e(x), mbrt.fill_(o, 2.5))),
        of("strided_copy", lambda: (o := torch.empty(96, 33, device="cuda"), mbrt.strided_copy(x.t(), o))),
        of("pad const", lambda: (o := torch.empty(33, 110, device="cuda"), mbrt.pad(x, o, [0, 5], value=1.5))),
        of("pad reflect", lambda: (o := torch.empty(33, 110, device="cuda"), mbrt.pad(x, o, (0, 5), reflect=True))),
        of("cat", lambda: (o := torch.empty(33, 192, device="cuda"), mbrt.cat([x, r], -1, o))),
        of("rms_norm", lambda: (o := e(x), mbrt.rms_norm(x, gamma, o, 9.8))),
        of("residual_add_rms_norm",
           lambda: (o := e(x), s := e(x), mbrt.residual_add_rms_norm(x, r, gamma, s, o, 9.8, 1e-8))),
        of("residual_add_rms_norm, no sum", lambda: (o := e(x), mbrt.residual_add_rms_norm(x, r, gamma, None, o, 9.8))),
        of("bias_act", lambda: (o := e(wide), mbrt.bias_act(wide, gamma[:64].contiguous(), o, mbrt.ACT_TANH))),
        of("bias_act, no bias", lambda: (o := e(wide), mbrt.bias_act(wide, None, o, mbrt.ACT_GELU_STD))),
        of("glu", lambda: (o := torch.empty(33, 48, device="cuda"), mbrt.glu(x, o))),
        of("gate_merge", lambda: (o := b(2, 19, 256), mbrt.gate_merge(hn(q), gate, o))),
        of("gate_merge bnhd",
           lambda: (o := b(2, 19, 256), mbrt.gate_merge(q.contiguous(), gate, o, mbrt.LAYOUT_BNHD, False))),
        of("softmax", lambda: (o := e(x), mbrt.softmax(x, o, 0.5))),
        of("split_qkv_rotary",
           lambda: (o := [e(hn(q)) for _ in range(3)], mbrt.split_qkv_rotary(qkv, cos, sin, *o, 4))),
        of("attention", lambda: (o := b(8, 19, 64), mbrt.attention(*(hn(t).view(8, 19, 64) for t in (q, k, v)), o))),
        of("attention_bnhd", lambda: (o := b(2, 19, 256), mbrt.attention_bnhd(q, k, v, o, cos=cos, sin=sin, gate=gate,
                                                                              p_precision=mbrt.ATTN_P_BF16))),
        of("stft", lambda: (o := torch.empty(2, 1025, n, 2, device="cuda"), mbrt.stft(sig, win, 441, out=o))),
        of("istft", lambda: (mbrt.istft(spec, win, 441),)),
        of("chunk_accumulate",
           lambda: (o := [t.clone() for t in chunk], mbrt.chunk_accumulate(*o, 13))),
    ]


def _flat(x):
    if isinstance(x, torch.Tensor):
        return [x]
    return [] if x is None else [t for y in x for t in _flat(y)]


def test_native_and_ctypes_calls_agree(dev, monkeypatch):
    native = _abi.load_calls(_abi.calls_path(torch.__version__))
    for name, make in _cases():
        say(f"native and ctypes: {name}")
        outs = []
        for calls in (native, _calls):
            monkeypatch.setattr(mbrt, "_n", calls)
            outs.append(_flat(make()))
            torch.cuda.synchronize()
        assert len(outs[0]) == len(outs[1]) > 0
        for a, c in zip(*outs):
            assert torch.equal(a, c), name
