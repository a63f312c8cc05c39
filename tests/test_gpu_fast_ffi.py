"""The native form of the Python wrappers (exl3r/_fast.so, host/fast_ffi.cpp): it is there, it takes the calls of a
forward pass, and each call's results are the bits that the general form of the wrapper gives."""
import numpy as np
import pytest
import torch

import exl3r
import exl3r.ffi as ffi
from exl3r import _lib
from _gpu import dev_normal
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

F16, BF16, F32 = orc.F16, orc.BF16, orc.F32


def N(shape, dt, seed, mean=0.0, std=1.0):
    return dev_normal(shape, mean, std, dt, seed)


def E(shape, dtype=torch.float16):
    return torch.zeros(shape, device="cuda", dtype=dtype)


def rope_inputs(hd=128):
    s = dict(q=N((2, 3, 4, hd), F16, 1), k=N((2, 3, 2, hd), F16, 2), v=N((2, 3, 2, hd), F16, 3), qn=N((hd,), F16, 4, 1, 0.1),
             kn=N((hd,), F16, 5, 1, 0.1), inv=torch.rand(hd // 2, device="cuda"), lens=torch.tensor([3, 250], dtype=torch.int32, device="cuda"),
             kc=E((6, 256, 2, hd)), vc=E((6, 256, 2, hd)), bt=torch.arange(4, dtype=torch.int32, device="cuda").view(2, 2))
    s["oq"] = torch.zeros_like(s["q"])
    return s


def calls():
    """name -> (make inputs, call); every tensor of the inputs is compared afterwards."""
    x, r, w = (lambda: N((5, 640), F16, 1)), (lambda: N((5, 640), F32, 2, 0, 4)), (lambda: N((640,), F16, 3, 1, 0.1))
    signs = lambda n, seed: (N((n,), F16, seed) > 0).to(torch.float16) * 2 - 1
    wide = lambda seed: N((5, 1000), F16, seed)[:, :640]
    return {
        "rms_norm": (lambda: [wide(1), w(), E((5, 640))], lambda a: ffi.rms_norm(*a, 1e-6, 1.0)),
        "rms_norm_no_w": (lambda: [x(), E((5, 640))], lambda a: ffi.rms_norm(a[0], None, a[1], 1e-6)),
        "res_in": (lambda: [x(), w(), E((5, 640)), r()], lambda a: ffi.rms_norm_res_in(*a, 1e-6)),
        "silu": (lambda: [wide(4), N((5, 640), F16, 5), E((5, 640))], lambda a: ffi.silu_mul(*a, act_limit=2.0)),
        "gelu": (lambda: [N((5, 640), BF16, 4), N((5, 640), BF16, 5), E((5, 640), torch.bfloat16)], lambda a: ffi.gelu_mul(*a)),
        "sigmoid": (lambda: [x(), N((5, 640), F16, 5)], lambda a: ffi.mul_sigmoid_(*a)),
        "gated": (lambda: [N((6, 128), BF16, 1), N((2, 128), F32, 2), E((6, 128)), N((6, 128), F32, 3)],
                  lambda a: ffi.gated_rms_norm(*a, 1e-6, w_groups=2, gate_first=True, gate_act=1)),
        "gated_had": (lambda: [N((8, 128), BF16, 1), N((128,), F32, 2), N((8, 128), F32, 3), E((8, 128)), signs(512, 4)],
                      lambda a: ffi.gated_rms_norm_had(*a[:4], 1e-6, a[4], pre_rows=4)),
        "gated_had_exact_y": (lambda: [N((8, 256), BF16, 1), N((256,), F32, 2), N((8, 256), F32, 3), E((8, 256)), signs(512, 4), E((8, 256))],
                              lambda a: ffi.gated_rms_norm_had(*a[:4], 1e-6, a[4], y=a[5], pre_rows=2, exact=True)),
        "rms_norm_had": (lambda: [x(), w(), E((5, 640)), E((5, 640)), signs(640, 6), r(), E((5, 640)), signs(640, 7)],
                         lambda a: ffi.rms_norm_had(a[0], a[1], [a[2], a[3]], [a[4], None], 1e-6, r=a[5], y=a[6], rotate_x=True,
                                                    x_post_scale=a[7])),
        "act_mul_had": (lambda: [x(), N((5, 640), F16, 5), E((5, 640)), signs(640, 6), E((5, 640)), signs(640, 7)],
                        lambda a: ffi.act_mul_had("silu", a[0], a[1], a[2], a[3], z=a[4], rotate_x=True, rotate_y=True, x_post_scale=a[5],
                                                  exact=True)),
        "embedding": (lambda: [N((50, 640), BF16, 1), torch.tensor([3, 49, 3], device="cuda"), E((3, 640), torch.float32)],
                      lambda a: ffi.embedding(*a)),
        "embedding_norm": (lambda: [N((50, 640), BF16, 1), torch.tensor([3, 60, 3], device="cuda"), E((3, 640), torch.float32), w(),
                                    E((3, 640)), E((1,), torch.int32)], lambda a: ffi.embedding_rms_norm(*a[:5], 1e-6, err_flag=a[5])),
        "argmax": (lambda: [N((4, 999), F32, 1), E((4,), torch.int64)], lambda a: ffi.argmax_sample(*a, max_logit=800)),
        "gumbel": (lambda: [N((4, 999), F32, 1), E((4,), torch.int64)], lambda a: ffi.gumbel_sample(*a, random=2 ** 32 - 5)),
        "rope": (rope_inputs, lambda s: ffi.rope(s["q"], s["oq"], s["k"], s["k"], s["inv"], 3, None, s["qn"], s["kn"], 1e-6, 0.0,
                                                 exl3r.ROPE_NEOX, 1.0)),
        "rope_q_positions": (rope_inputs, lambda s: ffi.rope(s["q"], s["oq"], None, None, s["inv"], 0, s["lens"], None, None, 1e-6, 0.0,
                                                             exl3r.ROPE_GPTJ, 0.5)),
        "rope_table": (lambda: dict(rope_inputs(), t=torch.rand((2, 4, 64), device="cuda") * 9),
                       lambda s: ffi.rope(s["q"], s["q"], s["k"], s["k"], s["t"], 0, None, s["qn"], s["kn"], 1e-6, 0.0, exl3r.ROPE_NEOX, 1.0)),
        "rope_qg": (lambda: dict(rope_inputs(), qg=N((2, 3, 4, 256), F16, 8)),
                    lambda s: ffi.rope_qg(s["qg"], s["oq"], s["k"], s["k"], s["inv"], 5, None, s["qn"], s["kn"], 1e-6, 1.0, exl3r.ROPE_NEOX, 1.0)),
        "rope_paged_kv": (rope_inputs, lambda s: ffi.rope_paged_kv(s["q"], s["oq"], s["k"], None, s["v"], s["inv"], 0, s["lens"], s["qn"],
                                                                   s["kn"], 1e-6, 0.0, exl3r.ROPE_NEOX, 1.0, s["kc"], s["vc"], s["bt"], s["lens"])),
        "rope_paged_kv_had": (lambda: dict(rope_inputs(), sq=signs(512, 9), sk=signs(256, 10)),
                              lambda s: ffi.rope_paged_kv_had(s["q"], s["oq"], s["k"], s["k"], s["v"], s["inv"], 0, s["lens"], s["qn"], s["kn"],
                                                              1e-6, 0.0, exl3r.ROPE_NEOX, 1.0, s["kc"], s["vc"], s["bt"], s["lens"],
                                                              q_post_scale=s["sq"], k_post_scale=s["sk"], exact=True)),
    }


class Counting:
    """The native module, counting the calls it takes."""

    def __init__(self, fast):
        self.fast, self.taken = fast, 0

    def __getattr__(self, name):
        fn = getattr(self.fast, name)

        def counted(*a):
            rc = fn(*a)
            self.taken += rc is not None
            return rc
        return counted


def outcome(make, call):
    torch.manual_seed(7)
    a = make()
    call(a)
    torch.cuda.synchronize()
    return [t.clone() for t in (a.values() if isinstance(a, dict) else a)]


@pytest.mark.parametrize("name", list(calls()))
def test_native_equals_general(name, monkeypatch):
    _lib.load()
    assert _lib.fast is not None, "exl3r/_fast.so is not built"
    make, call = calls()[name]
    count = Counting(_lib.fast)
    monkeypatch.setattr(_lib, "fast", count)
    native = outcome(make, call)
    assert count.taken == 1, "declined"
    monkeypatch.setattr(_lib, "fast", None)
    general = outcome(make, call)
    for x, y in zip(native, general):
        assert torch.equal(x.view(torch.uint8) if x.dtype != torch.int64 else x, y.view(torch.uint8) if y.dtype != torch.int64 else y)


def test_errors_are_the_general_forms():
    x, w, y = N((4, 256), F16, 1), N((256,), F16, 2), E((4, 256))
    with pytest.raises(ValueError, match="x and y shapes differ"):
        ffi.rms_norm(x, w, E((4, 128)), 1e-6)
    with pytest.raises(TypeError, match="unsupported dtype"):
        ffi.rms_norm(x, w, E((4, 256), torch.float64), 1e-6)
    with pytest.raises(exl3r.Exl3rError, match="alias"):
        ffi.rms_norm_res_in(x, w, y, y, 1e-6)                                  # the entry point's own status
    with pytest.raises(ValueError):
        ffi.rms_norm(x.t(), w, y, 1e-6)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: ffi.rms_norm(a, w, y[0], 1e-6))(x)           # a batched tensor has no storage


def test_stream_and_device_of_the_call():
    """The current stream of the tensors' device is the one that the call goes to, and a stream given is used."""
    x, w = N((64, 4096), F16, 1), N((4096,), F16, 2, 1, 0.1)
    want = E((64, 4096))
    ffi.rms_norm(x, w, want, 1e-6)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for given in (None, side):
        y = E((64, 4096))
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            late = torch.zeros_like(x)
            for _ in range(20):
                late.add_(x).sub_(x)
            late.copy_(x)                                                      # what the norm must wait for on `side`
            if given is None:
                ffi.rms_norm(late, w, y, 1e-6)
        if given is not None:
            ffi.rms_norm(late, w, y, 1e-6, stream=given)
        side.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
