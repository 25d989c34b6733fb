"""The compiled call path (csrc/bind.cpp) against the Python wrappers it stands for: the same outputs for plain
arguments, arguments that it leaves to the wrapper, and the same errors; and what it holds after a failure."""

import contextlib
import functools

import pytest
import torch

from stblarge_amd import _lib, data, ops

pytestmark = pytest.mark.gpu


class _Sub(torch.Tensor):
    pass


class _Spy:
    """Records for each compiled call whether it took the arguments."""

    def __init__(self, native):
        self.native, self.took = native, []

    def __getattr__(self, name):
        fn = getattr(self.native, name)

        def call(*args):
            y = fn(*args)
            self.took.append(y is not NotImplemented)
            return y
        return call


@contextlib.contextmanager
def _path(native):
    _lib.load()
    was, _lib.native = _lib.native, native
    try:
        yield native
    finally:
        _lib.native = was


def _run(call, native):
    """What call() returns on that path, or the type and text of the error it raises."""
    with _path(native):
        try:
            return call()
        except Exception as e:
            return type(e), str(e)


def _flat(y):
    return [t for v in y for t in _flat(v)] if isinstance(y, (list, tuple)) else [y]


def _same(a, b):
    a, b = _flat(a), _flat(b)
    assert len(a) == len(b)
    for x, y in zip(a, b):
        if not isinstance(x, torch.Tensor):
            assert x == y
            continue
        assert type(x) is type(y) and x.dtype == y.dtype and x.shape == y.shape and x.device == y.device
        assert torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8))


def _weights(gpu, fmt, n, k, seed):
    w = data.weight(n, k, seed=seed).to(gpu)
    return ops.quant_fp4(w) if fmt == ops.FP4 else ops.quant_fp8_b128(w)


def _x(gpu, m, k, seed=1):
    return data.activation(m, k, seed=seed).to(gpu)


def _slot(gpu, fmt, dim, inter, seed):
    shapes = ((inter, dim), (inter, dim), (dim, inter))
    return ops.quant_expert(*(data.weight(r, k, seed=seed + i).to(gpu) for i, (r, k) in enumerate(shapes)), fmt)


def _gemv_calls(add, gpu, fmt):
    f, gemv, n, k = f"fmt{fmt}", ops.gemv_fp4 if fmt == ops.FP4 else ops.gemv_fp8, 272, 512
    w, s = _weights(gpu, fmt, n, k, 5 + fmt)
    x = _x(gpu, 3, k)
    add(f"gemv {f}", True, gemv, w, s, x)
    add(f"gemv {f} one token, fp32", True, gemv, w, s, x[0], out_f32=True)
    add(f"gemv {f} out", True, gemv, w, s, x, out_f32=True, out=torch.empty((3, n), device=gpu))
    add(f"gemv {f} parameter", True, gemv, torch.nn.Parameter(w, requires_grad=False), s, x)
    add(f"gemv {f} int flag", False, gemv, w, s, x, out_f32=1)
    add(f"gemv {f} subclass", False, gemv, w.as_subclass(_Sub), s, x)
    add(f"gemv {f} wrong k", None, gemv, w, s, x[:, :256].contiguous())
    add(f"gemv {f} strided", None, gemv, w, s, x[:, ::2])
    add(f"gemv {f} five tokens", None, gemv, w, s, _x(gpu, 5, k))
    add(f"gemv {f} no tokens", None, gemv, w, s, x[:0])
    add(f"gemv {f} fp32 x", None, gemv, w, s, x.float())
    add(f"gemv {f} host x", None, gemv, w, s, x.cpu())
    ws, xs = [_weights(gpu, fmt, n, k, 20 + i) for i in range(3)], [_x(gpu, 2, k, i) for i in range(3)]
    cs, ss = [c for c, _ in ws], [v for _, v in ws]
    add(f"batch {f}", True, ops.gemv_batch, cs, ss, xs, fmt)
    add(f"batch {f} outs", True, ops.gemv_batch, cs, ss, xs, fmt,
        outs=[torch.empty((2, n), dtype=torch.bfloat16, device=gpu) for _ in range(3)])
    add(f"batch {f} tuples", False, ops.gemv_batch, tuple(cs), tuple(ss), tuple(xs), fmt)
    add(f"batch {f} shapes", None, ops.gemv_batch, cs, ss, xs[:2] + [xs[0][:1]], fmt)
    add(f"batch {f} empty", None, ops.gemv_batch, [], [], [], fmt)


def _gemm_calls(add, gpu, fmt):
    n, k = 272, 512
    w, s = _weights(gpu, fmt, n, k, 7 + fmt)
    pk, small = ops.gemm_pack(w, fmt), torch.empty(16, dtype=torch.uint8, device=gpu)
    for block in (32, 128) if fmt == ops.FP4 else (128,):
        for m in (40, 130):
            x, g = _x(gpu, m, k, m), f"fmt{fmt} block {block} m {m}"
            aq, a_s = ops.act_quant_e4m3(x, block)
            add(f"gemm {g}", True, ops.gemm, w, s, x, fmt, block)
            add(f"gemm work {g}", True, ops.gemm, w, s, x, fmt, block, True, ops.gemm_work(m, n, k, gpu))
            add(f"gemm small work {g}", True, ops.gemm, w, s, x, fmt, block, work=small)
            add(f"gemm_packed {g}", True, ops.gemm_packed, pk, s, x, fmt, block, True)
            add(f"gemm_q {g}", True, ops.gemm_q, w, s, aq, a_s, fmt, block)
            add(f"gemm_q_packed {g}", True, ops.gemm_q_packed, pk, s, aq, a_s, fmt, block)
            add(f"gemm int flag {g}", False, ops.gemm, w, s, x, fmt, block, 1)
            add(f"gemm_q scales {g}", None, ops.gemm_q, w, s, aq, a_s[:-1], fmt, block)
    add(f"gemm fmt{fmt} block 64", None, ops.gemm, w, s, x, fmt, 64)
    add(f"gemm fmt{fmt} no rows", None, ops.gemm, w, s, x[:0], fmt)
    add(f"gemm fmt{fmt} k", None, ops.gemm, w, s, x[:, :256].contiguous(), fmt)
    if fmt == ops.FP8:
        add("gemm unknown format", None, ops.gemm, w, s, x, 7)


def _expert_calls(add, gpu, fmt):
    f, dim, inter = f"fmt{fmt}", 256, 128
    slots, x = [_slot(gpu, fmt, dim, inter, 10 * i) for i in range(4)], _x(gpu, 2, dim)
    pick, wt = [[2, 0], [1, 2]], [[0.5, 0.25], [0.75, 1]]
    add(f"ffn {f}", True, ops.expert_ffn, slots[0], x, fmt, dim, inter, 0.5, 10, True, True)
    add(f"ffn {f} int flag", False, ops.expert_ffn, slots[0], x[0], fmt, dim, inter, official=1)
    add(f"ffn {f} short slot", None, ops.expert_ffn, slots[0][:-256], x, fmt, dim, inter)
    add(f"ffn {f} tokens", None, ops.expert_ffn, slots[0], _x(gpu, 5, dim), fmt, dim, inter)
    add(f"ffn {f} dims", None, ops.expert_ffn, slots[0], x[:, :100].contiguous(), fmt, 100, inter)
    add(f"moe {f}", True, ops.moe_experts, x, slots, pick, wt, fmt, dim, inter, shared=3, limit=10)
    add(f"moe {f} addresses, work, out", True, ops.moe_experts, x, [v.data_ptr() for v in slots], pick, wt, fmt, dim, inter,
        shared=3, official=True, shared_fmt=fmt, out=torch.empty((2, dim), dtype=torch.bfloat16, device=gpu),
        work=torch.empty(ops.moe_work_bytes(2, 2, dim, inter), dtype=torch.uint8, device=gpu))
    add(f"moe {f} tuples", False, ops.moe_experts, x, tuple(slots), tuple(pick), tuple(wt), fmt, dim, inter)
    add(f"moe {f} pick", None, ops.moe_experts, x, slots, [[0, 9], [1, 2]], wt, fmt, dim, inter)
    add(f"moe {f} shared", None, ops.moe_experts, x, slots, pick, wt, fmt, dim, inter, shared=4)


def _other_calls(add, gpu):
    rows, k, g = 96, 256, torch.Generator(gpu).manual_seed(1)
    ws = [torch.randint(100, 130, (rows * k // 32 * 17,), dtype=torch.uint8, device=gpu, generator=g) for _ in range(2)]
    xs, ys = [_x(gpu, 1, k, i).float().view(-1) for i in range(2)], [torch.empty(rows, device=gpu) for _ in range(2)]
    add("mxfp4", True, ops.stbl_gemv_mxfp4_batch, ys, ws, xs, rows, k)
    add("mxfp4 tuple", False, ops.stbl_gemv_mxfp4_batch, tuple(ys), ws, xs, rows, k)
    add("mxfp4 short y", None, ops.stbl_gemv_mxfp4_batch, [ys[0], ys[1][:8]], ws, xs, rows, k)
    add("mxfp4 k", None, ops.stbl_gemv_mxfp4_batch, ys, ws, xs, rows, k + 32)
    lg, bias = torch.randn((5, 96), device=gpu, generator=g), torch.linspace(0, 0.1, 96, device=gpu)
    add("route", True, ops.route, lg, 4)
    add("route bias", True, ops.route, lg, 4, bias, 2, score_fn=ops.SCORE_SQRT_SOFTPLUS)
    add("route strided bias", None, ops.route, lg, 4, bias[::2])
    add("route top-k", None, ops.route, lg, 97)
    add("route fp64", None, ops.route, lg.double(), 4)
    x = _x(gpu, 6, 256).view(2, 3, 256)
    add("act_quant", True, ops.act_quant, x, 32, want_deq=True)
    add("act_quant any scale", True, ops.act_quant, x, 128, False)
    add("act_quant int flag", False, ops.act_quant, x, 32, 1)
    add("act_quant block", None, ops.act_quant, x, 96)
    add("act_quant_e4m3", True, ops.act_quant_e4m3, x.view(6, 256), 32)
    add("act_quant_e4m3 3-D", None, ops.act_quant_e4m3, x, 32)
    add("act_quant_e4m3 block", None, ops.act_quant_e4m3, x.view(6, 256), 64)


def _calls(gpu):
    """name -> (call, whether the compiled path takes it; None: it is refused)."""
    c = {}

    def add(name, takes, fn, *args, **kw):
        c[name] = functools.partial(fn, *args, **kw), takes

    for fmt in (ops.FP4, ops.FP8):
        _gemv_calls(add, gpu, fmt)
        _gemm_calls(add, gpu, fmt)
    for fmt in (ops.FP4, ops.FP8, ops.FP8_E8M0):
        _expert_calls(add, gpu, fmt)
    _other_calls(add, gpu)
    return c


def test_compiled_calls_equal_the_wrappers(gpu):
    assert _lib.load() and _lib.native.__name__ == "stblarge_amd._bind"
    _lib.last_error()
    used = set()
    for name, (call, takes) in _calls(gpu).items():
        spy = _Spy(_lib.native)
        got = _run(call, spy)
        got = [t.clone() if isinstance(t, torch.Tensor) else t for t in _flat(got)]  # outputs may be the caller's own
        want = _run(call, _lib._PythonPath())
        raised = isinstance(want, tuple) and isinstance(want[0], type)
        assert raised == (takes is None), (name, want)
        if takes is not None:
            assert spy.took == [takes], name
        try:
            _same(got, want)
        except AssertionError as e:
            raise AssertionError(f"{name}: {e}") from e
        used.add(name.split()[0])
    assert _lib.last_error()[0] == 0
    assert used == {"gemv", "batch", "gemm", "gemm_packed", "gemm_q", "gemm_q_packed", "mxfp4", "ffn", "moe", "route",
                    "act_quant", "act_quant_e4m3"}


def test_compiled_call_that_runs_out_of_memory_keeps_nothing(gpu):
    # a batch whose outputs do not all fit: those that were allocated are freed with the error
    rows, k = 1 << 20, 32
    w = torch.zeros((rows, k // 2), dtype=torch.uint8, device=gpu)
    s, x = torch.full((rows, 1), 127, dtype=torch.uint8, device=gpu), _x(gpu, 1, k)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    total = torch.cuda.get_device_properties(gpu).total_memory
    room = torch.cuda.memory_reserved() - before + (32 << 20)  # in blocks that other tensors keep, and in new ones
    assert room < 256 << 20
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (32 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            ops.gemv_batch([w] * 64, [s] * 64, [x] * 64, ops.FP4, out_f32=True)  # 256 MB of outputs
        assert torch.cuda.memory_allocated() == before
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
