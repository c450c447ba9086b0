"""GPU parity of the two passes for any column count (lpmm_nonfused_adamw_rank1_any_step_multi) and of the float16
step on states that are not quantised, through lpmm.optim.AdamW against the CPU oracle: codes with their padding,
scales and statistics bit for bit, parameters bit for bit in float16 and within 1e-6 in float32."""
import os

import numpy as np
import pytest
import torch

from util import assert_rel, to_dev, to_np

pytestmark = pytest.mark.gpu

H = dict(lr=1e-2, betas=(0.9, 0.999), eps=1e-3, weight_decay=0.01)
# column counts around the 128-column blocks and 16-column strides, odd and even: rows that start inside a code byte;
# fewer rows than a tile and more; one long row; one column; a row of several tiles; 34 tensors (two launches)
SHAPES = [(70, 61), (61, 70), (33, 127), (33, 129), (20, 255), (300, 257), (9, 1003), (131, 130), (65, 322), (64, 66),
          (1, 5001), (4099, 1), (130, 33), (40, 200), (25, 172)] + [(47, 90), (47, 91)] * 10
KINDS = {
    "codes4": ("default.yml", 4, np.float32),
    "float_m": ("2nd_moment_only_default.yml", 4, np.float32),
    "codes5": ("default_5b.yml", 5, np.float32),
    "codes8": ("default_8b.yml", 8, np.float32),
    "half": ("default.yml", 4, np.float16),
}


def _same(got, want, what):
    got, want = np.ascontiguousarray(got).reshape(-1), np.ascontiguousarray(want).reshape(-1)
    assert got.dtype == want.dtype, what
    ok = (got == want) | (np.isnan(got) & np.isnan(want))
    assert ok.all(), (what, int((~ok).sum()), np.flatnonzero(~ok)[:5], got[~ok][:5], want[~ok][:5])


def _setup(kind, shapes, rng):
    import lpmm

    config, bits, dtype = KINDS[kind]
    host = [(rng.standard_normal(s) * 0.5).astype(dtype) for s in shapes]
    # every third parameter starts one value off the allocation
    stores = [to_dev(np.concatenate([np.zeros(int(i % 3 == 2), dtype), h.reshape(-1)])) for i, h in enumerate(host)]
    params = [torch.nn.Parameter(s[int(i % 3 == 2):].view(h.shape)) for i, (s, h) in enumerate(zip(stores, host))]
    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    return host, params, lpmm.optim.AdamW(params, fused=False, qconfig=path, **H)


def _oracle_step(oracle, kind, h, g, state, qm, qv):
    if kind == "half":
        oracle.nonfused_step_f16(h, g, state, qm, qv, H["lr"], 0.9, 0.999, H["eps"], H["weight_decay"], device_ops=True)
    elif kind == "float_m":
        state.step += 1
        r, c = h.shape
        if state.m is None:
            state.m = np.zeros(h.size, np.float32)
        v = (np.zeros(h.size, np.float32) if state.v is None
             else np.ascontiguousarray(oracle.dequant_rank1(*state.v, qv, r, c)).reshape(-1))
        oracle.nonfused_update(h.reshape(-1), g.reshape(-1), state.m, v, 0.9, 0.999, H["lr"], H["weight_decay"], H["eps"],
                               float(state.step))
        rowmax, colmax = oracle.rank1_stats(v.reshape(r, c))
        state.v = (oracle.quant_rank1(v.reshape(r, c), rowmax, colmax, qv), rowmax, colmax)
    else:
        oracle.nonfused_step(h, g, state, qm, qv, H["lr"], 0.9, 0.999, H["eps"], H["weight_decay"])


def _check(kind, opt, p, h, before, state, what):
    s = opt.state[p]
    if kind == "float_m":
        _same(to_np(s["exp_avg"]).reshape(-1), state.m, what + ": m")
    else:
        _same(to_np(s["exp_avg_qstate"]["overhead"]["max1"]), state.m[1], what + ": m scales")
        _same(to_np(s["exp_avg"]).view(np.uint8), state.m[0], what + ": m codes")
    oh = s["exp_avg_sq_qstate"]["overhead"]
    _same(to_np(oh["max_dims"][0]), state.v[1], what + ": row statistics")
    _same(to_np(oh["max_dims"][1]), state.v[2], what + ": column statistics")
    _same(to_np(s["exp_avg_sq"]).view(np.uint8), state.v[0], what + ": v codes")
    if kind == "half":
        _same(to_np(p.detach()), h, what + ": p")
    else:
        assert_rel(to_np(p.detach()), h, what + ": p", scale=before)


@pytest.mark.parametrize("kind", list(KINDS))
def test_every_column_count(oracle, kind):
    bits = KINDS[kind][1]
    from lpmm.functional import create_general_qmap

    qm, qv = (create_general_qmap(*k).numpy() for k in (("nonlinear", bits, True), ("power-1", bits, False)))
    rng = np.random.default_rng(90)
    host, params, opt = _setup(kind, SHAPES, rng)
    states = [oracle.NonFusedState(s, "rank1", bits=bits) for s in SHAPES]
    for step in range(1, 4):
        grads = [(rng.standard_normal(s) * 0.3 * 10.0 ** (1 - step) * np.exp(rng.standard_normal((s[0], 1)))).astype(h.dtype)
                 for s, h in zip(SHAPES, host)]
        grads[3][5:12] = 0     # rows, a column and whole groups that never see a gradient: zero scales, NaN codes
        grads[3][:, 17] = 0
        grads[4][10:] = 0
        for p, g in zip(params, grads):
            p.grad = to_dev(g)
        opt.step()
        torch.cuda.synchronize()
        for i, (p, h, g, st) in enumerate(zip(params, host, grads, states)):
            before = h.copy()
            _oracle_step(oracle, kind, h, g, st, qm, qv)
            _check(kind, opt, p, h, before, st, f"step {step} tensor {i} {SHAPES[i]}")


# columns that are a multiple of 4 (runs of four a lane), on either side of a whole column block, with one run in the last block and one
# missing
RUN_SHAPES = [(70, 60), (61, 68), (33, 132), (20, 252), (300, 260), (9, 1004), (131, 196), (40, 132), (65, 388), (1030, 36)]


@pytest.mark.parametrize("kind", list(KINDS))
def test_columns_in_runs_of_four(oracle, kind, monkeypatch):
    monkeypatch.setitem(globals(), "SHAPES", RUN_SHAPES)
    test_every_column_count(oracle, kind)


def test_half_infinities_and_nans(oracle, qmaps):
    """Gradients whose squares overflow a half, an infinite one and a NaN: statistics, scales and codes as the chain of
    half ops leaves them (a NaN is the maximum of its row, its column and its group)."""
    qm, qv = qmaps
    rng = np.random.default_rng(91)
    shapes = [(70, 61), (40, 200)]
    host, params, opt = _setup("half", shapes, rng)
    states = [oracle.NonFusedState(s, "rank1") for s in shapes]
    for step in range(1, 4):
        grads = [(rng.standard_normal(s) * 0.1).astype(np.float16) for s in shapes]
        grads[0][3, 4] = 20000.0
        grads[1][7, 150] = 20000.0
        if step == 2:
            grads[0][20, 60] = np.inf
            grads[1][30, 5] = np.nan
        for p, g in zip(params, grads):
            p.grad = to_dev(g)
        opt.step()
        torch.cuda.synchronize()
        for i, (p, h, g, st) in enumerate(zip(params, host, grads, states)):
            with np.errstate(all="ignore"):
                _oracle_step(oracle, "half", h, g, st, qm, qv)
            _check("half", opt, p, h, None, st, f"step {step} tensor {i}")


class _NoWalk:
    """lpmm._native with a walk that serves nothing."""

    def __init__(self, native):
        self._native = native

    def __getattr__(self, name):
        return getattr(self._native, name)

    def walk(self):
        return self

    def collect(self, *args):
        return self._native.walk().collect(*args[:7], False, *args[8:])


def _tensors(opt, p):
    out = [p.detach()]
    for name in ("exp_avg", "exp_avg_sq"):
        out.append(opt.state[p][name])
        oh = opt.state[p][name + "_qstate"]["overhead"]
        out += ([oh["max1"]] if oh.get("max1") is not None else []) + list(oh.get("max_dims", ()))
    return [to_np(t) for t in out]


@pytest.mark.parametrize("kind", ["codes4", "float_m", "codes5", "codes8"])
def test_a_nan_gradient_costs_its_own_parameter(kind, monkeypatch):
    """One NaN gradient: parameters, statistics, scales and codes of the step after it and of two more are those of the
    staged route (dequantise, update, quantise), and every other parameter stays finite.  (Of more than two dimensions only
    the latter: the staged route's statistics keep a NaN there, and lose whole slices to it.)"""
    _nan_case(kind, [(70, 61), (33, 129), (40, 257)] + [(24, 10, 5, 5)] * (kind == "codes4"), monkeypatch)


@pytest.mark.parametrize("kind", ["codes4", "float_m", "codes5", "codes8"])
def test_a_nan_gradient_in_runs_of_four(kind, monkeypatch):
    _nan_case(kind, [(70, 60), (33, 132), (40, 260)], monkeypatch)


def _nan_case(kind, shapes, monkeypatch):
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    (_, params, opt), (_, staged_params, staged) = (_setup(kind, shapes, np.random.default_rng(94)) for _ in range(2))
    rng = np.random.default_rng(95)
    for step in range(4):
        grads = [(rng.standard_normal(s) * 0.1).astype(np.float32) for s in shapes]
        if step == 1:
            for g, at in zip(grads, (1250, 773, 0, 3001)):
                g.reshape(-1)[at] = np.nan
        for p, q, g in zip(params, staged_params, grads):
            p.grad, q.grad = to_dev(g), to_dev(g)
        opt.step()
        with monkeypatch.context() as patch:
            patch.setattr(adamw, "_any_columns", lambda rows, cols: False)
            patch.setattr(adamw, "_native", _NoWalk(_native))
            staged.step()
        torch.cuda.synchronize()
        for i, (p, q) in enumerate(zip(params, staged_params)):
            assert int(p.isnan().sum()) == (step > 0), f"step {step} tensor {i}"
            if p.dim() > 2:
                continue
            for j, (got, want) in enumerate(zip(_tensors(opt, p), _tensors(staged, q))):
                _same(got, want, f"step {step} tensor {i}, {j}")


@pytest.mark.parametrize("eps", [1e-3, 1e-8])
def test_half_states_that_are_not_quantised(oracle, eps):
    """lpmm_nonfused_update_f16_multi: sizes around the 2048-value tiles, odd offsets, more tensors than one launch; a
    gradient of zero under an eps that is zero as a half, one whose square overflows."""
    import lpmm

    rng = np.random.default_rng(92)
    sizes = [1, 2, 3, 255, 257, 2047, 2048, 2049, 4095, 4096] + [int(n) for n in rng.integers(2, 4097, 60)]
    host = [(rng.standard_normal(n) * 0.5).astype(np.float16) for n in sizes]
    stores = [to_dev(np.concatenate([np.zeros(i % 2, np.float16), h])) for i, h in enumerate(host)]
    params = [torch.nn.Parameter(s[i % 2:]) for i, s in enumerate(stores)]
    hyper = dict(H, eps=eps)
    opt = lpmm.optim.AdamW(params, fused=False, **hyper)
    ms, vs = [np.zeros_like(h) for h in host], [np.zeros_like(h) for h in host]
    for step in range(1, 4):
        grads = [(rng.standard_normal(n) * 0.1).astype(np.float16) for n in sizes]
        grads[4][7] = 0
        grads[5][9] = 20000.0
        for p, g in zip(params, grads):
            p.grad = to_dev(g)
        opt.step()
        torch.cuda.synchronize()
        for i, (p, h, g, m, v) in enumerate(zip(params, host, grads, ms, vs)):
            if h.size == 1:  # a one-element state counts as not created yet, on every step
                m[:], v[:] = 0, 0
            with np.errstate(all="ignore"):
                oracle.nonfused_update_f16(h, g, m, v, 0.9, 0.999, hyper["lr"], hyper["weight_decay"], eps, float(step), device_ops=True)
            _same(to_np(p.detach()), h, f"step {step} tensor {i}: p")
            _same(to_np(opt.state[p]["exp_avg"]), m, f"step {step} tensor {i}: m")
            _same(to_np(opt.state[p]["exp_avg_sq"]), v, f"step {step} tensor {i}: v")


@pytest.mark.parametrize("offset", [0, 1, 8])
@pytest.mark.parametrize("shape", [(300,), (2048,), (4095,), (70, 61), (64, 66), (33, 1000)])
def test_half_second_moment_at_ties(shape, offset):
    """Gradients whose square times 1 - beta2 lies half way between two halfs (odd multiples of 200 * 2^-14): the kernels
    round as the PyTorch ops on the device do, in whole blocks of 2048 values, behind them and off 16-byte boundaries."""
    import lpmm

    n = int(np.prod(shape))
    p = torch.nn.Parameter(to_dev(np.zeros(shape, np.float16)))
    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    opt = lpmm.optim.AdamW([p], fused=False, qconfig=path, **H)
    v = torch.zeros(shape, dtype=torch.float16, device="cuda")
    for step in range(3):
        g = np.zeros(offset + n, np.float16)
        g[offset:] = 200.0 * (1 + (np.arange(n) + 3 * step) % 10) * 2.0 ** -14
        p.grad = to_dev(g)[offset:].view(shape)
        opt.step()
        v.mul_(0.999).addcmul_(p.grad, p.grad, value=1 - 0.999)
        if len(shape) == 1:
            _same(to_np(opt.state[p]["exp_avg_sq"]), to_np(v), f"step {step}: second moment")
        else:
            rows, cols = opt.state[p]["exp_avg_sq_qstate"]["overhead"]["max_dims"]
            _same(to_np(rows), to_np(v.amax(1)), "row statistics")
            _same(to_np(cols), to_np(v.amax(0)), "column statistics")
            break  # the next second moment starts from the codes


def test_tensors_of_more_dimensions(oracle, qmaps):
    """The same passes on the shape[0] x rest view, one at a time: trailing products that are odd, a multiple of 8, and
    neither."""
    import lpmm

    qm, qv = qmaps
    rng = np.random.default_rng(93)
    shapes = [(64, 3, 7, 7), (40, 40, 3, 3), (24, 10, 5, 5), (600, 1, 3, 3), (33, 5, 27)] + [(32, 24, 3, 3)] * 33
    host = [(rng.standard_normal(s) * 0.5).astype(np.float32) for s in shapes]
    params = [torch.nn.Parameter(to_dev(h.copy())) for h in host]
    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    opt = lpmm.optim.AdamW(params, fused=False, qconfig=path, **H)
    states = [oracle.NonFusedState(s, "rank1") for s in shapes]
    for step in range(1, 4):
        grads = []
        for s in shapes:
            g = rng.standard_normal(s) * 1e-1
            for d in range(len(s)):
                g = g * np.exp(0.7 * rng.standard_normal([n if i == d else 1 for i, n in enumerate(s)]))
            grads.append(g.astype(np.float32))
        for p, g in zip(params, grads):
            p.grad = to_dev(g)
        opt.step()
        torch.cuda.synchronize()
        for i, (p, h, g, st) in enumerate(zip(params, host, grads, states)):
            before = h.copy()
            oracle.nonfused_step(h, g, st, qm, qv, H["lr"], 0.9, 0.999, H["eps"], H["weight_decay"])
            s, what, n = opt.state[p], f"step {step} tensor {i} {shapes[i]}", h.size
            for got, want in zip(s["exp_avg_sq_qstate"]["overhead"]["max_dims"], st.v[1]):
                _same(to_np(got), want, what + ": statistics")
            _same(to_np(s["exp_avg_qstate"]["overhead"]["max1"]), st.m[1], what + ": m scales")
            _same(to_np(s["exp_avg"]).view(np.uint8)[: (n + 1) // 2], st.m[0][: (n + 1) // 2], what + ": m codes")
            _same(to_np(s["exp_avg_sq"]).view(np.uint8)[: (n + 1) // 2], st.v[0][: (n + 1) // 2], what + ": v codes")
            assert_rel(to_np(p.detach()), h, what + ": p", scale=before)


@pytest.mark.parametrize("kind,shape", [("codes4", (4095, 4099)), ("float_m", (4095, 4099)), ("half", (4095, 4099)),
                                        ("codes4", (3000001, 7)), ("codes4", (1, 16777217))])
def test_large_odd_matrices_equal_the_staged_route(kind, shape, monkeypatch):
    """More than sixteen million values whose rows start inside a byte, over thousands of workgroups on every XCD: codes of
    both moments, scales, statistics and parameters are those of the staged route (float16: the chain of torch ops)."""
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    gen = torch.Generator(device="cuda").manual_seed(96)
    dtype = torch.float16 if kind == "half" else torch.float32
    path = os.path.join(os.path.dirname(adamw.__file__), "..", "configs", KINDS[kind][0])
    start = (torch.randn(shape, device="cuda", generator=gen) * 0.5).to(dtype)
    params = [torch.nn.Parameter(start.clone()) for _ in range(2)]
    opts = [adamw.AdamW([p], qconfig=path, **H) for p in params]
    for step in range(2):
        g = (torch.randn(shape, device="cuda", generator=gen) * 0.1).to(dtype)
        for i, (p, opt) in enumerate(zip(params, opts)):
            p.grad = g
            with monkeypatch.context() as patch:
                patch.setattr(adamw, "_any_columns", lambda rows, cols: i == 0)
                if i == 1:
                    patch.setattr(adamw, "_native", _NoWalk(_native))
                opt.step()
        for j, (got, want) in enumerate(zip(_tensors(opts[0], params[0]), _tensors(opts[1], params[1]))):
            if kind == "half" and j == 0:
                # the last op of the chain, p + value * (m / d), may be contracted there: one unit of the half, at ties
                off = got != want
                assert off.mean() < 1e-4
                assert (np.abs(got[off].astype(np.float32) - want[off]) <= np.spacing(np.abs(want[off]))).all()
                params[1].data.copy_(params[0])
                continue
            _same(got, want, f"step {step}, {j}")


@pytest.mark.parametrize("offset", [0, 1, 4])
def test_half_second_moment_with_gradients_off_a_boundary(offset, monkeypatch):
    """The product by beta2 is an op on the second moment alone, whose rounding the gradient's address does not change: a
    hundred thousand random values a step (one in ten thousand tells), in 64 tensors whose states are not quantised and, as the
    maxima of short rows, in a matrix; against torch's own ops and the chain of them."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    gen = torch.Generator(device="cuda").manual_seed(97)

    def gradient(shape):
        n = int(np.prod(shape))
        return (torch.randn(offset + n, device="cuda", generator=gen) * 0.1).half()[offset:].view(shape)

    plain = [torch.nn.Parameter(torch.zeros(4096 - i % 3, device="cuda", dtype=torch.float16)) for i in range(64)]
    moments = [torch.zeros_like(p) for p in plain]
    opt = lpmm.optim.AdamW(plain, fused=False, **H)
    for step in range(4):
        for p, v in zip(plain, moments):
            p.grad = gradient(p.shape)
            v.mul_(0.999).addcmul_(p.grad, p.grad, value=1 - 0.999)
        opt.step()
        for i, (p, v) in enumerate(zip(plain, moments)):
            _same(to_np(opt.state[p]["exp_avg_sq"]), to_np(v), f"step {step} tensor {i}: second moment")

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    params = [torch.nn.Parameter(torch.zeros(32768, 35, device="cuda", dtype=torch.float16)) for _ in range(2)]
    opts = [lpmm.optim.AdamW([p], qconfig=path, **H) for p in params]
    for step in range(4):
        params[0].grad = params[1].grad = gradient(params[0].shape)
        opts[0].step()
        with monkeypatch.context() as patch:
            patch.setattr(adamw, "_any_columns", lambda rows, cols: False)
            patch.setattr(adamw, "_native", _NoWalk(_native))
            opts[1].step()
        for j, (got, want) in enumerate(zip(_tensors(opts[0], params[0])[1:], _tensors(opts[1], params[1])[1:])):
            _same(got, want, f"step {step}, {j}")


@pytest.mark.parametrize("config, dtype", [("default.yml", torch.float32), ("2nd_moment_only_default.yml", torch.float32),
                                           ("default_8b.yml", torch.float32), ("1st_moment_group_256.yml", torch.float32),
                                           ("default.yml", torch.float16)])
def test_runs_and_single_values_in_one_call(config, dtype):
    """More tensors than a launch holds, in turn with columns that go in runs of four and columns that do not: alone they go together, one
    value at a time, and beside a tensor of 24M values that is worth it in launches of either kind.  The same bits."""
    import lpmm

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    shapes = [(70 + k, 60 + 4 * k) if k % 2 else (64 + k, 65 + 2 * k) for k in range(40)] + [(40, 7, 5, 5), (48, 4, 3, 3)]
    if dtype is torch.float16:
        shapes = [s for s in shapes if len(s) == 2]
    want = None
    for beside in ([], [(6004, 4004)]):
        gen = torch.Generator(device="cuda").manual_seed(6)
        params = [torch.nn.Parameter(torch.randn(s, device="cuda", generator=gen).to(dtype)) for s in shapes]
        grads = [[torch.randn(s, device="cuda", generator=gen).mul_(0.1).to(dtype) for s in shapes] for _ in range(3)]
        others = [torch.nn.Parameter(torch.zeros(s, dtype=dtype, device="cuda")) for s in beside]
        for p in others:
            p.grad = torch.ones_like(p)
        opt = lpmm.optim.AdamW(params[:7] + others + params[7:], lr=1e-3, eps=1e-3, weight_decay=0.01, fused=False, qconfig=path)
        for step in grads:
            for p, g in zip(params, step):
                p.grad = g
            opt.step()
        got = []
        for p in params:
            state = opt.state[p]
            got += [p.detach(), state["exp_avg"], state["exp_avg_sq"]]
            for name in ("exp_avg_qstate", "exp_avg_sq_qstate"):
                overhead = state[name]["overhead"]
                got += [t for t in [overhead.get("max1")] + list(overhead.get("max_dims") or ()) if t is not None]
        for p in others:
            assert torch.isfinite(p).all() and (p.detach() == p.detach().view(-1)[0]).all()
        want = want or got
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert torch.equal(a, b), (beside, tuple(a.shape))
