"""The host walk (csrc/walk.cpp) against the Python loops it stands in for: the same steps with and without it leave
the same bits everywhere, whatever the route, across missing gradients, strided tensors, a checkpoint load, an
overridden state and states the caller has moved."""
import copy
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MATRICES = [(64, 256), (48, 192), (33, 200), (33, 130), (5000,), (70,), (17, 16, 8), (32, 24, 3, 3), (40, 5, 7, 5), (90, 128)]
CASES = {
    "fused": dict(fused=True),
    "fused_factored": dict(fused=True, factor_second_moment=True),
    "default": dict(qconfig="default.yml"),
    "group": dict(qconfig="2nd_moment_group_128.yml"),
    "float_m": dict(qconfig="2nd_moment_only_default.yml"),
    "float_m_group": dict(qconfig="2nd_moment_only_group_128.yml"),
    "wide": dict(qconfig="1st_moment_group_512.yml"),
    "bits": dict(qconfig="default_6b.yml"),
    "half": dict(qconfig="default.yml", dtype=torch.float16),
    "half_group": dict(qconfig="2nd_moment_group_128.yml", dtype=torch.float16),
    "sgd": dict(sgd=True),
}


class _Native:
    """lpmm._native with a walk that serves nothing, or counts what it serves."""

    def __init__(self, native, serve):
        self._native, self._serve, self.served, self.rest = native, serve, 0, 0

    def __getattr__(self, name):
        return getattr(self._native, name)

    def walk(self):
        return self

    def collect(self, *args):
        args = list(args)
        args[7] = args[7] and self._serve
        plan = self._native.walk().collect(*args)
        self.served += plan.served
        self.rest += len(plan.rest)
        return plan


def _build(case, rng):
    import lpmm

    kw = dict(CASES[case])
    dtype, sgd = kw.pop("dtype", torch.float32), kw.pop("sgd", False)
    if "qconfig" in kw:
        kw["qconfig"] = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", kw["qconfig"])
    shapes = [s for s in MATRICES if dtype is torch.float32 or len(s) < 3]
    params = [torch.nn.Parameter(torch.from_numpy(rng.standard_normal(s) * 0.1).to(dtype).cuda()) for s in shapes]
    if not kw.get("fused"):  # the fused operators refuse strided parameters
        params.append(torch.nn.Parameter(torch.from_numpy(rng.standard_normal((96, 80))).float().cuda().t().to(dtype)))
    if sgd:
        return params, lpmm.optim.SGD(params, lr=1e-2, momentum=0.9, weight_decay=1e-3, nesterov=True)
    return params, lpmm.optim.AdamW(params, lr=1e-2, eps=1e-3, **kw)


def _state(opt, p):
    out = {}
    for k, v in opt.state[p].items():
        if torch.is_tensor(v):
            out[k] = v
        else:
            for name, o in v["overhead"].items():
                for i, t in enumerate(o if isinstance(o, list) else [o]):
                    if torch.is_tensor(t):
                        out[k, name, i] = t
    return out


@pytest.mark.parametrize("case", list(CASES))
def test_walk_equals_the_loops(case, monkeypatch):
    import lpmm.optim.adamw as adamw
    import lpmm.optim.sgd as sgd
    from lpmm import _native

    sides = [_build(case, np.random.default_rng(5)) for _ in range(2)]
    rng = np.random.default_rng(6)
    natives = [_Native(_native, True), _Native(_native, False)]
    for step in range(6):
        grads = [rng.standard_normal(p.shape) * 0.1 for p in sides[0][0]]
        for side, ((params, opt), native) in enumerate(zip(sides, natives)):
            monkeypatch.setattr(adamw, "_native", native)
            monkeypatch.setattr(sgd, "_native", native)
            for i, (p, g) in enumerate(zip(params, grads)):
                p.grad = None if (step + i) % 5 == 4 else torch.from_numpy(g).to(p.dtype).cuda()
            if step == 3:  # a checkpoint round trip in the middle
                opt.load_state_dict(copy.deepcopy(opt.state_dict()))
            if step == 4:  # a state in other memory
                for s in opt.state.values():
                    for k, v in s.items():
                        if torch.is_tensor(v) and v.dtype is torch.int8:
                            s[k] = v.clone()
            opt.step()
        torch.cuda.synchronize()
        for i, (p, q) in enumerate(zip(sides[0][0], sides[1][0])):
            assert torch.equal(p.detach(), q.detach()), (step, i)
            a, b = _state(sides[0][1], p), _state(sides[1][1], q)
            assert a.keys() == b.keys()
            for k in a:
                assert a[k].shape == b[k].shape and a[k].dtype == b[k].dtype, (step, i, k)
                assert torch.equal(a[k].nan_to_num(), b[k].nan_to_num()) if a[k].is_floating_point() else torch.equal(a[k], b[k]), \
                    (step, i, k)
    assert natives[0].served > 0 and natives[1].served == 0
    # the steady state: everything but the strided tensor (and what is named below) is served
    native = natives[0]
    monkeypatch.setattr(adamw, "_native", native)
    monkeypatch.setattr(sgd, "_native", native)
    params, opt = sides[0]
    for _ in range(2):
        native.rest = 0
        for p, g in zip(params, grads):
            p.grad = torch.from_numpy(g).to(p.dtype).cuda()
        opt.step()
    nd = sum(p.dim() > 2 for p in params)  # factored stacks of matrices go one by one
    # other N-D routes than the default configuration's are the staged path's
    staged = 2 if case in ("float_m", "wide", "bits") else 0
    staged += {"wide": 1, "bits": 1}.get(case, 0)  # the 5000-long vector
    assert native.rest == (nd if case == "fused_factored" else 0 if case == "fused" else staged + 1), native.rest


def test_walk_leaves_overridden_and_subclassed_parameters_to_the_loops():
    """An override is looked up by the parameter; a subclass of Parameter may define its own .grad."""
    import lpmm
    from lpmm import _native

    class Own(torch.nn.Parameter):
        pass

    class Module(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.a = torch.nn.Parameter(torch.randn(64, 128, device="cuda"))
            self.b = torch.nn.Parameter(torch.randn(64, 128, device="cuda"))
            self.c = Own(torch.randn(64, 128, device="cuda"))

    m = Module()
    opt = lpmm.optim.AdamW(list(m.parameters()), fused=True)
    opt.override_quantize_enable(m, "b", False)
    for _ in range(2):
        for p in m.parameters():
            p.grad = torch.randn_like(p)
        opt.step()
    assert opt.state[m.a]["exp_avg"].dtype is torch.int8 and opt.state[m.b]["exp_avg"].dtype is torch.float32
    plan = opt._walk(opt.param_groups[0], lpmm.optim.adamw._Routes(opt.get_qmetadata_by_state_name("exp_avg"),
                                                                    dict(opt.get_qmetadata_by_state_name("exp_avg_sq"), scale_type="group")))
    assert [p is m.c for p in plan.rest] == [True]
    kinds = {batch[0]: batch[5] for batch in plan.start()}
    assert kinds == {_native.WALK_FUSED4: 1, _native.WALK_PLAIN: 1}


@pytest.mark.parametrize("case", ["fused", "default", "half", "sgd"])
def test_tensors_dropped_during_the_step_outlive_it(case):
    """The .grad of a Parameter's subclass is the caller's code and runs after the walk: it may drop gradients and states
    that the walk's records point into, and allocate over them."""
    import lpmm

    rng = np.random.default_rng(8)
    drop = []

    class Own(torch.nn.Parameter):
        @property
        def grad(self):
            for p, state in drop:
                shapes = [t.shape for t in (p.grad, *state.values()) if torch.is_tensor(t) and t.is_cuda]
                p.grad = None
                state.clear()
                junk.extend(torch.full(s, 3.0, device="cuda", dtype=p.dtype) for s in shapes for _ in range(3))
            drop.clear()
            return None

    kw = dict(CASES[case])
    dtype, sgd = kw.pop("dtype", torch.float32), kw.pop("sgd", False)
    if "qconfig" in kw:
        kw["qconfig"] = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", kw["qconfig"])
    shapes = [(64, 128), (48, 192), (33, 130), (70,)]
    host = [rng.standard_normal(s) for s in shapes]
    results = []
    for dropping in (False, True):
        junk = []
        params = [torch.nn.Parameter(torch.from_numpy(h).to(dtype).cuda()) for h in host]
        own = Own(torch.zeros(4, device="cuda"))
        opt = (lpmm.optim.SGD(params + [own], lr=1e-2, momentum=0.9) if sgd
               else lpmm.optim.AdamW(params + [own], lr=1e-2, eps=1e-3, **kw))
        grads = np.random.default_rng(9)
        for step in range(3):
            for p in params:
                p.grad = torch.from_numpy(grads.standard_normal(p.shape)).to(dtype).cuda()
            if dropping and step == 2:
                drop.extend((p, opt.state[p]) for p in params)
            opt.step()
        torch.cuda.synchronize()
        results.append([p.detach().clone() for p in params])
    assert junk and not opt.state[params[0]].get("exp_avg_qstate")
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("case", [c for c in CASES if not c.startswith("fused")] + ["factored"])
def test_codes_without_their_padding(case, monkeypatch):
    """States whose code arrays end with the values (the fused operators' layout): the walk leaves them to the loops, the
    step completes them, and leaves what it leaves on the padded arrays."""
    import lpmm.optim.adamw as adamw
    import lpmm.optim.sgd as sgd
    from lpmm import _native

    monkeypatch.setitem(CASES, "factored", dict(factor_second_moment=True))
    sides = [_build(case, np.random.default_rng(5)) for _ in range(2)]
    rng = np.random.default_rng(7)
    for step in range(4):
        grads = [rng.standard_normal(p.shape) * 0.1 for p in sides[0][0]]
        for side, (params, opt) in enumerate(sides):
            for p, g in zip(params, grads):
                p.grad = torch.from_numpy(g).to(p.dtype).cuda()
            cut = 0
            if step == 2 and side == 1:
                for p in params:
                    if p.dtype is torch.float16 and not p.is_contiguous():
                        continue  # the chain of torch ops refuses short codes
                    for k, v in opt.state[p].items():
                        if torch.is_tensor(v) and v.dtype is torch.int8:
                            bytes_ = p.numel() if case == "bits" else (p.numel() + 1) // 2
                            opt.state[p][k], cut = v[:bytes_].clone(), cut + 1
                native = _Native(_native, True)
                with monkeypatch.context() as patch:
                    patch.setattr(adamw, "_native", native)
                    patch.setattr(sgd, "_native", native)
                    opt.step()
                assert 0 < cut <= 2 * native.rest
            else:
                opt.step()
        torch.cuda.synchronize()
        for i, (p, q) in enumerate(zip(sides[0][0], sides[1][0])):
            assert torch.equal(p.detach(), q.detach()), (step, i)
            a, b = _state(sides[0][1], p), _state(sides[1][1], q)
            for k in a:
                assert torch.equal(a[k].nan_to_num(), b[k].nan_to_num()) if a[k].is_floating_point() else torch.equal(a[k], b[k]), \
                    (step, i, k)


def test_rank1_scales_without_a_group_size():
    """Rank-1 scales for both moments and a group size of zero: the staged route, on every step."""
    import lpmm

    p = torch.nn.Parameter(torch.ones(70, 61, device="cuda"))
    opt = lpmm.optim.AdamW([p], lr=1e-2, qconfig=dict(QUANT=dict(M=dict(SCALE_TYPE=dict(DEFAULT="rank1"), GROUP_SIZE=0),
                                                                SQM=dict(SCALE_TYPE=dict(DEFAULT="rank1")))))
    for _ in range(3):
        p.grad = torch.ones_like(p)
        opt.step()
    # a constant gradient moves every value by lr a step, weight decay by lr * 0.01 at most
    assert torch.allclose(p, torch.full_like(p, 1 - 3e-2), atol=4e-4)
    assert len(opt.state[p]["exp_avg_qstate"]["overhead"]["max_dims"]) == 2


@pytest.mark.parametrize("case", [c for c in CASES if c != "sgd" and not c.startswith("half")])
def test_operands_off_a_16_byte_boundary(case, monkeypatch):
    """Parameters and gradients that are views at an odd offset of a flat buffer, one or both, on every route and column
    count: the step leaves what it leaves on aligned twins, through the walk and through the loops.  (float16 rounds by
    the addresses, as torch's ops: test_gpu_nonfused_rank1_any.py.)"""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    kw = dict(CASES[case])
    if "qconfig" in kw:
        kw["qconfig"] = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", kw["qconfig"])
    shapes = MATRICES + [(17, 8, 24), (40, 1024)]
    rng = np.random.default_rng(12)
    host = [rng.standard_normal(s) * 0.1 for s in shapes]

    def at(a, off):
        flat = torch.zeros(a.size + off, device="cuda")
        flat[off:] = torch.from_numpy(a.reshape(-1)).float()
        return flat[off:].view(a.shape)

    def build(off):
        params = [torch.nn.Parameter(at(h, off)) for h in host]
        return params, lpmm.optim.AdamW(params, lr=1e-2, eps=1e-3, **kw)

    sides = [build(0), build(1), build(0), build(3)]  # aligned; parameters, gradients, both off; the last without the walk
    for step in range(4):
        grads = [rng.standard_normal(s) * 0.1 for s in shapes]
        for k, (params, opt) in enumerate(sides):
            for p, g in zip(params, grads):
                p.grad = at(g, (0, 0, 2, 1)[k])
            with monkeypatch.context() as patch:
                patch.setattr(adamw, "_native", _Native(_native, k != 3))
                opt.step()
        torch.cuda.synchronize()
        for i, p in enumerate(sides[0][0]):
            a = _state(sides[0][1], p)
            for params, opt in sides[1:]:
                b = _state(opt, params[i])
                assert a.keys() == b.keys()
                for k in a:
                    assert torch.equal(a[k].nan_to_num(), b[k].nan_to_num()) if a[k].is_floating_point() else torch.equal(a[k], b[k]), \
                        (step, i, shapes[i], k)
                assert torch.allclose(p, params[i], rtol=1e-6, atol=1e-7), (step, i, shapes[i])


@pytest.mark.parametrize("case,shape", [("default", (300, 501)), ("half", (300, 501)), ("bits", (300, 501)), ("default", (100, 61, 5, 5)),
                                        ("fused_factored", (300, 501))])
@pytest.mark.parametrize("walk", [True, False])
def test_a_step_holds_one_launch_of_new_arrays(case, shape, walk, monkeypatch):
    """160 matrices of odd width, whose codes go to new arrays on every step: beside the states a step holds the
    arrays of one launch (at most 32 tensors), not a second set of all states.  The bound is a quarter of the codes
    (a launch's are a fifth; a factored step's workspaces are less still)."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    kw = dict(CASES[case])
    dtype = kw.pop("dtype", torch.float32)
    if "qconfig" in kw:
        kw["qconfig"] = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", kw["qconfig"])
    params = [torch.nn.Parameter(torch.full(shape, 0.1, device="cuda", dtype=dtype)) for _ in range(160)]
    opt = lpmm.optim.AdamW(params, lr=1e-3, eps=1e-3, **kw)
    for p in params:
        p.grad = torch.full_like(p, 0.01)
    with monkeypatch.context() as patch:
        patch.setattr(adamw, "_native", _Native(_native, walk))
        for _ in range(2):  # the states and the second buffers of their statistics exist
            opt.step()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        opt.step()
    grown = torch.cuda.max_memory_allocated() - before
    codes = sum(t.numel() for p in params for t in opt.state[p].values() if torch.is_tensor(t) and t.dtype is torch.int8)
    assert codes > 10 << 20 and grown <= codes // 4, (grown, codes)
    assert torch.cuda.memory_allocated() <= before


@pytest.mark.parametrize("kind", ["sgd", "half vector", "half matrix"])
def test_backward_over_tensors_saved_before_a_step_fails(kind):
    """Steps that stand for a chain of torch's in-place operations count as a modification of the parameter: on the first step
    and on later ones."""
    import lpmm

    dtype = torch.float32 if kind == "sgd" else torch.float16
    p = torch.nn.Parameter(torch.full((70, 61) if kind == "half matrix" else (70,), 0.5, device="cuda", dtype=dtype))
    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    opt = (lpmm.optim.SGD([p], lr=1e-2, momentum=0.9) if kind == "sgd" else lpmm.optim.AdamW([p], lr=1e-2, eps=1e-3, qconfig=path))
    for _ in range(3):
        before = p._version
        loss = (p * p).sum()
        p.grad = torch.full_like(p, 0.1)
        opt.step()
        assert p._version > before
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()


# (shape, configuration): both sides of every limit that the walk and the loops' routes share
LIMITS = [((32768, 31), "default.yml"), ((32769, 31), "default.yml"), ((32769, 32), "default.yml"), ((32769, 33), "default.yml"),
          ((32768, 31), "2nd_moment_only_default.yml"), ((32769, 31), "2nd_moment_only_default.yml"),
          ((32768, 31), "default_8b.yml"), ((32769, 31), "default_8b.yml"), ((32769, 24), "1st_moment_group_256.yml"),
          ((15, 64, 1093), "default.yml"), ((15, 64, 1092), "default.yml"), ((16, 64, 1093), "default.yml"),  # 2^20 values, 16 rows
          ((16, 8, 8184), "default.yml"), ((16, 8, 8185), "default.yml"),  # 8192 statistics of the trailing dimensions
          ((16, 256, 256), "default.yml"), ((16, 256, 257), "default.yml"), ((32, 255, 257), "default.yml"),  # 2^16 trailing values
          ((2,) * 13, "default.yml"), ((3, 3, 3, 3, 3, 3, 3, 3), "default.yml"), ((3, 3, 3, 3, 3, 3, 3, 3, 3), "default.yml"),
          ((64, 192), "default.yml"), ((63, 192), "default.yml"), ((4097,), "default.yml"), ((4096,), "default.yml")]


@pytest.mark.parametrize("shape,config", LIMITS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_walk_and_loops_choose_one_route_at_the_limits(shape, config, dtype, monkeypatch):
    """A step by the walk leaves what a step by the loops leaves, in the same arrays' shapes, on either side of each limit."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    gen = torch.Generator(device="cuda").manual_seed(31)
    start = (torch.randn(shape, device="cuda", generator=gen) * 0.1).to(dtype)
    sides = []
    for _ in range(2):
        p = torch.nn.Parameter(start.clone())
        sides.append((p, lpmm.optim.AdamW([p], lr=1e-2, eps=1e-3, qconfig=path)))
    for step in range(4):
        g = (torch.randn(shape, device="cuda", generator=gen) * 0.1).to(dtype)
        for serve, (p, opt) in zip((True, False), sides):
            p.grad = g
            with monkeypatch.context() as patch:
                patch.setattr(adamw, "_native", _Native(_native, serve))
                opt.step()
    (p, a), (q, b) = sides
    assert torch.equal(p, q)
    x, y = _state(a, p), _state(b, q)
    assert x.keys() == y.keys()
    for k in x:
        assert x[k].shape == y[k].shape and x[k].dtype == y[k].dtype, k
        assert torch.equal(x[k].nan_to_num(), y[k].nan_to_num()) if x[k].is_floating_point() else torch.equal(x[k], y[k]), k


@pytest.mark.parametrize("case", ["fused", "group", "default", "half_group"])
def test_which_tensors_share_launches(case, monkeypatch):
    """Quantised tensors and tensors with fp32 states go to the library in one call, as the walk's batches say; float16 tensors
    have no such call, and their batches stay apart."""
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    params, opt = _build(case, np.random.default_rng(7))
    batches, calls = [], []

    class Plan:
        def __init__(self, plan):
            self._plan = plan

        def __getattr__(self, name):
            return getattr(self._plan, name)

        def start(self):
            batches.append(self._plan.start())
            return batches[-1]

    class Lib:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(_native.lib(), name)

    class Native:
        def __getattr__(self, name):
            return getattr(_native, name)

        def walk(self):
            return self

        def lib(self):
            return Lib()

        def collect(self, *args):
            return Plan(_native.walk().collect(*args))

    for p in params:
        p.grad = torch.ones_like(p) if p.is_contiguous() else None  # a strided one goes by the loops
    for _ in range(2):
        opt.step()
    monkeypatch.setattr(adamw, "_native", Native())
    opt.step()
    (kinds,) = [{b[0]: b for b in batch} for batch in batches]
    quantised = kinds[{"fused": _native.WALK_FUSED4, "half_group": _native.WALK_HALF_FLAT}.get(case, _native.WALK_FLAT)]
    plain = kinds[_native.WALK_HALF_PLAIN if case == "half_group" else _native.WALK_PLAIN]
    if case == "half_group":
        assert quantised[5] > 0 and plain[5] > 0 and quantised[7:] == (0, 0) and plain[4] == 0
        assert {"lpmm_nonfused_adamw4bit_f16_step_multi", "lpmm_nonfused_update_f16_multi"} <= set(calls)
    else:
        assert quantised[5] > 0 and plain[5] > 0 and quantised[7:] == (plain[6], plain[5]) and plain[4] == 1
        one = "lpmm_adamw4bit_fp32_step_multi" if case == "fused" else "lpmm_nonfused_adamw4bit_fp32_step_multi"
        assert calls.count(one) == 1
        assert not {"lpmm_adamw4bit_step_multi", "lpmm_adamw_fp32_step_multi", "lpmm_nonfused_adamw4bit_step_multi",
                    "lpmm_nonfused_update_multi"} & set(calls)


@pytest.mark.parametrize("serve", [True, False])
def test_scratch_vectors_share_no_cache_line(serve, monkeypatch):
    """Tensors of more than two dimensions: the column scale and the column maxima of the passes, whatever the columns."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    params = [torch.nn.Parameter(torch.randn(s, device="cuda")) for s in [(300, 12, 6, 6), (90, 7, 7, 9), (40, 64, 3, 3), (64, 128, 1, 1)]]
    opt = lpmm.optim.AdamW(params, lr=1e-2, qconfig=path)
    monkeypatch.setattr(adamw, "_native", _Native(_native, serve))
    for step in range(3):
        for p in params:
            p.grad = torch.randn_like(p)
        opt.step()
    for p in params:
        work, cols = opt._nd_scratch[p]["work"], p.numel() // p.shape[0]
        assert work.dtype is torch.float32 and work.shape[0] == 3 and work.shape[1] >= cols
        assert all(work[r].data_ptr() % 128 == 0 for r in range(3))


@pytest.mark.parametrize("case", ["fused", "default", "half", "sgd"])
def test_states_under_equal_keys_that_are_other_strings(case):
    """A state's names are compared by address first; dictionaries with other strings of the same text, or with further
    entries, are served alike."""
    sides = [_build(case, np.random.default_rng(7)) for _ in range(2)]
    for step in range(3):
        for k, (params, opt) in enumerate(sides):
            rng = np.random.default_rng(8 + step)
            for p in params:
                p.grad = torch.from_numpy(rng.standard_normal(p.shape) * 0.1).to(p.dtype).cuda()
            if step == 1 and k == 1:
                def other(d):
                    return {"".join(list(key)): other(v) if isinstance(v, dict) else v for key, v in d.items()} | {"further": 0}
                for p in params:
                    opt.state[p] = other(opt.state[p])
            opt.step()
    for p, q in zip(sides[0][0], sides[1][0]):
        assert torch.equal(p.detach(), q.detach())
        a, b = _state(sides[0][1], p), {k: v for k, v in opt.state[q].items() if torch.is_tensor(v)}
        assert all(torch.equal(a[k], v) for k, v in b.items())


@pytest.mark.parametrize("config,shape", [("default.yml", (17, 256)), ("default.yml", (17, 32, 3, 3)), ("default.yml", (34, 192)),
                                          ("default.yml", (33, 130)), ("2nd_moment_only_default.yml", (17, 256)),
                                          ("1st_moment_group_256.yml", (17, 256)), ("default_8b.yml", (17, 256)),
                                          ("default_8b.yml", (33, 130))])
@pytest.mark.parametrize("matrices,vectors", [(1, 1), (33, 63), (97, 129)])
def test_float_states_beside_the_clearing(config, shape, matrices, vectors, monkeypatch):
    """Tensors with fp32 states go with the launch that clears the two-pass kernels' statistics: more of either than one launch takes
    (192 ranges, two a matrix; 64 tensors), against the loops."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    sides = []
    for _ in range(2):
        gen = torch.Generator(device="cuda").manual_seed(3)
        shapes = [(2 + 37 * k % 3000,) for k in range(vectors)] + [shape] * matrices
        params = [torch.nn.Parameter(torch.randn(s, device="cuda", generator=gen) * 0.1) for s in shapes]
        sides.append((params, lpmm.optim.AdamW(params, lr=1e-2, eps=1e-3, qconfig=path)))
    gen = torch.Generator(device="cuda").manual_seed(4)
    for step in range(3):
        grads = [torch.randn(p.shape, device="cuda", generator=gen) * 0.1 for p in sides[0][0]]
        for serve, (params, opt) in zip((True, False), sides):
            for p, g in zip(params, grads):
                p.grad = g
            with monkeypatch.context() as patch:
                native = _Native(_native, serve)
                patch.setattr(adamw, "_native", native)
                opt.step()
                assert step < 2 or native.rest == (0 if serve else len(params))
    for p, q in zip(sides[0][0], sides[1][0]):
        assert torch.equal(p, q)
        a, b = _state(sides[0][1], p), _state(sides[1][1], q)
        assert a.keys() == b.keys() and all(torch.equal(a[k], b[k]) for k in a)


@pytest.mark.parametrize("config", ["default.yml", "2nd_moment_only_default.yml", "default_8b.yml", "default_5b.yml",
                                    "1st_moment_group_256.yml", "1st_moment_group_1024.yml"])
@pytest.mark.parametrize("shape", [(1, 5000), (5, 1004), (33, 132), (70, 64), (31, 192), (97, 136), (64, 140), (129, 160), (257, 200), (1000, 408),
                                   (16, 576), (2047, 1600), (300, 3076), (33, 33, 2, 2), (88, 88, 3, 3), (45, 17, 8), (352, 132, 1, 1)])
def test_rows_of_several_tensor_rows(shape, config, monkeypatch):
    """Column counts of 4 to 64 modulo 128 on the kernels for whole column blocks (rank1_tiles.hpp: Fold), whole and partial last rows and
    groups, against the kernels for any column count, which the loops take; rows of zeros (0 / 0 in scales and codes), a
    not-a-number and an infinity among the gradients."""
    import lpmm
    import lpmm.optim.adamw as adamw

    float_m, in_place, wide = config.startswith("2nd"), config == "default.yml", config.startswith("1st")
    if not in_place and len(shape) > 2:
        pytest.skip("such tensors go by the loops")
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    gen = torch.Generator(device="cuda").manual_seed(41)
    start = [torch.randn(s, device="cuda", generator=gen) * 0.1 for s in (shape, (64, 256))]
    sides = []
    for _ in range(2):
        params = [torch.nn.Parameter(s.clone()) for s in start]
        sides.append((params, lpmm.optim.AdamW(params, lr=1e-2, eps=1e-3, qconfig=path)))
    for step in range(5):
        grads = [torch.randn(s.shape, device="cuda", generator=gen) * 0.1 for s in start]
        rows = grads[0].view(shape[0], -1)
        rows.mul_(torch.randn(shape[0], 1, device="cuda", generator=gen).exp())
        rows[shape[0] // 2:: 5] = 0
        if step < 2:
            rows[:, ::7] = 0
        if step == 3:
            rows[-1, -1], rows[0, 1] = float("inf"), float("nan")
        for serve, (params, opt) in zip((True, False), sides):
            for p, g in zip(params, grads):
                p.grad = g
            with monkeypatch.context() as patch:
                native = _Native(_native, serve)
                patch.setattr(adamw, "_native", native)
                opt.step()
                assert step < 2 or native.rest == (0 if serve else len(params))
        # the second step replaces scales and codes as the loops' kernels do, those after it write in place
        state = sides[0][1].state[sides[0][0][0]]
        held = state["exp_avg_sq"] if float_m else state["exp_avg_qstate"]["overhead"]["max1"]
        cols = start[0].numel() // shape[0]
        if wide:  # their scales trade places on every step
            held = state["exp_avg"]
        if start[0].numel() > 4096 and not (wide and cols % 8 == 0) and (not in_place or cols % 128 != 64 or shape[0] % 2):
            assert step == 0 or (held is last) == (step >= 2)
        last = held
        if step in (2, 4):
            for p, q in zip(*(params for params, _ in sides)):
                assert torch.equal(p.nan_to_num(), q.nan_to_num())
                a, b = _state(sides[0][1], p), _state(sides[1][1], q)
                assert a.keys() == b.keys()
                for k in a:
                    assert torch.equal(a[k].nan_to_num(), b[k].nan_to_num()) if a[k].is_floating_point() else torch.equal(a[k], b[k]), k


@pytest.mark.parametrize("config,shape", [("default.yml", (33, 132)), ("2nd_moment_only_default.yml", (33, 132)),
                                          ("2nd_moment_only_default.yml", (65, 200)), ("default_8b.yml", (33, 132)),
                                          ("default_8b.yml", (65, 200)), ("1st_moment_group_256.yml", (33, 132))])
@pytest.mark.parametrize("odd", ["state", "spare"])
def test_column_statistics_at_any_float(config, shape, odd, monkeypatch):
    """Column statistics behind an odd number of row statistics in one buffer, as a caller may hold them: such a matrix stays with the
    kernels for any column count on every step, the others' own state or their spare one."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    gen = torch.Generator(device="cuda").manual_seed(5)
    start = torch.randn(shape, device="cuda", generator=gen) * 0.1
    sides = []
    for _ in range(2):
        p = torch.nn.Parameter(start.clone())
        sides.append((p, lpmm.optim.AdamW([p], lr=1e-2, eps=1e-3, qconfig=path)))

    def moved(stats):
        rows, cols = shape
        flat = torch.empty(rows + cols, device="cuda")
        assert flat[rows:].data_ptr() % 16 != 0
        views = [flat[:rows].view(rows, 1), flat[rows:].view(1, cols)]
        for view, s in zip(views, stats):
            view.copy_(s)
        return views

    for step in range(6):
        grad = torch.randn(shape, device="cuda", generator=gen) * 0.1
        for serve, (p, opt) in zip((True, False), sides):
            if step == 1 and serve:
                oh = opt.state[p]["exp_avg_sq_qstate"]["overhead"]
                if odd == "state":
                    oh["max_dims"] = moved(oh["max_dims"])
                else:
                    opt._spare_stats[p] = moved(opt._spare_stats[p])
            p.grad = grad
            with monkeypatch.context() as patch:
                native = _Native(_native, serve)
                patch.setattr(adamw, "_native", native)
                opt.step()
                assert step < 2 or native.rest == (0 if serve else 1)
        assert torch.equal(sides[0][0], sides[1][0])
        a, b = (_state(opt, p) for p, opt in sides)
        assert a.keys() == b.keys() and all(torch.equal(a[k], b[k]) for k in a)


@pytest.mark.parametrize("config", ["default.yml", "2nd_moment_only_default.yml", "default_8b.yml", "1st_moment_group_256.yml"])
@pytest.mark.parametrize("shape,in_place", [((1, 100004), False), ((31, 20004), False), ((127, 20008), False), ((511, 4100), False),
                                            ((512, 4100), True), ((31, 4092), True), ((3, 8184), True)])
def test_few_rows_of_many_columns(shape, in_place, config, monkeypatch):
    """Rows of several tensor rows pay where the matrix has at least 16 of them, or no more than 512 tiles side by side: other shapes stay
    with the kernels that they had, which leave new codes (of an fp32 first moment those of the second) or scales in other arrays."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    gen = torch.Generator(device="cuda").manual_seed(6)
    start = torch.randn(shape, device="cuda", generator=gen) * 0.1
    sides = []
    for _ in range(2):
        p = torch.nn.Parameter(start.clone())
        sides.append((p, lpmm.optim.AdamW([p], lr=1e-2, eps=1e-3, qconfig=path)))
    for step in range(4):
        grad = torch.randn(shape, device="cuda", generator=gen) * 0.1
        held = dict(sides[0][1].state[sides[0][0]])
        scales = held["exp_avg_qstate"]["overhead"].get("max1") if step else None
        for serve, (p, opt) in zip((True, False), sides):
            p.grad = grad
            with monkeypatch.context() as patch:
                native = _Native(_native, serve)
                patch.setattr(adamw, "_native", native)
                opt.step()
                assert step < 2 or native.rest == (0 if serve else 1)
        if step >= 2:
            state = sides[0][1].state[sides[0][0]]
            same = state["exp_avg_sq"] is held["exp_avg_sq"] and (
                config.startswith("1st") or state["exp_avg_qstate"]["overhead"].get("max1") is scales)
            assert same == in_place or (config.startswith("1st") and shape[1] % 8 == 0)  # those go by other kernels, in place too
    assert torch.equal(sides[0][0], sides[1][0])
    a, b = (_state(opt, p) for p, opt in sides)
    assert a.keys() == b.keys() and all(torch.equal(a[k], b[k]) for k in a)


def test_a_parameter_that_becomes_another_tensor():
    """A matrix of rows of several tensor rows, then a tensor of more than two dimensions, then a matrix again, with a fresh state each
    time; and a state from a file: its first step leaves new arrays, as any state's does."""
    import lpmm

    gen = torch.Generator(device="cuda").manual_seed(7)
    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", "default.yml")
    p = torch.nn.Parameter(torch.randn(40, 132, device="cuda", generator=gen))
    opt = lpmm.optim.AdamW([p], lr=1e-2, eps=1e-3, qconfig=path)

    def steps(optimizer, q, count):
        out = []
        for _ in range(count):
            gen.manual_seed(8)
            before = optimizer.state[q].get("exp_avg_sq") if q in optimizer.state else None
            q.grad = torch.randn(q.shape, device="cuda", generator=gen)
            optimizer.step()
            out.append(optimizer.state[q]["exp_avg_sq"] is before)
        return out

    assert steps(opt, p, 4) == [False, False, True, True]
    for shape in [(66, 33, 2, 2), (40, 132), (33, 44, 3)]:
        p.grad = None
        p.data = torch.randn(shape, device="cuda", generator=gen)
        del opt.state[p]
        q = torch.nn.Parameter(p.detach().clone())
        other = lpmm.optim.AdamW([q], lr=1e-2, eps=1e-3, qconfig=path)
        assert steps(opt, p, 4) == steps(other, q, 4) == [False, False, True, True]
        assert torch.equal(p, q)
        opt.load_state_dict(copy.deepcopy(opt.state_dict()))
        # of more than two dimensions the loops take the first one
        assert steps(opt, p, 4) == [False, len(shape) == 2, True, True]


@pytest.mark.parametrize("config", ["default.yml", "2nd_moment_only_default.yml", "default_8b.yml", "1st_moment_group_256.yml"])
def test_launches_that_end_between_kinds_of_matrices(config, monkeypatch):
    """Whole column blocks, double rows and rows of several tensor rows in turn, beyond the 48M values from which on a launch ends where
    tensors that wrap meet others: every one of them is stepped, once, as by the loops."""
    import lpmm
    import lpmm.optim.adamw as adamw
    from lpmm import _native

    path = os.path.join(os.path.dirname(lpmm.config.__file__), "configs", config)
    whole, double, wraps = (4096, 4096), (4096, 4160), (4095, 4100)
    shapes = [whole, whole, whole, wraps, whole, double, wraps, (33, 132), wraps, double, double, whole, (17, 256), whole, wraps]
    gen = torch.Generator(device="cuda").manual_seed(11)
    sides = []
    for _ in range(2):
        gen.manual_seed(12)
        params = [torch.nn.Parameter(torch.randn(s, device="cuda", generator=gen) * 0.1) for s in shapes]
        sides.append((params, lpmm.optim.AdamW(params, lr=1e-2, eps=1e-3, qconfig=path)))
    for step in range(4):
        grads = [torch.randn(s, device="cuda", generator=gen) * 0.1 for s in shapes]
        for serve, (params, opt) in zip((True, False), sides):
            for p, g in zip(params, grads):
                p.grad = g
            with monkeypatch.context() as patch:
                native = _Native(_native, serve)
                patch.setattr(adamw, "_native", native)
                opt.step()
                assert step < 2 or native.rest == (0 if serve else len(params))
    for i, (p, q) in enumerate(zip(*(params for params, _ in sides))):
        assert torch.equal(p, q), i
        a, b = _state(sides[0][1], p), _state(sides[1][1], q)
        assert a.keys() == b.keys() and all(torch.equal(a[k], b[k]) for k in a), i
