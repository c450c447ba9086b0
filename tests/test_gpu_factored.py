"""GPU parity of the non-fused elementwise update and of the factored second-moment step
against the CPU oracle, through the C ABI."""
import numpy as np
import pytest
import torch

from util import assert_rel, to_dev, to_np

pytestmark = pytest.mark.gpu

H = dict(beta1=0.9, beta2=0.999, lr=1e-3, wd=0.01, eps=1e-8)


def _lib():
    from lpmm import _native

    return _native.lib()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def test_nonfused_update_matches_oracle(oracle):
    lib = _lib()
    rng = np.random.default_rng(5)
    for n in (1, 1000, 4096 * 33 + 5):
        p = (rng.standard_normal(n) * 0.02).astype(np.float32)
        m = (rng.standard_normal(n) * 1e-3).astype(np.float32)
        v = (rng.standard_normal(n) ** 2 * 1e-6).astype(np.float32)
        dp, dm, dv = to_dev(p), to_dev(m), to_dev(v)
        mismatches = 0
        for step in (1.0, 2.0, 77.0):
            g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
            dg = to_dev(g)
            st = lib.lpmm_nonfused_update(dp.data_ptr(), dg.data_ptr(), dm.data_ptr(), dv.data_ptr(), n, H["beta1"],
                                          H["beta2"], H["lr"], H["wd"], H["eps"], step, _stream())
            assert st == 0
            oracle.nonfused_update(p, g, m, v, H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"], step)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(to_np(dm), m)
            np.testing.assert_array_equal(to_np(dv), v)
            got_p = to_np(dp)
            assert_rel(got_p, p, "p", scale=p)
            mismatches += int(np.sum(got_p != p))
            dp.copy_(torch.from_numpy(p))
        # the update's sqrt and divisions are near-exact: at most a stray last-bit difference
        assert mismatches <= max(1, n // 100000), mismatches


def test_nonfused_update_multi_matches_oracle(oracle):
    """Many small fp32-state tensors in one call (more than one launch holds), each with its
    own step count."""
    from lpmm import _native

    lib = _lib()
    rng = np.random.default_rng(6)
    sizes = [int(n) for n in rng.integers(1, 5000, size=70)] + [4096 * 3 + 1]
    host, dev = [], []
    for n in sizes:
        arrs = [(rng.standard_normal(n) * 0.02).astype(np.float32), (rng.standard_normal(n) * 1e-3).astype(np.float32),
                (rng.standard_normal(n) * 1e-3).astype(np.float32), (rng.standard_normal(n) ** 2 * 1e-6).astype(np.float32)]
        host.append(arrs)
        dev.append([to_dev(a) for a in arrs])
    steps = [float(1 + i % 9) for i in range(len(sizes))]
    table = np.array([(d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), d[3].data_ptr(), n, st, 0.0)
                      for d, n, st in zip(dev, sizes, steps)], dtype=_native.ADAMW_FP32_TENSOR)
    st = lib.lpmm_nonfused_update_multi(table.ctypes.data, len(sizes), H["beta1"], H["beta2"], H["lr"], H["wd"],
                                        H["eps"], _stream())
    assert st == 0
    torch.cuda.synchronize()
    for (p, g, m, v), d, step in zip(host, dev, steps):
        oracle.nonfused_update(p, g, m, v, H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"], step)
        np.testing.assert_array_equal(to_np(d[2]), m)
        np.testing.assert_array_equal(to_np(d[3]), v)
        assert_rel(to_np(d[0]), p, "p", scale=p)


@pytest.mark.parametrize("shape", [(64, 128), (100, 70), (513, 1025), (1024, 2752), (2752, 1024)])
def test_factored_step_matches_oracle(oracle, qmaps, shape):
    lib = _lib()
    qm = qmaps[0]
    dqm = to_dev(qm)
    r, c = shape
    n = r * c
    rng = np.random.default_rng(r + c)
    p = (rng.standard_normal((r, c)) * 0.02).astype(np.float32)
    row, col = np.zeros(r, np.float32), np.zeros(c, np.float32)
    dp, drow, dcol = to_dev(p), to_dev(row), to_dev(col)
    groups = (n + 127) // 128
    nbytes = (groups * 128 + 2047) // 2048 * 1024 + 1
    codes = torch.full((nbytes,), 0x55, dtype=torch.uint8, device="cuda")
    max1 = torch.zeros(groups, dtype=torch.float32, device="cuda")
    mean_all = torch.zeros(1, dtype=torch.float32, device="cuda")
    work = torch.empty(lib.lpmm_factored_workspace_bytes(r, c), dtype=torch.uint8, device="cuda")
    m_state = None
    for step in range(1, 5):
        g = (rng.standard_normal((r, c)) * 1e-3 * (1 + rng.random((r, 1)) * 3)).astype(np.float32)
        dg = to_dev(g)
        assert lib.lpmm_factored_stats(dg.data_ptr(), r, c, drow.data_ptr(), dcol.data_ptr(), mean_all.data_ptr(),
                                       H["beta2"], work.data_ptr(), _stream()) == 0
        assert lib.lpmm_factored_update(dp.data_ptr(), dg.data_ptr(), codes.data_ptr(), max1.data_ptr(),
                                        dqm.data_ptr(), drow.data_ptr(), dcol.data_ptr(), mean_all.data_ptr(), r, c,
                                        H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"], float(step),
                                        1 if step == 1 else 0, _stream()) == 0
        # oracle
        row_mean, col_mean = oracle.factored_stats(g)
        mean_ref = oracle.factored_ema(row, col, row_mean, col_mean, H["beta2"])
        m = np.zeros(n, np.float32) if m_state is None else oracle.dequant_group(m_state[0], m_state[1], qm, n)
        oracle.factored_update(p, g, m, row, col, mean_ref, H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"],
                               float(step))
        m_state = oracle.quant_group(m, qm)
        torch.cuda.synchronize()
        # row/col sums are accumulated in double in a different (fixed) order than the oracle's
        # sequential loop: equal after rounding to float except for rare last-bit differences
        assert_rel(to_np(drow), row, f"row step {step}", tol=2e-7)
        assert_rel(to_np(dcol), col, f"col step {step}", tol=2e-7)
        assert_rel(to_np(mean_all), [mean_ref], f"mean step {step}", tol=2e-7)
        assert_rel(to_np(dp), p, f"p step {step}")
        # the first moment does not depend on the second: bit-exact
        np.testing.assert_array_equal(to_np(max1), m_state[1])
        np.testing.assert_array_equal(to_np(codes), m_state[0])
        # continue from the oracle's statistics so that the comparison stays one step deep
        drow.copy_(torch.from_numpy(row)); dcol.copy_(torch.from_numpy(col)); dp.copy_(torch.from_numpy(p))


def test_factored_step_multi_matches_oracle(oracle, qmaps):
    """Statistics + update of many tensors per call (more than one launch group holds), each
    with its own step count, against the oracle."""
    from lpmm import _native

    lib = _lib()
    qm = qmaps[0]
    dqm = to_dev(qm)
    rng = np.random.default_rng(9)
    shapes = [(64, 128), (1, 128), (33, 256), (513, 1024), (100, 2176), (300, 4224)]
    shapes += [(int(r), 128 * int(cb)) for r, cb in zip(rng.integers(1, 120, 24), rng.integers(1, 4, 24))]
    tensors = []
    for r, c in shapes:
        n = r * c
        t = dict(r=r, c=c, n=n, p=(rng.standard_normal((r, c)) * 0.02).astype(np.float32),
                 row=np.zeros(r, np.float32), col=np.zeros(c, np.float32), m_state=None,
                 step0=int(rng.integers(0, 5)))
        t["dp"], t["drow"], t["dcol"] = to_dev(t["p"]), to_dev(t["row"]), to_dev(t["col"])
        t["codes"] = torch.full(((n + 2047) // 2048 * 1024 + 1,), 0x55, dtype=torch.uint8, device="cuda")
        t["max1"] = torch.zeros(n // 128, dtype=torch.float32, device="cuda")
        t["work"] = torch.empty(lib.lpmm_factored_workspace_bytes(r, c), dtype=torch.uint8, device="cuda")
        tensors.append(t)
    for it in range(1, 4):
        grads, recs = [], []
        for t in tensors:
            g = (rng.standard_normal((t["r"], t["c"])) * 1e-3 * (1 + rng.random((t["r"], 1)) * 3)).astype(np.float32)
            t["g"], t["dg"] = g, to_dev(g)
            recs.append((t["dp"].data_ptr(), t["dg"].data_ptr(), t["codes"].data_ptr(), t["max1"].data_ptr(),
                         t["drow"].data_ptr(), t["dcol"].data_ptr(), t["work"].data_ptr(), t["r"], t["c"],
                         float(t["step0"] + it), 1 if it == 1 else 0))
        table = np.array(recs, dtype=_native.FACTORED_TENSOR)
        st = lib.lpmm_factored_step_multi(table.ctypes.data, len(recs), dqm.data_ptr(), H["beta1"], H["beta2"],
                                          H["lr"], H["wd"], H["eps"], _stream())
        assert st == 0, lib.lpmm_status_string(st)
        torch.cuda.synchronize()
        for t in tensors:
            what = f'{t["r"]}x{t["c"]} iteration {it}'
            row_mean, col_mean = oracle.factored_stats(t["g"])
            mean_ref = oracle.factored_ema(t["row"], t["col"], row_mean, col_mean, H["beta2"])
            m = (np.zeros(t["n"], np.float32) if t["m_state"] is None
                 else oracle.dequant_group(t["m_state"][0], t["m_state"][1], qm, t["n"]))
            oracle.factored_update(t["p"], t["g"], m, t["row"], t["col"], mean_ref, H["beta1"], H["beta2"], H["lr"],
                                   H["wd"], H["eps"], float(t["step0"] + it))
            t["m_state"] = oracle.quant_group(m, qm)
            assert_rel(to_np(t["drow"]), t["row"], f"row {what}", tol=2e-7)
            assert_rel(to_np(t["dcol"]), t["col"], f"col {what}", tol=2e-7)
            assert_rel(to_np(t["dp"]), t["p"], f"p {what}")
            np.testing.assert_array_equal(to_np(t["max1"]), t["m_state"][1], err_msg=what)
            np.testing.assert_array_equal(to_np(t["codes"]), t["m_state"][0], err_msg=what)
            t["drow"].copy_(torch.from_numpy(t["row"])); t["dcol"].copy_(torch.from_numpy(t["col"]))
            t["dp"].copy_(torch.from_numpy(t["p"]))


def test_factored_fp32m_matches_oracle(oracle):
    lib = _lib()
    r, c = 48, 64
    rng = np.random.default_rng(9)
    p = (rng.standard_normal((r, c)) * 0.02).astype(np.float32)
    m = np.zeros(r * c, np.float32)
    row, col = np.zeros(r, np.float32), np.zeros(c, np.float32)
    dp, dm, drow, dcol = to_dev(p), to_dev(m), to_dev(row), to_dev(col)
    mean_all = torch.zeros(1, dtype=torch.float32, device="cuda")
    work = torch.empty(lib.lpmm_factored_workspace_bytes(r, c), dtype=torch.uint8, device="cuda")
    for step in range(1, 4):
        g = (rng.standard_normal((r, c)) * 1e-3).astype(np.float32)
        dg = to_dev(g)
        assert lib.lpmm_factored_stats(dg.data_ptr(), r, c, drow.data_ptr(), dcol.data_ptr(), mean_all.data_ptr(),
                                       H["beta2"], work.data_ptr(), _stream()) == 0
        assert lib.lpmm_factored_update_fp32m(dp.data_ptr(), dg.data_ptr(), dm.data_ptr(), drow.data_ptr(),
                                              dcol.data_ptr(), mean_all.data_ptr(), r, c, H["beta1"], H["beta2"],
                                              H["lr"], H["wd"], H["eps"], float(step), _stream()) == 0
        row_mean, col_mean = oracle.factored_stats(g)
        mean_ref = oracle.factored_ema(row, col, row_mean, col_mean, H["beta2"])
        oracle.factored_update(p, g, m, row, col, mean_ref, H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"],
                               float(step))
        torch.cuda.synchronize()
        assert_rel(to_np(drow), row, "row", tol=2e-7)
        assert_rel(to_np(dp), p, "p")
        np.testing.assert_array_equal(to_np(dm), m)
        drow.copy_(torch.from_numpy(row)); dcol.copy_(torch.from_numpy(col)); dp.copy_(torch.from_numpy(p))


def test_factored_step_multi_large_batches_equal_single_tensor_calls(qmaps):
    """Tensors whose gradients exceed the byte budget of one launch batch: the multi-tensor
    call (several batches, update pass walking back to front) must leave exactly what
    lpmm_factored_stats + lpmm_factored_update leave tensor by tensor."""
    from lpmm import _native

    lib = _lib()
    dqm = to_dev(qmaps[0])
    gen = torch.Generator(device="cuda").manual_seed(77)
    shapes = [(4096, 8192), (2048, 11008), (4096, 8192), (8192, 4096), (4096, 8192), (1000, 1152), (4096, 8192)]
    assert sum(r * c * 4 for r, c in shapes) > (384 << 20) * 3 // 2  # at least two batches

    def fresh(r, c):
        n = r * c
        t = dict(r=r, c=c, p=torch.randn(r, c, device="cuda", generator=gen) * 0.02,
                 row=torch.rand(r, device="cuda", generator=gen) * 1e-6,
                 col=torch.rand(c, device="cuda", generator=gen) * 1e-6,
                 codes=torch.randint(0, 256, (n // 2048 * 1024 + (1024 if n % 2048 else 0) + 1,), dtype=torch.uint8,
                                     device="cuda", generator=gen),
                 max1=torch.rand(n // 128, device="cuda", generator=gen) * 1e-3,
                 g=torch.randn(r, c, device="cuda", generator=gen) * 1e-3,
                 work=torch.empty(lib.lpmm_factored_workspace_bytes(r, c), dtype=torch.uint8, device="cuda"))
        return t

    a = [fresh(r, c) for r, c in shapes]
    b = [{k: (v.clone() if torch.is_tensor(v) else v) for k, v in t.items()} for t in a]
    recs = [(t["p"].data_ptr(), t["g"].data_ptr(), t["codes"].data_ptr(), t["max1"].data_ptr(), t["row"].data_ptr(),
             t["col"].data_ptr(), t["work"].data_ptr(), t["r"], t["c"], 7.0, 0) for t in a]
    table = np.array(recs, dtype=_native.FACTORED_TENSOR)
    st = lib.lpmm_factored_step_multi(table.ctypes.data, len(recs), dqm.data_ptr(), H["beta1"], H["beta2"], H["lr"],
                                      H["wd"], H["eps"], _stream())
    assert st == 0, lib.lpmm_status_string(st)
    mean_all = torch.zeros(1, dtype=torch.float32, device="cuda")
    for t in b:
        assert lib.lpmm_factored_stats(t["g"].data_ptr(), t["r"], t["c"], t["row"].data_ptr(), t["col"].data_ptr(),
                                       mean_all.data_ptr(), H["beta2"], t["work"].data_ptr(), _stream()) == 0
        assert lib.lpmm_factored_update(t["p"].data_ptr(), t["g"].data_ptr(), t["codes"].data_ptr(),
                                        t["max1"].data_ptr(), dqm.data_ptr(), t["row"].data_ptr(), t["col"].data_ptr(),
                                        mean_all.data_ptr(), t["r"], t["c"], H["beta1"], H["beta2"], H["lr"], H["wd"],
                                        H["eps"], 7.0, 0, _stream()) == 0
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        for k in ("p", "row", "col", "codes", "max1"):
            assert torch.equal(x[k], y[k]), f'{k} of {x["r"]}x{x["c"]}'


def test_factored_any_step_multi_equals_single_tensor_calls(qmaps):
    """lpmm_factored_any_step_multi on column counts of every kind (whole groups, a multiple of 8, of 4, of 2, odd), one
    column, one row, unaligned operands, fp32 first moments and first steps, 26 tensors (two launch groups): bit for bit
    what the single-tensor calls leave."""
    from lpmm import _native

    lib = _lib()
    dqm = to_dev(qmaps[0])
    gen = torch.Generator(device="cuda").manual_seed(78)
    shapes = [(64, 128), (300, 190), (70, 1000), (65, 764), (33, 257), (1, 9000), (9000, 1), (257, 66)] * 3 + [(50, 60), (700, 520)]

    def fresh(i, r, c):
        n, off = r * c, int(i % 4 == 3)
        groups = (n + 127) // 128
        dense = lambda scale: (torch.randn(n + off, device="cuda", generator=gen) * scale)[off:]
        t = dict(r=r, c=c, fp32=i % 5 == 4, first=int(i % 5 == 2), p=dense(0.02), g=dense(1e-3), m=dense(1e-3),
                 row=torch.rand(r, device="cuda", generator=gen) * 1e-6, col=torch.rand(c + off, device="cuda", generator=gen)[off:] * 1e-6,
                 codes=torch.randint(0, 256, ((n + 2047) // 2048 * 1024 + 1,), dtype=torch.uint8, device="cuda", generator=gen),
                 max1=torch.rand(groups, device="cuda", generator=gen) * 1e-3,
                 work=torch.empty(lib.lpmm_factored_workspace_bytes(r, c), dtype=torch.uint8, device="cuda"))
        return t

    def copied(v):  # at the same offset within its 16 bytes
        off = v.data_ptr() % 16 // v.element_size()
        return torch.cat([v.new_zeros(off), v])[off:]

    a = [fresh(i, r, c) for i, (r, c) in enumerate(shapes)]
    b = [{k: (copied(v) if torch.is_tensor(v) and v.is_floating_point() else v.clone() if torch.is_tensor(v) else v)
          for k, v in t.items()} for t in a]
    recs = [(t["p"].data_ptr(), t["g"].data_ptr(), t["m"].data_ptr() if t["fp32"] else t["codes"].data_ptr(),
             0 if t["fp32"] else t["max1"].data_ptr(), t["row"].data_ptr(), t["col"].data_ptr(), t["work"].data_ptr(), t["r"], t["c"],
             7.0, t["first"]) for t in a]
    table = np.array(recs, dtype=_native.FACTORED_TENSOR)
    hyper = (H["beta1"], H["beta2"], H["lr"], H["wd"], H["eps"])
    assert lib.lpmm_factored_any_step_multi(table.ctypes.data, len(recs), dqm.data_ptr(), *hyper, _stream()) == 0
    mean_all = torch.zeros(1, dtype=torch.float32, device="cuda")
    for t in b:
        r, c = t["r"], t["c"]
        assert lib.lpmm_factored_stats(t["g"].data_ptr(), r, c, t["row"].data_ptr(), t["col"].data_ptr(), mean_all.data_ptr(),
                                       H["beta2"], t["work"].data_ptr(), _stream()) == 0
        if t["fp32"]:
            assert lib.lpmm_factored_update_fp32m(t["p"].data_ptr(), t["g"].data_ptr(), t["m"].data_ptr(), t["row"].data_ptr(),
                                                  t["col"].data_ptr(), mean_all.data_ptr(), r, c, *hyper, 7.0, _stream()) == 0
        else:
            assert lib.lpmm_factored_update(t["p"].data_ptr(), t["g"].data_ptr(), t["codes"].data_ptr(), t["max1"].data_ptr(),
                                            dqm.data_ptr(), t["row"].data_ptr(), t["col"].data_ptr(), mean_all.data_ptr(), r, c,
                                            *hyper, 7.0, t["first"], _stream()) == 0
    torch.cuda.synchronize()
    for i, (x, y) in enumerate(zip(a, b)):
        for k in ("p", "m", "row", "col", "codes", "max1"):
            assert torch.equal(x[k], y[k]), f'{k} of tensor {i}, {x["r"]}x{x["c"]}'
    bad = list(recs[1])
    bad[1] = 0
    table = np.array([tuple(bad)], dtype=_native.FACTORED_TENSOR)
    assert lib.lpmm_factored_any_step_multi(table.ctypes.data, 1, dqm.data_ptr(), *hyper, _stream()) != 0


@pytest.mark.parametrize("count,rows,cols", [(25, 64, 128), (49, 64, 96), (30, 256, 128), (30, 257, 128), (25, 1024, 72), (25, 1025, 128), (2, 1500, 128)])
def test_groups_of_small_tensors(count, rows, cols):
    """More than 24 tensors in a group, and means without their launch (up to 1024 rows), on either kind of kernels, against the
    single-tensor entry points (one tensor of more than 1024 rows beside each would change the route, not the result)."""
    import lpmm

    gen = torch.Generator(device="cuda").manual_seed(9)
    start = [torch.randn(rows, cols, device="cuda", generator=gen) * 0.1 for _ in range(count)]
    tall = torch.randn(1300, cols, device="cuda", generator=gen) * 0.1
    many, few = [[torch.nn.Parameter(s.clone()) for s in start] for _ in range(2)]
    tails = [torch.nn.Parameter(tall.clone()) for _ in few]
    make = lambda ps: lpmm.optim.AdamW(ps, lr=1e-2, factor_second_moment=True, fused=True)  # noqa: E731
    opt, apart = make(many), [make([p, t]) for p, t in zip(few, tails)]
    for step in range(4):
        for p, q, t in zip(many, few, tails):
            p.grad = q.grad = torch.randn(rows, cols, device="cuda", generator=gen)
            t.grad = torch.ones_like(t)
        for o in [opt] + apart:
            o.step()
    for k, (p, q) in enumerate(zip(many, few)):
        assert torch.equal(p, q)
        a, b = opt.state[p], apart[k].state[q]
        for name in ("exp_avg", "exp_avg_sq_row", "exp_avg_sq_col"):
            assert torch.equal(a[name], b[name]), name


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("matrices,vectors,rows", [(1, 1, 96), (24, 64, 96), (3, 70, 1100), (26, 5, 96)])
def test_float_states_beside_the_statistics(matrices, vectors, rows, fused):
    """Tensors with fp32 states go with the launch that finishes the factored ones' statistics: either arithmetic, with and without the
    launch for the means, more of them than one launch takes (64), against optimizers of their own."""
    import lpmm

    gen = torch.Generator(device="cuda").manual_seed(10)
    start = [torch.randn(s, device="cuda", generator=gen) * 0.1
             for s in [(2 + 37 * k % 3000,) for k in range(vectors)] + [(rows, 128 if k % 2 else 72) for k in range(matrices)]]
    both, apart = [[torch.nn.Parameter(s.clone()) for s in start] for _ in range(2)]
    make = lambda ps: lpmm.optim.AdamW(ps, lr=1e-2, factor_second_moment=True, fused=fused)  # noqa: E731
    opt, others = make(both), [make(apart[:vectors]), make(apart[vectors:])]
    for step in range(4):
        for p, q in zip(both, apart):
            p.grad = q.grad = torch.randn(p.shape, device="cuda", generator=gen)
        for o in [opt] + others:
            o.step()
    for k, (p, q) in enumerate(zip(both, apart)):
        assert torch.equal(p, q), k
        a, b = opt.state[p], others[k >= vectors].state[q]
        assert all(torch.equal(a[n], b[n]) for n in a if torch.is_tensor(a[n]))
