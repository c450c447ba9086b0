"""Host-side behaviour that needs no GPU: the C ABI's symbols and argument checks, the
config reader, the optimizer's state bookkeeping and error behaviour."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HEADER = os.path.join(ROOT, "include", "lpmm_hip.h")


def declared_functions():
    txt = open(HEADER).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(lpmm_[a-z0-9_]+)\s*\(", txt)))


def test_library_exports_every_declared_symbol():
    from lpmm import _native

    lib = ctypes.CDLL(_native.LIB_PATH)
    names = declared_functions()
    assert len(names) >= 17
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/lpmm_hip.h but not exported"
    assert sorted(_native.PROTOTYPES) == names, "lpmm/_native.py prototypes differ from the header"
    assert _native.lib().lpmm_abi_version() == _native.ABI_VERSION


def test_record_layouts_match_header():
    from lpmm import _native

    assert _native.ADAMW4BIT_TENSOR.itemsize == 64 and _native.ADAMW_FP32_TENSOR.itemsize == 48
    assert _native.ADAMW4BIT_TENSOR.fields["n"][1] == 48 and _native.ADAMW4BIT_TENSOR.fields["step"][1] == 56
    assert _native.ADAMW_FP32_TENSOR.fields["n"][1] == 32 and _native.ADAMW_FP32_TENSOR.fields["step"][1] == 40
    assert _native.NONFUSED_RANK1_F16_TENSOR.itemsize == 104 and _native.NONFUSED_RANK1_F16_TENSOR.fields["work"][1] == 72
    assert _native.NONFUSED_RANK1_F16_TENSOR.fields["rows"][1] == 80 and _native.NONFUSED_RANK1_F16_TENSOR.fields["step"][1] == 96
    header = open(os.path.join(ROOT, "include", "lpmm_hip.h")).read()
    assert int(re.search(r"#define LPMM_MULTI_MAX (\d+)", header).group(1)) == _native.MULTI_MAX


def test_argument_errors_without_gpu():
    """Validation precedes any HIP call: NULL, misaligned and out-of-range arguments are
    reported as status codes on a machine without a GPU."""
    from lpmm import _native

    lib = _native.lib()
    buf = np.zeros(64, np.float32)
    ptr = buf.ctypes.data
    NULL, ALIGN, SIZE = 1, 2, 3
    f6 = (0.9, 0.999, 1e-3, 0.01, 1e-8, 1.0)
    assert lib.lpmm_adamw4bit_step(None, ptr, ptr, ptr, ptr, ptr, ptr, ptr, 16, *f6, None) == NULL
    assert lib.lpmm_adamw4bit_step(ptr, ptr, ptr, ptr, ptr, ptr, None, ptr, 16, *f6, None) == NULL
    assert lib.lpmm_adamw4bit_step(ptr + 2, ptr, ptr, ptr, ptr, ptr, ptr, ptr, 16, *f6, None) == ALIGN
    assert lib.lpmm_adamw4bit_step(ptr, ptr, ptr, ptr, ptr, ptr, ptr, ptr, -1, *f6, None) == SIZE
    assert lib.lpmm_adamw4bit_step(ptr, ptr, ptr, ptr, ptr, ptr, ptr, ptr, 0, *f6, None) == 0  # nothing to do
    assert lib.lpmm_adamw4bit_step_multi(None, 3, ptr, ptr, *f6[:5], None) == NULL
    assert lib.lpmm_adamw4bit_step_multi(None, 0, ptr, ptr, *f6[:5], None) == 0
    assert lib.lpmm_adamw_fp32_step(ptr, None, ptr, ptr, 16, *f6, None) == NULL
    assert lib.lpmm_pack_nonlinear_4bit(ptr, ptr, 12, ptr, None) == SIZE  # not a multiple of 8
    assert lib.lpmm_pack_nonlinear_4bit(None, ptr, 16, ptr, None) == NULL
    assert lib.lpmm_unpack_nonlinear_4bit(ptr, ptr, -5, ptr, None) == SIZE
    assert lib.lpmm_quant_group(ptr, 64, 100, ptr, ptr, ptr, None) == SIZE  # group size not 128 * 2^k
    assert lib.lpmm_quant_group(ptr, 64, 8192, ptr, ptr, ptr, None) == SIZE
    assert lib.lpmm_quant_group(ptr, 0, 128, ptr, ptr, ptr, None) == SIZE
    assert lib.lpmm_dequant_group(ptr, ptr, ptr, 64, 64, ptr, None) == SIZE
    assert lib.lpmm_rank1_stats(ptr, 0, 8, ptr, ptr, None) == SIZE
    assert lib.lpmm_quant_rank1(ptr, 8, 8, None, ptr, ptr, ptr, None) == NULL
    assert lib.lpmm_dequant_rank1(ptr, ptr, ptr, ptr, 8, -8, ptr, None) == SIZE
    assert lib.lpmm_nonfused_update(ptr, ptr, ptr + 1, ptr, 16, 0.9, 0.999, 1e-3, 0.01, 1e-8, 1.0, None) == ALIGN
    assert lib.lpmm_factored_stats(ptr, 8, 8, ptr, ptr, ptr, 0.999, None, None) == NULL
    assert lib.lpmm_factored_update(ptr, ptr, ptr, ptr, ptr, ptr, ptr, ptr, 0, 8, 0.9, 0.999, 1e-3, 0.01, 1e-8, 1.0,
                                    0, None) == SIZE
    # 64 x 256 tiles: 64 row tiles of column partials, 43 column tiles of row partials, 16 row-block sums, the mean
    assert lib.lpmm_factored_workspace_bytes(4096, 11008) == (64 * 11008 + 43 * 4096 + 16 + 1) * 8
    assert lib.lpmm_status_string(NULL).decode().startswith("a required pointer")
    with pytest.raises(RuntimeError, match="status 3"):
        _native.check(SIZE, "probe")


@pytest.mark.parametrize("kind", ["RANK1_CODES4", "RANK1_FLOAT_M", "RANK1_CODES8", "RANK1_HALF"])
@pytest.mark.parametrize("field, change, status", [("v_codes_next", "null", 1), ("v_codes_next", "shift", 2),
                                                   ("v_codes_next", "v_codes", 5), ("p", "null", 1), ("g", "shift", 2),
                                                   ("v_rowmax_next", "v_rowmax", 5), ("rows", "negative", 3)])
def test_a_call_for_any_column_count_checks_every_record_first(kind, field, change, status):
    """A record that is taken in runs of four values, large enough for launches of its own beside the other kind, and an
    invalid one of the other kind: its status comes back, and not that of the first one's launch (there is no device here)."""
    from lpmm import _native

    lib, k = _native.lib(), getattr(_native, kind)
    memory = np.zeros(4096, np.uint8)  # never read: only the addresses count
    base = (memory.ctypes.data + 63) // 64 * 64
    records = np.zeros(2, _native.RANK1_ANY_TENSOR)
    for i, (rows, cols) in enumerate([(12000, 2004), (70, 61)]):
        for j, name in enumerate(_native.RANK1_ANY_TENSOR.names[:13]):
            records[i][name] = base + 1024 * i + 64 * j
        records[i]["rows"], records[i]["cols"], records[i]["step"] = rows, cols, 1.0
    bad = records[1]
    bad[field] = 0 if change == "null" else bad[field] + 1 if change == "shift" else -1 if change == "negative" else bad[change]
    bits = 8 if kind == "RANK1_CODES8" else 4
    for table in (records, records[::-1].copy()):
        assert lib.lpmm_nonfused_adamw_rank1_any_step_multi(table.ctypes.data, 2, k, 128, base, bits, None, base, bits, None, 0.9, 0.999,
                                                            1e-3, 0.01, 1e-8, 3, None) == status


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """launches(line, ...): per line (a call as tests/launches.cpp describes it) its status and the grids it launches, in order."""
    from lpmm import _native

    exe, libs, rocm = str(tmp_path_factory.mktemp("launches") / "launches"), os.path.dirname(_native.LIB_PATH), "/opt/rocm"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-rdynamic", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                           "-I" + os.path.join(ROOT, "include"), os.path.join(HERE, "launches.cpp"), "-L" + libs, "-llpmm_hip",
                           f"-L{rocm}/lib", "-lamdhip64", f"-Wl,-rpath,{libs}", f"-Wl,-rpath,{rocm}/lib", "-o", exe])

    def run(*lines):
        out = subprocess.run([exe], input="\n".join(lines), capture_output=True, text=True, check=True).stdout.splitlines()
        assert len(out) == len(lines)
        return [(int(words[0]), [tuple(map(int, w.split(","))) for w in words[1:]]) for words in map(str.split, out)]

    return run


def test_rank1_statistics_of_extreme_sizes(launches):
    """What lpmm_rank1_stats refuses it refuses before the launch that clears the caller's arrays, and a matrix of more tiles
    than a grid holds is taken in taller ones."""
    rows, limit = 65535 * 64, 0x7fffffff
    for status, grids in launches(f"stats {rows + 1} 1", f"stats 1 {limit * 256 + 1}", "stats 0 8", "stats 8 0", "stats -1 8"):
        assert (status, grids) == (3, [])
    for status, grids in launches(f"stats {rows} 1", f"stats {rows} {1 << 24}", f"stats 40 {1 << 36}", "stats 40 100"):
        assert status == 0 and len(grids) == 2 and all(0 < x <= limit and y == 1 for x, y in grids)


def test_rank1_quantisers_of_more_rows_than_a_grid_holds(launches):
    """Rows go along the grid's second dimension, which ends at 65535; a matrix with more takes the flat split, in one dimension."""
    limit = 65535 * 64  # rows of 128 columns: 16 side by side, four of each
    calls = [f"{way} {bits} {rows} 128" for way in ("quant", "dequant") for bits in (4, 8) for rows in (limit, limit + 1)]
    for call, (status, grids) in zip(calls, launches(*calls)):
        values = 128 * int(call.split()[2])
        rows_split, flat = (1, 65535), (-(-values // 4096), 1)
        assert status == 0 and grids == [rows_split if values == 128 * limit else flat], call


def test_chunks_of_the_rank1_dequantisers(launches):
    """Whole column groups: chunks that leave few lanes idle or cut few lines, and the flat split (0) for the others."""
    rows = 1000
    chunks = {1: 1, 2: 2, 4: 4, 3: 0, 5: 0, 6: 0, 9: 0, 12: 2, 13: 0, 18: 2, 33: 2, 43: 2, 8: 8, 16: 16, 40: 8, 64: 16, 86: 8, 250: 16}
    calls = {f"dequant {bits} {rows} {128 * groups}": (groups, wide) for groups, wide in chunks.items() for bits in (4, 8)}
    for (call, (groups, wide)), (status, grids) in zip(calls.items(), launches(*calls)):
        want = (-(-groups // wide), -(-rows // (4 * (16 // wide)))) if wide else (-(-rows * 128 * groups // 4096), 1)
        assert (status, grids) == (0, [want]), call


# matrices of one column of tiles, so that a pass's grid is its row blocks
NARROW = [(mode, rows, cols) for mode in ("codes4", "float_m", "codes8")
          for rows, cols in [(20000, 128), (21788, 256), (50257, 128), (70001, 256), (100000, 128)]]


def test_interleaved_groups_of_narrow_matrices(launches):
    """Groups of row blocks that work on neighbouring rows are of a multiple of 8 blocks where they are large: neighbours share
    cache lines of statistics and scales."""
    for case, (status, grids) in zip(NARROW, launches(*("rank1 %s %d %d" % case for case in NARROW))):
        assert status == 0 and len(grids) == 3, case
        for x, y in grids[1:]:
            assert y == 1 and x % 8 == 0 and x * 128 >= case[1], (case, grids)


def test_row_blocks_of_a_column(launches):
    """Atomics of a column's row blocks queue up on one address: the update pass of a tall narrow matrix keeps them few, alone
    and beside large matrices, below and above the sizes at which its tiles change."""
    cases = [(mode, rows, cols, beside) for mode in ("codes4", "float_m", "codes8") for cols in (128, 256, 512, 1024)
             for values in (6e6, 60e6, 70e6, 300e6) for rows in [int(values) // cols] for beside in ("", " 8192 8192")]
    for (mode, rows, cols, beside), (status, grids) in zip(cases, launches(*("rank1 %s %d %d%s" % case for case in cases))):
        assert status == 0 and len(grids) == 3
        tiles = grids[1][0]
        if beside:
            tiles -= 8192 * 8192 // 256 // 16  # at most: tiles of 16 rows by 256 columns
        col_tiles = (cols + 255) // 256
        # the rule, the tallest tiles, and the empty blocks of a group
        assert tiles // col_tiles <= max(512, rows * cols / 12000, rows / 128) + 256, (mode, rows, cols, beside, grids)


def test_second_pass_of_tiles_of_one_column_group(launches):
    """Five column groups go one to a tile; above 3M values such tiles have 32 rows in the second pass, as many values as the
    16-row tiles of two groups that matrices of up to 4M values take."""
    calls = ["rank1 %s %d %d" % (mode, rows, cols) for mode in ("codes4", "float_m", "codes8")
             for rows, cols in [(5000, 640), (4000, 640), (2500, 1280)]]
    for call, (status, grids) in zip(calls, launches(*calls)):
        rows = call.split()[2]
        tile_rows = 32 if rows == "5000" else 16
        blocks, tiles = -(-int(rows) // tile_rows), 5
        assert status == 0 and blocks * tiles <= grids[2][0] < (blocks + 64) * tiles, (call, grids)


def test_update_tiles_of_small_launches(launches):
    """Workgroups of the update pass (row blocks times column tiles; full groups, so that none is empty): tiles of one column group have 16
    rows only in the smallest launches, byte codes 32 rows at least from 14M values on."""
    want = {"rank1 codes4 2048 128": 2048 // 16, "rank1 codes4" + 24 * " 4096 128": 24 * 4096 // 32, "rank1 float_m" + 24 * " 4096 128": 24 * 4096 // 32,
            "rank1 codes8" + 24 * " 4096 128": 24 * 4096 // 64, "rank1 codes8 4096 4096": 4096 // 32 * 16, "rank1 codes4 4096 4096": 4096 // 16 * 16,
            "rank1 codes8 2048 2048": 2048 // 16 * 8}
    for (call, tiles), (status, grids) in zip(want.items(), launches(*want)):
        assert status == 0 and grids[1] == (tiles, 1), (call, grids)


def test_second_pass_tiles_of_odd_columns(launches):
    """Rows of an odd column count share code bytes: tiles of 16 rows, of 32 in between.  (The call takes any column count.)"""
    for values_of, tile_rows in (((1000, 2001), 16), ((2001, 3001), 32), ((2072, 4615), 16), ((5000, 5001), 16)):
        rows, cols = values_of
        (status, grids), = launches(f"any {rows} {cols}")
        blocks, tiles = -(-rows // tile_rows), -(-(-(-cols // 128)) // 2)
        assert status == 0 and blocks * tiles <= grids[2][0] < (blocks + 256 // tiles) * tiles, (values_of, grids)


def test_where_launches_end_between_kinds_of_matrices(launches):
    """A launch ends at 32 tensors (4-bit codes: 64 of at most 80M values in all), and from 48M values on before the first tensor that
    wraps among others or the other way round; double rows count as others.  In calls: the clearing, then two passes a launch."""
    whole, double, wraps = " 4096 4096", " 4096 4160", " 4096 4100"  # 17M values each
    for mode in ("codes4", "float_m", "codes8", "groups"):
        cases = {3 * whole + wraps: 2, 2 * whole + wraps + whole + wraps: 1, 3 * double + wraps: 2, 3 * whole + double: 1, 3 * wraps + double: 2,
                 3 * wraps + whole + 2 * wraps: 2, 3 * whole + wraps + 2 * whole + double: 2, 3 * whole + 3 * wraps + whole: 3, wraps: 1,
                 33 * " 512 512": 1 if mode == "codes4" else 2, 64 * " 512 516": 1 if mode == "codes4" else 2,
                 65 * " 512 516": 2 if mode == "codes4" else 3}
        for (shapes, count), (status, grids) in zip(cases.items(), launches(*(f"beside {mode}{shapes}" for shapes in cases))):
            assert status == 0 and len(grids) == 1 + 2 * count, (mode, shapes, grids)


def test_remainders_of_small_float16_launches(launches):
    """55 row blocks of 128 rows, 17 resident beside 15 column tiles: launches of few workgroups take four groups of 17, the last one's
    rows spread over all of its blocks; others take groups of equal size."""
    few, many = launches("rank1 half 6974 3840", "rank1 half" + 2 * " 6974 3840")
    assert few[0] == 0 and [x for x, y in few[1][1:3]] == [4 * 17 * 15] * 2
    assert many[0] == 0 and [x for x, y in many[1][1:3]] == [2 * 4 * 14 * 15] * 2


def test_config_defaults_and_yaml():
    from lpmm.config import CONFIG_DIR, get_config

    c = get_config(None)
    # built-in default for v is 'group', not 'rank1' (lpmm/config.py:58); README's default.yml says rank1
    assert c.QUANT.SQM.SCALE_TYPE.DEFAULT == "group" and c.QUANT.M.SCALE_TYPE.DEFAULT == "group"
    assert c.QUANT.M.BITS == 4 and c.QUANT.M.SIGNED is True and c.QUANT.M.QUANT_TYPE.DEFAULT == "nonlinear"
    assert c.QUANT.SQM.SIGNED is False and c.QUANT.SQM.QUANT_TYPE.DEFAULT == "power-1"
    assert c.QUANT.M.THRESHOLD == 4096 and c.QUANT.M.ROUND_TYPE == "real-nearest" and c.QUANT.M.GROUP_SIZE == 128
    d = get_config(os.path.join(CONFIG_DIR, "default.yml"))
    assert d.QUANT.SQM.SCALE_TYPE.DEFAULT == "rank1" and d.QUANT.SQM.SIGNED is False  # untouched keys survive
    assert get_config(os.path.join(CONFIG_DIR, "2nd_moment_group_128.yml")).QUANT.SQM.SCALE_TYPE.DEFAULT == "group"
    assert get_config(os.path.join(CONFIG_DIR, "1st_moment_group_512.yml")).QUANT.M.GROUP_SIZE == 512
    assert get_config(os.path.join(CONFIG_DIR, "2nd_moment_only_default.yml")).QUANT.M.ENABLE is False
    assert get_config(None).QUANT.SQM.SCALE_TYPE.DEFAULT == "group"  # defaults are not mutated by merges
    with pytest.raises(TypeError):
        get_config(42)


def test_config_base_inheritance(tmp_path):
    from lpmm.config import get_config

    (tmp_path / "base.yml").write_text("QUANT:\n  M:\n    GROUP_SIZE: 256\n  SQM:\n    THRESHOLD: 100\n")
    (tmp_path / "child.yml").write_text("BASE: ['base.yml']\nQUANT:\n  SQM:\n    SCALE_TYPE: {DEFAULT: rank1}\n")
    c = get_config(str(tmp_path / "child.yml"))
    assert c.QUANT.M.GROUP_SIZE == 256 and c.QUANT.SQM.THRESHOLD == 100 and c.QUANT.SQM.SCALE_TYPE.DEFAULT == "rank1"


def test_optimizer_argument_validation():
    import lpmm

    p = [torch.nn.Parameter(torch.zeros(4))]
    for kw in (dict(lr=-1.0), dict(eps=-1e-8), dict(betas=(1.0, 0.999)), dict(betas=(0.9, -0.1)), dict(weight_decay=-1)):
        with pytest.raises(ValueError):
            lpmm.optim.AdamW(p, **kw)
    opt = lpmm.optim.AdamW(p, lr=1e-3, fused=True, factor_second_moment=True)
    g = opt.param_groups[0]
    assert g["fused"] is True and g["factor_second_moment"] is True and g["use_first_moment"] is True
    assert g["betas"] == (0.9, 0.999) and g["eps"] == 1e-8 and g["weight_decay"] == 1e-2
    with pytest.raises(ValueError):
        opt.get_subqconfig("nope")
    md = opt.get_qmetadata_by_state_name("exp_avg")
    assert md == dict(b=4, scale_type="group", quant_type="nonlinear", round_type="real-nearest", gp_sz=128, signed=True)
    md = opt.get_qmetadata_by_state_name("exp_avg_sq")
    assert md == dict(b=4, scale_type="group", quant_type="power-1", round_type="real-nearest", gp_sz=128, signed=False)


def test_sgd_argument_validation():
    import lpmm

    p = [torch.nn.Parameter(torch.zeros(4))]
    for kw in (dict(lr=-1.0), dict(lr=0.1, momentum=-0.5), dict(lr=0.1, weight_decay=-1.0), dict(lr=0.1, fused=True)):
        with pytest.raises(ValueError):
            lpmm.optim.SGD(p, **kw)
    opt = lpmm.optim.SGD(p, lr=0.1, momentum=0.9)
    assert opt.get_qmetadata_by_state_name("momentum_buffer")["quant_type"] == "nonlinear"
    with pytest.raises(ValueError):
        opt.get_subqconfig("exp_avg")


def test_state_init_threshold_and_override():
    """State layout on first use (lpmm/optim/adamw.py:114-129) and the numel > 4096 rule
    (lpmm/optim/optimizer.py:156-163); needs no GPU because only the bookkeeping runs."""
    import lpmm

    big = torch.nn.Parameter(torch.zeros(64, 65))     # 4160 > 4096
    edge = torch.nn.Parameter(torch.zeros(64, 64))    # 4096: not quantised
    forced = torch.nn.Parameter(torch.zeros(100, 100))
    holder = torch.nn.Module()
    holder.w = forced
    opt = lpmm.optim.AdamW([big, edge, forced], factor_second_moment=False)
    opt.override_quantize_enable(holder, "w", False)
    group = opt.param_groups[0]
    for p in (big, edge, forced):
        state, factored = opt._state_of(group, p)
        assert not factored
        assert set(state) == {"step", "exp_avg", "exp_avg_sq", "exp_avg_qstate", "exp_avg_sq_qstate"}
        assert state["step"].device.type == "cpu" and float(state["step"]) == 0.0
        assert state["exp_avg"].dim() == 0 and state["exp_avg_sq"].dim() == 0
        assert set(state["exp_avg_qstate"]) == {"enable", "overhead", "qmap"}
        assert state["exp_avg_qstate"]["qmap"].numel() == 16
    assert opt.state[big]["exp_avg_qstate"]["enable"] is True
    assert opt.state[edge]["exp_avg_qstate"]["enable"] is False
    assert opt._enabled(forced, opt.state[forced], "exp_avg") is False
    assert opt.state[big]["exp_avg_qstate"]["qmap"] is opt.state[forced]["exp_avg_qstate"]["qmap"]  # cached
    with pytest.raises(ValueError):
        opt.override_quantize_enable(holder, "w", True)  # state already exists
    fopt = lpmm.optim.AdamW([torch.nn.Parameter(torch.zeros(3, 8, 16))], factor_second_moment=True)
    p = fopt.param_groups[0]["params"][0]
    state, factored = fopt._state_of(fopt.param_groups[0], p)
    assert factored and state["exp_avg_sq_row"].shape == (3, 8) and state["exp_avg_sq_col"].shape == (3, 16)
    assert "exp_avg_sq" not in state


def test_cpu_tensors_are_rejected_loudly():
    """There is no CPU path: a step on CPU parameters raises like the reference's operators
    (lpmm/cpp_extension/common.h:15-27)."""
    import lpmm
    from lpmm.cpp_extension import fused_adamw, quantization

    p = torch.nn.Parameter(torch.randn(100, 100))
    p.grad = torch.randn(100, 100)
    for fused in (True, False):
        opt = lpmm.optim.AdamW([p], fused=fused)
        with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
            opt.step()
    z = torch.zeros(8)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        fused_adamw.adamw_single_tensor(z, z, z, z, 0.9, 0.999, 1e-3, 0.01, 1e-8, 1.0)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        quantization.pack_nonlinear(torch.zeros(1, 8), torch.zeros(16), 4, False)
    with pytest.raises(RuntimeError):
        quantization.pack_nonlinear(torch.zeros(1, 8), torch.zeros(16), 9, False)  # bits <= 8
    sparse = torch.nn.Parameter(torch.randn(10, 10))
    sparse.grad = torch.randn(10, 10).to_sparse()
    with pytest.raises(RuntimeError, match="sparse"):
        lpmm.optim.AdamW([sparse]).step()


def test_state_dict_round_trip_keeps_packed_int8():
    """load_state_dict moves state to the parameter's device/dtype but never converts the
    packed int8 tensors or `step` (lpmm/optim/optimizer.py:95-115)."""
    import lpmm

    p = torch.nn.Parameter(torch.zeros(64, 65, dtype=torch.float64))
    opt = lpmm.optim.AdamW([p], fused=True)
    state, _ = opt._state_of(opt.param_groups[0], p)
    state["step"] += 3
    state["exp_avg"] = torch.arange(-100, 100, dtype=torch.int8)
    state["exp_avg_sq"] = torch.arange(0, 120, dtype=torch.int8)
    state["exp_avg_qstate"]["overhead"]["max1"] = torch.rand(33)
    state["exp_avg_sq_qstate"]["overhead"].update({"max1": None, "max_dims": [torch.rand(64, 1), torch.rand(1, 65)],
                                                   "scaled_shape": torch.Size((64, 65)), "dtype": torch.float32,
                                                   "stride": (65, 1), "dim": 2})
    sd = opt.state_dict()
    assert "qconfig" in sd
    opt2 = lpmm.optim.AdamW([torch.nn.Parameter(torch.zeros(64, 65, dtype=torch.float64))], fused=True)
    opt2.load_state_dict(sd)
    s2 = opt2.state[opt2.param_groups[0]["params"][0]]
    assert s2["exp_avg"].dtype == torch.int8 and torch.equal(s2["exp_avg"], state["exp_avg"])
    assert s2["exp_avg_sq"].dtype == torch.int8
    assert float(s2["step"]) == 3.0 and s2["step"].dtype == torch.float32
    assert s2["exp_avg_qstate"]["overhead"]["max1"].dtype == torch.float64  # float state follows the parameter
    # ... except the maps: the kernels read them as floats, and a rounded map would decode the codes differently
    assert s2["exp_avg_qstate"]["qmap"].dtype == torch.float32 and s2["exp_avg_sq_qstate"]["qmap"].dtype == torch.float32
    assert torch.equal(s2["exp_avg_qstate"]["qmap"], state["exp_avg_qstate"]["qmap"])
    oh = s2["exp_avg_sq_qstate"]["overhead"]
    assert oh["scaled_shape"] == torch.Size((64, 65)) and oh["dtype"] == torch.float32 and oh["dim"] == 2
    assert isinstance(oh["max_dims"], list) and oh["max_dims"][1].shape == (1, 65)
    assert opt2.qconfig.QUANT.M.BITS == 4
    with pytest.raises(ValueError):
        lpmm.optim.AdamW([torch.nn.Parameter(torch.zeros(2)), torch.nn.Parameter(torch.zeros(2))]).load_state_dict(sd)

    # the reference stores its yacs CfgNode under 'qconfig' (lpmm/optim/optimizer.py:68-71): a dict subclass with
    # attribute access, nested in itself.  Any such mapping is accepted and becomes this package's own node type.
    class CfgNodeLike(dict):
        def __getattr__(self, name):
            if name in self:
                return self[name]
            raise AttributeError(name)

    def wrap(value):
        return CfgNodeLike({k: wrap(v) for k, v in value.items()}) if isinstance(value, dict) else value

    sd3 = dict(sd, qconfig=wrap(sd["qconfig"]))
    sd3["qconfig"]["QUANT"]["SQM"]["SCALE_TYPE"]["DEFAULT"] = "rank1"
    opt3 = lpmm.optim.AdamW([torch.nn.Parameter(torch.zeros(64, 65, dtype=torch.float64))], fused=True)
    opt3.load_state_dict(sd3)
    assert type(opt3.qconfig) is lpmm.config.Node and type(opt3.qconfig.QUANT.SQM) is lpmm.config.Node
    assert opt3.qconfig.QUANT.SQM.SCALE_TYPE.DEFAULT == "rank1"
    assert type(opt3.state_dict()["qconfig"]) is dict
    with pytest.raises(ValueError, match="lacks QUANT.M"):
        opt3.load_state_dict(dict(sd, qconfig={"QUANT": {"SQM": sd["qconfig"]["QUANT"]["SQM"]}}))


def test_oracle_under_sanitizers(tmp_path):
    """The oracle's C code under AddressSanitizer + UBSan on ragged sizes (host only)."""
    exe = str(tmp_path / "oracle_sanitize")
    subprocess.check_call(["gcc", "-O1", "-g", "-std=c11", "-ffp-contract=off", "-fsanitize=address,undefined",
                           "-fno-sanitize-recover=all", "-fno-omit-frame-pointer", "-static-libasan",
                           os.path.join(HERE, "oracle_sanitize_driver.c"), os.path.join(ROOT, "oracle", "lpmm_oracle.c"),
                           "-lm", "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    assert "ok" in out.stdout


def test_utils_metrics_and_bookkeeping():
    """lpmm.utils: closed forms of the error metrics, byte counting, rank helpers."""
    from lpmm import utils

    x = torch.tensor([3.0, 4.0])
    qx = torch.tensor([3.0, 3.0])
    assert utils.relerr(x, qx).item() == pytest.approx(1.0 / 5.0)
    assert utils.abserr(x, qx).item() == pytest.approx(0.5)
    assert utils.sqnr(x, qx).item() == pytest.approx(20 * np.log10(5.0), rel=1e-6)
    assert utils.compute_tensor_bytes([torch.zeros(10), torch.zeros(6, dtype=torch.int8),
                                       torch.zeros(4, dtype=torch.bfloat16)]) == 40 + 6 + 8
    assert utils.compute_tensor_bytes(torch.zeros(3, dtype=torch.float64)) == 0  # a type the reference does not list
    assert utils.get_rank() == 0 and utils.get_world_size() == 1
    assert utils.get_metric_fn("min")(1, 2) and utils.get_metric_fn("max")(2, 1)
    with pytest.raises(NotImplementedError):
        utils.get_metric_fn("median")


def test_every_shipped_configuration_merges_to_the_reference_settings():
    """The 13 files under lpmm/configs carry the reference's names; merged over the defaults each
    must give the settings of the reference's file of that name (lpmm/configs/*.yml there):
    (m enabled, m bits, m block size, v bits, v scale type)."""
    import lpmm
    from lpmm.config import get_config

    want = {
        "default.yml": (True, 4, 128, 4, "rank1"),
        "default_5b.yml": (True, 5, 128, 5, "rank1"),
        "default_6b.yml": (True, 6, 128, 6, "rank1"),
        "default_7b.yml": (True, 7, 128, 7, "rank1"),
        "default_8b.yml": (True, 8, 128, 8, "rank1"),
        "1st_moment_group_256.yml": (True, 4, 256, 4, "rank1"),
        "1st_moment_group_512.yml": (True, 4, 512, 4, "rank1"),
        "1st_moment_group_1024.yml": (True, 4, 1024, 4, "rank1"),
        "1st_moment_group_2048.yml": (True, 4, 2048, 4, "rank1"),
        "1st_moment_group_4096.yml": (True, 4, 4096, 4, "rank1"),
        "2nd_moment_group_128.yml": (True, 4, 128, 4, "group"),
        "2nd_moment_only_default.yml": (False, 4, 128, 4, "rank1"),
        "2nd_moment_only_group_128.yml": (False, 4, 128, 4, "group"),
    }
    cfg_dir = os.path.join(os.path.dirname(lpmm.config.__file__), "configs")
    assert sorted(os.listdir(cfg_dir)) == sorted(want)
    for name, (m_on, m_bits, m_gp, v_bits, v_scale) in want.items():
        q = get_config(os.path.join(cfg_dir, name)).QUANT
        got = (q.M.ENABLE, q.M.BITS, q.M.GROUP_SIZE, q.SQM.BITS, q.SQM.SCALE_TYPE.DEFAULT)
        assert got == (m_on, m_bits, m_gp, v_bits, v_scale), name
        # everything else stays at the defaults the two files share
        assert q.SQM.ENABLE is True and q.SQM.GROUP_SIZE == 128 and q.M.SCALE_TYPE.DEFAULT == "group"
        assert q.M.QUANT_TYPE.DEFAULT == "nonlinear" and q.SQM.QUANT_TYPE.DEFAULT == "power-1"
        assert q.M.ROUND_TYPE == "real-nearest" and q.SQM.ROUND_TYPE == "real-nearest"
        assert q.M.SIGNED is True and q.SQM.SIGNED is False and q.M.THRESHOLD == 4096


@pytest.mark.parametrize("shape", [(6, 40), (6, 5, 40), (2, 3, 5, 8)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("count", [-1, 0, 1])
def test_rank1_dequantise_takes_one_statistic_a_dimension(shape, bits, count, monkeypatch):
    """A rank-1 state with a statistic too few or too many, as a truncated or foreign state dictionary holds it, is refused before the
    library sees an address; the library is a stand-in that takes them."""
    from lpmm import _native, functional

    class Reached(Exception):
        pass

    class Lib:
        def lpmm_dequant_rank1_nd(self, codes, dims, shape, stats, *rest):
            assert dims == len(shape) == len(stats)
            raise Reached

    monkeypatch.setattr(functional, "_require_supported", lambda kwargs, x: None)
    monkeypatch.setattr(torch.cuda, "device", lambda index: torch.no_grad())
    monkeypatch.setattr(_native, "lib", Lib)
    monkeypatch.setattr(_native, "current_stream", lambda index: 0)
    stats = [torch.ones([d if i == k else 1 for k in range(len(shape))]) for i, d in enumerate(shape)]
    stats = stats[:-1] if count < 0 else stats + stats[:count]
    size = torch.Size(shape)
    kw = dict(qmap=torch.zeros(2 ** bits), b=bits, scale_type="rank1", quant_type="power-1", round_type="real-nearest", gp_sz=128, signed=False,
              dtype=torch.float32, stride=None, dim=len(shape), max1=None, max_dims=stats, scaled_shape=size, shape=size)
    with pytest.raises(ValueError, match="statistics do not belong") if count else pytest.raises(Reached):
        functional.vectorwise_dequant(torch.zeros(functional.packed_nbytes(size.numel(), bits), dtype=torch.int8), **kw)


@pytest.mark.parametrize("first,second", [((66, 33, 2, 2), (40, 132)), ((40, 132), (40, 200)), ((200, 40), (132, 132)), ((40, 132), (66, 33, 4)),
                                          ((66, 33, 2), (66, 34, 2)), ((66, 8, 8), (66, 64, 1))])
@pytest.mark.parametrize("half", [False, True])
def test_spare_statistics_of_a_parameter_that_changed_its_shape(first, second, half):
    """A parameter given another shape and a fresh state: what the kernels write the next statistics to, and the vectors between the
    passes, have the new sizes."""
    import lpmm
    from lpmm.optim.adamw import _Batch, _nd_pitch

    p = torch.nn.Parameter(torch.zeros(first, dtype=torch.float16 if half else torch.float32))
    opt = lpmm.optim.AdamW([p])
    for shape in (first, second, second):
        if half and len(shape) != 2:
            continue
        p.data = torch.zeros(shape, dtype=p.dtype)
        opt.state.clear()
        state, _ = opt._state_of(opt.param_groups[0], p)
        for step in range(2):
            batch = _Batch()
            (opt._rank1_state_f16 if half else opt._rank1_state if len(shape) == 2 else opt._rank1_nd_state)(p, state, batch)
            batch.launched()
            stats = state["exp_avg_sq_qstate"]["overhead"]["max_dims"]
            for pair in (stats, opt._spare_stats[p]):
                assert [t.numel() for t in pair] == list(shape) and all(t.dtype == p.dtype for t in pair)
        if len(shape) > 2:
            cols = p.numel() // shape[0]
            assert opt._nd_scratch_of(p, cols)["work"].shape == (3, _nd_pitch(cols)) and opt._nd_scratch_of(p, cols) is opt._nd_scratch[p]


HYPER = (0.9, 0.999, 1e-3, 0.01, 1e-8)


def _records(dtype, count, **values):
    """Records whose pointers are distinct addresses of a buffer that nothing reads; the buffer has to be kept."""
    memory = np.zeros(64 * 32 * count + 64, np.uint8)
    base = (memory.ctypes.data + 63) // 64 * 64
    records = np.zeros(count, dtype)
    for i in range(count):
        for j, name in enumerate(n for n in dtype.names if dtype[n] == np.dtype("<u8")):
            records[i][name] = base + 64 * (32 * i + j)
        for name, value in values.items():
            records[i][name] = value
    return records, memory, base


def _spoil(record, field, change):
    record[field] = {"null": 0, "shift": record[field] + 2, "shift4": record[field] + 4}.get(change, change) if not (
        isinstance(change, str) and change in record.dtype.names) else record[change]


# kind of the two-pass steps (LPMM_STEP_* of the header): its records, columns that it takes, columns that it refuses
STEPS = {0: ("NONFUSED_RANK1_TENSOR", (128, 64, 132, 1600), (130, 60, 12)), 1: ("NONFUSED_RANK1_TENSOR", (128, 132), (130, 60)),
         2: ("NONFUSED_RANK1_TENSOR", (128, 132), (130, 60)), 3: ("RANK1_V4BIT_TENSOR", (128, 132), (130, 60)),
         4: ("RANK1_MGROUP_TENSOR", (128, 8, 200), (12, 130)), 5: ("RANK1_MGROUP_TENSOR", (128, 132), (130, 8, 60)),
         8: ("RANK1_ANY_TENSOR", (128, 61), ()), 9: ("RANK1_ANY_TENSOR", (128, 61), ()), 10: ("RANK1_ANY_TENSOR", (128, 61), ())}


@pytest.mark.parametrize("kind", list(STEPS))
def test_errors_of_the_two_pass_steps_beside_float_states(kind):
    """lpmm_nonfused_rank1_fp32_step_multi: every record of either array is looked at before the first launch (which has a status of its
    own on a machine without a GPU)."""
    from lpmm import _native

    name, taken, refused = STEPS[kind]
    lib, dtype = _native.lib(), getattr(_native, name)
    bits = 8 if kind in (1, 10) else 4
    plain, keep_plain, base = _records(_native.ADAMW_FP32_TENSOR, 3, n=100, step=1.0)

    def call(records, count=None, plain=plain, plain_count=3, group=128, bits=(bits, bits), tables=(None, None), maps=(base, base), folds=None):
        folds = None if folds is None else folds.ctypes.data
        return lib.lpmm_nonfused_rank1_fp32_step_multi(
            kind, None if records is None else records.ctypes.data, folds, len(records) if count is None else count,
            None if plain is None else plain.ctypes.data, plain_count, group, maps[0], bits[0], tables[0], maps[1], bits[1], tables[1], *HYPER, None)

    def fresh(cols=taken[0]):
        records, *keep = _records(dtype, 40, rows=70, cols=cols, step=1.0)
        return records, (np.zeros(40, _native.RANK1_SMALL_VECTOR) if kind == 2 else None), keep  # ndim 0: matrices

    records, folds, keep = fresh()
    assert call(None, 3, folds=folds) == 1 and call(records, -1, folds=folds) == 3 and call(records, plain_count=-1, folds=folds) == 3
    assert call(records, plain=None, folds=folds) == 1
    assert call(records, bits=(9 if bits == 8 else 5, bits), folds=folds) == 5 and call(records, bits=(bits, 3), folds=folds) == 5
    assert call(records, tables=(base + 8, None), folds=folds) == 2 and call(records, tables=(None, base + 4), folds=folds) == 2
    assert call(records, group=192, folds=folds) == 3 and call(records, group=8192, folds=folds) == 3
    if kind not in (4, 5, 8):  # those take wide groups of the first moment
        assert call(records, group=256, folds=folds) == 3
    assert call(records, maps=(base, None), folds=folds) == 1 and call(records, maps=(base, base + 2), folds=folds) == 2
    if kind == 2:
        assert call(records) == 1  # without the vectors
    for field, change, status in (("p", "null", 1), ("n", -1, 3), ("g", "shift", 2), ("v", "null", 1)):
        bad = plain.copy()
        _spoil(bad[2], field, change)
        assert call(records, plain=bad, folds=folds) == status, field
    whole = kind < 8
    for field, change, status in (("p", "null", 1), ("g", "shift4" if whole else "shift", 2), ("v_codes", "shift", 2), ("v_rowmax", "null", 1),
                                  ("v_rowmax_next", "v_rowmax", 5), ("v_colmax_next", "v_colmax", 5), ("rows", -1, 3), ("cols", -1, 3),
                                  ("v_colmax", "shift4" if whole else "shift", 2), ("v_colmax_next", "shift4" if whole else "shift", 2)):
        for cols in taken:
            records, folds, keep = fresh(cols)
            _spoil(records[39], field, change)  # beyond what one launch takes
            assert call(records, folds=folds) == status, (field, cols)
    for cols in refused:
        records, folds, keep = fresh()
        records[39]["cols"] = cols
        assert call(records, folds=folds) == 3, cols


def test_errors_of_kinds_that_there_are_not():
    from lpmm import _native

    records, keep, base = _records(_native.RANK1_ANY_TENSOR, 1, rows=70, cols=61, step=1.0)
    for kind in (-1, 6, 7, 11, 12):  # 11: float16 has no such call
        assert _native.lib().lpmm_nonfused_rank1_fp32_step_multi(kind, records.ctypes.data, None, 1, None, 0, 128, base, 4, None, base, 4, None,
                                                                 *HYPER, None) == 5


def test_errors_of_the_steps_on_tensors_of_more_than_two_dimensions():
    """lpmm_nonfused_adamw4bit_rank1_nd_step_multi: a vector between the passes that is not its tensor's."""
    from lpmm import _native

    lib = _native.lib()
    records, keep, base = _records(_native.NONFUSED_RANK1_TENSOR, 40, rows=70, cols=9 * 128, step=1.0)
    folds, keep_folds, _ = _records(_native.RANK1_SMALL_VECTOR, 40, ndim=2)
    stats = np.zeros(4096, np.float32)
    scales = (stats.ctypes.data + 63) // 64 * 64
    folds["shape"][:, :2], folds["stats"][:, :2], folds["x"], folds["scale"] = (128, 9), scales + 4096, records["v_colmax_next"], scales

    def call(records=records, folds=folds, count=40):
        return lib.lpmm_nonfused_adamw4bit_rank1_nd_step_multi(None if records is None else records.ctypes.data,
                                                               None if folds is None else folds.ctypes.data, count, base, base, *HYPER, None)

    assert call(count=0) == 0 and call(None, None, 0) == 0 and call(count=-1) == 3 and call(None) == 1 and call(folds=None) == 1
    for field, value, status in (("x", scales + 1024, 5), ("x", 0, 1), ("scale", scales + 4, 2), ("scale", 0, 1), ("ndim", 8, 5), ("ndim", -1, 5)):
        bad = folds.copy()
        bad[39][field] = value
        assert call(folds=bad) == status, field
    for shape, status in (((128, 8), 3), ((0, 9), 3), ((8192, 9), 3)):
        bad = folds.copy()
        bad["shape"][39, :2] = shape
        assert call(folds=bad) == status, shape
    bad = folds.copy()
    bad["scale"][39] = bad["x"][39]  # in the place of what the second pass still needs
    assert call(folds=bad) == 5
    bad = folds.copy()
    bad["scale"][39] = records["v_colmax"][39]
    assert call(folds=bad) == 5
    bad = folds.copy()
    bad["stats"][39, 1] = 0
    assert call(folds=bad) == 1
    bad = records.copy()
    bad["v_codes"][39] = 0
    assert call(bad) == 1


@pytest.mark.parametrize("general", [0, 1])
@pytest.mark.parametrize("plain_fused", [0, 1])
def test_errors_of_the_factored_steps_beside_float_states(general, plain_fused):
    from lpmm import _native

    lib = _native.lib()
    plain, keep_plain, base = _records(_native.ADAMW_FP32_TENSOR, 3, n=100, step=1.0)
    records, keep, _ = _records(_native.FACTORED_TENSOR, 60, rows=70, cols=128, step=1.0)

    def call(records=records, count=60, plain=plain, plain_count=3, qmap=base):
        return lib.lpmm_factored_fp32_step_multi(None if records is None else records.ctypes.data, count, general,
                                                 None if plain is None else plain.ctypes.data, plain_count, plain_fused, qmap, *HYPER, None)

    assert call(count=-1) == 3 and call(plain_count=-1) == 3 and call(None) == 1 and call(plain=None) == 1 and call(qmap=None) == 1
    assert call(None, 0, None, 0) == 0  # nothing to do
    for field, change, status in (("m", "null", 1), ("n", -1, 3), ("g", "shift", 2)):
        bad = plain.copy()
        _spoil(bad[2], field, change)
        assert call(plain=bad) == status and call(None, 0, bad) == status, field
    for field, change, status in (("p", "null", 1), ("row", "shift", 2), ("workspace", "shift4", 2), ("rows", 0, 3), ("cols", -1, 3),
                                  ("col", "shift" if general else "shift4", 2)) + (() if general else (("cols", 136, 3), ("m_max1", "null", 1))):
        bad = records.copy()
        _spoil(bad[59], field, change)
        assert call(bad) == status, field


def test_errors_of_the_sgd_steps_beside_float_buffers():
    from lpmm import _native

    lib = _native.lib()
    plain, keep_plain, base = _records(_native.SGD_FP32_TENSOR, 70, n=100)
    records, keep, _ = _records(_native.SGD4BIT_TENSOR, 70, n=5000)

    def call(records=records, count=70, plain=plain, plain_count=70, qmap=base):
        return lib.lpmm_sgd4bit_fp32_step_multi(None if records is None else records.ctypes.data, count, None if plain is None else plain.ctypes.data,
                                                plain_count, qmap, 0.9, 0.0, 0.1, 0.0, 0, 0, None)

    assert call(count=-1) == 3 and call(plain_count=-1) == 3 and call(None) == 1 and call(plain=None) == 1 and call(qmap=None) == 1
    assert call(None, 0, None, 0, None) == 0  # nothing to do
    for field, change, status in (("buf", "null", 1), ("n", -1, 3), ("g", "shift", 2)):
        bad = plain.copy()
        _spoil(bad[69], field, change)
        assert call(plain=bad) == status and call(None, 0, bad) == status, field
    for field, change, status in (("m_codes", "null", 1), ("n", -1, 3), ("m_max1", "shift", 2)):
        bad = records.copy()
        _spoil(bad[69], field, change)
        assert call(bad) == status and call(bad, plain=None, plain_count=0) == status, field


@pytest.mark.parametrize("shape", [(12, 40), (3, 4, 40), (3, 5, 2, 7)])
@pytest.mark.parametrize("bits", [4, 2, 8])
@pytest.mark.parametrize("back", [False, True])
def test_errors_of_whole_rank1_quantisations(shape, bits, back):
    """lpmm_quant_rank1_nd and lpmm_dequant_rank1_nd are several calls to the device: what the last would refuse is refused before the
    first (whose status is another on a machine without a GPU)."""
    from lpmm import _native

    lib, memory = _native.lib(), np.zeros(4096, np.uint8)  # never read: only the addresses count
    base = (memory.ctypes.data + 63) // 64 * 64
    stats = [base + 64 * i for i in range(len(shape))]
    fine = dict(values=base + 512, shape=shape, dims=len(shape), stats=stats, work=base + 1024 if len(shape) > 2 else None, qmap=base + 1536, bits=bits,
                table=None, codes=base + 2048)

    def call(**kw):
        a = {**fine, **kw}
        sizes = None if a["shape"] is None else (ctypes.c_int64 * len(a["shape"]))(*a["shape"])
        pointers = None if a["stats"] is None else (ctypes.c_void_p * len(a["stats"]))(*a["stats"])
        if back:
            return lib.lpmm_dequant_rank1_nd(a["codes"], a["dims"], sizes, pointers, a["work"], a["qmap"], a["bits"], a["values"], None)
        return lib.lpmm_quant_rank1_nd(a["values"], a["dims"], sizes, pointers, a["work"], a["qmap"], a["bits"], a["table"], a["codes"], None)

    assert call(dims=1) == 5 and call(dims=9) == 5
    for name in ("values", "shape", "stats", "qmap", "codes") + (("work",) if len(shape) > 2 else ()):
        assert call(**{name: None}) == 1, name
    for name in ("values", "qmap") + (("work",) if len(shape) > 2 else ()):
        assert call(**{name: fine[name] + 2}) == 2, name
    for i in range(len(shape)):
        assert call(stats=stats[:i] + [None] + stats[i + 1:]) == 1 and call(stats=stats[:i] + [stats[i] + 1] + stats[i + 1:]) == 2
        assert call(shape=shape[:i] + (0,) + shape[i + 1:]) == 3 and call(shape=shape[:i] + (-4,) + shape[i + 1:]) == 3
    assert call(shape=(1 << 40,) * len(shape)) == 3
    assert call(bits=0) == 3 and call(bits=9) == 3
    if bits != 4:
        assert call(codes=fine["codes"] + 4) == 2
        assert back or call(table=base + 8) == 2
    elif not back:
        assert call(codes=fine["codes"] + 2) == 2
