// Prints what the library would launch, on a machine without a GPU: this program's own launch functions stand before the HIP
// runtime's and record the grids.  The arguments' addresses are made up and never read.  One line of standard input is one call,
//   stats ROWS COLS                     lpmm_rank1_stats
//   quant BITS ROWS COLS                lpmm_quant_rank1 (4 bits) or lpmm_quant_rank1_bits
//   dequant BITS ROWS COLS              the way back
//   rank1 MODE ROWS COLS [ROWS COLS]... one step on these matrices; MODE: codes4, float_m (fp32 first moment), codes8 or
//                                       half (float16)
//   beside MODE ROWS COLS [ROWS COLS]...  the same but for half, by the entry point for steps beside tensors with fp32 states (of which
//                                       there are none); groups as well (first moment in groups of 256 values)
//   any ROWS COLS [ROWS COLS]...        one step with 4-bit codes by the kernels for any column count
// and one line of output its status and the grids, "x,y" each.
// Build: g++ -O1 -rdynamic -D__HIP_PLATFORM_AMD__ -I<rocm>/include -I<include> launches.cpp -llpmm_hip
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "lpmm_hip.h"

static std::vector<dim3> launches;
static dim3 next_grid, next_block;

extern "C" hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t)
{
    next_grid = grid;
    next_block = block;
    return hipSuccess;
}

extern "C" hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
    *grid = next_grid;
    *block = next_block;
    *shared = 0;
    *stream = nullptr;
    return hipSuccess;
}

extern "C" hipError_t hipLaunchKernel(const void *, dim3 grid, dim3, void **, size_t, hipStream_t)
{
    launches.push_back(grid);
    return hipSuccess;
}

extern "C" hipError_t hipGetLastError() { return hipSuccess; }

// distinct addresses on a 256-byte boundary
static char *made_up()
{
    static uintptr_t at = 1u << 20;
    return reinterpret_cast<char *>(at += uintptr_t(1) << 30);
}

static int rank1(const std::string &mode, const std::vector<std::pair<int64_t, int64_t>> &shapes, bool beside = false)
{
    std::vector<lpmm_nonfused_rank1_tensor> coded;
    std::vector<lpmm_rank1_v4bit_tensor> plain;
    std::vector<lpmm_nonfused_rank1_f16_tensor> halfs;
    std::vector<lpmm_rank1_mgroup_tensor> groups;
    for (const auto &[rows, cols] : shapes) {
        lpmm_nonfused_rank1_tensor t;
        lpmm_rank1_v4bit_tensor f;
        memset(&t, 0, sizeof t);
        memset(&f, 0, sizeof f);
        f.p = t.p = (float *)made_up();
        f.g = t.g = (const float *)made_up();
        t.m_codes = (uint8_t *)made_up();
        f.m = (float *)made_up();
        t.m_max1 = (float *)made_up();
        f.v_codes = t.v_codes = (uint8_t *)made_up();
        f.v_rowmax = t.v_rowmax = (const float *)made_up();
        f.v_colmax = t.v_colmax = (const float *)made_up();
        f.v_rowmax_next = t.v_rowmax_next = (float *)made_up();
        f.v_colmax_next = t.v_colmax_next = (float *)made_up();
        f.rows = t.rows = rows;
        f.cols = t.cols = cols;
        f.step = t.step = 1.0f;
        coded.push_back(t);
        plain.push_back(f);
        groups.push_back({t.p, t.g, t.m_codes, t.m_max1, (float *)made_up(), t.v_codes, t.v_rowmax, t.v_colmax, t.v_rowmax_next,
                          t.v_colmax_next, rows, cols, 1.0f, 0.0f});
        halfs.push_back({t.p, t.g, t.m_codes, t.m_max1, t.v_codes, t.v_rowmax, t.v_colmax, t.v_rowmax_next, t.v_colmax_next,
                         (float *)made_up(), rows, cols, 1.0f, 0.0f});
    }
    const float *map = (const float *)made_up();
    const int64_t n = (int64_t)shapes.size();
    if (beside) {
        const int kind = mode == "codes4" ? LPMM_STEP_MATRIX : mode == "codes8" ? LPMM_STEP_BITS : mode == "float_m" ? LPMM_STEP_FLOAT_M : LPMM_STEP_GROUPS_WRAP;
        const void *records = mode == "float_m" ? (const void *)plain.data() : mode == "groups" ? (const void *)groups.data() : coded.data();
        const int bits = mode == "codes8" ? 8 : 4;
        return lpmm_nonfused_rank1_fp32_step_multi(kind, records, nullptr, n, nullptr, 0, mode == "groups" ? 256 : 128, map, bits, nullptr, map,
                                                   bits, nullptr, 0.9, 0.999, 1e-3, 0.01, 1e-8, nullptr);
    }
    if (mode == "float_m")
        return lpmm_nonfused_adamw_v4bit_rank1_step_multi(plain.data(), n, map, 0.9, 0.999, 1e-3, 0.01, 1e-8, nullptr);
    if (mode == "half")
        return lpmm_nonfused_adamw4bit_rank1_f16_step_multi(halfs.data(), n, map, map, 0.9, 0.999, 1e-3, 0.01, 1e-8, nullptr);
    if (mode == "codes8")
        return lpmm_nonfused_adamw_bits_rank1_step_multi(coded.data(), n, map, 8, map, 8, 0.9, 0.999, 1e-3, 0.01, 1e-8, nullptr);
    return lpmm_nonfused_adamw4bit_rank1_step_multi(coded.data(), n, map, map, 0.9, 0.999, 1e-3, 0.01, 1e-8, nullptr);
}

static int any_columns(const std::vector<std::pair<int64_t, int64_t>> &shapes)
{
    std::vector<lpmm_rank1_any_tensor> records;
    for (const auto &[rows, cols] : shapes) {
        lpmm_rank1_any_tensor t;
        memset(&t, 0, sizeof t);
        t.p = made_up();
        t.g = made_up();
        t.m = made_up();
        t.m_codes_next = (uint8_t *)made_up();
        t.m_max1 = made_up();
        t.m_max1_next = made_up();
        t.v_codes = (const uint8_t *)made_up();
        t.v_codes_next = (uint8_t *)made_up();
        t.v_rowmax = made_up();
        t.v_colmax = made_up();
        t.v_rowmax_next = made_up();
        t.v_colmax_next = made_up();
        t.rows = rows;
        t.cols = cols;
        t.step = 1.0f;
        records.push_back(t);
    }
    const float *map = (const float *)made_up();
    return lpmm_nonfused_adamw_rank1_any_step_multi(records.data(), (int64_t)records.size(), LPMM_RANK1_CODES4, 128, map, 4, nullptr, map, 4,
                                                    nullptr, 0.9, 0.999, 1e-3, 0.01, 1e-8, 3, nullptr);
}

static int quantiser(bool back, int bits, int64_t rows, int64_t cols)
{
    const float *x = (const float *)made_up(), *rowmax = (const float *)made_up(), *colmax = (const float *)made_up();
    const float *map = (const float *)made_up();
    uint8_t *codes = (uint8_t *)made_up();
    if (back)
        return bits == 4 ? lpmm_dequant_rank1(codes, rowmax, colmax, map, rows, cols, const_cast<float *>(x), nullptr)
                         : lpmm_dequant_rank1_bits(codes, rowmax, colmax, map, bits, rows, cols, const_cast<float *>(x), nullptr);
    return bits == 4 ? lpmm_quant_rank1(x, rows, cols, rowmax, colmax, map, codes, nullptr)
                     : lpmm_quant_rank1_bits(x, rows, cols, rowmax, colmax, map, bits, codes, nullptr);
}

int main()
{
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string call, mode;
        std::vector<std::pair<int64_t, int64_t>> shapes;
        int64_t rows, cols;
        in >> call;
        if (call != "stats" && call != "any")
            in >> mode;
        while (in >> rows >> cols)
            shapes.push_back({rows, cols});
        launches.clear();
        const auto &[r, c] = shapes.at(0);
        const int status = call == "stats"   ? lpmm_rank1_stats((const float *)made_up(), r, c, (float *)made_up(), (float *)made_up(),
                                                                nullptr)
                           : call == "rank1" ? rank1(mode, shapes)
                           : call == "beside" ? rank1(mode, shapes, true)
                           : call == "any"   ? any_columns(shapes)
                                             : quantiser(call == "dequant", std::stoi(mode), r, c);
        printf("%d", status);
        for (const dim3 &grid : launches)
            printf(" %u,%u", grid.x, grid.y);
        printf("\n");
    }
    return 0;
}
