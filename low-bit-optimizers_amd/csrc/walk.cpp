// The host side of a step on a model whose optimizer states exist: one walk over a parameter group's tensors
// that writes the records of the multi-tensor launches.  In Python the same walk is dozens of attribute and
// dictionary reads a tensor -- 3 to 15 us a tensor, against 0.15 here, while the kernels take 1 us for a tensor of a
// million values -- and bound every model of small tensors: fifty tensors of a few thousand to a million values
// 186 -> 43 us a step, the 203 of a wide ResNet-152 1634 -> 1054, GPT-2-XL's 580 1.8 -> 0.23 ms of host time.
// What counts here is dictionary reads: names compared by address (read), a parameter's hash without its call into Python
// (hash_of), one allocation for a launch's scratch (prepare): 52 tensors 10.3 -> 7.2 us, and with fewer attribute reads in Python
// their fused step 31.8 -> 25.1 us, 576 tensors of width 64 on the two-pass route 277 -> 209, 18 float16 matrices 70 -> 49.
// lpmm/optim/adamw.py and sgd.py keep that walk for what is not served here: first steps, other data types,
// strided operands, other routes; and for every error.
//
// collect() decides for each tensor, from the tensor and its state alone and anew on every step, whether it is
// served, and reads its pointers; no state changes.  Plan.start() advances the step counts, Plan.prepare()
// allocates what a launch's records need; after it is on the stream, Plan.commit() lets the states point to their new
// statistics (and, on the kernels for any column count, codes).  A Plan lives for one step.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstddef>
#include <cstring>
#include <memory>
#include <vector>

#include "lpmm_hip.h"

namespace {

enum Kind : int { kFused4, kPlain, kFlat, kRank1, kNd, kFlatM32, kRank1M32, kRank1Bits, kRank1Wide, kSgd4, kSgdPlain,
                  kAny, kNdAny, kHalfPlain, kHalfFlat, kHalfRank1, kFactored, kFactoredAny, kKinds };

constexpr size_t kRecordBytes[kKinds] = {
    sizeof(lpmm_adamw4bit_tensor),     sizeof(lpmm_adamw_fp32_tensor),     sizeof(lpmm_adamw4bit_tensor),
    sizeof(lpmm_nonfused_rank1_tensor), sizeof(lpmm_nonfused_rank1_tensor), sizeof(lpmm_adamw_v4bit_tensor),
    sizeof(lpmm_rank1_v4bit_tensor),   sizeof(lpmm_nonfused_rank1_tensor), sizeof(lpmm_rank1_mgroup_tensor),
    sizeof(lpmm_sgd4bit_tensor),       sizeof(lpmm_sgd_fp32_tensor),       sizeof(lpmm_rank1_any_tensor),
    sizeof(lpmm_rank1_any_tensor),     sizeof(lpmm_adamw_fp32_tensor),     sizeof(lpmm_adamw4bit_f16_tensor),
    sizeof(lpmm_nonfused_rank1_f16_tensor), sizeof(lpmm_factored_tensor), sizeof(lpmm_factored_tensor)};

struct Names {
    PyObject *step, *exp_avg, *exp_avg_sq, *exp_avg_qstate, *exp_avg_sq_qstate, *exp_avg_sq_row, *exp_avg_sq_col, *enable, *overhead, *qmap, *max1,
        *max_dims, *work, *scale_of, *row, *momentum_buffer, *momentum_buffer_qstate, *dtype;
} N;

// dict[key] = value, once the launch is on the stream; strong references.  hash: of a key that is a parameter, else -1
struct Swap {
    PyObject *dict, *key, *value;
    Py_hash_t hash = -1;
};

// memory of a record, allocated when its launch is next (prepare): n floats of this step's scratch, or the array that
// becomes the state which swap number `swap` replaces
struct Need {
    size_t at;  // of the pointer in the record
    int64_t n;
    int swap;
    at::Tensor like;
};

// a record in the making
struct Item {
    PyObject *step = nullptr;
    const at::Tensor *grad = nullptr;
    size_t held = 0;  // its objects in the plan's begin here
    Swap swap[9];
    int swaps = 0, needs = 0;
    Need need[3];
};

// what belongs to a record: ranges of the plan's and the batch's lists
struct Record {
    float *step;
    at::Tensor grad, scratch;
    uint32_t held, held_end, swaps, swaps_end, needs, needs_end;
};

struct Batch {
    Kind kind;
    int device, flag;  // flag: kRank1Wide: ragged rows; kAny: the kind of its entry point; plan_start: kPlain
    PyObject *qm, *qv;  // the maps' tensors (borrowed from held references)
    std::vector<uint8_t> records, second;
    std::vector<lpmm_rank1_small_vector> fold;
    std::vector<Record> items;
    std::vector<Swap> swaps;
    std::vector<Need> needs;
    bool wraps = false;  // kRank1, kRank1M32, kRank1Bits, kRank1Wide: a tensor that the kernels take as rows of several of its own
};

struct Plan {
    PyObject_HEAD
    std::vector<Batch> *batches;
    // what the records point into (parameters, step counts, states), until their launch is on the stream:
    // between collect() and then runs the loop over the other tensors, and with it code of the caller's (a gradient that is a
    // property), which may drop gradients or states.  References of the Python objects: with copies of the tensors instead,
    // counted atomically, 580 tensors took 60 us more a step.
    std::vector<PyObject *> *held;
    std::vector<PyObject *> *others;  // the maps, and objects made for the swaps: until the step is over
    PyObject *rest;
};

// a Python object that is a tensor (borrowed), or none
struct Ref {
    PyObject *o = nullptr;

    Ref() = default;
    Ref(std::nullptr_t) {}
    explicit Ref(PyObject *tensor) : o(tensor) {}
    const at::Tensor &operator*() const { return THPVariable_Unpack(o); }
    const at::Tensor *operator->() const { return &THPVariable_Unpack(o); }
    bool operator==(std::nullptr_t) const { return o == nullptr; }
    bool operator!=(std::nullptr_t) const { return o != nullptr; }
};

Ref tensor_of(PyObject *o) { return o != nullptr && THPVariable_Check(o) ? Ref(o) : Ref(); }

PyObject *get(PyObject *dict, PyObject *key)  // borrowed; null where absent (a Python error stays set)
{
    return dict != nullptr && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, key) : nullptr;
}

// Values of `count` names in a dictionary of a few entries (borrowed; null where absent): one pass over the entries, whose keys are
// as a rule these very strings.  Only a dictionary that holds other keys as well, or equal strings that are other objects (from a
// file), is searched name by name.
template <int COUNT>
void read(PyObject *dict, PyObject *const (&names)[COUNT], PyObject *(&values)[COUNT])
{
    for (int i = 0; i < COUNT; ++i)
        values[i] = nullptr;
    if (dict == nullptr || !PyDict_Check(dict))
        return;
    PyObject *key, *value;
    Py_ssize_t at = 0, found = 0;
    while (PyDict_Next(dict, &at, &key, &value))
        for (int i = 0; i < COUNT; ++i)
            if (key == names[i]) {
                values[i] = value;
                ++found;
                break;
            }
    if (found != PyDict_GET_SIZE(dict))
        for (int i = 0; i < COUNT; ++i)
            if (values[i] == nullptr)
                values[i] = PyDict_GetItemWithError(dict, names[i]);
}

// A tensor's hash, its id: torch computes it in Python, 0.1 us a time.  (Were it another one, no state would be found with this and
// every tensor would go to the loops in Python.)
Py_hash_t hash_of(PyObject *tensor)
{
    const Py_hash_t id = (Py_hash_t)(uintptr_t)tensor;
    return id == -1 ? -2 : id;
}
// The dictionary calls that take a hash are private to the interpreter from Python 3.13 on, which gets the public ones.
PyObject *of_parameter(PyObject *dict, PyObject *p)  // dict[p]; borrowed, or null
{
    if (dict == nullptr || !PyDict_Check(dict))
        return nullptr;
#if PY_VERSION_HEX < 0x030d0000
    return _PyDict_GetItem_KnownHash(dict, p, hash_of(p));
#else
    return PyDict_GetItemWithError(dict, p);
#endif
}
int set_item(const Swap &swap)  // dict[key] = value
{
#if PY_VERSION_HEX < 0x030d0000
    if (swap.hash != -1)
        return _PyDict_SetItem_KnownHash(swap.dict, swap.key, swap.value, swap.hash);
#endif
    return PyDict_SetItem(swap.dict, swap.key, swap.value);
}

// the settings of a state, state[name + "_qstate"]
struct QState {
    PyObject *enable, *overhead, *qmap;

    explicit QState(PyObject *qstate)
    {
        PyObject *const names[] = {N.enable, N.overhead, N.qmap};
        PyObject *of[3];
        read(qstate, names, of);
        enable = of[0];
        overhead = of[1];
        qmap = of[2];
    }
};

bool on_gpu(const at::Tensor &t)
{
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided &&
           !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) && t.is_contiguous();
}

bool floats(const at::Tensor &t) { return on_gpu(t) && t.scalar_type() == at::kFloat; }
bool halfs(const at::Tensor &t) { return on_gpu(t) && t.scalar_type() == at::kHalf; }

template <typename T = void>
T *ptr(const at::Tensor &t)
{
    return static_cast<T *>(t.unsafeGetTensorImpl()->mutable_data());
}

// Bytes of a state's codes as the kernels write them: whole groups, rounded up to pack groups, and one more
// (lpmm/functional.py: packed_nbytes).  The fused operators alone ask for no more than the values.
int64_t packed(int64_t n, int64_t group, bool bytes)
{
    const int64_t scaled = (n + group - 1) / group * group;
    const int64_t all = (scaled + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP;
    return (bytes ? all : all / 2) + 1;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Does a matrix gain as rows of 2^lg tensor rows (Fold, rank1_tiles.hpp), which are as many times wider?  The kernels take tiles of 16 such
// rows and 256 columns: with fewer rows there are up to 32 times as many tiles, and 5.5 ns each, mostly empty.  So it has 16, or at
// most 512 tiles side by side, which cost less than the host saves.  Steps by the kernels for any column count -> as such rows, us:
// one of 1 x 1000004 72 -> 701, of 31 x 50004 35 -> 88, of 64 x 50008 32 -> 82; sixteen of 256 x 20004 (8 rows) 384 -> 457, of
// 512 x 20004 (16) 745 -> 676; of 64 x 5004 (626 tiles side by side) 74 -> 94, of 64 x 5008 (313) 42 -> 41, of 64 x 1004 (126) 76 -> 35.
bool worth_folding(int64_t rows, int64_t cols)
{
    int lg = 0;
    while ((cols << lg) % 128 != 0)
        ++lg;
    return rows >= (int64_t)16 << lg || (cols << lg) / 128 <= 1024;
}

struct Settings {
    int fused;  // 0: the non-fused path, 1: the fused operators, 2: settings the fused operators warn about or refuse
    int m_group128, v_group128, v_rank1, m_wide, bits_rank1;
    int64_t m_group;  // values per group of the first moment's scales; 0: scaled in a way that is not served here
};

struct Walk {
    Plan *plan;
    PyObject *state, *override_, *spare_stats, *spare_scales, *nd_scratch, *in_place;
    Settings s;
    size_t most;  // records of a batch: the group's tensors, fewer at first where they are many
    int64_t (*workspace_bytes)(int64_t, int64_t);  // lpmm_factored_workspace_bytes

    // a dense tensor of n values beside p and of its type (parameters on the kernels are float or half)
    static Ref reals_of(PyObject *o, const at::Tensor &p, int64_t n)
    {
        const Ref t = tensor_of(o);
        return t != nullptr && on_gpu(*t) && t->scalar_type() == p.scalar_type() && t->numel() == n && t->get_device() == p.get_device() ? t : nullptr;
    }
    // a state of p's values; a single value: not created yet
    static Ref reals_like(PyObject *o, const at::Tensor &p) { return p.numel() > 1 ? reals_of(o, p, p.numel()) : nullptr; }
    // a state's codes, at least `bytes` of them
    static Ref codes(PyObject *o, const at::Tensor &p, int64_t bytes)
    {
        const Ref t = tensor_of(o);
        return t != nullptr && t->numel() > 1 && t->numel() >= bytes && on_gpu(*t) && t->scalar_type() == at::kChar &&
                       t->get_device() == p.get_device()
                   ? t
                   : nullptr;
    }
    // the scales of `groups` groups
    static Ref scales(PyObject *overhead, const at::Tensor &p, int64_t groups) { return reals_of(get(overhead, N.max1), p, groups); }
    // one tensor per dimension
    template <typename T>
    bool statistics(PyObject *list, const at::Tensor &p, T **out)
    {
        if (list == nullptr || !PyList_Check(list) || PyList_GET_SIZE(list) != p.dim())
            return false;
        for (Py_ssize_t i = 0; i < p.dim(); ++i) {
            const Ref t = reals_of(PyList_GET_ITEM(list, i), p, p.size(i));
            if (t == nullptr)
                return false;
            out[i] = use<T>(t);
        }
        return true;
    }

    Batch &batch(Kind kind, const at::Tensor &p, PyObject *qm, PyObject *qv, int flag = 0)
    {
        const int device = p.get_device();
        for (Batch &b : *plan->batches)
            if (b.kind == kind && b.device == device && b.qm == qm && b.qv == qv && b.flag == flag)
                return b;
        plan->batches->push_back(Batch{kind, device, flag, qm, qv, {}, {}, {}, {}, {}, {}});
        plan->batches->back().records.reserve(most * kRecordBytes[kind]);
        plan->batches->back().items.reserve(most);
        for (PyObject *map : {qm, qv})
            if (map != nullptr) {
                Py_INCREF(map);
                plan->others->push_back(map);
            }
        return plan->batches->back();
    }
    void keep(PyObject *o)
    {
        Py_INCREF(o);
        plan->held->push_back(o);
    }
    template <typename R>
    static void append(std::vector<uint8_t> &to, const R &record)
    {
        const uint8_t *r = reinterpret_cast<const uint8_t *>(&record);
        to.insert(to.end(), r, r + sizeof(R));
    }
    template <typename R>
    void add(Batch &b, const R &record, Item &item)
    {
        append(b.records, record);
        const uint32_t swaps = (uint32_t)b.swaps.size(), needs = (uint32_t)b.needs.size();
        for (int i = 0; i < item.needs; ++i) {
            item.need[i].swap += item.need[i].swap >= 0 ? (int)swaps : 0;
            b.needs.push_back(std::move(item.need[i]));
        }
        for (int i = 0; i < item.swaps; ++i) {
            Py_INCREF(item.swap[i].dict);
            Py_INCREF(item.swap[i].key);
            Py_XINCREF(item.swap[i].value);
            b.swaps.push_back(item.swap[i]);
        }
        b.items.push_back(Record{item.step != nullptr ? ptr<float>(THPVariable_Unpack(item.step)) : nullptr, *item.grad, at::Tensor(),
                                 (uint32_t)item.held, (uint32_t)plan->held->size(), swaps, (uint32_t)b.swaps.size(), needs,
                                 (uint32_t)b.needs.size()});
    }
    // the data of a tensor that the plan holds from here on
    template <typename T = void>
    T *use(const Ref &t)
    {
        keep(t.o);
        return ptr<T>(*t);
    }
    // an item for a parameter with its gradient; step: its count, or null
    Item item_of(PyObject *po, const at::Tensor &g, const Ref &step)
    {
        Item item;
        item.held = plan->held->size();
        item.grad = &g;
        keep(po);
        if (step != nullptr)
            keep(item.step = step.o);
        return item;
    }

    int enabled(PyObject *p, PyObject *e)  // e: of the state's settings; -1: not decided here
    {
        if (override_ != nullptr && PyDict_GET_SIZE(override_) != 0) {
            PyObject *id = PyLong_FromVoidPtr(p);
            if (id == nullptr)
                return -1;
            PyObject *o = PyDict_GetItemWithError(override_, id);
            Py_DECREF(id);
            if (o != nullptr)
                return PyObject_IsTrue(o);
        }
        return e != nullptr ? PyObject_IsTrue(e) : -1;
    }

    // where a state's new codes go: a tensor that becomes the state (st[name])
    static void next_codes(Item &item, size_t at, PyObject *st, PyObject *name, const at::Tensor &codes)
    {
        item.need[item.needs++] = Need{at, 0, item.swaps, codes};
        item.swap[item.swaps++] = Swap{st, name, nullptr, -1};
    }
    static void scratch(Item &item, size_t at, int64_t n) { item.need[item.needs++] = Need{at, n, -1, at::Tensor()}; }

    bool adamw(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st);
    bool factored(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, const Ref &step, PyObject *mo,
                  PyObject *row_of, const QState &m_of);
    bool half(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, Item &item, PyObject *mo, PyObject *vo,
              const QState &m_of, const QState &v_of, int en_m, int en_v);
    bool any(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, Item &item, int kind, const Ref &mc,
             const Ref &ms, const Ref &vc, PyObject *oh_m, PyObject *oh_v, PyObject *qm, PyObject *qv);
    bool nd(PyObject *po, const at::Tensor &p, Item &item, lpmm_nonfused_rank1_tensor &r, PyObject *st, Ref any_mc, bool may_wrap,
            PyObject *oh_m, const Ref &vc, PyObject *oh_v, PyObject *qm, PyObject *qv);
    bool sgd(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st);
};

void swap_later(Item &item, PyObject *dict, PyObject *key, PyObject *value, Py_hash_t hash = -1)
{
    item.swap[item.swaps++] = Swap{dict, key, value, hash};
}

// true: a record was added.  Every return before that leaves the plan as it was.
bool Walk::adamw(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st)
{
    if (!g.defined() || !on_gpu(p) || !on_gpu(g) || p.device() != g.device() || p.numel() != g.numel() ||
        g.scalar_type() != p.scalar_type())
        return false;
    PyObject *const names[] = {N.step, N.exp_avg, N.exp_avg_qstate, N.exp_avg_sq, N.exp_avg_sq_qstate, N.exp_avg_sq_row};
    PyObject *state_of[6];
    read(st, names, state_of);
    const Ref step = tensor_of(state_of[0]);
    if (step == nullptr || !step->is_cpu() || step->scalar_type() != at::kFloat || step->dim() != 0)
        return false;
    const bool is_factored = state_of[5] != nullptr;
    if (floats(p) ? !is_factored && s.fused == 2 : !halfs(p) || s.fused || is_factored)
        return false;
    PyObject *const mo = state_of[1], *const vo = state_of[3];
    const QState m_of(state_of[2]), v_of(state_of[4]);
    if (is_factored)
        return factored(po, p, g, st, step, mo, state_of[5], m_of);
    const int en_m = enabled(po, m_of.enable), en_v = enabled(po, v_of.enable);
    if (en_m < 0 || en_v < 0)
        return false;
    Item item = item_of(po, g, step);
    if (!floats(p))
        return half(po, p, g, st, item, mo, vo, m_of, v_of, en_m, en_v);
    const int64_t n = p.numel();
    if (!en_m && !en_v) {
        const Ref m = reals_like(mo, p), v = reals_like(vo, p);
        if (m == nullptr || v == nullptr)
            return false;
        lpmm_adamw_fp32_tensor r = {ptr<float>(p), ptr<float>(g), use<float>(m), use<float>(v), n, 0.0f, 0.0f};
        add(batch(kPlain, p, nullptr, nullptr), r, item);
        return true;
    }
    PyObject *const qm = m_of.qmap, *const qv = v_of.qmap;
    const Ref map_m = tensor_of(qm), map_v = tensor_of(qv);
    const Ref vc = codes(vo, p, s.fused ? (n + 1) / 2 : packed(n, 128, s.bits_rank1));
    if (map_m == nullptr || map_v == nullptr || !floats(*map_m) || !floats(*map_v) || vc == nullptr || !en_v)
        return false;
    PyObject *const oh_m = m_of.overhead, *const oh_v = v_of.overhead;
    if (s.fused || s.v_group128 || (s.v_rank1 && p.dim() == 1)) {
        const Ref vs = scales(oh_v, p, (n + 127) / 128);
        if (vs == nullptr)
            return false;
        if (!en_m) {
            const Ref m = reals_like(mo, p);
            if (s.fused || m == nullptr)
                return false;
            lpmm_adamw_v4bit_tensor r = {ptr<float>(p), ptr<float>(g), use<float>(m), use<uint8_t>(vc), use<float>(vs), n, 0.0f, 0.0f};
            add(batch(kFlatM32, p, nullptr, qv), r, item);
            return true;
        }
        const Ref mc = codes(mo, p, s.fused ? (n + 1) / 2 : packed(n, 128, false)), ms = scales(oh_m, p, (n + 127) / 128);
        if (!(s.fused ? n % 2 == 0 : s.m_group128 != 0) || mc == nullptr || ms == nullptr)
            return false;
        lpmm_adamw4bit_tensor r;
        memset(&r, 0, sizeof r);
        r.p = ptr<float>(p);
        r.g = ptr<float>(g);
        r.m_codes = use<uint8_t>(mc);
        r.v_codes = use<uint8_t>(vc);
        r.m_scale = use<float>(ms);
        r.v_scale = use<float>(vs);
        r.n = n;
        add(batch(s.fused ? kFused4 : kFlat, p, qm, qv), r, item);
        return true;
    }
    PyObject *cur = get(oh_v, N.max_dims);
    if (!(s.v_rank1 || s.bits_rank1) || cur == nullptr || p.dim() < 2 || p.size(0) == 0)
        return false;
    lpmm_nonfused_rank1_tensor r;
    memset(&r, 0, sizeof r);
    r.p = ptr<float>(p);
    r.g = ptr<float>(g);
    r.v_codes = use<uint8_t>(vc);
    r.rows = p.size(0);
    r.cols = n / r.rows;
    Ref mc, ms;
    if (en_m) {
        if (s.m_group <= 0)
            return false;
        mc = codes(mo, p, packed(n, s.m_group, s.bits_rank1));
        ms = scales(oh_m, p, (n + s.m_group - 1) / s.m_group);
        if (mc == nullptr || ms == nullptr)
            return false;
        r.m_codes = use<uint8_t>(mc);
        r.m_max1 = use<float>(ms);
    }
    // the kernels that take 16 bytes an access; other operands go to the kernels for any column count
    const bool aligned = aligned16(r.p) && aligned16(r.g);
    const bool whole = aligned && r.cols % 128 == 0, folds = en_m && s.m_group128 && aligned && r.cols % 128 == 64 && r.rows % 2 == 0;
    // Rows of several tensor rows (Fold, rank1_tiles.hpp; the entry points that take them are those beside fp32 states and folds), in
    // place.  A state's first step here still goes the way of the steps in Python, whose kernels leave new scales, and of some columns
    // new codes, in arrays of their own.  in_place says for which state that is done: the second moment's overhead.
    const Ref m32 = en_m ? Ref() : reals_like(mo, p);
    const bool may_wrap = (en_m ? s.m_group128 || s.bits_rank1 || s.m_wide : m32 != nullptr && aligned16(ptr(*m32))) &&
                          (s.v_rank1 || s.bits_rank1) && aligned && !whole && !folds && r.cols % 4 == 0 &&
                          (r.cols >= 128 || r.cols == 64) && r.cols <= (1 << 24) && worth_folding(r.rows, r.cols);
    const auto wraps_next = [&] {
        if (may_wrap)
            swap_later(item, in_place, po, oh_v, hash_of(po));
    };
    const bool served = r.cols >= 32 || r.rows <= 32768;  // _any_columns
    if (p.dim() > 2)
        return en_m && s.m_group128 && s.v_rank1 && served &&
               nd(po, p, item, r, st, whole || folds ? Ref() : mc, may_wrap, oh_m, vc, oh_v, qm, qv);
    PyObject *nxt = of_parameter(spare_stats, po);
    float *now[2], *next[2];
    if (!statistics(cur, p, now) || !statistics(nxt, p, next))
        return false;
    r.v_rowmax = now[0];
    r.v_colmax = now[1];
    r.v_rowmax_next = next[0];
    r.v_colmax_next = next[1];
    // (their entry points take column statistics at 16 bytes, those for any column count at any float)
    const bool wraps = may_wrap && of_parameter(in_place, po) == oh_v && aligned16(r.v_colmax) && aligned16(r.v_colmax_next);
    swap_later(item, spare_stats, po, cur, hash_of(po));
    swap_later(item, oh_v, N.max_dims, nxt);
    if (!en_m) {
        const Ref &m = m32;
        if (!s.v_rank1 || m == nullptr)
            return false;
        if (!whole && !wraps) {
            item.swaps = 0;
            wraps_next();
            return served && any(po, p, g, st, item, LPMM_RANK1_FLOAT_M, m, nullptr, vc, nullptr, oh_v, qm, qv);
        }
        if (!aligned16(ptr(*m)))
            return false;
        lpmm_rank1_v4bit_tensor f = {r.p, r.g, use<float>(m), r.v_codes, r.v_rowmax, r.v_colmax, r.v_rowmax_next, r.v_colmax_next,
                                     r.rows, r.cols, 0.0f, 0.0f};
        Batch &b = batch(kRank1M32, p, nullptr, qv);
        add(b, f, item);
        b.wraps = b.wraps || wraps;
        return true;
    }
    if (s.bits_rank1) {
        if (!whole && !wraps) {
            item.swaps = 0;
            wraps_next();
            return served && any(po, p, g, st, item, LPMM_RANK1_CODES8, mc, ms, vc, oh_m, oh_v, qm, qv);
        }
        Batch &b = batch(kRank1Bits, p, qm, qv);
        add(b, r, item);
        b.wraps = b.wraps || wraps;
        return true;
    }
    if (s.m_group128 && (whole || folds || wraps)) {
        Batch &b = batch(kRank1, p, qm, qv);
        add(b, r, item);
        b.wraps = b.wraps || wraps;
        return true;
    }
    const bool ragged = aligned && !whole && !wraps && r.cols % 8 == 0;
    if (!whole && !ragged && !wraps) {
        item.swaps = 0;
        wraps_next();
        return served && (s.m_wide || s.m_group128) && any(po, p, g, st, item, LPMM_RANK1_CODES4, mc, ms, vc, oh_m, oh_v, qm, qv);
    }
    PyObject *spare = of_parameter(spare_scales, po);
    const Ref ms_next = reals_of(spare, p, ms->numel());
    if (!((s.m_wide && (whole || wraps)) || ((s.m_wide || s.m_group128) && ragged)) || ms_next == nullptr)
        return false;
    lpmm_rank1_mgroup_tensor w = {r.p,        r.g,        r.m_codes,       r.m_max1,        use<float>(ms_next), r.v_codes, r.v_rowmax,
                                  r.v_colmax, r.v_rowmax_next, r.v_colmax_next, r.rows, r.cols, 0.0f, 0.0f};
    swap_later(item, spare_scales, po, get(oh_m, N.max1), hash_of(po));
    swap_later(item, oh_m, N.max1, spare);
    if (!wraps)
        wraps_next();
    Batch &b = batch(kRank1Wide, p, qm, qv, ragged);
    add(b, w, item);
    b.wraps = b.wraps || wraps;
    return true;
}

// a matrix of any column count (lpmm_nonfused_adamw_rank1_any_step_multi); mc: the first moment's codes or values
bool Walk::any(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, Item &item, int kind, const Ref &mc,
               const Ref &ms, const Ref &vc, PyObject *oh_m, PyObject *oh_v, PyObject *qm, PyObject *qv)
{
    PyObject *cur = get(oh_v, N.max_dims), *nxt = of_parameter(spare_stats, po), *spare = of_parameter(spare_scales, po);
    void *now[2], *next[2];
    const Ref ms_next = ms != nullptr ? reals_of(spare, p, ms->numel()) : nullptr;
    if (!statistics(cur, p, now) || !statistics(nxt, p, next) || (ms != nullptr && ms_next == nullptr))
        return false;
    lpmm_rank1_any_tensor r;
    memset(&r, 0, sizeof r);
    r.p = ptr(p);
    r.g = ptr(g);
    r.m = use<>(mc);
    r.v_codes = use<uint8_t>(vc);
    r.v_rowmax = now[0];
    r.v_colmax = now[1];
    r.v_rowmax_next = next[0];
    r.v_colmax_next = next[1];
    r.rows = p.size(0);
    r.cols = p.size(1);
    if (kind == LPMM_RANK1_HALF)
        scratch(item, offsetof(lpmm_rank1_any_tensor, work), r.rows + r.cols + (p.numel() + 127) / 128);
    swap_later(item, spare_stats, po, cur, hash_of(po));
    swap_later(item, oh_v, N.max_dims, nxt);
    next_codes(item, offsetof(lpmm_rank1_any_tensor, v_codes_next), st, N.exp_avg_sq, *vc);
    if (ms != nullptr) {
        r.m_max1 = use<>(ms);
        r.m_max1_next = use<>(ms_next);
        next_codes(item, offsetof(lpmm_rank1_any_tensor, m_codes_next), st, N.exp_avg, *mc);
        swap_later(item, spare_scales, po, get(oh_m, N.max1), hash_of(po));
        swap_later(item, oh_m, N.max1, spare);
    }
    add(batch(kAny, p, qm, qv, kind), r, item);
    return true;
}

// a matrix with a factored second moment, its first moment 4-bit in groups of 128 values or not quantised
bool Walk::factored(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, const Ref &step, PyObject *mo,
                    PyObject *row_of, const QState &m_of)
{
    if (p.dim() != 2 || p.numel() == 0 || workspace_bytes == nullptr)
        return false;
    const int64_t rows = p.size(0), cols = p.size(1), n = p.numel();
    PyObject *const qm = m_of.qmap;
    const Ref row = reals_of(row_of, p, rows), col = reals_of(get(st, N.exp_avg_sq_col), p, cols);
    const Ref map = tensor_of(qm);
    const int en = enabled(po, m_of.enable);
    if (en < 0 || row == nullptr || col == nullptr || map == nullptr || !floats(*map))
        return false;
    Item item = item_of(po, g, step);
    lpmm_factored_tensor r;
    memset(&r, 0, sizeof r);
    r.p = ptr<float>(p);
    r.g = ptr<float>(g);
    r.row = use<float>(row);
    r.col = use<float>(col);
    r.rows = rows;
    r.cols = cols;
    if (en) {
        const Ref mc = codes(mo, p, packed(n, 128, false)), ms = scales(m_of.overhead, p, (n + 127) / 128);
        if (!s.m_group128 || mc == nullptr || ms == nullptr)
            return false;
        r.m_codes = use<uint8_t>(mc);
        r.m_max1 = use<float>(ms);
    } else {
        const Ref m = reals_like(mo, p);
        if (m == nullptr)
            return false;
        r.m_codes = use<uint8_t>(m);
    }
    scratch(item, offsetof(lpmm_factored_tensor, workspace), (workspace_bytes(rows, cols) + 3) / 4);
    const bool tuned = en && cols % 128 == 0 && aligned16(r.p) && aligned16(r.g) && aligned16(r.col);
    add(batch(tuned ? kFactored : kFactoredAny, p, qm, nullptr), r, item);
    return true;
}

// float16 parameters on the non-fused path (lpmm/optim/adamw.py: _half_kernel_kind)
bool Walk::half(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st, Item &item, PyObject *mo, PyObject *vo,
                const QState &m_of, const QState &v_of, int en_m, int en_v)
{
    const int64_t n = p.numel(), groups = (n + 127) / 128;
    if (en_m == 0 && en_v == 0) {
        const Ref m = reals_like(mo, p), v = reals_like(vo, p);
        if (m == nullptr || v == nullptr || m->sizes() != p.sizes() || v->sizes() != p.sizes())
            return false;
        lpmm_adamw_fp32_tensor r = {ptr<float>(p), ptr<float>(g), use<float>(m), use<float>(v), n, 0.0f, 0.0f};
        add(batch(kHalfPlain, p, nullptr, nullptr), r, item);
        return true;
    }
    PyObject *const qm = m_of.qmap, *const qv = v_of.qmap, *const oh_m = m_of.overhead, *const oh_v = v_of.overhead;
    const Ref map_m = tensor_of(qm), map_v = tensor_of(qv);
    const Ref mc = codes(mo, p, packed(n, 128, false)), vc = codes(vo, p, packed(n, 128, false)), ms = scales(oh_m, p, groups);
    PyObject *const half_type = reinterpret_cast<PyObject *>(torch::getTHPDtype(at::kHalf));
    if (en_m != 1 || en_v != 1 || !s.m_group128 || map_m == nullptr || map_v == nullptr || !floats(*map_m) || !floats(*map_v) ||
        mc == nullptr || vc == nullptr || ms == nullptr || get(oh_m, N.dtype) != half_type || get(oh_v, N.dtype) != half_type)
        return false;
    if (s.v_group128 || (s.v_rank1 && p.dim() == 1)) {
        const Ref vs = scales(oh_v, p, groups);
        if (vs == nullptr)
            return false;
        lpmm_adamw4bit_f16_tensor r = {ptr(p), ptr(g), use<uint8_t>(mc), use<uint8_t>(vc), use<>(ms), use<>(vs), n, 0.0f, 0.0f};
        add(batch(kHalfFlat, p, qm, qv), r, item);
        return true;
    }
    if (!s.v_rank1 || p.dim() != 2 || p.size(0) == 0)
        return false;
    const int64_t rows = p.size(0), cols = p.size(1);
    if (cols % 128 != 0 || !aligned16(ptr(p)) || !aligned16(ptr(g)))
        return (cols >= 32 || rows <= 32768) && any(po, p, g, st, item, LPMM_RANK1_HALF, mc, ms, vc, oh_m, oh_v, qm, qv);
    PyObject *cur = get(oh_v, N.max_dims), *nxt = of_parameter(spare_stats, po);
    void *now[2], *next[2];
    if (!statistics(cur, p, now) || !statistics(nxt, p, next))
        return false;
    swap_later(item, spare_stats, po, cur, hash_of(po));
    swap_later(item, oh_v, N.max_dims, nxt);
    lpmm_nonfused_rank1_f16_tensor r = {ptr(p), ptr(g), use<uint8_t>(mc), use<>(ms), use<uint8_t>(vc), now[0], now[1], next[0], next[1],
                                        nullptr, rows, cols, 0.0f, 0.0f};
    scratch(item, offsetof(lpmm_nonfused_rank1_f16_tensor, work), (rows + 3) / 4 * 4 + cols);
    add(batch(kHalfRank1, p, qm, qv), r, item);
    return true;
}

// a tensor of 3 to 8 dimensions on its shape[0] x rest view, where the fold between the passes takes one workgroup
// and the column scale the last step left still holds (lpmm/optim/adamw.py: _rank1_nd_steps)
bool Walk::nd(PyObject *po, const at::Tensor &p, Item &item, lpmm_nonfused_rank1_tensor &r, PyObject *st, Ref any_mc, bool may_wrap,
              PyObject *oh_m, const Ref &vc, PyObject *oh_v, PyObject *qm, PyObject *qv)
{
    const int dims = (int)p.dim();
    if (dims > LPMM_RANK1_ND_MAX || (r.rows < 16 && p.numel() > (1 << 20)) || r.cols > (1 << 16))
        return false;
    PyObject *cur = get(oh_v, N.max_dims), *nxt = of_parameter(spare_stats, po), *scratch = of_parameter(nd_scratch, po);
    PyObject *row = get(scratch, N.row);
    if (may_wrap && of_parameter(in_place, po) == oh_v)
        any_mc = nullptr;
    const int64_t pitch = (r.cols + 31) / 32 * 32;  // _nd_pitch
    const Ref work = reals_of(get(scratch, N.work), p, 3 * pitch);
    float *now[LPMM_RANK1_ND_MAX], *next[LPMM_RANK1_ND_MAX];
    if (!statistics(cur, p, now) || !statistics(nxt, p, next) || work == nullptr || get(scratch, N.scale_of) != cur || row == nullptr || !PyLong_Check(row))
        return false;
    const long old_row = PyLong_AsLong(row);
    if (old_row < 0 || old_row > 2)
        return false;
    const int raw_row = old_row == 0 ? 1 : 0, new_row = old_row == 2 ? 1 : 2;
    lpmm_rank1_small_vector fold;
    memset(&fold, 0, sizeof fold);
    int64_t slots = 0;
    for (int i = 0; i < LPMM_RANK1_ND_MAX - 1; ++i) {
        fold.shape[i] = i + 1 < dims ? p.size(i + 1) : 1;
        fold.stats[i] = i + 1 < dims ? next[i + 1] : nullptr;
        slots += i + 1 < dims ? fold.shape[i] : 0;
    }
    if (slots > 8192)
        return false;
    float *const rows = use<float>(work);
    fold.ndim = dims - 1;
    fold.x = rows + raw_row * pitch;
    fold.scale = rows + new_row * pitch;
    r.v_rowmax = now[0];
    r.v_rowmax_next = next[0];
    r.v_colmax = rows + old_row * pitch;
    r.v_colmax_next = rows + raw_row * pitch;
    // any_mc: a column count for the general kernels, which also need the next scales
    PyObject *spare = of_parameter(spare_scales, po);
    const Ref ms_next = any_mc != nullptr ? reals_of(spare, p, (p.numel() + 127) / 128) : nullptr;
    if (any_mc != nullptr && ms_next == nullptr)
        return false;
    PyObject *row_obj = PyLong_FromLong(new_row);
    if (row_obj == nullptr)
        return false;
    plan->others->push_back(row_obj);
    swap_later(item, spare_stats, po, cur, hash_of(po));
    swap_later(item, oh_v, N.max_dims, nxt);
    swap_later(item, scratch, N.scale_of, nxt);
    swap_later(item, scratch, N.row, row_obj);
    if (may_wrap && any_mc != nullptr)
        swap_later(item, in_place, po, oh_v, hash_of(po));
    if (any_mc == nullptr) {
        Batch &b = batch(kNd, p, qm, qv);
        add(b, r, item);
        b.fold.push_back(fold);
        return true;
    }
    lpmm_rank1_any_tensor w = {r.p, r.g, r.m_codes, nullptr, r.m_max1, use<>(ms_next), r.v_codes, nullptr, r.v_rowmax, r.v_colmax,
                               r.v_rowmax_next, r.v_colmax_next, nullptr, r.rows, r.cols, 0.0f, 0.0f};
    next_codes(item, offsetof(lpmm_rank1_any_tensor, m_codes_next), st, N.exp_avg, *any_mc);
    next_codes(item, offsetof(lpmm_rank1_any_tensor, v_codes_next), st, N.exp_avg_sq, *vc);
    swap_later(item, spare_scales, po, get(oh_m, N.max1), hash_of(po));
    swap_later(item, oh_m, N.max1, spare);
    Batch &b = batch(kNdAny, p, qm, qv);
    add(b, w, item);
    w.v_colmax_next = rows + new_row * pitch;
    append(b.second, w);
    b.fold.push_back(fold);
    return true;
}

bool Walk::sgd(PyObject *po, const at::Tensor &p, const at::Tensor &g, PyObject *st)
{
    if (!g.defined() || !floats(p) || !floats(g) || p.device() != g.device() || p.numel() != g.numel())
        return false;
    PyObject *const names[] = {N.momentum_buffer, N.momentum_buffer_qstate};
    PyObject *state_of[2];
    read(st, names, state_of);
    PyObject *const bo = state_of[0];
    const QState of(state_of[1]);
    Item item = item_of(po, g, nullptr);
    const int en = enabled(po, of.enable);
    if (en < 0)
        return false;
    if (!en) {
        const Ref buf = reals_like(bo, p);
        if (buf == nullptr || buf->sizes() != p.sizes())
            return false;
        lpmm_sgd_fp32_tensor r = {ptr<float>(p), ptr<float>(g), use<float>(buf), p.numel(), 0, 0};
        add(batch(kSgdPlain, p, nullptr, nullptr), r, item);
        return true;
    }
    PyObject *const qm = of.qmap;
    const Ref map = tensor_of(qm), mc = codes(bo, p, packed(p.numel(), 128, false)), ms = scales(of.overhead, p, (p.numel() + 127) / 128);
    if (!s.m_group128 || map == nullptr || !floats(*map) || mc == nullptr || ms == nullptr)
        return false;
    lpmm_sgd4bit_tensor r = {ptr<float>(p), ptr<float>(g), use<uint8_t>(mc), use<float>(ms), p.numel(), 0, 0};
    add(batch(kSgd4, p, qm, nullptr), r, item);
    return true;
}

// ---- the Plan object ---------------------------------------------------------------------------
void plan_dealloc(PyObject *self)
{
    Plan *plan = reinterpret_cast<Plan *>(self);
    if (plan->batches != nullptr)
        for (Batch &b : *plan->batches)
            for (Swap &swap : b.swaps) {
                Py_DECREF(swap.dict);
                Py_DECREF(swap.key);
                Py_XDECREF(swap.value);
            }
    for (std::vector<PyObject *> *list : {plan->held, plan->others})
        if (list != nullptr)
            for (PyObject *o : *list)
                Py_XDECREF(o);
    delete plan->batches;
    delete plan->held;
    delete plan->others;
    Py_XDECREF(plan->rest);
    Py_TYPE(self)->tp_free(self);
}

PyObject *plan_rest(PyObject *self, void *)
{
    PyObject *rest = reinterpret_cast<Plan *>(self)->rest;
    Py_INCREF(rest);
    return rest;
}

// Can a batch's launches take tensors with fp32 states along, and how well: 2, the one-pass kernels, 1, the launch that clears the
// two-pass kernels' statistics or the one that finishes the factored ones', 0.
int takes_plain(const Batch &b)
{
    switch (b.kind) {
    case kFused4:
    case kFlat:
    case kSgd4:
        return 2;
    case kRank1:
    case kNd:
    case kRank1M32:
    case kRank1Bits:
    case kRank1Wide:
    case kFactored:
    case kFactoredAny:
        return b.items.empty() ? 0 : 1;
    case kAny:
        return b.flag != LPMM_RANK1_HALF ? 1 : 0;
    default:
        return 0;
    }
}

// The tensors with fp32 states that share the launches of the quantised tensors b (lpmm_adamw4bit_fp32_step_multi, its
// non-fused form, lpmm_nonfused_rank1_fp32_step_multi, lpmm_factored_fp32_step_multi, lpmm_sgd4bit_fp32_step_multi), or null; they go with the first batch that takes them best.
// Decided here: a loop over the batches in Python cost every step 1.0 us, of 34 on three layers of width 128.
const Batch *joined(const std::vector<Batch> &batches, const Batch &b)
{
    const int best = takes_plain(b);
    if (best == 0)
        return nullptr;
    const Batch *plain = nullptr;
    for (const Batch &other : batches) {
        if (other.device != b.device)
            continue;
        const int takes = takes_plain(other);
        if (takes > best || (takes == best && &other < &b))
            return nullptr;
        if (other.kind == (b.kind == kSgd4 ? kSgdPlain : kPlain))
            plain = &other;
    }
    return plain;
}

// Matrices go with the tensors of more than two dimensions that have the same maps: their launches are the same (records with
// no vector to fold).  A classifier's own clearing, update and second pass cost an image model's step 28 of 860 us.
void join_matrices(std::vector<Batch> &batches)
{
    for (Batch &nd : batches)
        for (Batch &flat : batches) {
            if (nd.kind != kNd || flat.kind != kRank1 || flat.device != nd.device || flat.qm != nd.qm || flat.qv != nd.qv)
                continue;
            const uint32_t swaps = (uint32_t)nd.swaps.size();
            nd.records.insert(nd.records.end(), flat.records.begin(), flat.records.end());
            nd.swaps.insert(nd.swaps.end(), flat.swaps.begin(), flat.swaps.end());
            for (Record &item : flat.items) {  // records of these kinds need no memory
                item.swaps += swaps;
                item.swaps_end += swaps;
                nd.items.push_back(std::move(item));
            }
            nd.fold.resize(nd.items.size());  // ndim 0
            flat.records.clear();
            flat.swaps.clear();
            flat.items.clear();
        }
}

// advances the step counts, completes the records; the batches: (kind, device, first map, second map, flag, count,
// address of the records, address of the second pass's records or 0, address of the fold records or 0).  Quantised tensors
// that others share launches with: the latter's records in the place of a second pass's, their count in that of the fold's (beside
// a fold, in that of the flag), and flag 1 in the latter's own batch.  kRank1, kRank1M32, kRank1Bits, kRank1Wide: flag 1 where tensors wrap;
// the factored kinds: how many to launch at a time, whose scratch is then held.
PyObject *plan_start(PyObject *self, PyObject *)
{
    Plan *plan = reinterpret_cast<Plan *>(self);
    PyObject *out = PyList_New(0);
    if (out == nullptr)
        return nullptr;
    for (Batch &b : *plan->batches) {
        const size_t bytes = kRecordBytes[b.kind];
        const bool has_step = b.kind != kSgd4 && b.kind != kSgdPlain;
        // steps that stand for in-place operations of torch count as one for autograd's check of saved tensors
        if (b.kind == kSgdPlain || b.kind == kHalfPlain || (b.kind == kAny && b.flag == LPMM_RANK1_HALF))
            for (const Record &item : b.items) {
                const at::Tensor &p = THPVariable_Unpack((*plan->held)[item.held]);
                if (!p.is_inference())
                    p.unsafeGetTensorImpl()->bump_version();
            }
        for (size_t i = 0; i < b.items.size() && has_step; ++i) {
            const float step = *b.items[i].step += 1.0f;
            // every record ends in  float step  and four more bytes
            memcpy(&b.records[(i + 1) * bytes - 8], &step, 4);
            if (!b.second.empty())
                memcpy(&b.second[(i + 1) * bytes - 8], &step, 4);
        }
        const Batch *const plain = joined(*plan->batches, b);
        bool elsewhere = false;
        if (b.kind == kPlain || b.kind == kSgdPlain)
            for (const Batch &other : *plan->batches)
                elsewhere = elsewhere || joined(*plan->batches, other) == &b;
        int flag = elsewhere ? 1 : plain != nullptr && b.kind == kNd ? (int)plain->items.size() : b.wraps ? 1 : b.kind == kRank1Wide ? 0 : b.flag;
        if (b.kind == kFactored || b.kind == kFactoredAny) {
            int64_t scratch = 0;  // floats
            for (const Need &need : b.needs)
                scratch += need.n;
            flag = scratch <= (1 << 24) ? 48 : 24;
        }
        PyObject *t = Py_BuildValue("(iiOOinKKK)", (int)b.kind, b.device, b.qm != nullptr ? b.qm : Py_None,
                                    b.qv != nullptr ? b.qv : Py_None, flag, (Py_ssize_t)b.items.size(),
                                    (unsigned long long)(uintptr_t)b.records.data(),
                                    (unsigned long long)(uintptr_t)(plain != nullptr ? plain->records.data() : b.second.data()),
                                    plain != nullptr && b.kind != kNd ? (unsigned long long)plain->items.size()
                                                     : (unsigned long long)(uintptr_t)b.fold.data());
        if (t == nullptr || PyList_Append(out, t) != 0) {
            Py_XDECREF(t);
            Py_DECREF(out);
            return nullptr;
        }
        Py_DECREF(t);
    }
    return out;
}

// the arguments (batch, first, count) of the two methods below
Batch *batch_of(PyObject *self, PyObject *args, Py_ssize_t *first, Py_ssize_t *end)
{
    Plan *plan = reinterpret_cast<Plan *>(self);
    Py_ssize_t k, count;
    if (!PyArg_ParseTuple(args, "nnn", &k, first, &count))
        return nullptr;
    if (k < 0 || (size_t)k >= plan->batches->size() || *first < 0 || count < 0 ||
        (size_t)(*first + count) > (*plan->batches)[k].items.size()) {
        PyErr_SetString(PyExc_IndexError, "no such records");
        return nullptr;
    }
    *end = *first + count;
    return &(*plan->batches)[k];
}

// prepare(batch, first, count): these records are launched next.  Their memory is allocated now and not in collect():
// what the launches before them have released, old codes and scratch, is used again, so that a step holds
// one launch's arrays beside the states and not a second set of them.
PyObject *plan_prepare(PyObject *self, PyObject *args)
{
    HANDLE_TH_ERRORS
    Py_ssize_t first, end;
    Batch *b = batch_of(self, args, &first, &end);
    if (b == nullptr)
        return nullptr;
    const size_t bytes = kRecordBytes[b->kind];
    const auto floats = at::TensorOptions().dtype(at::kFloat).device(at::Device(at::kCUDA, (at::DeviceIndex)b->device));
    // scratch of little size comes out of one allocation for all (1 us each otherwise), at the alignment the allocator gives
    constexpr int64_t kLittle = 1 << 18, kAlign = 128;  // floats
    const auto little = [](const Need &need) { return !need.like.defined() && need.n > 0 && need.n < kLittle; };
    int64_t all = 0, used = 0;
    for (Py_ssize_t i = first; i < end; ++i)
        for (uint32_t j = b->items[i].needs; j < b->items[i].needs_end; ++j)
            if (little(b->needs[j]))
                all += (b->needs[j].n + kAlign - 1) / kAlign * kAlign;
    at::Tensor block;
    if (all != 0)
        block = at::empty({all}, floats);
    for (Py_ssize_t i = first; i < end; ++i) {
        Record &item = b->items[i];
        for (uint32_t j = item.needs; j < item.needs_end; ++j) {
            Need &need = b->needs[j];
            if (little(need)) {
                const void *const p = ptr<float>(block) + used;
                used += (need.n + kAlign - 1) / kAlign * kAlign;
                item.scratch = block;
                memcpy(&b->records[i * bytes + need.at], &p, sizeof p);
                if (!b->second.empty())
                    memcpy(&b->second[i * bytes + need.at], &p, sizeof p);
                continue;
            }
            const at::Tensor t = need.like.defined() ? at::empty_like(need.like) : at::empty({need.n}, floats);
            if (need.like.defined()) {
                PyObject *o = THPVariable_Wrap(t);
                if (o == nullptr)
                    return nullptr;
                Py_XDECREF(b->swaps[need.swap].value);
                b->swaps[need.swap].value = o;
            } else {
                item.scratch = t;
            }
            need.like.reset();
            const void *const p = ptr(t);
            memcpy(&b->records[i * bytes + need.at], &p, sizeof p);
            if (!b->second.empty())
                memcpy(&b->second[i * bytes + need.at], &p, sizeof p);
        }
        item.needs = item.needs_end;
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// commit(batch, first, count): the launch of these records is on the stream
PyObject *plan_commit(PyObject *self, PyObject *args)
{
    Py_ssize_t first, end;
    Plan *plan = reinterpret_cast<Plan *>(self);
    Batch *b = batch_of(self, args, &first, &end);
    if (b == nullptr)
        return nullptr;
    for (Py_ssize_t i = first; i < end; ++i) {
        Record &item = b->items[i];
        item.grad.reset();
        item.scratch.reset();
        for (uint32_t j = item.held; j < item.held_end; ++j)
            Py_CLEAR((*plan->held)[j]);
        for (uint32_t j = item.swaps; j < item.swaps_end; ++j)
            if (b->swaps[j].value == nullptr) {
                PyErr_SetString(PyExc_RuntimeError, "records that were not prepared");
                return nullptr;
            } else if (set_item(b->swaps[j]) != 0) {
                return nullptr;
            }
    }
    Py_RETURN_NONE;
}

PyMethodDef plan_methods[] = {{"start", plan_start, METH_NOARGS, "advance the step counts and return the batches"},
                              {"prepare", plan_prepare, METH_VARARGS, "allocate for records [first, first + count) of a batch"},
                              {"commit", plan_commit, METH_VARARGS, "records [first, first + count) of a batch are on the stream"},
                              {nullptr, nullptr, 0, nullptr}};
PyObject *plan_served(PyObject *self, void *) { return PyBool_FromLong(!reinterpret_cast<Plan *>(self)->batches->empty()); }

PyGetSetDef plan_getset[] = {{"served", plan_served, nullptr, "are there records", nullptr},
                             {"rest", plan_rest, nullptr, "parameters with a gradient that are not served here", nullptr},
                             {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// collect(sgd, params, state, override, spare_stats, spare_scales, nd_scratch, serve, settings,
// address of lpmm_factored_workspace_bytes or 0, in_place)
PyObject *collect(PyObject *, PyObject *args)
{
    int is_sgd, serve;
    PyObject *params, *state, *override_, *spare_stats, *spare_scales, *nd_scratch, *in_place;
    Walk w;
    int m_group;
    unsigned long long workspace;
    if (!PyArg_ParseTuple(args, "iO!O!O!O!O!O!p(iiiiiii)KO!", &is_sgd, &PyList_Type, &params, &PyDict_Type, &state, &PyDict_Type,
                          &override_, &PyDict_Type, &spare_stats, &PyDict_Type, &spare_scales, &PyDict_Type, &nd_scratch, &serve,
                          &w.s.fused, &w.s.m_group128, &w.s.v_group128, &w.s.v_rank1, &w.s.m_wide, &w.s.bits_rank1, &m_group, &workspace,
                          &PyDict_Type, &in_place))
        return nullptr;
    w.s.m_group = m_group;
    w.workspace_bytes = reinterpret_cast<int64_t (*)(int64_t, int64_t)>((uintptr_t)workspace);
    Plan *plan = reinterpret_cast<Plan *>(PlanType.tp_alloc(&PlanType, 0));
    if (plan == nullptr)
        return nullptr;
    std::unique_ptr<PyObject, void (*)(PyObject *)> owner(reinterpret_cast<PyObject *>(plan), [](PyObject *o) { Py_DECREF(o); });
    try {
        plan->batches = new std::vector<Batch>();
        plan->held = new std::vector<PyObject *>();
        plan->others = new std::vector<PyObject *>();
        plan->held->reserve(8 * PyList_GET_SIZE(params));
        plan->rest = PyList_New(0);
        if (plan->rest == nullptr)
            return nullptr;
        plan->batches->reserve(16);
        w.plan = plan;
        w.most = (size_t)(PyList_GET_SIZE(params) < 1024 ? PyList_GET_SIZE(params) : 1024);
        w.state = state;
        w.override_ = override_;
        w.spare_stats = spare_stats;
        w.spare_scales = spare_scales;
        w.nd_scratch = nd_scratch;
        w.in_place = in_place;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(params); ++i) {
            PyObject *po = PyList_GET_ITEM(params, i);
            bool served = false;
            if (THPVariable_Check(po)) {
                const at::Tensor &p = THPVariable_Unpack(po);
                const at::Tensor &g = p.grad();
                const bool own = THPVariable_CheckExact(po);  // a Tensor or a Parameter, no subclass of either
                if (!g.defined() && own)
                    continue;
                if (serve && own) {
                    PyObject *st = of_parameter(state, po);
                    if (st != nullptr && PyDict_Check(st) && PyDict_GET_SIZE(st) != 0)
                        served = is_sgd ? w.sgd(po, p, g, st) : w.adamw(po, p, g, st);
                }
            }
            if (PyErr_Occurred())
                return nullptr;
            if (!served && PyList_Append(plan->rest, po) != 0)
                return nullptr;
        }
        join_matrices(*plan->batches);
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
    return owner.release();
}

PyMethodDef methods[] = {{"collect", collect, METH_VARARGS, "walk a parameter group"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_walk", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__walk()
{
    PlanType.tp_name = "lpmm._walk.Plan";
    PlanType.tp_basicsize = sizeof(Plan);
    PlanType.tp_dealloc = plan_dealloc;
    PlanType.tp_flags = Py_TPFLAGS_DEFAULT;
    PlanType.tp_methods = plan_methods;
    PlanType.tp_getset = plan_getset;
    if (PyType_Ready(&PlanType) < 0)
        return nullptr;
#define LPMM_NAME(n) N.n = PyUnicode_InternFromString(#n)
    LPMM_NAME(step);
    LPMM_NAME(exp_avg);
    LPMM_NAME(exp_avg_sq);
    LPMM_NAME(exp_avg_qstate);
    LPMM_NAME(exp_avg_sq_qstate);
    LPMM_NAME(exp_avg_sq_row);
    LPMM_NAME(exp_avg_sq_col);
    LPMM_NAME(enable);
    LPMM_NAME(overhead);
    LPMM_NAME(qmap);
    LPMM_NAME(max1);
    LPMM_NAME(max_dims);
    LPMM_NAME(work);
    LPMM_NAME(scale_of);
    LPMM_NAME(row);
    LPMM_NAME(dtype);
    LPMM_NAME(momentum_buffer);
    LPMM_NAME(momentum_buffer_qstate);
#undef LPMM_NAME
    return PyModule_Create(&module);
}
