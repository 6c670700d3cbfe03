// The ordinary call of an operator from Python, without the Python: operands checked, descriptor filled in, launcher called.
//
// A call of a small launch is bound by what it does on the host (16x1024x8192 bf16 all-reduce of eight ranks: 6 to 7.5 us on the GPU, 10.8 us per
// call through Python and ctypes, of which the launch itself is 2.9).  call() takes the arguments of one operator call, and either launches
// it or returns None without having done anything: it accepts only what it has checked to the last condition the Python path
// checks, and everything else -- subclasses, wrapped tensors, numbers that are no Python integers, and all that is wrong -- goes through
// that path, which also says what is wrong.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string.h>

#include "catcoc_hip.h"

namespace {

// Addresses of the library the package has loaded (a second copy would have error state of its own).
decltype(&catcoc_get_kernel) getKernel;
decltype(&catcoc_launch_quant_matmul_reduce_scatter) launchQuant;
decltype(&catcoc_get_task_count) getTaskCount;
decltype(&catcoc_default_tiling) defaultTiling;
decltype(&catcoc_last_status) lastStatus;
decltype(&catcoc_last_error) lastError;
PyObject *errorType, *tilingType;   // CatcocError, CocTilingParams

PyObject *attach(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    if (n != 8) return PyErr_Format(PyExc_TypeError, "attach takes six addresses and two types");
    void *p[6];
    for (int i = 0; i < 6; ++i) {
        p[i] = PyLong_AsVoidPtr(v[i]);
        if (p[i] == nullptr) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "address %d is null", i);
    }
    getKernel = (decltype(getKernel))p[0];
    launchQuant = (decltype(launchQuant))p[1];
    getTaskCount = (decltype(getTaskCount))p[2];
    defaultTiling = (decltype(defaultTiling))p[3];
    lastStatus = (decltype(lastStatus))p[4];
    lastError = (decltype(lastError))p[5];
    Py_INCREF(v[6]);
    Py_INCREF(v[7]);
    Py_XDECREF(errorType);
    Py_XDECREF(tilingType);
    errorType = v[6];
    tilingType = v[7];
    Py_RETURN_NONE;
}

// The arguments of call(), in order.  KIND is the CocCommType, or DECODE: the W8A8 operator with explicit kept rows.
enum { KIND, A, B, SCALE_A, SCALE_B, BIAS, PEERS, RANK, RANKS, TILING, TRANS_A, TRANS_B, PEER_ROW, FLAGS, OUTBOUND, CHECKSUM, DUMP, ACCUM, WORKSPACE, OUT,
       OUT_DTYPE, BLOCK_NUM, STAGES, SWIZZLE, SPLIT_K, KEPT_BEGIN, KEPT_ROWS, N0, ARGS };
constexpr int64_t DECODE = 4;

struct Other {};   // a call for the Python path

int64_t number(PyObject *o, int64_t hi = 0xffffffffll)
{
    if (!PyLong_Check(o)) throw Other{};
    int over = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &over);
    if (over || v < 0 || v > hi) throw Other{};
    return v;
}

// A plain tensor on the GPU without gaps, of the given type (Undefined: any) and dimensions (0: any).
const at::Tensor &tensor(PyObject *o, at::ScalarType type, int64_t dims, int64_t atLeast = 0)
{
    if (!THPVariable_CheckExact(o)) throw Other{};
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || !t.is_contiguous() || !t.has_storage() || (type != at::ScalarType::Undefined && t.scalar_type() != type) || (dims && t.dim() != dims) ||
        t.numel() < atLeast)
        throw Other{};
    return t;
}

uint8_t *address(const at::Tensor &t) { return (uint8_t *)t.mutable_data_ptr(); }

uint8_t *optional(PyObject *o, at::ScalarType type, int64_t dims, int64_t atLeast) { return o == Py_None ? nullptr : address(tensor(o, type, dims, atLeast)); }

PyObject *launch(PyObject *const *v)
{
    const int64_t kind = number(v[KIND], DECODE);
    const bool quant = kind >= QUANT_MATMUL_REDUCE_SCATTER, decode = kind == DECODE;
    const int comm = decode ? QUANT_MATMUL_REDUCE_SCATTER : (int)kind;
    const at::Tensor &a = tensor(v[A], quant ? at::kChar : at::ScalarType::Undefined, 2), &b = tensor(v[B], a.scalar_type(), 2);
    if (!quant && a.scalar_type() != at::kHalf && a.scalar_type() != at::kBFloat16) throw Other{};
    const int64_t P = number(v[RANKS], CATCOC_MAX_RANKS), rank = number(v[RANK], P - 1);   // (no rank: nothing is in range)
    const bool transA = number(v[TRANS_A], 1) != 0, transB = number(v[TRANS_B], 1) != 0;
    const int64_t m = a.size(transA ? 1 : 0), k = a.size(transA ? 0 : 1), n = b.size(transB ? 0 : 1);
    if (b.size(transB ? 1 : 0) != k || m > 0x7fffffff || k > 0x7fffffff || n > 0x7fffffff) throw Other{};
    const int64_t peerRow = number(v[PEER_ROW], 0x7fffffff);

    CatcocSymmetricDesc d{};
    d.magic = CATCOC_DESC_MAGIC;
    d.rankIdx = (uint32_t)rank;
    d.rankSize = (uint32_t)P;
    d.flags = (uint32_t)number(v[FLAGS]);
    d.blockNum = (uint32_t)number(v[BLOCK_NUM]);
    d.workspaceStages = (uint32_t)number(v[STAGES]);
    d.splitK = (uint32_t)number(v[SPLIT_K]);
    if (v[SWIZZLE] != Py_None) {
        if (!PyTuple_CheckExact(v[SWIZZLE]) || PyTuple_GET_SIZE(v[SWIZZLE]) != 2) throw Other{};
        d.swizzleOffset = (uint32_t)number(PyTuple_GET_ITEM(v[SWIZZLE], 0));
        d.swizzleDirection = (uint32_t)number(PyTuple_GET_ITEM(v[SWIZZLE], 1));
    }
    // ---- rows that are kept and written
    int64_t rows;
    if (decode) {
        const int64_t begin = number(v[KEPT_BEGIN]);
        rows = v[KEPT_ROWS] == Py_None ? m : number(v[KEPT_ROWS]);
        if (rows < 1 || begin + rows > m) throw Other{};
        d.keptRowBegin = (uint32_t)begin;
        d.keptRows = (uint32_t)rows;
    } else if (comm == MATMUL_ALLREDUCE) {
        rows = m;
    } else if (comm == ALLGATHER_MATMUL) {
        rows = m * P;
    } else {
        if (m % P != 0) throw Other{};
        rows = m / P;
    }
    // ---- peers
    const bool list = PyList_CheckExact(v[PEERS]);
    if (!list && !PyTuple_CheckExact(v[PEERS])) throw Other{};
    const Py_ssize_t peers = list ? PyList_GET_SIZE(v[PEERS]) : PyTuple_GET_SIZE(v[PEERS]);
    if (peers != P - 1) throw Other{};
    const at::ScalarType peerType = comm == ALLGATHER_MATMUL ? a.scalar_type() : quant && (d.flags & CATCOC_FLAG_REDUCE_INT32) ? at::kInt : at::kFloat;
    for (Py_ssize_t i = 0; i < peers; ++i) {
        const at::Tensor &p = tensor(list ? PyList_GET_ITEM(v[PEERS], i) : PyTuple_GET_ITEM(v[PEERS], i), peerType, 2);
        if (comm == ALLGATHER_MATMUL ? p.size(0) != m || p.size(1) != k : p.size(0) < peerRow + rows || p.size(1) < n || (i && p.size(1) != d.peerLd)) throw Other{};
        d.peers[i] = address(p);
        d.peerLd = p.size(1);
    }
    d.peerRowOffset = peerRow;
    // ---- the W8A8 operator's vectors, and what both kinds may be given
    uint8_t *scaleA = nullptr, *scaleB = nullptr, *bias = nullptr, *accum = nullptr;
    if (quant) {
        scaleA = address(tensor(v[SCALE_A], at::kFloat, 1, m));
        scaleB = address(tensor(v[SCALE_B], at::kFloat, 1, n));
        bias = optional(v[BIAS], at::kInt, 1, n);
        accum = optional(v[ACCUM], at::kInt, 0, rows * n);
    }
    d.accDump = optional(v[DUMP], quant ? at::kInt : at::kFloat, 0, (comm == ALLGATHER_MATMUL ? rows : m) * n);
    if (v[OUTBOUND] != Py_None) {
        const at::Tensor &t = tensor(v[OUTBOUND], at::ScalarType::Undefined, 0);
        if (t.scalar_type() != at::kFloat && !(quant && t.scalar_type() == at::kInt)) throw Other{};
        d.outbound = address(t);
        d.outboundBytes = (uint64_t)t.nbytes();
    }
    if (v[WORKSPACE] != Py_None) {
        const at::Tensor &t = tensor(v[WORKSPACE], at::ScalarType::Undefined, 0);
        d.workspace = address(t);
        d.workspaceBytes = (uint64_t)t.nbytes();
    }
    // ---- tiling: the caller's, or the library's tiles
    CocTilingParams tiling;
    if (v[TILING] == Py_None) {
        const int64_t n0 = number(v[N0]);
        defaultTiling(&tiling, (uint32_t)m, (uint32_t)k, (uint32_t)n, (uint32_t)P);
        tiling.commInterval = 1;
        tiling.m0 = n0 ? 128 : 0;
        tiling.n0 = (uint32_t)n0;
        tiling.k0 = 0;
    } else {
        Py_buffer view;
        if ((PyObject *)Py_TYPE(v[TILING]) != tilingType || PyObject_GetBuffer(v[TILING], &view, PyBUF_SIMPLE) != 0) {
            PyErr_Clear();
            throw Other{};
        }
        memcpy(&tiling, view.buf, sizeof tiling);
        PyBuffer_Release(&view);
        if (tiling.m != m || tiling.k != k || tiling.n != n) throw Other{};
    }
    if (v[CHECKSUM] != Py_None) {
        int64_t need;
        if (decode) {
            need = (m + 127) / 128 * ((n + 127) / 128);
        } else {
            need = getTaskCount(comm, &tiling, &d);
            if (lastStatus() != 0) throw Other{};
        }
        d.checksum = (int64_t *)address(tensor(v[CHECKSUM], quant ? at::kLong : at::kDouble, 0, need));
    }
    // ---- output
    at::Tensor made;
    const at::Tensor *out = &made;
    if (v[OUT] != Py_None) {
        out = &tensor(v[OUT], quant ? at::ScalarType::Undefined : a.scalar_type(), 2);
        if ((out->scalar_type() != at::kHalf && out->scalar_type() != at::kBFloat16) || out->size(0) != rows || out->size(1) != n) throw Other{};
    } else {
        at::ScalarType type = a.scalar_type();
        if (quant) {
            if (!THPDtype_Check(v[OUT_DTYPE])) throw Other{};
            type = ((THPDtype *)v[OUT_DTYPE])->scalar_type;
            if (type != at::kHalf && type != at::kBFloat16) throw Other{};
        }
        made = at::empty({rows, n}, a.options().dtype(type));
    }
    uint8_t *const pa = address(a), *const pb = address(b), *const po = address(*out);
    const uint32_t outType = out->scalar_type() == at::kHalf ? FP16 : BF16;
    void *const stream = (void *)c10::hip::getCurrentHIPStream().stream();
    const auto kernel = quant ? nullptr : getKernel(comm, (int)outType);
    if (!quant && kernel == nullptr) throw Other{};
    Py_BEGIN_ALLOW_THREADS
    if (quant) launchQuant(stream, 0, pa, pb, scaleA, scaleB, bias, accum, po, (uint8_t *)&d, &tiling, transA, transB, outType);
    else kernel(stream, 0, pa, pb, po, nullptr, nullptr, (uint8_t *)&d, &tiling, transA, transB);
    Py_END_ALLOW_THREADS
    if (lastStatus() != 0) {
        PyErr_SetString(errorType, lastError());
        return nullptr;
    }
    if (v[OUT] == Py_None) return THPVariable_Wrap(std::move(made));
    Py_INCREF(v[OUT]);
    return v[OUT];
}

PyObject *call(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    if (n != ARGS || errorType == nullptr) return PyErr_Format(PyExc_TypeError, "call takes %d arguments, after attach", (int)ARGS);
    try {
        return launch(v);
    } catch (const Other &) {
    } catch (const std::exception &) {   // (a tensor without memory of its own, no memory for the output: the Python path meets it again)
        PyErr_Clear();
    }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"attach", (PyCFunction)(void *)attach, METH_FASTCALL, "addresses of the library's functions, CatcocError, CocTilingParams"},
                         {"call", (PyCFunction)(void *)call, METH_FASTCALL, "one operator call: the output, or None for the Python path"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
