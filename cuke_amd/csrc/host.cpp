// The eager surface's host path: what KGEModel.score / backward, margin_loss, the sparse optimizer steps, the
// positional score functions and the sampler do between Python and the library's entry points, in native code.
//
// A batch of a few hundred triples is 50 to 100 us of small kernels; the same calls issued through Python's
// ctypes -- argument checks, structure building, a dozen torch.empty calls, one synchronisation per distinct-row
// count -- took the host 250 to 300 us, which is what such a loop then ran at.  Every function here
// handles the ordinary case (tensors on the current device, right types, contiguous) and returns None for anything
// else, so that kge.py's own code converts or rejects it: the checks and their messages live in one place.
//
// Outputs are torch tensors; workspaces that no later call needs come straight from torch's caching allocator and go
// back to it when the call returns (stream-ordered, as a tensor that goes out of scope is).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/kge_mi355.h"

namespace {

PyObject *g_error = nullptr;  // kge.KgeError

int64_t up256(int64_t x) { return (x + 255) & ~int64_t(255); }

bool fail(int rc, const char *what)
{
    PyErr_Format(g_error ? g_error : PyExc_RuntimeError, "%s: %s (%d)", what, kge_strerror(rc), rc);
    return true;
}

// Runs a library call without the GIL, as ctypes does.
template <typename F>
int nogil(F &&f)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = f();
    Py_END_ALLOW_THREADS return rc;
}

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

const at::Tensor *tensor(PyObject *o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

bool is_f32(const at::Tensor *t, int64_t ndim, int dev)
{
    return t && t->is_cuda() && t->device().index() == dev && t->scalar_type() == at::kFloat && t->dim() == ndim && t->is_contiguous();
}

// An id array this module can hand on: on the device, contiguous, 64 or 32 bits wide.
bool is_ids(const at::Tensor *t, int dev)
{
    return t && t->is_cuda() && t->device().index() == dev && (t->scalar_type() == at::kLong || t->scalar_type() == at::kInt) &&
           t->is_contiguous();
}

bool number(PyObject *o, double *out)
{
    *out = PyFloat_AsDouble(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();  // (the caller converts it, or raises)
    return false;
}

PyObject *wrap(const at::Tensor &t)
{
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}

c10::DataPtr scratch(size_t bytes) { return c10::hip::HIPCachingAllocator::get()->allocate(bytes ? bytes : 1); }

// 32-bit ids of up to four arrays widened to 64 bits in one launch; 64-bit ones are passed on.
int widen(at::Tensor *ids, int n, void *st)
{
    const int32_t *src[4];
    int64_t *dst[4], len[4];
    int m = 0;
    for (int i = 0; i < n; ++i)
        if (ids[i].defined() && ids[i].scalar_type() == at::kInt) {
            at::Tensor w = at::empty(ids[i].sizes(), ids[i].options().dtype(at::kLong));
            src[m] = ids[i].data_ptr<int32_t>(), dst[m] = w.data_ptr<int64_t>(), len[m] = w.numel();
            ids[i] = w, ++m;
        }
    return m ? kge_widen_ids(src, dst, len, m, st) : KGE_OK;
}

// An inspection whose arrays live in two tensors: the ids and one block
//   [num_unique, padded to 256 bytes][seg_offsets n + 1][perm n][inverse n][sorted_seg n][workspace]
// each part on a 256-byte boundary (kge.py's _PackedInspection names the parts on demand).
struct Packed {
    at::Tensor ids, block;
    kge_inspection c;
    void *ws;
    size_t ws_bytes;
};

Packed make_packed(int64_t n, int64_t n_rows, const at::TensorOptions &bytes)
{
    Packed p;
    const int64_t m = n > 0 ? n : 1, i4 = up256(4 * m);
    p.ws_bytes = kge_inspect_workspace(n, n_rows);
    p.ids = at::empty({m}, bytes.dtype(at::kLong));
    p.block = at::empty({256 + up256(4 * (n + 1)) + 3 * i4 + (int64_t)p.ws_bytes + 256}, bytes.dtype(at::kByte));
    char *b = static_cast<char *>(p.block.data_ptr());
    p.c.n = n, p.c.n_rows = n_rows;
    p.c.num_unique = reinterpret_cast<int32_t *>(b);
    p.c.unique_ids = p.ids.data_ptr<int64_t>();
    b += 256;
    p.c.seg_offsets = reinterpret_cast<int32_t *>(b), b += up256(4 * (n + 1));
    p.c.perm = reinterpret_cast<int32_t *>(b), b += i4;
    p.c.inverse = reinterpret_cast<int32_t *>(b), b += i4;
    p.c.sorted_seg = reinterpret_cast<int32_t *>(b), b += i4;
    p.ws = b;
    return p;
}

kge_inspect_job make_job(const Packed &p, const at::Tensor *const *parts, int n_parts)
{
    kge_inspect_job j;
    std::memset(&j, 0, sizeof(j));
    for (int q = 0; q < n_parts; ++q) j.parts[q] = parts[q]->data_ptr<int64_t>(), j.part_len[q] = parts[q]->numel();
    j.n_parts = n_parts, j.n_rows = p.c.n_rows, j.out = p.c, j.workspace = p.ws, j.workspace_bytes = p.ws_bytes;
    return j;
}

// (ids, block, kge_inspection as bytes)
PyObject *packed_tuple(const Packed &p)
{
    return Py_BuildValue("(NNy#)", wrap(p.ids), wrap(p.block), reinterpret_cast<const char *>(&p.c), (Py_ssize_t)sizeof(p.c));
}

// ---- distinct-row counts on the host -------------------------------------------------------------------
// The sizes of the gradient arrays are device data.  A one-thread kernel behind the inspection writes both counts
// to a slot of pinned memory as one 64-bit word; the host goes on enqueueing the backward pass and only then
// reads the slot, by which time the word has usually arrived: it waits for the inspection alone, never for the
// gradient kernels, and the device does not run dry.
struct Slots {
    std::mutex m;
    std::vector<volatile uint64_t *> free_;
    volatile uint64_t *take()
    {
        std::lock_guard<std::mutex> g(m);
        if (free_.empty()) {
            constexpr size_t kSlots = 64, kStride = 128;  // one line each
            void *p = nullptr;
            if (hipHostMalloc(&p, kSlots * kStride, hipHostMallocPortable) != hipSuccess) return nullptr;
            for (size_t i = 0; i < kSlots; ++i) free_.push_back(reinterpret_cast<volatile uint64_t *>(static_cast<char *>(p) + i * kStride));
        }
        volatile uint64_t *s = free_.back();
        free_.pop_back();
        return s;
    }
    void give(volatile uint64_t *s)
    {
        std::lock_guard<std::mutex> g(m);
        free_.push_back(s);
    }
} g_slots;

constexpr uint64_t kEmpty = ~uint64_t(0);  // no pair of counts (they are below 2^31)

// Waits (without the GIL) for the word; after a tenth of a second asks the stream instead, which also ends the wait if
// the device has failed.
bool await(volatile uint64_t *slot, void *st, uint64_t *out)
{
    bool ok = true;
    Py_BEGIN_ALLOW_THREADS
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(100);
    uint64_t v;
    for (unsigned spin = 0; (v = *slot) == kEmpty; ++spin) {
        __builtin_ia32_pause();
        if ((spin & 1023) == 1023 && std::chrono::steady_clock::now() > until) {
            ok = hipStreamSynchronize(static_cast<hipStream_t>(st)) == hipSuccess && (v = *slot) != kEmpty;
            break;
        }
    }
    *out = v;
    Py_END_ALLOW_THREADS
    return ok;
}

#define NOT_HERE Py_RETURN_NONE  // not the ordinary case: the caller's own code takes it

// set_error(type)
PyObject *py_set_error(PyObject *, PyObject *o)
{
    Py_XINCREF(o);
    Py_XSETREF(g_error, o);
    Py_RETURN_NONE;
}

// inspect(parts tuple, n_rows) -> (ids, block, struct) or None
PyObject *py_inspect(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    if (!PyTuple_Check(args[0]) && !PyList_Check(args[0])) NOT_HERE;
    const Py_ssize_t n_parts = PySequence_Fast_GET_SIZE(args[0]);
    if (n_parts < 1 || n_parts > 4) NOT_HERE;
    const int dev = c10::hip::current_device();
    at::Tensor ids[4];
    int64_t n = 0;
    for (Py_ssize_t q = 0; q < n_parts; ++q) {
        const at::Tensor *t = tensor(PySequence_Fast_GET_ITEM(args[0], q));
        if (!is_ids(t, dev) || t->dim() != 1) NOT_HERE;
        ids[q] = *t, n += t->numel();
    }
    if (!PyLong_Check(args[1])) NOT_HERE;  // (a count of another type: converted by the caller)
    const int64_t n_rows = PyLong_AsLongLong(args[1]);
    if (n_rows == -1 && PyErr_Occurred()) return nullptr;
    void *st = stream();
    if (int rc = widen(ids, (int)n_parts, st)) return fail(rc, "kge_widen_ids"), nullptr;
    const Packed p = make_packed(n, n_rows, ids[0].options());
    const at::Tensor *parts[4] = {&ids[0], &ids[1], &ids[2], &ids[3]};
    const kge_inspect_job job = make_job(p, parts, (int)n_parts);
    if (int rc = nogil([&] { return kge_inspect_batch(&job, 1, st); })) return fail(rc, "kge_inspect"), nullptr;
    return packed_tuple(p);
    END_HANDLE_TH_ERRORS
}

struct Ids {
    at::Tensor h, r, t, neg;
};

// h, r, t (and neg) of a batch; false: not the ordinary case
bool take_ids(PyObject *const *o, bool has_neg, int dev, Ids *out)
{
    at::Tensor *dst[4] = {&out->h, &out->r, &out->t, &out->neg};
    for (int i = 0; i < (has_neg ? 4 : 3); ++i) {
        const at::Tensor *x = tensor(o[i]);
        if (!is_ids(x, dev) || (i < 3 && x->dim() != 1)) return false;
        *dst[i] = *x;
    }
    return out->r.numel() == out->h.numel() && out->t.numel() == out->h.numel();
}

int widen_batch(Ids *i, void *st)
{
    at::Tensor ids[4] = {i->h, i->r, i->t, i->neg};
    const int rc = widen(ids, 4, st);
    i->h = ids[0], i->r = ids[1], i->t = ids[2], i->neg = ids[3];
    return rc;
}

float *fptr(const at::Tensor &t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

// score(tables address, E, h, r, t, neg|None, chunk|None, head, ent_insp address, rel_insp address, for_backward)
//   -> (pos, neg, side_pos, side_neg, residual, workspace, back_rows, (h, r, t, neg, C, N), packed rel_insp | None)
PyObject *py_score(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    const auto *tab = static_cast<const kge_tables *>(PyLong_AsVoidPtr(args[0]));
    const int dev = c10::hip::current_device();
    const at::Tensor &E = THPVariable_Unpack(args[1]);
    if (E.device().index() != dev) NOT_HERE;
    const bool has_neg = args[5] != Py_None;
    Ids ids;
    if (!take_ids(args + 2, has_neg, dev, &ids)) NOT_HERE;
    kge_batch bat;
    std::memset(&bat, 0, sizeof(bat));
    const int64_t B = ids.h.numel(), d = tab->dim;
    bat.batch = B;
    const bool projected = tab->model == KGE_TRANSR || tab->model == KGE_RESCAL;
    if (has_neg) {
        int64_t chunk = 0;
        if (args[6] != Py_None) {
            if (!PyLong_Check(args[6])) NOT_HERE;
            chunk = PyLong_AsLongLong(args[6]);
        }
        chunk = chunk ? chunk : B;
        if (chunk <= 0 || B == 0 || B % chunk || ids.neg.numel() % (B / chunk)) NOT_HERE;
        if (projected && (d % 4 || d > 1024)) NOT_HERE;
        bat.chunk = chunk, bat.n_neg = ids.neg.numel() / (B / chunk);
        bat.neg_mode = PyObject_IsTrue(args[7]) ? KGE_NEG_HEAD : KGE_NEG_TAIL;
        if (ids.neg.dim() != 1) ids.neg = ids.neg.view({-1});
    }
    void *st = stream();
    if (int rc = widen_batch(&ids, st)) return fail(rc, "kge_widen_ids"), nullptr;
    bat.h = ids.h.data_ptr<int64_t>(), bat.r = ids.r.data_ptr<int64_t>(), bat.t = ids.t.data_ptr<int64_t>();
    bat.neg = has_neg ? ids.neg.data_ptr<int64_t>() : nullptr;
    bat.ent_insp = static_cast<const kge_inspection *>(PyLong_AsVoidPtr(args[8]));
    bat.rel_insp = static_cast<const kge_inspection *>(PyLong_AsVoidPtr(args[9]));
    Packed rel;
    const bool own_rel = has_neg && projected && !bat.rel_insp;
    if (own_rel) {
        rel = make_packed(B, tab->n_rel, ids.r.options());
        bat.rel_insp = &rel.c;
    }
    if (has_neg && tab->model == KGE_TRANSR && kge_score_bwd_workspace(tab, &bat) == 0) NOT_HERE;  // flattened by the caller
    if (own_rel) {
        const at::Tensor *parts[1] = {&ids.r};
        const kge_inspect_job job = make_job(rel, parts, 1);
        if (int rc = nogil([&] { return kge_inspect_batch(&job, 1, st); })) return fail(rc, "kge_inspect"), nullptr;
    }
    const auto f32 = E.options().requires_grad(false);
    at::Tensor pos = at::empty({B}, f32), neg, side_pos, side_neg, residual, back, fws;
    if (has_neg) neg = at::empty({B, bat.n_neg}, f32);
    if (tab->model == KGE_TRANSH || (tab->model == KGE_TRANSF && has_neg)) {
        side_pos = at::empty({B}, f32);
        if (has_neg && tab->model == KGE_TRANSH) side_neg = at::empty({2, B, bat.n_neg}, f32);
    }
    if (projected || tab->model == KGE_ROTATE) residual = at::empty({B, d}, f32);
    if (PyObject_IsTrue(args[10]) && B > 0 && kge_back_rows_ok(tab, &bat)) {
        back = at::empty({B, d}, f32);
        bat.back_rows = back.data_ptr<float>();
    }
    const size_t ws_bytes = kge_score_fwd_workspace(tab, &bat);
    c10::DataPtr tmp;
    void *ws;
    if (has_neg && tab->model == KGE_TRANSR) {  // group list and projected rows, read again by backward
        fws = at::empty({(int64_t)(ws_bytes ? ws_bytes : 1)}, f32.dtype(at::kByte));
        ws = fws.data_ptr();
    } else {
        if (ws_bytes) tmp = scratch(ws_bytes);
        ws = tmp.get();
    }
    const int rc = nogil([&] {
        return kge_score_fwd(tab, &bat, fptr(pos), fptr(neg), fptr(side_pos), fptr(side_neg), fptr(residual), ws, ws_bytes, st);
    });
    if (rc) return fail(rc, "kge_score_fwd"), nullptr;
    PyObject *batch = Py_BuildValue("(NNNNLL)", wrap(ids.h), wrap(ids.r), wrap(ids.t), wrap(ids.neg), (long long)bat.chunk, (long long)bat.n_neg);
    PyObject *ins = own_rel ? packed_tuple(rel) : Py_NewRef(Py_None);
    return Py_BuildValue("(NNNNNNNNN)", wrap(pos), wrap(neg), wrap(side_pos), wrap(side_neg), wrap(residual), wrap(fws), wrap(back), batch, ins);
    END_HANDLE_TH_ERRORS
}

// backward(tables address, E, (h, r, t, neg, C, N), head, ent_insp address, rel_insp address, (U_ent, U_rel) known or -1,
//          (pos, neg, side_pos, side_neg, residual, fwd_ws, back_rows), dpos|None, dneg|None, factor_max)
//   -> (packed ent | None, packed rel | None, U_ent, U_rel, ent_rows, rel_rows, aux_rows, aux_x, aux_q, kge_grads as bytes)
// Rows come back whole; the caller narrows them to the distinct rows.
PyObject *py_backward(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    const auto *tab = static_cast<const kge_tables *>(PyLong_AsVoidPtr(args[0]));
    const int dev = c10::hip::current_device();
    const at::Tensor &E = THPVariable_Unpack(args[1]);
    if (E.device().index() != dev) NOT_HERE;
    PyObject *bt = args[2];
    kge_batch bat;
    std::memset(&bat, 0, sizeof(bat));
    const at::Tensor *ids[4];
    for (int i = 0; i < 4; ++i) {
        ids[i] = tensor(PyTuple_GET_ITEM(bt, i));
        if (ids[i] && (!is_ids(ids[i], dev) || ids[i]->scalar_type() != at::kLong)) NOT_HERE;
    }
    if (!ids[0] || !ids[1] || !ids[2]) NOT_HERE;
    const int64_t B = ids[0]->numel(), d = tab->dim;
    if (B == 0) NOT_HERE;
    bat.batch = B, bat.h = ids[0]->data_ptr<int64_t>(), bat.r = ids[1]->data_ptr<int64_t>(), bat.t = ids[2]->data_ptr<int64_t>();
    if (ids[3]) {
        bat.neg = ids[3]->data_ptr<int64_t>();
        bat.chunk = PyLong_AsLongLong(PyTuple_GET_ITEM(bt, 4)), bat.n_neg = PyLong_AsLongLong(PyTuple_GET_ITEM(bt, 5));
    }
    bat.neg_mode = PyObject_IsTrue(args[3]) ? KGE_NEG_HEAD : KGE_NEG_TAIL;
    const at::Tensor *sv[7];
    for (int i = 0; i < 7; ++i) sv[i] = tensor(PyTuple_GET_ITEM(args[7], i));
    const at::Tensor *dpos = tensor(args[8]), *dneg = tensor(args[9]);
    if ((args[8] != Py_None && !is_f32(dpos, 1, dev)) || (args[9] != Py_None && !is_f32(dneg, 2, dev))) NOT_HERE;
    if ((dpos && dpos->numel() != B) || (dneg && (!ids[3] || dneg->numel() != B * bat.n_neg))) NOT_HERE;
    const int factor_max = (int)PyLong_AsLong(args[10]);
    void *st = stream();
    bat.ent_insp = static_cast<const kge_inspection *>(PyLong_AsVoidPtr(args[4]));
    bat.rel_insp = static_cast<const kge_inspection *>(PyLong_AsVoidPtr(args[5]));
    int64_t ue = PyLong_AsLongLong(PyTuple_GET_ITEM(args[6], 0)), ur = PyLong_AsLongLong(PyTuple_GET_ITEM(args[6], 1));
    Packed ent, rel;
    kge_inspect_job jobs[2];
    int n_jobs = 0;
    const bool own_ent = !bat.ent_insp, own_rel = !bat.rel_insp;
    if (own_ent) {
        const at::Tensor *parts[3] = {ids[0], ids[2], ids[3]};
        ent = make_packed(2 * B + (ids[3] ? ids[3]->numel() : 0), tab->n_ent, ids[0]->options());
        jobs[n_jobs++] = make_job(ent, parts, ids[3] ? 3 : 2);
        bat.ent_insp = &ent.c;
    }
    if (own_rel) {
        const at::Tensor *parts[1] = {ids[1]};
        rel = make_packed(B, tab->n_rel > 1 ? tab->n_rel : 1, ids[0]->options());
        jobs[n_jobs++] = make_job(rel, parts, 1);
        bat.rel_insp = &rel.c;
    }
    const auto f32 = E.options().requires_grad(false);
    const int64_t n_occ = bat.ent_insp->n;
    at::Tensor ent_rows = at::empty({n_occ, d}, f32), rel_rows, aux_rows, aux_x, aux_q;
    if (tab->rel_dim) rel_rows = at::empty({B, tab->rel_dim}, f32);
    if (tab->model == KGE_TRANSH) aux_rows = at::empty({B, d}, f32);
    else if (tab->model == KGE_TRANSR || tab->model == KGE_RESCAL) aux_rows = at::empty({B < tab->n_rel ? B : tab->n_rel, d * d}, f32);
    if (factor_max) aux_x = at::empty({B, d}, f32), aux_q = at::empty({B, d}, f32);
    kge_grads grads{fptr(ent_rows), fptr(rel_rows), fptr(aux_rows), fptr(aux_x), fptr(aux_q), factor_max, 0};
    auto sp = [&](int i) { return sv[i] ? sv[i]->data_ptr<float>() : nullptr; };
    kge_saved saved{sp(0), sp(1), sp(2), sp(3), sp(4), nullptr, 0, sp(6)};
    if (sv[5]) saved.fwd_workspace = sv[5]->data_ptr(), saved.fwd_workspace_bytes = (size_t)sv[5]->numel();
    const size_t ws_bytes = kge_score_bwd_workspace(tab, &bat);
    const c10::DataPtr ws = scratch(ws_bytes);
    const bool ask = ue < 0 || ur < 0;
    volatile uint64_t *slot = nullptr;
    if (ask) {
        if (!(slot = g_slots.take())) return fail(KGE_ELAUNCH, "hipHostMalloc"), nullptr;
        *slot = kEmpty;
    }
    const char *what = "kge_inspect";
    const int rc = nogil([&] {
        int e = n_jobs ? kge_inspect_batch(jobs, n_jobs, st) : KGE_OK;
        if (!e && ask) what = "kge_publish_counts", e = kge_publish_counts(bat.ent_insp->num_unique, bat.rel_insp->num_unique, const_cast<uint64_t *>(slot), st);
        if (!e)
            what = "kge_score_bwd", e = kge_score_bwd(tab, &bat, &saved, dpos ? dpos->data_ptr<float>() : nullptr,
                                                     dneg ? dneg->data_ptr<float>() : nullptr, &grads, ws.get(), ws_bytes, st);
        return e;
    });
    if (ask) {
        uint64_t v = 0;
        // (after an error the publishing kernel may or may not be under way: the slot is not used again then)
        if (!rc) {
            if (!await(slot, st, &v)) return fail(KGE_ELAUNCH, "waiting for the distinct-row counts"), nullptr;
            g_slots.give(slot);
            ue = (int64_t)(uint32_t)v, ur = (int64_t)(v >> 32);
        }
    }
    if (rc) return fail(rc, what), nullptr;
    PyObject *pe = own_ent ? packed_tuple(ent) : Py_NewRef(Py_None), *pr = own_rel ? packed_tuple(rel) : Py_NewRef(Py_None);
    const auto head = [](const at::Tensor &t, int64_t n) { return t.defined() && t.size(0) != n ? t.narrow(0, 0, n) : t; };
    return Py_BuildValue("(NNLLNNNNNy#)", pe, pr, (long long)ue, (long long)ur, wrap(head(ent_rows, ue)), wrap(head(rel_rows, ur)), wrap(head(aux_rows, ur)),
                         wrap(aux_x), wrap(aux_q), reinterpret_cast<const char *>(&grads), (Py_ssize_t)sizeof(grads));
    END_HANDLE_TH_ERRORS
}

// call(model, E, R|None, A|None, h, r, t, batch, dim, residual) -> tensor or None: one positional score call.  TransR / RESCAL run on
// the relation groups of r.
PyObject *py_call(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    const int model = (int)PyLong_AsLong(args[0]);
    const int dev = c10::hip::current_device();
    const at::Tensor *E = tensor(args[1]), *R = tensor(args[2]), *A = tensor(args[3]);
    const bool projected = model == KGE_TRANSR || model == KGE_RESCAL;
    if (!is_f32(E, 2, dev)) NOT_HERE;
    const int64_t d = E->size(1);
    if (model != KGE_RESCAL && (!is_f32(R, 2, dev) || R->size(1) != d)) NOT_HERE;
    if (model == KGE_TRANSH && (!is_f32(A, 2, dev) || A->size(0) != R->size(0) || A->size(1) != d)) NOT_HERE;
    if (projected && (!is_f32(A, 3, dev) || A->size(1) != d || A->size(2) != d || (R && A->size(0) != R->size(0)))) NOT_HERE;
    Ids ids;
    if (!take_ids(args + 4, false, dev, &ids)) NOT_HERE;
    const int64_t B = ids.h.numel();
    if (!PyLong_Check(args[7]) || !PyLong_Check(args[8]) || PyLong_AsLongLong(args[7]) != B || PyLong_AsLongLong(args[8]) != d) NOT_HERE;
    const bool resid = PyObject_IsTrue(args[9]);
    void *st = stream();
    if (int rc = widen_batch(&ids, st)) return fail(rc, "kge_widen_ids"), nullptr;
    kge_tables tab{model, 2, 0.0f, 0, d, model == KGE_RESCAL ? 0 : d, E->size(0), projected ? A->size(0) : R->size(0), E->data_ptr<float>(),
                   model == KGE_RESCAL ? nullptr : R->data_ptr<float>(), A ? A->data_ptr<float>() : nullptr};
    kge_batch bat;
    std::memset(&bat, 0, sizeof(bat));
    bat.batch = B, bat.h = ids.h.data_ptr<int64_t>(), bat.r = ids.r.data_ptr<int64_t>(), bat.t = ids.t.data_ptr<int64_t>();
    const auto f32 = E->options().requires_grad(false);
    at::Tensor out = resid ? at::empty({B, d}, f32) : at::empty({B}, f32);
    Packed rel;
    kge_inspect_job job;
    if (projected) {
        rel = make_packed(B, tab.n_rel, ids.r.options());
        const at::Tensor *parts[1] = {&ids.r};
        job = make_job(rel, parts, 1);
        bat.rel_insp = &rel.c;
    }
    const size_t ws_bytes = projected ? kge_score_fwd_workspace(&tab, &bat) : 0;
    c10::DataPtr ws;
    if (ws_bytes) ws = scratch(ws_bytes);
    const char *what = "kge_inspect";
    const int rc = nogil([&] {
        int e = projected ? kge_inspect_batch(&job, 1, st) : KGE_OK;
        if (e) return e;
        what = resid ? "kge_residual_fwd" : "kge_score_fwd";
        return resid ? kge_residual_fwd(&tab, &bat, out.data_ptr<float>(), ws.get(), ws_bytes, st)
                     : kge_score_fwd(&tab, &bat, out.data_ptr<float>(), nullptr, nullptr, nullptr, nullptr, ws.get(), ws_bytes, st);
    });
    if (rc) return fail(rc, what), nullptr;
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// margin_loss(pos, neg, margin, sign) -> (loss, dpos, dneg) or None
PyObject *py_margin_loss(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    const int dev = c10::hip::current_device();
    const at::Tensor *pos = tensor(args[0]), *neg = tensor(args[1]);
    if (!is_f32(pos, 1, dev) || !is_f32(neg, 2, dev) || neg->size(0) != pos->numel()) NOT_HERE;
    double margin, sign;
    if (!number(args[2], &margin) || !number(args[3], &sign)) NOT_HERE;
    const int64_t B = neg->size(0), N = neg->size(1);
    const auto f32 = pos->options().requires_grad(false);
    at::Tensor loss = at::empty({1}, f32), dpos = at::empty({B}, f32), dneg = at::empty({B, N}, f32);
    const size_t ws_bytes = kge_margin_loss_workspace(B, N);
    const c10::DataPtr ws = scratch(ws_bytes);
    void *st = stream();
    const int rc = nogil([&] {
        return kge_margin_loss(pos->data_ptr<float>(), neg->data_ptr<float>(), B, N, (float)margin, (float)sign, loss.data_ptr<float>(),
                               dpos.data_ptr<float>(), dneg.data_ptr<float>(), ws.get(), ws_bytes, st);
    });
    if (rc) return fail(rc, "kge_margin_loss"), nullptr;
    return Py_BuildValue("(NNN)", wrap(loss), wrap(dpos), wrap(dneg));
    END_HANDLE_TH_ERRORS
}

// sparse_step(table, state, inspection address, rows, lr, eps, adagrad) -> True, or None; SGD takes no state
PyObject *py_sparse_step(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    const int dev = c10::hip::current_device();
    const at::Tensor *table = tensor(args[0]), *state = tensor(args[1]), *rows = tensor(args[3]);
    if (!table || !is_f32(table, table->dim(), dev) || !is_f32(rows, 2, dev)) NOT_HERE;
    const bool adagrad = PyObject_IsTrue(args[6]);
    if (adagrad && !is_f32(state, 1, dev)) NOT_HERE;
    const auto *ins = static_cast<const kge_inspection *>(PyLong_AsVoidPtr(args[2]));
    if (!ins) NOT_HERE;  // (no inspection was given)
    double lr, eps;
    if (!number(args[4], &lr) || !number(args[5], &eps)) NOT_HERE;
    void *st = stream();
    const int rc = nogil([&] {
        return adagrad ? kge_sparse_adagrad(table->data_ptr<float>(), state->data_ptr<float>(), rows->size(1), ins->unique_ids, ins->num_unique,
                                            rows->size(0), rows->data_ptr<float>(), (float)lr, (float)eps, st)
                       : kge_sparse_sgd(table->data_ptr<float>(), rows->size(1), ins->unique_ids, ins->num_unique, rows->size(0),
                                        rows->data_ptr<float>(), (float)lr, st);
    });
    if (rc) return fail(rc, adagrad ? "kge_sparse_adagrad" : "kge_sparse_sgd"), nullptr;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// A one-dimensional array of 64-bit ids in host memory (numpy), read where it lies.
struct HostIds {
    Py_buffer b{};
    bool held = false;
    const char *base = nullptr;
    int64_t stride = 0;
    bool take(PyObject *o)
    {
        if (PyObject_GetBuffer(o, &b, PyBUF_FORMAT | PyBUF_STRIDES)) return PyErr_Clear(), false;
        held = true, base = static_cast<const char *>(b.buf), stride = b.ndim == 1 ? b.strides[0] : 0;
        return b.ndim == 1 && b.itemsize == 8 && b.format && (!std::strcmp(b.format, "l") || !std::strcmp(b.format, "q"));
    }
    int64_t size() const { return b.shape[0]; }
    int64_t at(int64_t i) const { return *reinterpret_cast<const int64_t *>(base + i * stride); }
    HostIds() = default;
    HostIds(const HostIds &) = delete;
    ~HostIds()
    {
        if (held) PyBuffer_Release(&b);
    }
};

// The pinned memory of one sampler: slots of [KGE_STAGED_BATCH_WORDS done words][3][batch] ids.  A slot is free when the launch
// that reads it has marked every word; a host that is further ahead gets another, up to 64 slots and 32 MB in all.
// They are freed with the sampler, behind the launches that still read them.  (Callers hold the GIL.)
struct Stage {
    struct Slot {
        uint32_t *done;
        int64_t *ids;
        uint32_t mark;
        bool idle(int words) const
        {
            for (int w = 0; w < words; ++w)
                if (__atomic_load_n(done + w, __ATOMIC_ACQUIRE) != mark) return false;
            return true;
        }
    };
    static constexpr size_t kHead = sizeof(uint32_t) * KGE_STAGED_BATCH_WORDS, kMaxSlots = 64, kMaxBytes = size_t(32) << 20;
    int64_t batch = 0;
    std::vector<Slot> slots;
    size_t at = 0;

    int words() const { return (int)std::min<int64_t>(KGE_STAGED_BATCH_WORDS, (batch + 255) / 256); }
    size_t bytes() const { return kHead + sizeof(int64_t) * 3 * (size_t)batch; }
    Slot *take()
    {
        for (size_t k = 0; k < slots.size(); ++k) {  // oldest first
            Slot &s = slots[(at + k) % slots.size()];
            if (s.idle(words())) return at = (at + k + 1) % slots.size(), &s;
        }
        if (slots.size() >= kMaxSlots || (slots.size() + 1) * bytes() > kMaxBytes) return nullptr;
        void *p = nullptr;
        if (hipHostMalloc(&p, bytes(), hipHostMallocPortable) != hipSuccess) return (void)hipGetLastError(), nullptr;
        std::memset(p, 0, kHead);
        slots.push_back(Slot{static_cast<uint32_t *>(p), reinterpret_cast<int64_t *>(static_cast<char *>(p) + kHead), 0});
        return &slots.back();
    }
    ~Stage()
    {
        for (const Slot &s : slots) {
            const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(100);
            bool idle;
            while (!(idle = s.idle(words())) && std::chrono::steady_clock::now() < until) __builtin_ia32_pause();
            if (!idle && hipDeviceSynchronize() == hipSuccess) idle = s.idle(words());
            if (idle) (void)hipHostFree(s.done);  // (what a failed launch was to read is kept)
        }
    }
};

constexpr const char *kStageName = "cuke_amd.sampler_stage";

// sampler_stage(batch): a handle for sample_batch
PyObject *py_sampler_stage(PyObject *, PyObject *o)
{
    HANDLE_TH_ERRORS
    const int64_t batch = PyLong_AsLongLong(o);
    if (batch == -1 && PyErr_Occurred()) return nullptr;
    Stage *s = new Stage;
    s->batch = batch;
    return PyCapsule_New(s, kStageName, [](PyObject *c) { delete static_cast<Stage *>(PyCapsule_GetPointer(c, kStageName)); });
    END_HANDLE_TH_ERRORS
}

// sample_batch(stage, h, r, t, order: host arrays, position, count, n_ent, seed, step, device) -> (h, r, t, neg) or None.  The triples
// order[position ..) are gathered into the stage's pinned memory, which one launch reads where it draws the negatives:
// no copy for the host to wait for, and the arrays are read as they are at this call.
PyObject *py_sample_batch(PyObject *, PyObject *const *args, Py_ssize_t)
{
    HANDLE_TH_ERRORS
    Stage *stage = static_cast<Stage *>(PyCapsule_GetPointer(args[0], kStageName));
    if (!stage) return nullptr;
    HostIds col[3], order;
    for (int k = 0; k < 3; ++k)
        if (!col[k].take(args[1 + k])) NOT_HERE;
    if (!order.take(args[4])) NOT_HERE;
    const int64_t at0 = PyLong_AsLongLong(args[5]), count = PyLong_AsLongLong(args[6]), n_ent = PyLong_AsLongLong(args[7]);
    const uint64_t seed = PyLong_AsUnsignedLongLongMask(args[8]), step = PyLong_AsUnsignedLongLongMask(args[9]);
    const int64_t asked = PyLong_AsLongLong(args[10]);  // device index, -1: the current one
    if (PyErr_Occurred()) return nullptr;
    const int dev = c10::hip::current_device();
    const int64_t B = stage->batch;
    if ((asked >= 0 && asked != dev) || at0 < 0 || B <= 0 || count < 0 || at0 > order.size() - B) NOT_HERE;
    void *st = stream();
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(static_cast<hipStream_t>(st), &capture) != hipSuccess || capture != hipStreamCaptureStatusNone)
        NOT_HERE;  // (a replay would read what a later batch has left there)
    const auto i64 = at::TensorOptions().dtype(at::kLong).device(at::kCUDA, (c10::DeviceIndex)dev);
    at::Tensor h = at::empty({B}, i64), r = at::empty({B}, i64), t = at::empty({B}, i64), neg = at::empty({count}, i64);
    Stage::Slot *slot = stage->take();  // (nothing lets another thread in between here and the new mark below)
    if (!slot) NOT_HERE;
    int64_t *ids = slot->ids;
    const uint64_t rows = (uint64_t)std::min({col[0].size(), col[1].size(), col[2].size()});
    bool inside = true;
    for (int64_t i = 0; i < B; ++i) {
        const uint64_t q = (uint64_t)order.at(at0 + i);
        if (!(inside = q < rows)) break;
        ids[i] = col[0].at(q), ids[B + i] = col[1].at(q), ids[2 * B + i] = col[2].at(q);
    }
    if (!inside) NOT_HERE;  // (numpy's indexing raises, or counts from the end)
    uint32_t *done = slot->done;
    const uint32_t mark = ++slot->mark;  // (taken from here on, also for a thread that comes in while the launch is under way)
    const int rc = nogil([&] {
        return kge_sample_staged_batch(ids, B, h.data_ptr<int64_t>(), r.data_ptr<int64_t>(), t.data_ptr<int64_t>(), neg.data_ptr<int64_t>(), count,
                                       n_ent, seed, step, done, mark, st);
    });
    if (rc) return fail(rc, "kge_sample_staged_batch"), nullptr;
    return Py_BuildValue("(NNNN)", wrap(h), wrap(r), wrap(t), wrap(neg));
    END_HANDLE_TH_ERRORS
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"set_error", py_set_error, METH_O, nullptr},
                         FAST(inspect),
                         FAST(score),
                         FAST(backward),
                         FAST(call),
                         FAST(margin_loss),
                         FAST(sparse_step),
                         {"sampler_stage", py_sampler_stage, METH_O, nullptr},
                         FAST(sample_batch),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
