// The host side of one call: checks, output and workspace tensors, strides and the launch through the C ABI
// (include/sparseattn.h), for the Python wrappers of sparse_attn_kernel.py and mask_utils.py.
//
// Why native: a small call's kernels take 10 to 40 us, and the same steps in Python with ctypes took 27 us for a forward
// with metadata, 68 us with the mask classified on the way and 220 us for a training step, so the device waited for the
// host.  Nothing is kept between calls; every workspace is a tensor of the caching allocator, ordered by the stream.
//
// The interpreter's lock is held while Python objects are read (arguments, metadata) and let go of for the rest, so that a
// launch that waits for room in a queue, or an allocation that waits for the device, stops no other thread.
//
// Errors are the Python exceptions the wrappers document: ValueError, TypeError, AssertionError, RuntimeError, and
// SparseAttnError for the library's own error codes.
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <cmath>
#include <memory>
#include <optional>
#include <string>

#include "sparseattn.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

[[noreturn]] void value_error(const std::string &m) { throw py::value_error(m); }
[[noreturn]] void type_error(const std::string &m) { throw py::type_error(m); }
[[noreturn]] void assertion(const char *m) {
    const py::gil_scoped_acquire gil;
    PyErr_SetString(PyExc_AssertionError, m);
    throw py::error_already_set();
}

std::string str(at::IntArrayRef s) {
    std::string out = "(";
    for (size_t i = 0; i < s.size(); i++) out += (i ? ", " : "") + std::to_string(s[i]);
    return out + (s.size() == 1 ? ",)" : ")");
}
std::string str(const Tensor &t) { return std::string(c10::toString(t.scalar_type())) + " " + str(t.sizes()) + " on " + t.device().str(); }

void check_rc(int rc) {
    if (rc == SA_OK) return;
    if (rc == SA_ERR_INVALID_ARGUMENT) value_error(std::string("libsparseattn_hip: ") + sa_last_error());
    const py::gil_scoped_acquire gil;
    const py::object cls = py::module_::import("sparseattention_amd._native").attr("SparseAttnError");
    const py::object err = cls(rc, py::str(sa_last_error()));
    PyErr_SetObject(cls.ptr(), err.ptr());
    throw py::error_already_set();
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

const int64_t *st(const Tensor &t) { return t.strides().data(); }
const int64_t *st(const OptTensor &t) { return t ? t->strides().data() : nullptr; }
template <class T>
T *ptr(const Tensor &t) { return static_cast<T *>(t.data_ptr()); }
template <class T>
T *ptr(const OptTensor &t) { return t ? static_cast<T *>(t->data_ptr()) : nullptr; }

int dtype_code(at::ScalarType t) {
    return t == at::kBFloat16 ? SA_DTYPE_BF16 : t == at::kHalf ? SA_DTYPE_FP16 : t == at::kFloat ? SA_DTYPE_FP32 : -1;
}

// Every tensor whose address goes to a kernel must live where `ref` lives.
void same_device(const Tensor &ref, const char *name, const Tensor &t) {
    if (t.device() != ref.device())
        value_error(std::string(name) + " is on " + t.device().str() + ", expected " + ref.device().str() +
                    " (every tensor argument must be on q's device)");
}
void same_device(const Tensor &ref, const char *name, const OptTensor &t) {
    if (t) same_device(ref, name, *t);
}

// The kernels want a unit stride in D and 16-byte aligned rows; copied only when that does not hold.
Tensor kernel_ready(const Tensor &t) {
    const int64_t per16 = 16 / t.element_size();
    bool ok = t.stride(-1) == 1 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
    for (int64_t d = 0; d + 1 < t.dim(); d++) ok = ok && t.stride(d) % per16 == 0;
    return ok ? t : t.contiguous();
}
// The head dim the kernels run a request for D with: the smallest that holds it (q, k, v are then padded with zero columns,
// which change neither the scores nor the first D columns of the result; the softmax scale stays that of D).  A D beyond
// all of them is passed on, for the library to refuse.
int64_t kernel_head_dim(int64_t D, bool has256) { return D <= 64 ? 64 : D <= 128 ? 128 : has256 && D <= 256 ? 256 : D; }
Tensor pad_head_dim(const Tensor &t, int64_t Dk) {
    return t.size(-1) == Dk ? t : at::constant_pad_nd(t, {0, Dk - t.size(-1)});
}
Tensor cut_head_dim(const Tensor &t, int64_t D) { return t.size(-1) == D ? t : t.narrow(-1, 0, D).contiguous(); }

bool pow2_from_16(int64_t n) { return n >= 16 && (n & (n - 1)) == 0; }
double scale_log2(int64_t D) { return 1.0 / std::sqrt((double)D) * 1.0 / std::log(2.0); }  // exp2 replaces exp (sparse_attn_kernel.py:152)

// ---- the tile lists of a mask -------------------------------------------------------------------------------------
struct Lists {
    Tensor fid, fl, pid, pl;
    OptTensor packed;
};

// Attribute of a metadata object: a new reference, or an empty object where there is none or it is None.  Names are interned
// once, or every look-up would make a string and miss the type's cache of attributes.
struct Name {
    const char *text;
    mutable PyObject *str = nullptr;
};
py::object attr(py::handle o, const Name &name) {
    if (!name.str) name.str = PyUnicode_InternFromString(name.text);
    PyObject *v = name.str ? PyObject_GetAttr(o.ptr(), name.str) : nullptr;
    if (!v) {
        if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw py::error_already_set();
        PyErr_Clear();
        return py::object();
    }
    if (v == Py_None) {
        Py_DECREF(v);
        return py::object();
    }
    return py::reinterpret_steal<py::object>(v);
}
// (read under the interpreter's lock)
const Name kFullIds{"unmasked_kv_ids"}, kFullLens{"unmasked_lens"}, kPartIds{"masked_kv_ids"}, kPartLens{"masked_lens"}, kPacked{"packed_masks"},
    kValidatedFor{"_validated_for"}, kSchedule{"schedule"}, kScheduleMode{"schedule_mode"}, kListStats{"list_stats"}, kListRotation{"list_rotation"},
    kByQuery{"by_query"}, kByKey{"by_key"}, kTransposedMask{"transposed_mask"}, kAgreeing{"_agreeing"};
Tensor tensor_attr(py::handle o, const Name &name) {
    const py::object v = attr(o, name);
    if (!v || !THPVariable_Check(v.ptr())) type_error(std::string("mask_metadata.") + name.text + " is not a tensor");
    return THPVariable_Unpack(v.ptr());
}
OptTensor opt_tensor_attr(py::handle o, const Name &name) {
    const py::object v = attr(o, name);
    if (!v) return std::nullopt;
    if (!THPVariable_Check(v.ptr())) type_error(std::string("mask_metadata.") + name.text + " is not a tensor");
    return THPVariable_Unpack(v.ptr());
}

Lists lists_of(py::handle md) {
    return {tensor_attr(md, kFullIds), tensor_attr(md, kFullLens), tensor_attr(md, kPartIds),
            tensor_attr(md, kPartLens), opt_tensor_attr(md, kPacked)};
}

bool int_is(PyObject *o, unsigned long long want) { return (PyLong_Check(o) ? PyLong_AsUnsignedLongLongMask(o) : ~want) == want; }

// Whether md._validated_for is mask_utils.validation_key(md, Sk, BK): the sizes, then address and version counter of the
// four list tensors.
bool validated(py::handle md, const Lists &l, int64_t Sk, int64_t BK) {
    const py::object key = attr(md, kValidatedFor);
    if (!key || !PyTuple_Check(key.ptr()) || PyTuple_GET_SIZE(key.ptr()) != 6) return false;
    if (!int_is(PyTuple_GET_ITEM(key.ptr(), 0), (unsigned long long)Sk) || !int_is(PyTuple_GET_ITEM(key.ptr(), 1), (unsigned long long)BK)) return false;
    const Tensor *t[4] = {&l.fid, &l.fl, &l.pid, &l.pl};
    for (int i = 0; i < 4; i++) {
        PyObject *e = PyTuple_GET_ITEM(key.ptr(), 2 + i);
        if (!PyTuple_Check(e) || PyTuple_GET_SIZE(e) != 2 || !int_is(PyTuple_GET_ITEM(e, 0), (unsigned long long)(uintptr_t)t[i]->data_ptr()) ||
            !int_is(PyTuple_GET_ITEM(e, 1), (unsigned long long)t[i]->_version()))
            return false;
    }
    return true;
}
void checked_metadata(py::handle md, const Lists &l, int64_t Sk, int64_t BK) {
    if (!validated(md, l, Sk, BK))
        py::module_::import("sparseattention_amd.sparse_attn_kernel").attr("_checked_metadata")(md, Sk, BK);
}

void check_lists(const Lists &l, const Tensor &ref, int64_t B, int64_t H, int64_t nQ, int64_t nK, const char *what) {
    const int64_t ids[4] = {B, H, nQ, nK};
    const Tensor *t[4] = {&l.fid, &l.pid, &l.fl, &l.pl};
    const char *name[4] = {"unmasked_kv_ids", "masked_kv_ids", "unmasked_lens", "masked_lens"};
    for (int i = 0; i < 4; i++) {
        const at::IntArrayRef want(ids, i < 2 ? 4 : 3);
        if (t[i]->sizes() != want || t[i]->scalar_type() != at::kInt || t[i]->device() != ref.device())
            value_error(std::string(what) + "." + name[i] + ": expected int32 " + str(want) + " on " + ref.device().str() + ", got " + str(*t[i]));
    }
}
void check_packed(const Tensor &pk, const Tensor &ref, int64_t B, int64_t H, int64_t nQ, int64_t nK, int64_t tile_bytes, const char *what) {
    const int64_t want[5] = {B, H, nQ, nK, tile_bytes};
    if (pk.sizes() != at::IntArrayRef(want, 5) || pk.scalar_type() != at::kByte || pk.device() != ref.device() ||
        pk.stride(2) != nK * tile_bytes || pk.stride(3) != tile_bytes || pk.stride(4) != 1)
        value_error(std::string(what) + ".packed_masks: expected uint8 " + str(at::IntArrayRef(want, 5)) + " on " + ref.device().str() +
                    " with contiguous tiles, got " + str(pk) + " strides " + str(pk.strides()));
}

// The tensors a classification fills: distinct planes only, seen through the whole [B,H] by stride 0.
Lists empty_lists(int64_t uB, int64_t uH, int64_t B, int64_t H, int64_t nQ, int64_t nK, int64_t tile_bytes, bool pack, const at::Device &dev) {
    const auto i32 = at::TensorOptions().dtype(at::kInt).device(dev);
    // (one allocation for the four: offsets are multiples of four bytes, and the views keep it alive)
    const int64_t planes = uB * uH, ids = planes * nQ * nK, lens = planes * nQ;
    const Tensor all = at::empty({2 * ids + 2 * lens}, i32);
    const int64_t sB = uB == 1 && B > 1 ? 0 : uH * nQ, sH = uH == 1 && H > 1 ? 0 : nQ;
    auto ids_at = [&](int64_t o) { return all.as_strided({B, H, nQ, nK}, {sB * nK, sH * nK, nK, 1}, o); };
    auto lens_at = [&](int64_t o) { return all.as_strided({B, H, nQ}, {sB, sH, 1}, o); };
    Lists l{ids_at(0), lens_at(2 * ids), ids_at(ids), lens_at(2 * ids + lens), std::nullopt};
    if (pack)
        l.packed = at::empty({uB, uH, nQ, nK, tile_bytes}, at::TensorOptions().dtype(at::kByte).device(dev)).expand({B, H, nQ, nK, tile_bytes});
    return l;
}

Lists classify_lists(const Tensor &mask, int64_t BQ, int64_t BK, std::optional<bool> pack_partial) {
    if (mask.dim() != 4) value_error("mask must be [B,H,Sq,Sk] (got " + str(mask.sizes()) + "); use mask.expand(B,H,Sq,Sk)");
    const int64_t B = mask.size(0), H = mask.size(1), Sq = mask.size(2), Sk = mask.size(3);
    // the reference asserts these (mask_utils.py:18-20, :89-90)
    if (mask.scalar_type() != at::kBool) assertion("mask must be a torch.bool tensor");
    if (BQ <= 0 || Sq % BQ) assertion("Sq must be a multiple of BLOCK_Q");
    if (BK <= 0 || Sk % BK) assertion("Sk must be a multiple of BLOCK_K");
    if (!mask.is_cuda()) throw std::runtime_error("compute_mask_kernel needs the mask on a ROCm GPU; compute_mask_slow runs anywhere");
    const bool pack = pack_partial.value_or(BK % 8 == 0);
    if (pack && BK % 8) value_error("pack_partial needs BLOCK_K to be a multiple of 8 (got " + std::to_string(BK) + ")");
    const int64_t uB = mask.stride(0) == 0 || B == 1 ? 1 : B, uH = mask.stride(1) == 0 || H == 1 ? 1 : H;
    const int64_t nQ = Sq / BQ, nK = Sk / BK;
    const c10::DeviceGuard guard(mask.device());
    void *const stream = stream_of(mask);
    Lists l = empty_lists(uB, uH, B, H, nQ, nK, BQ * BK / 8, pack, mask.device());
    const size_t need = sa_mask_classify_workspace_bytes(st(mask), B, H, Sq, Sk, BQ, BK);
    // (dropped at the end of this call: the allocator hands the block out again only behind these launches on the stream)
    const Tensor ws = at::empty({(int64_t)std::max<size_t>(need, 1)}, at::TensorOptions().dtype(at::kByte).device(mask.device()));
    if (pack)
        check_rc(sa_mask_classify_packed(ptr<uint8_t>(mask), st(mask), B, H, Sq, Sk, BQ, BK, ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl),
                                         ptr<int32_t>(l.pid), st(l.pid), ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(*l.packed), st(*l.packed),
                                         ws.data_ptr(), ws.numel(), stream));
    else
        check_rc(sa_mask_classify(ptr<uint8_t>(mask), st(mask), B, H, Sq, Sk, BQ, BK, ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl),
                                  ptr<int32_t>(l.pid), st(l.pid), ptr<int32_t>(l.pl), st(l.pl), ws.data_ptr(), ws.numel(), stream));
    return l;
}

py::tuple as_tuple(const Lists &l) { return py::make_tuple(l.fid, l.fl, l.pid, l.pl, l.packed ? py::cast(*l.packed) : py::none()); }

// compute_mask_kernel: (unmasked_kv_ids, unmasked_lens, masked_kv_ids, masked_lens, packed_masks or None)
py::tuple classify(const Tensor &mask, int64_t BQ, int64_t BK, std::optional<bool> pack_partial) {
    Lists l;
    {
        const py::gil_scoped_release unlocked;
        l = classify_lists(mask, BQ, BK, pack_partial);
    }
    return as_tuple(l);
}

// compute_mask_terms: the same from terms, eight int32 each (their and the documents' shapes are checked by the caller)
int64_t terms_planes(int64_t B, const OptTensor &doc_q, const OptTensor &doc_k) {
    const bool per_batch = B > 1 && ((doc_q && doc_q->stride(0) != 0) || (doc_k && doc_k->stride(0) != 0));
    return per_batch ? B : 1;
}

py::tuple classify_terms(const std::vector<int32_t> &terms, int64_t B, int64_t H, int64_t Sq, int64_t Sk, int64_t BQ, int64_t BK,
                         const OptTensor &doc_q, const OptTensor &doc_k, bool pack, const at::Device &dev) {
    const int64_t nQ = Sq / BQ, nK = Sk / BK;
    const int64_t uB = terms_planes(B, doc_q, doc_k);
    Lists l;
    {
        const py::gil_scoped_release unlocked;
        const c10::DeviceGuard guard(dev);
        l = empty_lists(uB, 1, B, H, nQ, nK, BQ * BK / 8, pack, dev);
        const size_t need = sa_mask_terms_workspace_bytes(uB, Sq, Sk, BQ, BK);
        const Tensor ws = at::empty({(int64_t)std::max<size_t>(need, 1)}, at::TensorOptions().dtype(at::kByte).device(dev));
        check_rc(sa_mask_classify_terms(terms.data(), (int)(terms.size() / 8), ptr<int32_t>(doc_q), st(doc_q), ptr<int32_t>(doc_k), st(doc_k), B, H, Sq,
                                        Sk, BQ, BK, ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl), ptr<int32_t>(l.pid), st(l.pid),
                                        ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(l.packed), st(l.packed), ws.data_ptr(), ws.numel(), stream_of(l.fid)));
    }
    return as_tuple(l);
}

// compute_backward_metadata_terms: the mask by query rows and, from its transposed terms, by keys (tiles of 128 x 64 both), packed
py::tuple classify_terms_backward(const std::vector<int32_t> &terms, const std::vector<int32_t> &transposed, int64_t B, int64_t H, int64_t Sq,
                                  int64_t Sk, const OptTensor &doc_q, const OptTensor &doc_k, const at::Device &dev) {
    constexpr int64_t BQ = 128, BK = 64;
    const int64_t uB = terms_planes(B, doc_q, doc_k);
    Lists l[2];
    {
        const py::gil_scoped_release unlocked;
        const c10::DeviceGuard guard(dev);
        const size_t need[2] = {sa_mask_terms_workspace_bytes(uB, Sq, Sk, BQ, BK), sa_mask_terms_workspace_bytes(uB, Sk, Sq, BQ, BK)};
        const Tensor ws = at::empty({(int64_t)std::max<size_t>(need[0] + need[1], 1)}, at::TensorOptions().dtype(at::kByte).device(dev));
        sa_mask_terms_call call[2];
        for (int i = 0; i < 2; i++) {
            const int64_t rows = i == 0 ? Sq : Sk, keys = i == 0 ? Sk : Sq;
            const std::vector<int32_t> &t = i == 0 ? terms : transposed;
            const OptTensor &dr = i == 0 ? doc_q : doc_k, &dk = i == 0 ? doc_k : doc_q;
            l[i] = empty_lists(uB, 1, B, H, rows / BQ, keys / BK, BQ * BK / 8, true, dev);
            call[i] = {t.data(), (int)(t.size() / 8), ptr<int32_t>(dr), st(dr), ptr<int32_t>(dk), st(dk), (int)B, (int)H, (int)rows, (int)keys,
                       (int)BQ, (int)BK, ptr<int32_t>(l[i].fid), st(l[i].fid), ptr<int32_t>(l[i].fl), st(l[i].fl), ptr<int32_t>(l[i].pid),
                       st(l[i].pid), ptr<int32_t>(l[i].pl), st(l[i].pl), ptr<uint8_t>(l[i].packed), st(l[i].packed),
                       ptr<uint8_t>(ws) + (i == 0 ? 0 : need[0]), need[i]};
        }
        check_rc(sa_mask_classify_terms_pair(&call[0], &call[1], stream_of(l[0].fid)));
    }
    return py::make_tuple(as_tuple(l[0]), as_tuple(l[1]));
}

// ---- decode -------------------------------------------------------------------------------------------------------
struct Out {
    Tensor o;
    OptTensor lse;
};
py::object as_object(const Out &r) { return r.lse ? py::object(py::make_tuple(r.o, *r.lse)) : py::cast(r.o); }

void check_qkv(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask, const char *what) {
    if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) value_error("q, k, v must be [B,H,S,D]");
    const int64_t want[4] = {q.size(0), q.size(1), k.size(2), q.size(3)};
    if (k.sizes() != at::IntArrayRef(want, 4) || v.sizes() != k.sizes())
        value_error("k/v shapes " + str(k.sizes()) + "/" + str(v.sizes()) + " do not match q " + str(q.sizes()));
    if (!q.is_cuda()) throw std::runtime_error(std::string(what) + " needs q, k, v on a ROCm GPU; there is no CPU path");
    same_device(q, "k", k);
    same_device(q, "v", v);
    same_device(q, "mask", mask);
}

Out decode_impl(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask_in, int64_t BK, py::handle md, int64_t num_splits, bool return_lse) {
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Sk = k.size(2);
    const int dt = dtype_code(q.scalar_type());
    if ((dt != SA_DTYPE_BF16 && dt != SA_DTYPE_FP16) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
        type_error(std::string("q, k, v must share dtype bfloat16 or float16 (got ") + c10::toString(q.scalar_type()) + ", " +
                   c10::toString(k.scalar_type()) + ", " + c10::toString(v.scalar_type()) + ")");
    OptTensor mask = mask_in;
    if (mask) mask = mask->expand({B, H, Sq, Sk});
    Lists l;
    const bool has_md = !md.is_none();
    if (has_md) {
        l = lists_of(md);
        if (BK <= 0) value_error("BLOCK_K must be positive");
        check_lists(l, q, B, H, 1, Sk / BK, "mask_metadata");
        checked_metadata(md, l, Sk, BK);
        if (l.packed) check_packed(*l.packed, q, B, H, 1, Sk / BK, Sq * BK / 8, "mask_metadata");
    }
    const py::gil_scoped_release unlocked;
    // (a small mask without lists: the decode kernel finds its tiles in it; what the classification refuses goes there)
    const bool direct = !has_md && mask && mask->scalar_type() == at::kBool && BK > 0 && BK <= Sk &&
                        sa_decode_mask_fits(ptr<uint8_t>(*mask), st(*mask), B, H, Sq, Sk, BK);
    if (!has_md && !direct) {
        if (!mask) value_error("sparse_attention_decode needs the mask or mask_metadata with packed_masks");
        l = classify_lists(*mask, Sq, BK, std::nullopt);
    }
    if (l.packed && BK == 16 && Sq % 2) l.packed.reset();  // (halfword rows: the kernels want an even number of them)
    if (!l.packed) {
        if (!mask)
            value_error("sparse_attention_decode without a mask tensor needs mask_metadata with packed_masks (and an even number of query rows at BLOCK_K = 16)");
        if (mask->scalar_type() != at::kBool) assertion("mask must be a torch.bool tensor");
    }
    const int64_t Dk = kernel_head_dim(D, false);
    const c10::DeviceGuard guard(q.device());
    const Tensor qc = kernel_ready(pad_head_dim(q, Dk)), kc = kernel_ready(pad_head_dim(k, Dk)), vc = kernel_ready(pad_head_dim(v, Dk));
    const Tensor o = at::empty_like(qc);
    const auto f32 = at::TensorOptions().dtype(at::kFloat).device(q.device());
    if (num_splits == 0) num_splits = sa_decode_num_splits(B, H, Sq, Sk, BK);
    const size_t ws_bytes = sa_decode_workspace_bytes_ex(B, H, Sq, Dk, num_splits);
    Tensor ws;
    if (ws_bytes) ws = at::empty({(int64_t)(ws_bytes / 4)}, f32);
    OptTensor lse;
    if (return_lse) lse = at::empty({B, H, Sq}, f32);
    if (direct) {
        check_rc(sa_sparse_attention_decode_mask(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o),
                                                 ptr<uint8_t>(*mask), st(*mask), B, H, Sq, Sk, Dk, BK, dt, (float)scale_log2(D), num_splits,
                                                 ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, ptr<float>(lse), st(lse), stream_of(q)));
        return {cut_head_dim(o, D), lse};
    }
    check_rc(sa_sparse_attention_decode_ex(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o), ptr<uint8_t>(mask),
                                           st(mask), ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl), ptr<int32_t>(l.pid), st(l.pid),
                                           ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(l.packed), st(l.packed), B, H, Sq, Sk, Dk, BK, dt,
                                           (float)scale_log2(D), num_splits, ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, ptr<float>(lse), st(lse),
                                           stream_of(q)));
    return {cut_head_dim(o, D), lse};
}

py::object decode(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask, int64_t BK, py::object md, int64_t num_splits, bool return_lse) {
    check_qkv(q, k, v, mask, "sparse_attention_decode");
    return as_object(decode_impl(q, k, v, mask, BK, md, num_splits, return_lse));
}

// ---- forward ------------------------------------------------------------------------------------------------------
// Whether the kernels tile by the caller's own sizes (kernel_tiles of sparse_attn_kernel.py returns them unchanged).
bool tiles_as_asked(int64_t Sq, int64_t Sk, int64_t D, int64_t BQ, int64_t BK, bool f32) {
    if (BQ < 1 || BK < 1 || Sq % BQ || Sk % BK) return false;
    if (f32 && BQ <= (D <= 128 ? 256 : 128)) return true;  // the float32 kernels tile by any sizes up to that
    if (!pow2_from_16(BK)) return false;
    if (Sq < 32) return D <= 128 && BQ == Sq;
    return BQ == 128 || BQ == 64 || (D <= 128 && (BQ == 32 || BQ == 256));
}

// Below this many listed keys per Q tile (mean over the Q tiles) the forward runs its short-list kernel when the
// metadata says so (MaskMetadata.list_stats) and the kernel has the sizes.  Measured on MI355X (B8 H32 S4096 D128,
// tiles 128x32, default / short-list kernel): 448 keys per Q tile 0.343 / 0.340 ms, 1222 keys 0.709 / 0.719 ms,
// 2100 keys and more +5 ... +8 %: the third workgroup per compute unit pays for itself on the shortest lists only.
constexpr double kShortListKeys = 512;

// What a metadata object says besides its lists.
struct Hints {
    OptTensor sched;
    int sched_mode = 0;
    bool stats = false;  // list_stats: mean and longest number of listed tiles per Q tile
    double mean_list = 0;
    int64_t longest_list = 0, rotation = 0;
};
Hints hints_of(py::handle md) {
    Hints h;
    h.sched = opt_tensor_attr(md, kSchedule);
    if (h.sched)
        if (const py::object m = attr(md, kScheduleMode)) h.sched_mode = m.cast<int>();
    if (const py::object s = attr(md, kListStats)) {
        h.stats = true;
        h.mean_list = s[py::int_(0)].cast<double>();
        h.longest_list = s[py::int_(1)].cast<int64_t>();
    }
    if (const py::object r = attr(md, kListRotation)) h.rotation = r.cast<int64_t>();
    return h;
}

// Which of the forward kernels a call runs, as a code of the C ABI.
int choose_kernel(const std::string &kernel, bool f32, int64_t Dk, int64_t BQ, int64_t BK, bool packed, const Hints &h) {
    if (kernel != "auto" && kernel != "default" && kernel != "short" && kernel != "rotated")
        value_error("kernel must be 'auto', 'default', 'rotated' or 'short' (got '" + kernel + "')");
    if (kernel == "rotated" && (h.sched || f32)) value_error("kernel='rotated' needs bf16/fp16 and mask_metadata without a schedule");
    const bool short_has = !f32 && Dk == 128 && BQ == 128 && pow2_from_16(BK) && packed && !h.sched;
    const bool short_fits = h.stats && h.longest_list <= SA_FWD_SHORT_LISTS_MAX_ENTRIES;
    if (kernel == "short") {
        if (!(short_has && short_fits))
            value_error("kernel='short' needs bf16/fp16, head dim 128, BLOCK_Q 128, mask_metadata with packed_masks, no schedule, and list_stats whose longest list has at most " +
                        std::to_string(SA_FWD_SHORT_LISTS_MAX_ENTRIES) + " entries");
        return SA_FWD_KERNEL_SHORT_LISTS;
    }
    if (kernel == "auto" && short_has && short_fits && h.mean_list * (double)BK < kShortListKeys) return SA_FWD_KERNEL_SHORT_LISTS;
    // the default kernel with the FULL entries of Q tile qt walked from a start that depends on qt
    if (!h.sched && !f32 && (kernel == "rotated" || (kernel == "auto" && h.rotation > 0)))
        return SA_FWD_KERNEL_ROTATED | ((int)(h.rotation ? h.rotation : 16) << 8);
    return SA_FWD_KERNEL_DEFAULT;
}
// The same by name ("default", "short" or "rotated"), for reports on what a call with this metadata runs.
std::string forward_kernel(const Tensor &q, int64_t BQ, int64_t BK, py::object md, const std::string &kernel) {
    const bool packed = (bool)attr(md, kPacked);
    const int code = choose_kernel(kernel, q.scalar_type() == at::kFloat, kernel_head_dim(q.size(-1), true), BQ, BK, packed, hints_of(md)) & 0xff;
    return code == SA_FWD_KERNEL_SHORT_LISTS ? "short" : code == SA_FWD_KERNEL_ROTATED ? "rotated" : "default";
}

// How a call with the default kernel hands its lists out: one workgroup each, or as sa_sparse_attention_fwd_split does (which needs
// ws_bytes).  Metadata that says that no list is long enough to gain by it (list_stats) keeps them whole: 128 tiles of 16 chunks
// 22.9 -> 20.0 us, no merge that finds nothing; 256 tiles of 64 rows, lists of 4 chunks 10.9 -> 10.2, of 128 rows and 8 chunks
// 14.9 -> 13.6, no workgroups of twice the waves.  So does metadata that says that they are too much alike for assistants.
struct ListsShared {
    bool whole;
    size_t ws_bytes = 0;
    bool assistants = false;  // only they need the workspace: a call whose parts find no place goes without
};
ListsShared lists_shared(const Hints &h, int64_t B, int64_t H, int64_t Sq, int64_t Sk, int64_t Dk, int64_t BQ, int64_t BK, int dt) {
    if (h.stats && h.longest_list * BK <= sa_fwd_split_least_keys(B, H, Sq, Sk, Dk, BQ, BK, dt)) return {true};
    const size_t bytes = sa_fwd_split_workspace_bytes(B, H, Sq, Sk, Dk, BQ, BK, dt);
    const int uneven = bytes != 0 ? sa_fwd_split_uneven_keys(B, H, Sq, Sk, Dk, BQ, BK, dt) : 0;
    if (h.stats && ((double)h.longest_list - h.mean_list) * (double)BK < uneven) return {true};
    return {false, bytes, uneven > 0};
}
// The same by name, for reports on what a call without a schedule runs: "whole", "halves" or "shared".
std::string forward_lists(const Tensor &q, int64_t Sk, int64_t BQ, int64_t BK, py::object md) {
    const c10::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), Dk = kernel_head_dim(q.size(3), true);
    const int dt = dtype_code(q.scalar_type());
    const ListsShared s = lists_shared(hints_of(md), B, H, Sq, Sk, Dk, BQ, BK, dt);
    if (s.whole || (s.ws_bytes == 0 && sa_fwd_split_least_keys(B, H, Sq, Sk, Dk, BQ, BK, dt) == Sk)) return "whole";
    return s.ws_bytes ? "shared" : "halves";
}

// Whether tensors of these sizes run on a larger tile grid as they are (sa_sparse_attention_fwd_ragged): nothing is padded.
bool ragged_has(const Tensor &q, int64_t BQ, int64_t BK, const Lists &l) {
    const int dt = dtype_code(q.scalar_type());
    return (dt == SA_DTYPE_BF16 || dt == SA_DTYPE_FP16) && q.size(3) % 8 == 0 && q.size(3) <= 128 && (BQ == 32 || BQ == 64 || BQ == 128) &&
           pow2_from_16(BK) && l.packed.has_value();
}
// (called without the interpreter's lock)
Out ragged_forward(const Tensor &q, const Tensor &k, const Tensor &v, const Lists &l, int64_t BQ, int64_t BK, int64_t q0, int64_t k0, int64_t Pq,
                   int64_t Pk, bool return_lse) {
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Sk = k.size(2);
    const c10::DeviceGuard guard(q.device());
    const Tensor qc = kernel_ready(q), kc = kernel_ready(k), vc = kernel_ready(v), o = at::empty_like(qc);
    OptTensor lse;
    if (return_lse) lse = at::empty({B, H, Sq}, at::TensorOptions().dtype(at::kFloat).device(q.device()));
    check_rc(sa_sparse_attention_fwd_ragged(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o), ptr<int32_t>(l.fid),
                                            st(l.fid), ptr<int32_t>(l.fl), st(l.fl), ptr<int32_t>(l.pid), st(l.pid), ptr<int32_t>(l.pl), st(l.pl),
                                            ptr<uint8_t>(*l.packed), st(*l.packed), ptr<float>(lse), st(lse), B, H, Sq, Sk, D, BQ, BK, q0, k0, Pq, Pk,
                                            dtype_code(q.scalar_type()), (float)scale_log2(D), stream_of(q)));
    return {o, lse};
}

// The forward where the kernels tile by the caller's sizes, or nothing (then the wrapper makes other tiles of the mask).
std::optional<Out> forward_impl(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask_in, int64_t BQ, int64_t BK, py::handle md,
                                bool return_lse, const std::string &kernel) {
    check_qkv(q, k, v, mask_in, "sparse_attention");
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Sk = k.size(2);
    const int dt = dtype_code(q.scalar_type());
    if (dt < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
        type_error(std::string("q, k, v must share dtype bfloat16, float16 or float32 (got ") + c10::toString(q.scalar_type()) + ", " +
                   c10::toString(k.scalar_type()) + ", " + c10::toString(v.scalar_type()) + ")");
    const bool f32 = dt == SA_DTYPE_FP32, has_md = !md.is_none();
    if (!mask_in && !(has_md && attr(md, kPacked)))
        value_error("sparse_attention without a mask tensor needs mask_metadata with packed_masks");
    OptTensor mask = mask_in;
    if (mask) mask = mask->expand({B, H, Sq, Sk});
    if (!tiles_as_asked(Sq, Sk, D, BQ, BK, f32)) return std::nullopt;
    // one Q tile of fewer rows than the forward kernels tile by: the split-KV kernels (they use no schedule)
    if (Sq == BQ && Sq < 32 && BK >= 16 && !f32) return decode_impl(q, k, v, mask, BK, md, 0, return_lse);

    const int64_t nQ = Sq / BQ, nK = Sk / BK;
    Lists l;
    Hints hints;
    if (has_md) {
        l = lists_of(md);
        check_lists(l, q, B, H, nQ, nK, "mask_metadata");
        checked_metadata(md, l, Sk, BK);
        if (l.packed) check_packed(*l.packed, q, B, H, nQ, nK, BQ * BK / 8, "mask_metadata");
        hints = hints_of(md);
        if (hints.sched && (hints.sched->scalar_type() != at::kInt || hints.sched->device() != q.device() || !hints.sched->is_contiguous()))
            value_error("mask_metadata.schedule: expected a contiguous int32 tensor on q's device");
    }
    const py::gil_scoped_release unlocked;
    if (!has_md) l = classify_lists(*mask, BQ, BK, std::nullopt);
    if (mask && mask->scalar_type() != at::kBool) assertion("mask must be a torch.bool tensor");

    const int64_t Dk = kernel_head_dim(D, true);
    const OptTensor &sched = hints.sched;
    const int code = choose_kernel(kernel, f32, Dk, BQ, BK, l.packed.has_value(), hints);

    if (D != Dk && !sched && code == SA_FWD_KERNEL_DEFAULT && ragged_has(q, BQ, BK, l))
        return ragged_forward(q, k, v, l, BQ, BK, 0, 0, Sq, Sk, return_lse);

    const c10::DeviceGuard guard(q.device());
    const Tensor qc = kernel_ready(pad_head_dim(q, Dk)), kc = kernel_ready(pad_head_dim(k, Dk)), vc = kernel_ready(pad_head_dim(v, Dk));
    const Tensor o = at::empty_like(qc);
    const auto opt_f32 = at::TensorOptions().dtype(at::kFloat).device(q.device());
    OptTensor lse;
    if (return_lse) lse = at::empty({B, H, Sq}, opt_f32);
    const float scale = (float)scale_log2(D);
    void *const stream = stream_of(q);
    if (sched) {
        check_rc(sa_sparse_attention_fwd_lse(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o), ptr<uint8_t>(mask),
                                             st(mask), ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl), ptr<int32_t>(l.pid), st(l.pid),
                                             ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(l.packed), st(l.packed), ptr<int32_t>(*sched),
                                             sched->numel() * 4, hints.sched_mode, ptr<float>(lse), st(lse), B, H, Sq, Sk, Dk, BQ, BK, dt, scale, stream));
        return Out{cut_head_dim(o, D), lse};
    }
    ListsShared shared{true};
    if (code == SA_FWD_KERNEL_DEFAULT) shared = lists_shared(hints, B, H, Sq, Sk, Dk, BQ, BK, dt);
    Tensor ws;
    if (!shared.whole && shared.ws_bytes != 0) {
        try {
            ws = at::empty({(int64_t)(shared.ws_bytes / 4)}, opt_f32);
        } catch (const c10::OutOfMemoryError &) {  // (shared lists of one workgroup each would be several times as long: for the caller to know)
            if (!shared.assistants) throw;
            shared.whole = true;
        }
    }
    if (shared.whole) {
        check_rc(sa_sparse_attention_fwd_kernel(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o),
                                                ptr<uint8_t>(mask), st(mask), ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl),
                                                ptr<int32_t>(l.pid), st(l.pid), ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(l.packed), st(l.packed),
                                                ptr<float>(lse), st(lse), B, H, Sq, Sk, Dk, BQ, BK, dt, scale, code, stream));
    } else {
        // (too few Q tiles to fill the device: lists are shared by several workgroups, which need a workspace, or walked in halves)
        const size_t ws_bytes = shared.ws_bytes;
        check_rc(sa_sparse_attention_fwd_split(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), o.data_ptr(), st(o),
                                               ptr<uint8_t>(mask), st(mask), ptr<int32_t>(l.fid), st(l.fid), ptr<int32_t>(l.fl), st(l.fl),
                                               ptr<int32_t>(l.pid), st(l.pid), ptr<int32_t>(l.pl), st(l.pl), ptr<uint8_t>(l.packed), st(l.packed),
                                               ptr<float>(lse), st(lse), B, H, Sq, Sk, Dk, BQ, BK, dt, scale, ws_bytes ? ws.data_ptr() : nullptr,
                                               ws_bytes, stream));
    }
    return Out{cut_head_dim(o, D), lse};
}

py::object forward(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask, int64_t BQ, int64_t BK, py::object md, bool return_lse,
                   const std::string &kernel) {
    const auto r = forward_impl(q, k, v, mask, BQ, BK, md, return_lse, kernel);
    return r ? as_object(*r) : py::none();
}

// The forward on the tile grid of a padded mask (sparse_attention_tiled), or None where the wrapper has to pad the tensors.
py::object forward_tiled(const Tensor &q, const Tensor &k, const Tensor &v, int64_t BQ, int64_t BK, int64_t q0, int64_t k0, int64_t Pq, int64_t Pk,
                         py::object md, bool return_lse) {
    check_qkv(q, k, v, std::nullopt, "sparse_attention");
    if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || BQ < 1 || BK < 1 || Pq % BQ || Pk % BK) return py::none();
    const Lists l = lists_of(md);
    if (!ragged_has(q, BQ, BK, l) || attr(md, kSchedule)) return py::none();
    check_lists(l, q, q.size(0), q.size(1), Pq / BQ, Pk / BK, "tiling.metadata");
    checked_metadata(md, l, Pk, BK);
    check_packed(*l.packed, q, q.size(0), q.size(1), Pq / BQ, Pk / BK, BQ * BK / 8, "tiling.metadata");
    Out r;
    {
        const py::gil_scoped_release unlocked;
        r = ragged_forward(q, k, v, l, BQ, BK, q0, k0, Pq, Pk, return_lse);
    }
    return as_object(r);
}

// ---- backward -----------------------------------------------------------------------------------------------------
// What the backward walks: the lists of the mask per 128 queries (KV tiles of 64) and of the transposed mask per 128 keys.
struct BackwardLists {
    Lists by_query, by_key;
    OptTensor transposed_mask;
    bool agree = false;  // both are known to say the same of every entry
};

// The note that a BackwardMetadata carries (_agreeing) when this package made both its lists of one mask: the ten tensors, with
// the addresses and in-place versions they had then.  It keeps them alive, so that nothing else can stand in their place.
// Native, and looked at without a reference taken to any of them, its lists used as they stand: the backward does so on the
// autograd thread, where every object whose count of references changes is a cache line that the two threads take from
// each other.
const Name *const kListNames[5] = {&kFullIds, &kFullLens, &kPartIds, &kPartLens, &kPacked};
struct OneMask {
    BackwardLists lists;
    struct {
        py::object object;
        const void *data;
        int64_t version;
    } was[10];

    const Tensor &tensor(int i) const {
        const Lists &l = i < 5 ? lists.by_query : lists.by_key;
        const Tensor *const t[5] = {&l.fid, &l.fl, &l.pid, &l.pl, &*l.packed};
        return *t[i % 5];
    }
};
// (None for lists without packed tiles, which no path needs it for, and for tensors that do not count their edits)
std::shared_ptr<OneMask> of_one_mask(py::object by_query, py::object by_key) {
    auto n = std::make_shared<OneMask>();
    n->lists = {lists_of(by_query), lists_of(by_key), std::nullopt, true};
    if (!n->lists.by_query.packed || !n->lists.by_key.packed) return nullptr;
    for (int i = 0; i < 10; i++) {
        const Tensor &t = n->tensor(i);
        if (t.is_inference()) return nullptr;
        n->was[i] = {attr(i < 5 ? by_query : by_key, *kListNames[i % 5]), t.data_ptr(), (int64_t)t._version()};
    }
    return n;
}
// The note of bmd where its lists are still those tensors, unedited, or nothing.
std::shared_ptr<OneMask> lists_agree(py::handle bmd, py::handle by_query, py::handle by_key) {
    const py::object made = attr(bmd, kAgreeing);
    if (!made || !py::isinstance<OneMask>(made)) return nullptr;
    auto n = made.cast<std::shared_ptr<OneMask>>();
    for (int l = 0; l < 2; l++) {
        const py::object dict = py::reinterpret_steal<py::object>(PyObject_GenericGetDict((l ? by_key : by_query).ptr(), nullptr));
        if (!dict || !PyDict_Check(dict.ptr())) {
            PyErr_Clear();
            return nullptr;
        }
        for (int i = 5 * l; i < 5 * l + 5; i++) {
            const Tensor &t = n->tensor(i);
            if (PyDict_GetItem(dict.ptr(), kListNames[i % 5]->str) != n->was[i].object.ptr() || t.data_ptr() != n->was[i].data ||
                (int64_t)t._version() != n->was[i].version)
                return nullptr;
        }
    }
    return n;
}

// The lists of a BackwardMetadata: those of its note, or else its own.
struct ReadLists {
    std::shared_ptr<const OneMask> note;
    BackwardLists own;
    const BackwardLists &get() const { return note ? note->lists : own; }
};
ReadLists backward_lists_of(py::handle bmd, const Tensor &q, int64_t Sk) {
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2);
    const py::object mq = attr(bmd, kByQuery), mk = attr(bmd, kByKey);
    if (!mq || !mk) type_error("bwd_metadata has no by_query / by_key lists");
    ReadLists r;
    r.note = lists_agree(bmd, mq, mk);
    const OptTensor mt = opt_tensor_attr(bmd, kTransposedMask);
    if (!r.note || mt) {
        r.own = {lists_of(mq), lists_of(mk), mt, r.note != nullptr};
        r.note.reset();
    }
    const BackwardLists &l = r.get();
    check_lists(l.by_query, q, B, H, Sq / 128, Sk / 64, "bwd_metadata");
    check_lists(l.by_key, q, B, H, Sk / 128, Sq / 64, "bwd_metadata");
    if (!r.note) {  // (lists of this package fit the sizes that their shapes have)
        checked_metadata(mq, l.by_query, Sk, 64);
        checked_metadata(mk, l.by_key, Sq, 64);
    }
    if (l.by_query.packed) check_packed(*l.by_query.packed, q, B, H, Sq / 128, Sk / 64, 1024, "bwd_metadata");
    if (l.by_key.packed) check_packed(*l.by_key.packed, q, B, H, Sk / 128, Sq / 64, 1024, "bwd_metadata");
    if (mt) {
        const int64_t want[4] = {B, H, Sk, Sq};
        if (mt->sizes() != at::IntArrayRef(want, 4) || mt->scalar_type() != at::kBool || mt->device() != q.device())
            value_error("bwd_metadata.transposed_mask: expected bool " + str(at::IntArrayRef(want, 4)) + " on " + q.device().str());
    }
    return r;
}

// The lists made from the mask itself (compute_backward_metadata with packed tiles; Sq and Sk multiples of 128).
BackwardLists backward_lists_from(const Tensor &mask) {
    const int64_t B = mask.size(0), H = mask.size(1);
    const Tensor distinct = mask.narrow(0, 0, mask.stride(0) == 0 ? 1 : B).narrow(1, 0, mask.stride(1) == 0 ? 1 : H);
    const Tensor transposed = distinct.transpose(-1, -2).contiguous().expand({B, H, mask.size(3), mask.size(2)});
    return {classify_lists(mask, 128, 64, true), classify_lists(transposed, 128, 64, true), std::nullopt, true};
}

// What the backward takes of `room` bytes of device memory: a quarter, so that a program near the card's capacity keeps its
// room, and its allocator need not give back what it holds (which waits for the device) to find a block of this size.
int64_t backward_workspace_bytes(int64_t B, int64_t H, int64_t Sq, int64_t Sk, int64_t D, int64_t room) {
    return (int64_t)sa_bwd_workspace_bytes_within(B, H, Sq, Sk, D, (size_t)room / 4);
}
// Bytes that this process can still get on `dev`: free ones, and those its allocator holds without a use for them.
int64_t device_room(const at::Device &dev) {
    int64_t idle = 0;
    try {
        const auto s = c10::hip::HIPCachingAllocator::getDeviceStats(dev.index());
        constexpr auto all = static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE);
        idle = s.reserved_bytes[all].current - s.allocated_bytes[all].current;
    } catch (const c10::Error &) {  // an allocator without statistics
    }
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) free = 0;
    return idle + (int64_t)free;
}

std::tuple<Tensor, Tensor, Tensor> backward_impl(const Tensor &do_, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o, const Tensor &lse,
                                                 const OptTensor &mask, const BackwardLists &l) {
    const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Sk = k.size(2);
    if (!mask && !(l.by_query.packed && l.by_key.packed))
        value_error("sparse_attention_backward without a mask needs packed_masks in both lists of bwd_metadata");
    const int64_t Dk = kernel_head_dim(D, false);
    const c10::DeviceGuard guard(q.device());
    const Tensor qc = kernel_ready(pad_head_dim(q, Dk)), kc = kernel_ready(pad_head_dim(k, Dk)), vc = kernel_ready(pad_head_dim(v, Dk));
    const Tensor oc = kernel_ready(pad_head_dim(o, Dk)), doc = kernel_ready(pad_head_dim(do_, Dk));
    const Tensor dq = at::empty_like(qc), dk = at::empty_like(kc), dv = at::empty_like(vc);
    const Lists &a = l.by_query, &b = l.by_key;
    const auto workspace = [&](size_t bytes) { return at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(q.device())); };
    // dQ from stored dS takes a dS of every entry of by_query that attends, which lists that do not agree do not give
    size_t ws_bytes = sa_bwd_workspace_bytes(B, H, Sq);
    if (a.packed && b.packed && l.agree && sa_bwd_workspace_bytes_ex(B, H, Sq, Sk, Dk) > ws_bytes)
        ws_bytes = backward_workspace_bytes(B, H, Sq, Sk, Dk, device_room(q.device()));
    if (ws_bytes == sa_bwd_workspace_bytes(B, H, Sq)) ws_bytes += sa_bwd_order_bytes(B, H, Sq, Sk, Dk);
    Tensor ws;
    try {
        ws = workspace(ws_bytes);
    } catch (const c10::OutOfMemoryError &) {  // dS finds no place after all: the passes that make it anew
        ws_bytes = sa_bwd_workspace_bytes(B, H, Sq);
        ws = workspace(ws_bytes);
    }
    check_rc(sa_sparse_attention_bwd(qc.data_ptr(), st(qc), kc.data_ptr(), st(kc), vc.data_ptr(), st(vc), oc.data_ptr(), st(oc), doc.data_ptr(), st(doc),
                                     ptr<float>(lse), st(lse), dq.data_ptr(), st(dq), dk.data_ptr(), st(dk), dv.data_ptr(), st(dv), ptr<uint8_t>(mask),
                                     st(mask), ptr<uint8_t>(l.transposed_mask), st(l.transposed_mask), ptr<uint8_t>(a.packed), st(a.packed),
                                     ptr<uint8_t>(b.packed), st(b.packed), ptr<int32_t>(a.fid), st(a.fid), ptr<int32_t>(a.fl), st(a.fl),
                                     ptr<int32_t>(a.pid), st(a.pid), ptr<int32_t>(a.pl), st(a.pl), ptr<int32_t>(b.fid), st(b.fid), ptr<int32_t>(b.fl),
                                     st(b.fl), ptr<int32_t>(b.pid), st(b.pid), ptr<int32_t>(b.pl), st(b.pl), ws.data_ptr(), ws_bytes, B, H, Sq, Sk, Dk,
                                     dtype_code(q.scalar_type()), (float)scale_log2(D), stream_of(q)));
    return {cut_head_dim(dq, D), cut_head_dim(dk, D), cut_head_dim(dv, D)};
}

void check_backward(const Tensor &do_, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o, const Tensor &lse, const OptTensor &mask) {
    if (q.dim() != 4 || k.dim() != 4) value_error("q, k, v must be [B,H,S,D]");
    if (!q.is_cuda()) throw std::runtime_error("sparse_attention_backward needs its tensors on a ROCm GPU; there is no CPU path");
    same_device(q, "k", k);
    same_device(q, "v", v);
    same_device(q, "o", o);
    same_device(q, "do", do_);
    same_device(q, "lse", lse);
    same_device(q, "mask", mask);
    const int dt = dtype_code(q.scalar_type());
    if (dt != SA_DTYPE_BF16 && dt != SA_DTYPE_FP16) type_error("q, k, v, o, do must share dtype bfloat16 or float16");
    for (const Tensor *t : {&k, &v, &o, &do_})
        if (t->scalar_type() != q.scalar_type()) type_error("q, k, v, o, do must share dtype bfloat16 or float16");
    const int64_t kw[4] = {q.size(0), q.size(1), k.size(2), q.size(3)}, lw[3] = {q.size(0), q.size(1), q.size(2)};
    if (k.sizes() != at::IntArrayRef(kw, 4) || v.sizes() != k.sizes() || o.sizes() != q.sizes() || do_.sizes() != q.sizes())
        value_error("shapes: q/o/do must be " + str(q.sizes()) + " and k/v " + str(at::IntArrayRef(kw, 4)) + " (got q " + str(q.sizes()) + ", k " +
                    str(k.sizes()) + ", v " + str(v.sizes()) + ", o " + str(o.sizes()) + ", do " + str(do_.sizes()) + ")");
    if (lse.scalar_type() != at::kFloat || lse.sizes() != at::IntArrayRef(lw, 3))
        value_error("lse: expected float32 " + str(at::IntArrayRef(lw, 3)) + ", got " + str(lse));
    if (mask && mask->scalar_type() != at::kBool) assertion("mask must be a torch.bool tensor");
}

// (dq, dk, dv), or None where Sq or Sk is no multiple of the kernels' 128 rows (then the wrapper pads)
py::object backward(const Tensor &do_, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o, const Tensor &lse, const OptTensor &mask_in,
                    py::object bmd) {
    check_backward(do_, q, k, v, o, lse, mask_in);
    const int64_t Sq = q.size(2), Sk = k.size(2);
    OptTensor mask = mask_in;
    if (mask) mask = mask->expand({q.size(0), q.size(1), Sq, Sk});
    if (Sq % 128 || Sk % 128) return py::none();
    if (bmd.is_none() && !mask) value_error("sparse_attention_backward needs the mask or a BackwardMetadata with packed tiles");
    const bool has_bmd = !bmd.is_none();
    ReadLists l;
    if (has_bmd) l = backward_lists_of(bmd, q, Sk);
    std::tuple<Tensor, Tensor, Tensor> g;
    {
        const py::gil_scoped_release unlocked;
        if (!has_bmd) l.own = backward_lists_from(*mask);
        g = backward_impl(do_, q, k, v, o, lse, mask, l.get());
    }
    return py::make_tuple(std::get<0>(g), std::get<1>(g), std::get<2>(g));
}

// ---- autograd -----------------------------------------------------------------------------------------------------
// What the caller passed is kept as it was passed: the mask unexpanded, so that hooks on saved tensors see the tensor the
// program has and not B * H planes of it, and the metadata object itself, whose lists are looked at (and checked) when the
// backward runs.  Autograd runs that on a thread of its own, without the interpreter's lock.
struct Metadata : torch::CustomClassHolder {
    PyObject *object;
    explicit Metadata(py::object o) : object(o.release().ptr()) {}
    ~Metadata() override {
        if (!Py_IsInitialized()) return;
        const py::gil_scoped_acquire gil;
        Py_DECREF(object);
    }
};

// Runs f; its exceptions become Python's own, which alone keep their type on the way out of a backward.
template <class F>
auto with_python_errors(F &&f) {
    try {
        return f();
    } catch (const py::builtin_exception &e) {
        const py::gil_scoped_acquire gil;
        e.set_error();
        throw py::error_already_set();
    }
}

struct AttentionFunction : public torch::autograd::Function<AttentionFunction> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask, const Out &r,
                          const py::object &bmd) {
        if (!bmd.is_none()) ctx->saved_data["bwd_metadata"] = c10::IValue::make_capsule(c10::make_intrusive<Metadata>(bmd));
        ctx->save_for_backward({q, k, v, r.o, *r.lse, mask.value_or(Tensor())});
        return r.o;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &q = s[0], &k = s[1];
        const auto g = with_python_errors([&] {
            OptTensor mask;
            if (s[5].defined()) mask = s[5].expand({q.size(0), q.size(1), q.size(2), k.size(2)});
            check_backward(grads[0], q, k, s[2], s[3], s[4], mask);
            const auto run = [&](const BackwardLists &l) { return backward_impl(grads[0], q, k, s[2], s[3], s[4], mask, l); };
            const auto it = ctx->saved_data.find("bwd_metadata");
            if (it == ctx->saved_data.end()) return run(backward_lists_from(*mask));
            const auto kept = it->second.toCapsule();
            const py::gil_scoped_acquire gil;
            // (let go of with the lock: tensors that the program has too would each take it for themselves)
            const ReadLists l = backward_lists_of(static_cast<const Metadata &>(*kept).object, q, k.size(2));
            const py::gil_scoped_release unlocked;
            return run(l.get());
        });
        return {std::get<0>(g), std::get<1>(g), std::get<2>(g), Tensor(), Tensor(), Tensor()};
    }
};

// sparse_attention_trainable, or None where the wrapper has to pad or to make other tiles.  Under torch.jit.trace too: a
// trace records the wrapper's Python function as one step, of this one it would keep the allocations and not the launches.
py::object trainable(const Tensor &q, const Tensor &k, const Tensor &v, const OptTensor &mask, int64_t BQ, int64_t BK, py::object md, py::object bmd) {
    if (q.dim() != 4 || k.dim() != 4 || q.size(2) % 128 || k.size(2) % 128 || q.scalar_type() == at::kFloat || (bmd.is_none() && !mask) ||
        torch::jit::tracer::isTracing())
        return py::none();
    std::optional<Out> r;
    {
        const at::NoGradGuard no_grad;
        r = forward_impl(q, k, v, mask, BQ, BK, md, true, "auto");
    }
    if (!r) return py::none();
    return py::cast(AttentionFunction::apply(q, k, v, mask, *r, bmd));
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    m.doc() = "Checks, allocations and launches of the wrappers in sparse_attn_kernel.py and mask_utils.py.";
    py::class_<OneMask, std::shared_ptr<OneMask>>(m, "OneMask");
    m.def("of_one_mask", &of_one_mask);
    m.def("forward", &forward);
    m.def("forward_lists", &forward_lists);
    m.def("forward_kernel", &forward_kernel);
    m.def("forward_tiled", &forward_tiled);
    m.def("decode", &decode);
    m.def("classify", &classify);
    m.def("classify_terms", &classify_terms);
    m.def("classify_terms_backward", &classify_terms_backward);
    m.def("backward", &backward);
    m.def("backward_workspace_bytes", &backward_workspace_bytes);
    m.def("kernel_head_dim", &kernel_head_dim);
    m.def("trainable", &trainable);
}
