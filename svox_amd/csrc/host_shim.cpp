// host_shim.cpp -- the operator calls of svox_amd.csrc in native code: checks, specs, outputs, launch.
//
// A call that works on a few thousand points or rays lasts as long as the host needs to make it.  In Python the checks
// of some ten tensors, the packing of the specs through ctypes and the launch took 20 to 60 us a call; here they take
// 3 to 5.  The functions take the Python objects (TreeSpec, RaysSpec, CameraSpec, RenderOptions) as they are, check
// them as svox/csrc/include/data_spec.hpp:37-126 does and call the C ABI of libsvox_hip.so, which init() opens.
// Every function that returns an integer status to Python is a helper of svox_amd/csrc/__init__.py.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>

#include <cstdarg>
#include <stdexcept>
#include <string>

#include "../../include/svox_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- the library
#define SVOX_CALLS(X)                                                                                                   \
    X(svox_last_error) X(svox_status_string) X(svox_out_data_dim) X(svox_query_vertical_ws) \
    X(svox_query_vertical_workspace_bytes)                                                            \
    X(svox_query_vertical_backward_ids) X(svox_query_vertical_backward_workspace_bytes)                                  \
    X(svox_assign_vertical) X(svox_calc_corners) X(svox_volume_render) X(svox_volume_render_images)                     \
    X(svox_volume_render_noted) X(svox_volume_render_images_noted) X(svox_volume_render_backward_ws)                    \
    X(svox_volume_render_images_backward_ws) X(svox_volume_render_backward_noted_with)                                  \
    X(svox_volume_render_images_backward_noted_with) X(svox_se_grad_ws) X(svox_se_grad_image_ws) X(svox_notes_serve)    \
    X(svox_mark_leaves_below) X(svox_walk_table_bytes) X(svox_walk_table)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    SVOX_CALLS(X)
#undef X
} lib;

void init(const std::string& path) {
    void* const handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (!handle) throw std::runtime_error(std::string("svox: ") + dlerror());
#define X(name)                                                                       \
    lib.name = reinterpret_cast<decltype(&::name)>(dlsym(handle, #name));             \
    if (!lib.name) throw std::runtime_error(path + " does not export " #name ": it was built from other sources, build it again");
    SVOX_CALLS(X)
#undef X
}

[[noreturn]] void fail(const std::string& what) { throw std::runtime_error(what); }
void status(int rc, const char* name) {
    if (rc != SVOX_OK) fail(std::string("svox.") + name + ": " + lib.svox_last_error() + " (" + lib.svox_status_string(rc) + ")");
}
// What allocates and launches runs without the interpreter's lock: a launch may wait for room in its queue, an allocation for
// memory, and other Python threads go on meanwhile.  No Python object is touched while one of these lives; those that a function
// holds are declared before it and so released after it.
using Unlocked = py::gil_scoped_release;

// ---- attributes of the spec objects
struct Name {
    PyObject* s;
    explicit Name(const char* text) : s(PyUnicode_InternFromString(text)) {}
};
#define NAME(var, text) static const Name var(text)

py::object attribute(py::handle obj, const Name& name) {
    PyObject* const v = PyObject_GetAttr(obj.ptr(), name.s);
    if (!v) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(v);
}
py::object attribute_or_none(py::handle obj, const Name& name) {
    PyObject* const v = PyObject_GetAttr(obj.ptr(), name.s);
    if (v) return py::reinterpret_steal<py::object>(v);
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw py::error_already_set();
    PyErr_Clear();
    return py::none();
}
double number(py::handle obj, const Name& name) {
    const double v = PyFloat_AsDouble(attribute(obj, name).ptr());
    if (v == -1.0 && PyErr_Occurred()) throw py::error_already_set();
    return v;
}
int32_t whole(py::handle obj, const Name& name) { return (int32_t)py::cast<int64_t>(py::int_(attribute(obj, name))); }
bool truth(py::handle obj, const Name& name) { return PyObject_IsTrue(attribute(obj, name).ptr()) == 1; }

const Tensor& tensor(const py::object& x, const char* name) {
    if (!THPVariable_Check(x.ptr())) fail(std::string(name) + " must be a tensor");
    return THPVariable_Unpack(x.ptr());
}

// ---- checks (CHECK_INPUT and friends, data_spec.hpp:37-42)
void check_input(const Tensor& x, const char* name) {
    if (!x.is_cuda()) fail(std::string(name) + " must be a CUDA tensor");
    if (!x.is_contiguous()) fail(std::string(name) + " must be contiguous");
}
std::string dtype_text(at::ScalarType t) {
    if (t == at::kFloat) return "torch.float32";
    if (t == at::kDouble) return "torch.float64";
    if (t == at::kHalf) return "torch.float16";
    if (t == at::kBFloat16) return "torch.bfloat16";
    return std::string("torch.") + c10::toString(t);
}
void same_dtype(const Tensor& x, at::ScalarType t, const char* name) {
    if (x.scalar_type() != t)
        fail("expected scalar type " + dtype_text(t) + " for " + name + " but found " + dtype_text(x.scalar_type()));
}
int32_t dtype_code(at::ScalarType t, const char* name) {
    if (t == at::kFloat) return SVOX_F32;
    if (t == at::kDouble) return SVOX_F64;
    fail(std::string(name) + " must be a float32 or float64 tensor, got " + dtype_text(t));
}
void check_floating(const Tensor& x, const char* name) {
    if (!x.is_floating_point()) fail(std::string(name) + " must be a floating point tensor");
}

// ---- specs
// TreeSpec::check, data_spec.hpp:75-88, plus the shape facts the kernels rely on.  The tensors stay alive with the
// Python object.  want: the scalar type the call works in (Undefined: that of tree.data).
struct Tree {
    SvoxTreeSpec spec;
    Tensor data, child;
};
Tree pack_tree(py::handle tree, at::ScalarType want, bool need_data) {
    NAME(n_data, "data"); NAME(n_child, "child"); NAME(n_parent_depth, "parent_depth"); NAME(n_extra, "extra_data");
    NAME(n_offset, "offset"); NAME(n_scaling, "scaling"); NAME(n_accum, "_weight_accum");
    NAME(n_accum_max, "_weight_accum_max"); NAME(n_marks, "child_marks"); NAME(n_marks_thresh, "child_marks_thresh");
    NAME(n_marks_softplus, "child_marks_softplus");
    const py::object o_data = attribute(tree, n_data), o_child = attribute(tree, n_child),
                     o_depth = attribute(tree, n_parent_depth), o_extra = attribute(tree, n_extra),
                     o_accum = attribute(tree, n_accum), o_marks = attribute_or_none(tree, n_marks);
    const py::object o_affine[2] = {attribute(tree, n_offset), attribute(tree, n_scaling)};
    const char* const affine_names[2] = {"offset", "scaling"};
    Tree t;
    t.data = tensor(o_data, "data");
    check_input(t.data, "data");
    t.child = tensor(o_child, "child");
    check_input(t.child, "child");
    const Tensor& depth = tensor(o_depth, "parent_depth");
    check_input(depth, "parent_depth");
    const bool has_extra = !o_extra.is_none() && tensor(o_extra, "extra_data").numel() > 0;
    if (has_extra) check_input(tensor(o_extra, "extra_data"), "extra_data");
    for (int i = 0; i < 2; ++i)
        if (!o_affine[i].is_none()) check_input(tensor(o_affine[i], affine_names[i]), affine_names[i]);
    const bool has_accum = !o_accum.is_none() && tensor(o_accum, "_weight_accum").numel() > 0;
    if (has_accum) check_input(tensor(o_accum, "_weight_accum"), "_weight_accum");
    if (t.data.dim() != 5 || t.child.dim() != 4 || depth.dim() != 2)
        fail("data must be 5-D, child 4-D and parent_depth 2-D");
    if (t.child.scalar_type() != at::kInt || depth.scalar_type() != at::kInt)
        fail("child and parent_depth must be int32 tensors");
    for (int i = 0; i < 4; ++i)
        if (t.data.size(i) != t.child.size(i)) fail("data and child disagree on (capacity, N, N, N)");

    const at::ScalarType dt = want == at::ScalarType::Undefined ? t.data.scalar_type() : want;
    SvoxTreeSpec& s = t.spec;
    s = SvoxTreeSpec{};
    s.dtype = dtype_code(dt, "data");
    if (need_data) same_dtype(t.data, dt, "data");
    s.data = t.data.data_ptr();
    s.child = (const int32_t*)t.child.data_ptr();
    s.parent_depth = (const int32_t*)depth.data_ptr();
    if (has_extra) {
        const Tensor& extra = tensor(o_extra, "extra_data");
        same_dtype(extra, dt, "extra_data");
        if (extra.dim() != 2) fail("extra_data must be 2-D");
        s.extra_data = extra.data_ptr();
        s.extra_rows = (int32_t)extra.size(0);
        s.extra_cols = (int32_t)extra.size(1);
    }
    const void* affine[2] = {nullptr, nullptr};
    for (int i = 0; i < 2; ++i) {
        if (o_affine[i].is_none()) continue;
        const Tensor& x = tensor(o_affine[i], affine_names[i]);
        same_dtype(x, dt, affine_names[i]);
        if (x.numel() != 3) fail(std::string(affine_names[i]) + " must have 3 elements");
        affine[i] = x.data_ptr();
    }
    s.offset = affine[0];
    s.scaling = affine[1];
    if (has_accum) {
        const Tensor& accum = tensor(o_accum, "_weight_accum");
        same_dtype(accum, dt, "_weight_accum");
        if (accum.numel() != t.child.numel()) fail("_weight_accum must have one entry per cell of child");
        s.weight_accum = accum.data_ptr();
    }
    s.weight_accum_max = truth(tree, n_accum_max);
    if (!o_marks.is_none()) {
        const Tensor& marks = tensor(o_marks, "child_marks");
        check_input(marks, "child_marks");
        if (marks.scalar_type() != at::kInt || marks.sizes() != t.child.sizes())
            fail("child_marks must be an int32 tensor shaped like child");
        s.child_marks = (const int32_t*)marks.data_ptr();
        const py::object thresh = attribute_or_none(tree, n_marks_thresh), soft = attribute_or_none(tree, n_marks_softplus);
        s.child_marks_thresh = thresh.is_none() ? 0.0f : (float)py::cast<double>(py::float_(thresh));
        s.child_marks_softplus = !soft.is_none() && PyObject_IsTrue(soft.ptr()) == 1;
    }
    s.capacity = t.child.size(0);
    s.N = (int32_t)t.child.size(1);
    s.data_dim = (int32_t)t.data.size(4);
    return t;
}

// marks made for this call alone: (tensor, threshold, softplus) or None
void attach_marks(Tree& t, const py::object& made) {
    if (made.is_none()) return;
    const auto m = py::cast<py::tuple>(made);
    t.spec.child_marks = (const int32_t*)THPVariable_Unpack(m[0].ptr()).data_ptr();
    t.spec.child_marks_thresh = (float)py::cast<double>(m[1]);
    t.spec.child_marks_softplus = py::cast<bool>(m[2]);
}

// RaysSpec::check, data_spec.hpp:56-63
struct Rays {
    SvoxRaysSpec spec;
    Tensor origins;
};
Rays pack_rays(py::handle rays, at::ScalarType dt) {
    NAME(n_origins, "origins"); NAME(n_dirs, "dirs"); NAME(n_vdirs, "vdirs");
    const Name* const names[3] = {&n_origins, &n_dirs, &n_vdirs};
    const char* const texts[3] = {"origins", "dirs", "vdirs"};
    Tensor t[3];
    for (int i = 0; i < 3; ++i) {
        t[i] = tensor(attribute(rays, *names[i]), texts[i]);
        check_input(t[i], texts[i]);
        check_floating(t[i], texts[i]);
        same_dtype(t[i], dt, texts[i]);
        if (t[i].dim() != 2 || t[i].size(1) != 3) fail(std::string(texts[i]) + " must be (B, 3)");
    }
    const int64_t n = t[0].size(0);
    if (t[1].size(0) != n || t[2].size(0) != n) fail("origins, dirs and vdirs must have the same number of rays");
    return Rays{SvoxRaysSpec{t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), n}, t[0]};
}

// CameraSpec::check, data_spec.hpp:98-103.  batched: c2w is (n, 3 or 4, 4); either (-1) takes both.
struct Camera {
    SvoxCameraSpec spec;
    bool single;
    int32_t n;
    int64_t stride;
    int64_t rays() const { return (int64_t)n * spec.width * spec.height; }
    std::vector<int64_t> shape(int64_t channels) const {
        if (single) return {spec.height, spec.width, channels};
        return {n, spec.height, spec.width, channels};
    }
};
Camera pack_camera(py::handle cam, at::ScalarType dt, int batched) {
    NAME(n_c2w, "c2w"); NAME(n_fx, "fx"); NAME(n_fy, "fy"); NAME(n_width, "width"); NAME(n_height, "height");
    const py::object o = attribute(cam, n_c2w);
    const Tensor& c2w = tensor(o, "c2w");
    check_input(c2w, "c2w");
    if (!c2w.is_floating_point()) fail("c2w must be a floating point tensor");
    const int64_t d = c2w.dim();
    const bool many = batched < 0 ? d != 2 : batched > 0;
    if (d != (many ? 3 : 2) || c2w.size(d - 1) != 4 || (c2w.size(d - 2) != 3 && c2w.size(d - 2) != 4))
        fail(many ? "c2w must be (n, 3, 4) or (n, 4, 4)" : "c2w must be (3, 4) or (4, 4)");
    same_dtype(c2w, dt, "c2w");
    Camera c;
    c.spec = SvoxCameraSpec{c2w.data_ptr(), (float)number(cam, n_fx), (float)number(cam, n_fy), whole(cam, n_width),
                            whole(cam, n_height)};
    c.single = !many;
    c.n = many ? (int32_t)c2w.size(0) : 1;
    c.stride = many ? c2w.size(1) * 4 : 12;
    return c;
}

SvoxRenderOptions pack_options(py::handle opt) {
    NAME(n_step, "step_size"); NAME(n_bg, "background_brightness"); NAME(n_format, "format"); NAME(n_basis, "basis_dim");
    NAME(n_nw, "ndc_width"); NAME(n_nh, "ndc_height"); NAME(n_nf, "ndc_focal"); NAME(n_min, "min_comp");
    NAME(n_max, "max_comp"); NAME(n_sigma, "sigma_thresh"); NAME(n_stop, "stop_thresh"); NAME(n_soft, "density_softplus");
    NAME(n_pad, "rgb_padding");
    SvoxRenderOptions o;
    o.step_size = (float)number(opt, n_step);
    o.background_brightness = (float)number(opt, n_bg);
    o.format = whole(opt, n_format);
    o.basis_dim = whole(opt, n_basis);
    o.ndc_width = whole(opt, n_nw);
    o.ndc_height = whole(opt, n_nh);
    o.ndc_focal = (float)number(opt, n_nf);
    o.min_comp = whole(opt, n_min);
    o.max_comp = whole(opt, n_max);
    o.sigma_thresh = (float)number(opt, n_sigma);
    o.stop_thresh = (float)number(opt, n_stop);
    o.density_softplus = truth(opt, n_soft);
    o.rgb_padding = (float)number(opt, n_pad);
    return o;
}

int64_t out_dim(const Tree& t, const SvoxRenderOptions& o) {
    const int od = lib.svox_out_data_dim(o.format, o.basis_dim, t.spec.data_dim);
    if (od < 0) fail("invalid data format / basis_dim for this tree");
    return od;
}

// the device of `x` made current, and torch's stream there
struct On {
    c10::DeviceGuard guard;
    void* stream;
    explicit On(const Tensor& x)
        : guard(x.device()), stream((void*)c10::hip::getCurrentHIPStream(x.device().index()).stream()) {}
};

Tensor like(const Tensor& x, at::IntArrayRef shape) { return at::empty(shape, x.options().requires_grad(false)); }
// (torch.empty_like of a contiguous tensor, without its autograd node)
Tensor like_data(const Tree& t) { return at::empty(t.data.sizes(), t.data.options().requires_grad(false)); }

struct Space {   // an optional tensor of bytes
    void* at = nullptr;
    int64_t bytes = 0;
    explicit Space(const py::object& x) {
        if (x.is_none()) return;
        const Tensor& t = tensor(x, "workspace");
        at = t.data_ptr();
        bytes = t.numel() * t.element_size();
    }
};
void check_shaped(const Tensor& x, const char* name, at::ScalarType dt, at::IntArrayRef shape) {
    check_input(x, name);
    same_dtype(x, dt, name);
    if (x.sizes() != shape) {
        auto text = [](at::IntArrayRef s) {
            std::string t = "(";
            for (size_t i = 0; i < s.size(); ++i) t += (i ? ", " : "") + std::to_string(s[i]);
            return t + (s.size() == 1 ? ",)" : ")");
        };
        fail(std::string(name) + " must have shape " + text(shape) + ", got " + text(x.sizes()));
    }
}

// The walk table of a call of n rays, where one pays and there is memory for it: it goes with what is returned.  (every_positive_leaf: svox_walk_table)
// Marks leave the march no way back to the child table where the rays of a picture run close together, as one pose's do from close up: on trees of few
// nodes such a picture is marched on its marks.  (128^3 shell, RGBA and SH9, 800x800, marks / walk table: from afar 118, 182 / 109, 172 us, closer 123, 167 / 127,
// 164, 264, 323 / 305, 344, 417, 491 / 486, 539; eight poses of 400x400, from afar and closer, 149, 192, 290, 345 / 141, 186, 316, 352.)
Tensor attach_walk(Tree& t, const SvoxRenderOptions& c, int64_t n_rays, int64_t n_images, bool every_positive_leaf, void* stream) {
    Tensor table;
    const bool image = n_images > 0;
    if (n_images == 1 && t.spec.child_marks && t.spec.capacity < 65536) return table;
    const int64_t bytes = lib.svox_walk_table_bytes(&t.spec, &c, n_rays, image, every_positive_leaf);
    if (bytes <= 0) return table;
    try {
        table = at::empty({bytes / 4}, t.child.options());
    } catch (const c10::OutOfMemoryError&) {
        return table;   // (the march does without)
    }
    const SvoxTreeSpec plain = t.spec;
    status(lib.svox_walk_table(&plain, &c, every_positive_leaf, (int32_t*)table.data_ptr(), &t.spec, stream), "walk_table");
    return table;
}

// ---- point queries
py::tuple query_vertical(py::handle tree, const py::object& points) {
    const Tensor& p = tensor(points, "indices");
    check_input(p, "indices");
    if (p.dim() != 2) fail("indices must be 2-D");
    check_floating(p, "indices");
    const Tree t = pack_tree(tree, p.scalar_type(), true);
    if (p.size(1) != 3) fail("indices must be (Q, 3)");
    Tensor values, ids;
    {
        const Unlocked unlocked;
        values = like(p, {p.size(0), t.spec.data_dim});
        ids = at::empty({p.size(0)}, t.child.options().dtype(at::kLong));
        const On on(p);
        const int64_t bytes = lib.svox_query_vertical_workspace_bytes(&t.spec, p.size(0));
        Tensor space;
        if (bytes > 0) space = at::empty({bytes}, t.child.options().dtype(at::kByte));
        status(lib.svox_query_vertical_ws(&t.spec, p.data_ptr(), p.size(0), values.data_ptr(), (int64_t*)ids.data_ptr(),
                                          bytes > 0 ? space.data_ptr() : nullptr, bytes, on.stream),
               "query_vertical");
    }
    return py::make_tuple(values, ids);
}

// node_ids: the leaves of the points as query_vertical left them, or None
Tensor query_vertical_backward(py::handle tree, const py::object& points, const py::object& grad_output, const py::object& node_ids) {
    const Tensor &p = tensor(points, "indices"), &g = tensor(grad_output, "grad_output");
    check_input(p, "indices");
    if (p.dim() != 2) fail("indices must be 2-D");
    check_floating(p, "indices");
    check_input(g, "grad_output");
    if (g.dim() != 2) fail("grad_output must be 2-D");
    check_floating(g, "grad_output");
    same_dtype(g, p.scalar_type(), "grad_output");
    const Tree t = pack_tree(tree, p.scalar_type(), false);
    if (g.size(0) != p.size(0)) fail("grad_output must have one row per point");
    const int64_t* ids = nullptr;
    if (!node_ids.is_none()) {
        const Tensor& i = tensor(node_ids, "node_ids");
        check_shaped(i, "node_ids", at::kLong, {p.size(0)});
        ids = (const int64_t*)i.data_ptr();
    }
    const Unlocked unlocked;
    Tensor grad = like(g, {t.spec.capacity, t.spec.N, t.spec.N, t.spec.N, g.size(1)});
    const On on(p);
    const int64_t bytes = lib.svox_query_vertical_backward_workspace_bytes(&t.spec, p.size(0), (int32_t)g.size(1));
    Tensor space;
    if (bytes > 0) space = at::empty({bytes}, p.options().dtype(at::kByte));
    status(lib.svox_query_vertical_backward_ids(&t.spec, p.data_ptr(), ids, p.size(0), g.data_ptr(), (int32_t)g.size(1),
                                                grad.data_ptr(), 0, bytes > 0 ? space.data_ptr() : nullptr, bytes, on.stream),
           "query_vertical_backward");
    return grad;
}

// ---- rendering
Tensor volume_render(py::handle tree, py::handle rays, py::handle opt, const py::object& marks) {
    NAME(n_origins, "origins");
    const py::object o = attribute(rays, n_origins);
    Tree t = pack_tree(tree, THPVariable_Check(o.ptr()) ? THPVariable_Unpack(o.ptr()).scalar_type() : at::ScalarType::Undefined,
                       true);
    const Rays r = pack_rays(rays, t.data.scalar_type());
    const SvoxRenderOptions c = pack_options(opt);
    attach_marks(t, marks);
    const Unlocked unlocked;
    Tensor out = like(r.origins, {r.spec.n_rays, out_dim(t, c)});
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, r.spec.n_rays, 0, false, on.stream);
    status(lib.svox_volume_render(&t.spec, &r.spec, &c, out.data_ptr(), on.stream), "volume_render");
    return out;
}

Tensor volume_render_images(py::handle tree, py::handle cam, py::handle opt, bool batched, const py::object& marks) {
    Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const Camera k = pack_camera(cam, t.data.scalar_type(), batched ? 1 : 0);
    const SvoxRenderOptions c = pack_options(opt);
    attach_marks(t, marks);
    const Unlocked unlocked;
    Tensor out = like(t.data, k.shape(out_dim(t, c)));
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, k.rays(), k.n, false, on.stream);
    status(lib.svox_volume_render_images(&t.spec, &k.spec, k.n, k.stride, &c, out.data_ptr(), on.stream), "volume_render_images");
    return out;
}

Tensor volume_render_noted(py::handle tree, py::handle rays, py::handle opt, const py::object& workspace,
                           const py::object& marks) {
    NAME(n_origins, "origins");
    const py::object o = attribute(rays, n_origins);
    Tree t = pack_tree(tree, THPVariable_Check(o.ptr()) ? THPVariable_Unpack(o.ptr()).scalar_type() : at::ScalarType::Undefined,
                       true);
    const Rays r = pack_rays(rays, t.data.scalar_type());
    const SvoxRenderOptions c = pack_options(opt);
    attach_marks(t, marks);
    const Space ws(workspace);
    const Unlocked unlocked;
    Tensor out = like(r.origins, {r.spec.n_rays, out_dim(t, c)});
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, r.spec.n_rays, 0, ws.at != nullptr, on.stream);
    status(lib.svox_volume_render_noted(&t.spec, &r.spec, &c, out.data_ptr(), ws.at, ws.bytes, on.stream), "volume_render_noted");
    return out;
}

Tensor volume_render_images_noted(py::handle tree, py::handle cam, py::handle opt, const py::object& workspace,
                                  const py::object& marks) {
    Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const Camera k = pack_camera(cam, t.data.scalar_type(), -1);
    const SvoxRenderOptions c = pack_options(opt);
    attach_marks(t, marks);
    const Space ws(workspace);
    const Unlocked unlocked;
    Tensor out = like(t.data, k.shape(out_dim(t, c)));
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, k.rays(), k.n, ws.at != nullptr, on.stream);
    status(lib.svox_volume_render_images_noted(&t.spec, &k.spec, k.n, k.stride, &c, out.data_ptr(), ws.at, ws.bytes, on.stream),
           "volume_render_images_noted");
    return out;
}

// from notes, or (`noted` false) in a workspace of the call's own, or without one
Tensor volume_render_backward(py::handle tree, py::handle rays, py::handle opt, const py::object& grad_output,
                              const py::object& workspace, bool noted, int64_t report, const py::object& marks) {
    Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const Rays r = pack_rays(rays, t.data.scalar_type());
    const SvoxRenderOptions c = pack_options(opt);
    const Tensor& g = tensor(grad_output, "grad_output");
    check_shaped(g, "grad_output", t.data.scalar_type(), {r.spec.n_rays, out_dim(t, c)});
    attach_marks(t, marks);
    const Space ws(workspace);
    const Unlocked unlocked;
    Tensor grad = like_data(t);
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, noted ? 0 : r.spec.n_rays, 0, true, on.stream);
    SvoxNotesExtras extras{};
    extras.report = (int64_t*)report;
    if (noted)
        status(lib.svox_volume_render_backward_noted_with(&t.spec, &r.spec, &c, g.data_ptr(), grad.data_ptr(), 0, ws.at,
                                                          ws.bytes, &extras, on.stream),
               "volume_render_backward_noted");
    else
        status(lib.svox_volume_render_backward_ws(&t.spec, &r.spec, &c, g.data_ptr(), grad.data_ptr(), 0, ws.at, ws.bytes,
                                                  on.stream),
               "volume_render_backward");
    return grad;
}

Tensor volume_render_images_backward(py::handle tree, py::handle cam, py::handle opt, const py::object& grad_output,
                                     const py::object& workspace, bool noted, int64_t report, int batched,
                                     const py::object& marks) {
    Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const Camera k = pack_camera(cam, t.data.scalar_type(), batched);
    const SvoxRenderOptions c = pack_options(opt);
    const Tensor& g = tensor(grad_output, "grad_output");
    check_shaped(g, "grad_output", t.data.scalar_type(), k.shape(out_dim(t, c)));
    attach_marks(t, marks);
    const Space ws(workspace);
    const Unlocked unlocked;
    Tensor grad = like_data(t);
    const On on(t.data);
    const Tensor walk = attach_walk(t, c, noted ? 0 : k.rays(), k.n, true, on.stream);
    SvoxNotesExtras extras{};
    extras.report = (int64_t*)report;
    if (noted)
        status(lib.svox_volume_render_images_backward_noted_with(&t.spec, &k.spec, k.n, k.stride, &c, g.data_ptr(),
                                                                 grad.data_ptr(), 0, ws.at, ws.bytes, &extras, on.stream),
               "volume_render_images_backward_noted");
    else
        status(lib.svox_volume_render_images_backward_ws(&t.spec, &k.spec, k.n, k.stride, &c, g.data_ptr(), grad.data_ptr(), 0,
                                                         ws.at, ws.bytes, on.stream),
               "volume_render_images_backward");
    return grad;
}

// ---- squared error.  rays_or_cam: RaysSpec or, with `image`, CameraSpec
py::tuple se_grad(py::handle tree, py::handle rays_or_cam, py::handle opt, const py::object& color, bool image,
                  const py::object& workspace) {
    Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const SvoxRenderOptions c = pack_options(opt);
    Rays r{};
    Camera k{};
    if (image)
        k = pack_camera(rays_or_cam, t.data.scalar_type(), 0);
    else
        r = pack_rays(rays_or_cam, t.data.scalar_type());
    const int64_t od = out_dim(t, c);
    if (od > 4) fail("Tree's output dim cannot be > 4 for se_grad");   // rt_kernel.cu:1123-1125
    const std::vector<int64_t> shape = image ? k.shape(od) : std::vector<int64_t>{r.spec.n_rays, od};
    const Tensor& ref = tensor(color, "color");
    check_shaped(ref, "color", t.data.scalar_type(), shape);
    const Space ws(workspace);
    Tensor result, grad, hess;
    {
        const Unlocked unlocked;
        result = like(t.data, shape);
        grad = like_data(t);
        hess = like_data(t);
        const On on(t.data);
        const Tensor walk = attach_walk(t, c, image ? k.rays() : r.spec.n_rays, image ? k.n : 0, true, on.stream);
        if (image)
            status(lib.svox_se_grad_image_ws(&t.spec, &k.spec, &c, ref.data_ptr(), result.data_ptr(), grad.data_ptr(),
                                             hess.data_ptr(), ws.at, ws.bytes, on.stream),
                   "se_grad_persp");
        else
            status(lib.svox_se_grad_ws(&t.spec, &r.spec, &c, ref.data_ptr(), result.data_ptr(), grad.data_ptr(), hess.data_ptr(),
                                       ws.at, ws.bytes, on.stream),
                   "se_grad");
    }
    return py::make_tuple(result, grad, hess);
}

int notes_serve(py::handle tree, py::handle opt) {
    const Tree t = pack_tree(tree, at::ScalarType::Undefined, true);
    const SvoxRenderOptions c = pack_options(opt);
    return lib.svox_notes_serve(&t.spec, &c);
}

// The bytes torch holds on a device that no tensor has: torch.cuda.memory_reserved - memory_allocated.  (Each of these makes a dictionary of
// every figure the allocator keeps, 37 us: the training step of 50 001 rays of a 256^3 SH9 shell, whose kernels take 165 us, waited for its host.  In turn with the step
// as it was 206 / 178 and 210 / 189 us, where two runs of one side differ by 11 to 17 %.)
int64_t cached_bytes(int device) {
    const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats((c10::DeviceIndex)device);
    constexpr size_t all = (size_t)c10::CachingAllocator::StatType::AGGREGATE;
    return stats.reserved_bytes[all].current - stats.allocated_bytes[all].current;
}

// ---- the specs for callers that go through ctypes: filled at the address of a ctypes structure
void fill_tree(int64_t at, py::handle tree, const py::object& dtype, bool need_data) {
    const auto want = dtype.is_none() ? at::ScalarType::Undefined : torch::python::detail::py_object_to_dtype(dtype);
    *(SvoxTreeSpec*)at = pack_tree(tree, want, need_data).spec;
}
void fill_rays(int64_t at, py::handle rays, const py::object& dtype) {
    *(SvoxRaysSpec*)at = pack_rays(rays, torch::python::detail::py_object_to_dtype(dtype)).spec;
}
void fill_camera(int64_t at, py::handle cam, const py::object& dtype, bool batched) {
    *(SvoxCameraSpec*)at = pack_camera(cam, torch::python::detail::py_object_to_dtype(dtype), batched ? 1 : 0).spec;
}
void fill_options(int64_t at, py::handle opt) { *(SvoxRenderOptions*)at = pack_options(opt); }

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("init", &init);
    m.def("query_vertical", &query_vertical);
    m.def("query_vertical_backward", &query_vertical_backward);
    m.def("volume_render", &volume_render);
    m.def("volume_render_images", &volume_render_images);
    m.def("volume_render_noted", &volume_render_noted);
    m.def("volume_render_images_noted", &volume_render_images_noted);
    m.def("volume_render_backward", &volume_render_backward);
    m.def("volume_render_images_backward", &volume_render_images_backward);
    m.def("se_grad", &se_grad);
    m.def("notes_serve", &notes_serve);
    m.def("cached_bytes", &cached_bytes);
    m.def("fill_tree", &fill_tree);
    m.def("fill_rays", &fill_rays);
    m.def("fill_camera", &fill_camera);
    m.def("fill_options", &fill_options);
}
