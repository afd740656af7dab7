// optim.hip -- SGD / Adam / AdamW with device-resident float64 moments.
//
// Reference: optimizers_c.c:64-562.  The handle keeps the hyper-parameters,
// the step count and per-parameter float64 moment buffers that are allocated
// (zeroed) on the first step and sized by numel(param).  Here the buffers
// live in HBM and each step is one fused launch for up to kStepTab parameter
// tensors of a dtype, which reads param, grad, m, v once and writes param, m, v
// once.
//
// Per-element arithmetic is the reference's, in double, in the same order,
// without FMA contraction; the bias corrections bc1 = 1 - pow(beta1, t),
// bc2 = 1 - pow(beta2, t) are computed on the host with libm pow as in
// optimizers_c.c:258-260,302-304 and passed in, so params, m and v match the
// reference bit for bit.
//
// OPTS state blob (optimizers_c.c:84-100,391-562): 80-byte header, then
// int64 sizes, then f64 velocities (SGD) or all m followed by all v.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <new>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"

namespace nh {

enum { OPT_SGD = 0, OPT_ADAM = 1, OPT_ADAMW = 2 };

struct OptHandle {
    int type;
    double lr, momentum, beta1, beta2, eps, wd;
    int64_t t;
    int64_t n_params;
    std::vector<int64_t> sizes;
    std::vector<double *> m, v, vel;  // device buffers
    std::vector<NeuralTensor *> last_grads;  // gradient tensors of the latest opt_step
};

struct OptStateHeader {
    uint32_t magic;
    uint32_t version;
    int32_t type;
    int32_t reserved;
    int64_t n_params;
    double lr, momentum, beta1, beta2, epsilon, weight_decay;
    int64_t t;
};
static_assert(sizeof(OptStateHeader) == 80, "OPTS header is 80 bytes");
constexpr uint32_t kOptsMagic = 0x5354504Fu;  // 'OPTS'
constexpr uint32_t kOptsVersion = 1u;

static void free_moments(OptHandle *o)
{
    for (double *p : o->m) dev_free(p);
    for (double *p : o->v) dev_free(p);
    for (double *p : o->vel) dev_free(p);
    o->m.clear();
    o->v.clear();
    o->vel.clear();
    o->sizes.clear();
    o->n_params = 0;
}

static double *alloc_zeroed(int64_t n)
{
    double *p = static_cast<double *>(dev_alloc(size_t(n > 0 ? n : 1) * sizeof(double)));
    if (p && n > 0 && launch_fill(p, NEURAL_DTYPE_FLOAT64, n, 0.0) != NEURAL_OK) {
        dev_free(p);
        return nullptr;
    }
    return p;
}

// ---- kernels -------------------------------------------------------------------------

struct AdamArgs {
    double lr, b1, b2, eps, wd, bc1, bc2;
};

// adamw_step_impl f32 body (optimizers_c.c:313-330).
NH_DEV float adamw_f32(float pd, float gd, double &m, double &v, const AdamArgs &a)
{
    double param = double(pd);
    const double grad = double(gd);
    param -= a.lr * a.wd * param;
    m = a.b1 * m + (1.0 - a.b1) * grad;
    v = a.b2 * v + (1.0 - a.b2) * grad * grad;
    const double mh = m / a.bc1;
    const double vh = v / a.bc2;
    param -= a.lr * mh / (sqrt(vh) + a.eps);
    return float(param);
}

NH_DEV double adamw_f64(double pd, double gd, double &m, double &v, const AdamArgs &a)
{
    double param = pd;
    param -= a.lr * a.wd * param;
    m = a.b1 * m + (1.0 - a.b1) * gd;
    v = a.b2 * v + (1.0 - a.b2) * gd * gd;
    const double mh = m / a.bc1;
    const double vh = v / a.bc2;
    param -= a.lr * mh / (sqrt(vh) + a.eps);
    return param;
}

// adam_step_impl (optimizers_c.c:270-291): the f32 step is rounded to float and
// subtracted in float.
NH_DEV float adam_f32(float pd, float gd, double &m, double &v, const AdamArgs &a)
{
    const double grad = double(gd);
    m = a.b1 * m + (1.0 - a.b1) * grad;
    v = a.b2 * v + (1.0 - a.b2) * grad * grad;
    const double mh = m / a.bc1;
    const double vh = v / a.bc2;
    return pd - float(a.lr * mh / (sqrt(vh) + a.eps));
}

NH_DEV double adam_f64(double pd, double gd, double &m, double &v, const AdamArgs &a)
{
    m = a.b1 * m + (1.0 - a.b1) * gd;
    v = a.b2 * v + (1.0 - a.b2) * gd * gd;
    const double mh = m / a.bc1;
    const double vh = v / a.bc2;
    return pd - a.lr * mh / (sqrt(vh) + a.eps);
}

constexpr int kOBlock = 256;

// The tensors of one launch, in its kernel arguments (no upload, nothing kept
// between calls): 44 bytes per tensor within the 4 KiB of arguments.
struct StepEntry {
    void *p;
    const void *g;
    double *m, *v;  // SGD: m holds the velocity
    int64_t n;
};
constexpr int kStepTab = 88;
struct StepTab {
    StepEntry e[kStepTab];
    int32_t first[kStepTab];  // first block of each tensor
    int32_t count;
    int32_t tiles;            // 256-element tiles per block
};
static_assert(sizeof(StepTab) + sizeof(AdamArgs) + 64 <= 4096, "kernel arguments");

// One element per lane.
template <typename T, int TYPE>
NH_DEV void step_elem(const StepEntry &e, int64_t j, const AdamArgs &a)
{
    T *__restrict__ p = static_cast<T *>(e.p);
    const T *__restrict__ g = static_cast<const T *>(e.g);
    if constexpr (TYPE == OPT_SGD) {  // sgd_step_impl (optimizers_c.c:218-249)
        const T pv = ld_nt(p + j);  // with the other loads: after the store to m it waits (50 M f64 302 us, 310)
        const double nv = a.b1 * ld_nt(e.m + j) + double(ld_nt(g + j));
        st_nt(e.m + j, nv);
        st_nt(p + j, pv - T(a.lr * nv));
    } else {
        const T pd = ld_nt(p + j), gd = ld_nt(g + j);
        double mm = ld_nt(e.m + j), vq = ld_nt(e.v + j);
        T r;
        if constexpr (sizeof(T) == 4) r = TYPE == OPT_ADAMW ? adamw_f32(pd, gd, mm, vq, a) : adam_f32(pd, gd, mm, vq, a);
        else r = TYPE == OPT_ADAMW ? adamw_f64(pd, gd, mm, vq, a) : adam_f64(pd, gd, mm, vq, a);
        st_nt(p + j, r);
        st_nt(e.m + j, mm);
        st_nt(e.v + j, vq);
    }
}

// `tiles` 256-lane tiles per block (1 unless the grid would pass
// kMaxGridBlocks); a block finds its tensor with one compare of its index per
// lane and two ballots.
// Bound by HBM, 44 B per element (f32 Adam).  A launch per tensor let the chip
// drain and refill between tensors: norm pass and step over 85 M values in 144
// tensors 1072 -> 718 us (70 of them the norm), 1.2 M values in 288 tensors
// 1033 -> 90 us, 50 M in 12 413 -> 389 us.
template <typename T, int TYPE>
__global__ __launch_bounds__(kOBlock) void k_opt_step(const StepTab tab, AdamArgs a)
{
    const int b = int(blockIdx.x);
    int i = 0;
    if (tab.count > 1) {
        const int lane = int(threadIdx.x & 63);
        static_assert(kStepTab <= 128, "two ballots");
        const bool c0 = lane < tab.count && tab.first[lane] <= b;
        const bool c1 = lane + 64 < tab.count && tab.first[lane + 64 < kStepTab ? lane + 64 : 0] <= b;
        i = __builtin_amdgcn_readfirstlane(int(__popcll(__ballot(c0)) + __popcll(__ballot(c1))) - 1);
    }
    const StepEntry &e = tab.e[i];
    const int64_t j0 = int64_t(b - tab.first[i]) * tab.tiles * kOBlock + threadIdx.x;
    for (int k = 0; k < tab.tiles; k++) {
        const int64_t j = j0 + int64_t(k) * kOBlock;
        if (j >= e.n) return;
        step_elem<T, TYPE>(e, j, a);
    }
}

// One tensor whose grid fits a launch: no table to look up before the first
// load.  100 M f32 values, AdamW 682 -> 679 us, SGD 477 -> 450; 2 or 4 elements in
// flight per lane or a grid of 16 blocks per CU striding over the tensor took
// 2-18% longer than one element per lane.
template <typename T, int TYPE>
__global__ __launch_bounds__(kOBlock) void k_opt_step_one(const StepEntry e, AdamArgs a)
{
    const int64_t j = int64_t(blockIdx.x) * kOBlock + threadIdx.x;
    if (j < e.n) step_elem<T, TYPE>(e, j, a);
}

template <typename T, int TYPE>
static void launch_step_of(const StepTab &tab, unsigned blocks, const AdamArgs &a)
{
    if (tab.count == 1 && tab.tiles == 1)
        NH_LAUNCH((k_opt_step_one<T, TYPE>), dim3(blocks), dim3(kOBlock), 0, stream(), tab.e[0], a);
    else
        NH_LAUNCH((k_opt_step<T, TYPE>), dim3(blocks), dim3(kOBlock), 0, stream(), tab, a);
}

template <typename T>
static int launch_step(int type, const StepTab &tab, unsigned blocks, const AdamArgs &a)
{
    if (type == OPT_SGD) launch_step_of<T, OPT_SGD>(tab, blocks, a);
    else if (type == OPT_ADAM) launch_step_of<T, OPT_ADAM>(tab, blocks, a);
    else launch_step_of<T, OPT_ADAMW>(tab, blocks, a);
    return check_launch();
}

// The tensors e[0..n) of one dtype, as few launches as the argument table and
// the grid allow.
static int launch_steps(int type, int dtype, const StepEntry *e, size_t n, const AdamArgs &a)
{
    for (size_t i = 0; i < n;) {
        StepTab tab;
        tab.count = 0;
        tab.tiles = 1;
        while (ceil_div(e[i].n, int64_t(tab.tiles) * kOBlock) > kMaxGridBlocks) tab.tiles *= 2;
        int64_t blocks = 0;
        for (; i < n && tab.count < kStepTab; i++) {
            const int64_t nb = ceil_div(e[i].n, int64_t(tab.tiles) * kOBlock);
            if (blocks + nb > kMaxGridBlocks) break;
            tab.e[tab.count] = e[i];
            tab.first[tab.count++] = int32_t(blocks);
            blocks += nb;
        }
        NH_TRY(dtype == NEURAL_DTYPE_FLOAT32 ? launch_step<float>(type, tab, unsigned(blocks), a)
                                             : launch_step<double>(type, tab, unsigned(blocks), a));
    }
    return NEURAL_OK;
}

// One parameter of the step, made ready on the device (nothing launched).
static int step_prepare(OptHandle *o, size_t i, NeuralTensor *p, const NeuralTensor *g, StepEntry &e)
{
    const int64_t sz = o->sizes[i];
    e.n = 0;
    if (!p || !g) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(check_tensor(p));
    if (g->dtype != p->dtype) return set_error(NEURAL_ERR_DTYPE_MISMATCH);
    if (numel(p) != sz || numel(g) != sz) return set_error(NEURAL_ERR_SHAPE_MISMATCH);
    if (!is_contiguous(p) || !is_contiguous(g)) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    if (sz == 0) return NEURAL_OK;
    const void *pr = nullptr;
    NH_TRY(dev_read(g, &e.g));
    NH_TRY(dev_read(p, &pr));
    NH_TRY(dev_write(p, &e.p, false));
    e.m = o->type == OPT_SGD ? o->vel[i] : o->m[i];
    e.v = o->type == OPT_SGD ? nullptr : o->v[i];
    e.n = sz;
    return NEURAL_OK;
}

// True when the order of the parameters' updates could show: a parameter
// tensor that shares bytes with another parameter or with a gradient (tied
// weights passed twice), or a tensor whose bytes are the caller's host memory.
static bool step_order_matters(void **params, void **grads, int64_t n)
{
    struct Span {
        uintptr_t lo, hi;
        bool write;
    };
    std::vector<Span> s;
    s.reserve(size_t(2 * n));
    for (int64_t i = 0; i < n; i++) {
        const NeuralTensor *t[2] = {static_cast<const NeuralTensor *>(params[i]),
                                    static_cast<const NeuralTensor *>(grads[i])};
        for (int k = 0; k < 2; k++) {
            if (!t[k]) continue;
            if (t[k]->st->kind == KIND_EXT_HOST) return true;
            const uintptr_t lo = reinterpret_cast<uintptr_t>(t[k]->dev);
            s.push_back({lo, lo + uintptr_t(numel(t[k])) * elem_size(t[k]->dtype), k == 0});
        }
    }
    std::sort(s.begin(), s.end(), [](const Span &a, const Span &b) { return a.lo < b.lo; });
    uintptr_t end_any = 0, end_write = 0;
    for (const Span &x : s) {
        if (x.lo < x.hi && (x.lo < end_write || (x.write && x.lo < end_any))) return true;
        end_any = x.hi > end_any ? x.hi : end_any;
        if (x.write) end_write = x.hi > end_write ? x.hi : end_write;
    }
    return false;
}

// Every parameter's update.  The first parameter that cannot be updated ends
// the step with its error, after the ones before it have been updated (the
// reference's loop, optimizers_c.c:218-348).
static int step_all(OptHandle *o, void **params, void **grads, int64_t n, const AdamArgs &a)
{
    const bool ordered = n > 1 && step_order_matters(params, grads, n);
    std::vector<StepEntry> list[2];  // by dtype
    std::vector<NeuralTensor *> written;
    if (!ordered)
        for (auto &l : list) l.reserve(size_t(n));
    written.reserve(size_t(n));
    int rc = NEURAL_OK;
    for (int64_t i = 0; i < n && rc == NEURAL_OK; i++) {
        NeuralTensor *p = static_cast<NeuralTensor *>(params[i]);
        StepEntry e;
        rc = step_prepare(o, size_t(i), p, static_cast<const NeuralTensor *>(grads[i]), e);
        if (rc != NEURAL_OK || e.n == 0) continue;
        if (ordered) {
            rc = launch_steps(o->type, p->dtype, &e, 1, a);
            if (rc == NEURAL_OK) rc = dev_written(p);
        } else {
            list[p->dtype == NEURAL_DTYPE_FLOAT32 ? 0 : 1].push_back(e);
            written.push_back(p);
        }
    }
    for (int d = 0; d < 2; d++) {
        const int lrc = launch_steps(o->type, d == 0 ? NEURAL_DTYPE_FLOAT32 : NEURAL_DTYPE_FLOAT64, list[d].data(),
                                     list[d].size(), a);
        rc = rc == NEURAL_OK ? lrc : rc;
    }
    for (NeuralTensor *p : written) {
        const int wrc = dev_written(p);
        rc = rc == NEURAL_OK ? wrc : rc;
    }
    return rc == NEURAL_OK ? NEURAL_OK : set_error(rc);
}

static OptHandle *make(int type)
{
    if (ensure_init() != NEURAL_OK) return nullptr;
    OptHandle *o = new (std::nothrow) OptHandle();
    if (!o) return nullptr;
    o->type = type;
    o->lr = o->momentum = o->beta1 = o->beta2 = o->eps = o->wd = 0.0;
    o->t = 0;
    o->n_params = 0;
    return o;
}

static int64_t total_elems(const OptHandle *o)
{
    int64_t t = 0;
    for (int64_t s : o->sizes) {
        if (s < 0) return -1;
        t += s;
    }
    return t;
}

}  // namespace nh

using namespace nh;

extern "C" {

void *opt_sgd_create(double lr, double momentum)
{
    OptHandle *o = make(OPT_SGD);
    if (o) { o->lr = lr; o->momentum = momentum; }
    return o;
}

void *opt_adam_create(double lr, double beta1, double beta2, double epsilon)
{
    OptHandle *o = make(OPT_ADAM);
    if (o) { o->lr = lr; o->beta1 = beta1; o->beta2 = beta2; o->eps = epsilon; o->wd = 0.0; }
    return o;
}

void *opt_adamw_create(double lr, double beta1, double beta2, double epsilon, double weight_decay)
{
    OptHandle *o = make(OPT_ADAMW);
    if (o) { o->lr = lr; o->beta1 = beta1; o->beta2 = beta2; o->eps = epsilon; o->wd = weight_decay; }
    return o;
}

// opt_step (optimizers_c.c:353-368): NULL -> 1; n < 0 or n != first-call count -> 3.
static int opt_step_impl(void *opt, void **params, void **grads, int64_t n)
{
    if (!opt || !params || !grads) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(ensure_init());
    OptHandle *o = static_cast<OptHandle *>(opt);
    if (n < 0) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    if (o->n_params > 0 && n != o->n_params) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    if (o->type < OPT_SGD || o->type > OPT_ADAMW) return set_error(NEURAL_ERR_NULL_POINTER);
    if (o->n_params == 0 && n > 0) {
        // Lazy moment allocation on the first step (optimizers_c.c:179-212).
        o->n_params = n;
        o->sizes.resize(size_t(n));
        for (int64_t i = 0; i < n; i++) {
            const NeuralTensor *p = static_cast<const NeuralTensor *>(params[i]);
            const int64_t sz = p ? numel(p) : 0;
            o->sizes[size_t(i)] = sz;
            if (o->type == OPT_SGD) {
                double *b = alloc_zeroed(sz);
                if (!b) { free_moments(o); return set_error(NEURAL_ERR_OUT_OF_MEMORY); }
                o->vel.push_back(b);
            } else {
                double *bm = alloc_zeroed(sz), *bv = alloc_zeroed(sz);
                if (!bm || !bv) { dev_free(bm); dev_free(bv); free_moments(o); return set_error(NEURAL_ERR_OUT_OF_MEMORY); }
                o->m.push_back(bm);
                o->v.push_back(bv);
            }
        }
    }
    o->last_grads.assign(reinterpret_cast<NeuralTensor **>(grads), reinterpret_cast<NeuralTensor **>(grads) + n);
    AdamArgs a{o->lr, o->beta1, o->beta2, o->eps, o->wd, 0.0, 0.0};
    if (o->type != OPT_SGD) {
        o->t++;
        a.bc1 = 1.0 - std::pow(o->beta1, double(o->t));
        a.bc2 = 1.0 - std::pow(o->beta2, double(o->t));
    }
    if (o->type == OPT_SGD) a.b1 = o->momentum;
    NH_TRY(step_all(o, params, grads, n, a));
    return set_error(NEURAL_OK);
}

// C++ exceptions (a failed vector growth) end as an error code at the C
// boundary, never as an abort.
int opt_step(void *opt, void **params, void **grads, int64_t n)
{
    try {
        return opt_step_impl(opt, params, grads, n);
    } catch (const std::bad_alloc &) {
        free_moments(static_cast<OptHandle *>(opt));
        return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    } catch (...) {
        return set_error(NEURAL_ERR_INTERNAL);
    }
}

void opt_free(void *opt)
{
    if (!opt) return;
    OptHandle *o = static_cast<OptHandle *>(opt);
    if (ensure_init() == NEURAL_OK) (void)sync();
    free_moments(o);
    delete o;
}

// neural_clip_grad_norm / neural_clip_grad_value (neural_api.h:731,741;
// neural_api.asm:1677-1720 -> clip_grad_norm_ / clip_grad_value_,
// optimizers.asm:1370-1620).  The reference's optimizer holds its parameter
// nodes and clips their gradients.  This handle learns its gradients from
// opt_step, so it clips the gradient tensors passed to its most recent
// opt_step (the caller keeps them alive, as the reference keeps its nodes).
// Before the first step there are none: NEURAL_OK with nothing done, as
// clip_grad_norm_ does for an optimizer without parameter nodes
// (optimizers.asm:1386-1388).
int neural_clip_grad_norm(void *opt, double max_norm)
{
    if (!opt) return set_error(NEURAL_ERR_NULL_POINTER);
    OptHandle *o = static_cast<OptHandle *>(opt);
    if (o->last_grads.empty()) return set_error(NEURAL_OK);
    return clip_norm_list(o->last_grads.data(), int64_t(o->last_grads.size()), max_norm, nullptr);
}

int neural_clip_grad_value(void *opt, double min_val, double max_val)
{
    if (!opt) return set_error(NEURAL_ERR_NULL_POINTER);
    OptHandle *o = static_cast<OptHandle *>(opt);
    if (o->last_grads.empty()) return set_error(NEURAL_OK);
    return clip_value_list(o->last_grads.data(), int64_t(o->last_grads.size()), min_val, max_val);
}

double opt_get_lr(void *opt) { return opt ? static_cast<OptHandle *>(opt)->lr : 0.0; }

void opt_set_lr(void *opt, double lr)
{
    if (opt) static_cast<OptHandle *>(opt)->lr = lr;
}

int64_t opt_state_bytes(void *opt)
{
    if (!opt) return 0;
    const OptHandle *o = static_cast<const OptHandle *>(opt);
    int64_t total = int64_t(sizeof(OptStateHeader)) + o->n_params * int64_t(sizeof(int64_t));
    const int64_t e = total_elems(o);
    if (e < 0) return 0;
    if (o->type == OPT_SGD) total += e * int64_t(sizeof(double));
    else total += 2 * e * int64_t(sizeof(double));
    return total;
}

int opt_state_export(void *opt, void *buffer, int64_t size)
{
    if (!opt || !buffer || size <= 0) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(ensure_init());
    OptHandle *o = static_cast<OptHandle *>(opt);
    const int64_t need = opt_state_bytes(opt);
    if (need <= 0 || size < need) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    OptStateHeader h;
    std::memset(&h, 0, sizeof(h));
    h.magic = kOptsMagic;
    h.version = kOptsVersion;
    h.type = o->type;
    h.n_params = o->n_params;
    h.lr = o->lr;
    h.momentum = o->momentum;
    h.beta1 = o->beta1;
    h.beta2 = o->beta2;
    h.epsilon = o->eps;
    h.weight_decay = o->wd;
    h.t = o->t;
    uint8_t *p = static_cast<uint8_t *>(buffer);
    std::memcpy(p, &h, sizeof(h));
    p += sizeof(h);
    if (o->n_params > 0) {
        std::memcpy(p, o->sizes.data(), size_t(o->n_params) * sizeof(int64_t));
        p += size_t(o->n_params) * sizeof(int64_t);
    }
    auto dump = [&](std::vector<double *> &bufs) -> int {
        for (size_t i = 0; i < bufs.size(); i++) {
            const int64_t n = o->sizes[i];
            if (n <= 0) continue;
            NH_HIP(hipMemcpyAsync(p, bufs[i], size_t(n) * sizeof(double), hipMemcpyDeviceToHost, stream()));
            p += size_t(n) * sizeof(double);
        }
        return NEURAL_OK;
    };
    if (o->type == OPT_SGD) NH_TRY(dump(o->vel));
    else {
        NH_TRY(dump(o->m));
        NH_TRY(dump(o->v));
    }
    NH_TRY(sync());
    return set_error(NEURAL_OK);
}

static int opt_state_import_impl(void *opt, const void *buffer, int64_t size)
{
    if (!opt || !buffer || size <= 0) return set_error(NEURAL_ERR_NULL_POINTER);
    NH_TRY(ensure_init());
    OptHandle *o = static_cast<OptHandle *>(opt);
    if (size < int64_t(sizeof(OptStateHeader))) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    const uint8_t *base = static_cast<const uint8_t *>(buffer);
    const uint8_t *p = base;
    OptStateHeader h;
    std::memcpy(&h, p, sizeof(h));
    p += sizeof(h);
    if (h.magic != kOptsMagic || h.version != kOptsVersion) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    if (h.type != o->type || h.n_params < 0) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    NH_TRY(sync());
    free_moments(o);
    o->lr = h.lr;
    o->momentum = h.momentum;
    o->beta1 = h.beta1;
    o->beta2 = h.beta2;
    o->eps = h.epsilon;
    o->wd = h.weight_decay;
    o->t = h.t;
    if (h.n_params == 0) return set_error(NEURAL_OK);
    // Counts whose byte sizes overflow int64 end, in the reference, in a
    // calloc that fails (NEURAL_ERR_OUT_OF_MEMORY); counts that fit but run
    // past the blob are NEURAL_ERR_INVALID_ARGUMENT.  No product below can
    // overflow.
    constexpr int64_t kMaxCount = INT64_MAX / int64_t(sizeof(double));
    const auto remaining = [&]() { return size - int64_t(p - base); };
    if (h.n_params > kMaxCount) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    const int64_t sizes_bytes = h.n_params * int64_t(sizeof(int64_t));
    if (sizes_bytes > remaining()) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
    try {
        o->sizes.resize(size_t(h.n_params));
    } catch (...) {
        o->sizes.clear();
        return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    }
    o->n_params = h.n_params;
    std::memcpy(o->sizes.data(), p, size_t(sizes_bytes));
    p += sizes_bytes;
    auto load = [&](std::vector<double *> &bufs) -> int {
        for (int64_t i = 0; i < o->n_params; i++) {
            const int64_t n = o->sizes[size_t(i)];
            if (n < 0) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
            if (n > kMaxCount) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
            const int64_t bytes = n * int64_t(sizeof(double));
            if (bytes > remaining()) return set_error(NEURAL_ERR_INVALID_ARGUMENT);
            double *d = static_cast<double *>(dev_alloc(size_t(n > 0 ? n : 1) * sizeof(double)));
            if (!d) return set_error(NEURAL_ERR_OUT_OF_MEMORY);
            try {
                bufs.push_back(d);
            } catch (...) {
                dev_free(d);
                return set_error(NEURAL_ERR_OUT_OF_MEMORY);
            }
            if (n == 0) continue;
            NH_HIP(hipMemcpyAsync(d, p, size_t(bytes), hipMemcpyHostToDevice, stream()));
            p += bytes;
        }
        return NEURAL_OK;
    };
    int rc = NEURAL_OK;
    if (o->type == OPT_SGD) rc = load(o->vel);
    else {
        rc = load(o->m);
        if (rc == NEURAL_OK) rc = load(o->v);
    }
    if (rc != NEURAL_OK) {
        (void)sync();
        free_moments(o);
        return rc;
    }
    NH_TRY(sync());
    return set_error(NEURAL_OK);
}

int opt_state_import(void *opt, const void *buffer, int64_t size)
{
    try {
        return opt_state_import_impl(opt, buffer, size);
    } catch (const std::bad_alloc &) {
        (void)sync();
        free_moments(static_cast<OptHandle *>(opt));
        return set_error(NEURAL_ERR_OUT_OF_MEMORY);
    } catch (...) {
        (void)sync();
        free_moments(static_cast<OptHandle *>(opt));
        return set_error(NEURAL_ERR_INTERNAL);
    }
}

}  // extern "C"
