// C ABI of the batched integrator (include/sodecl.h, no reference
// counterpart): orbits of several system sizes and individual step counts,
// one kernel per size class with a workgroup per work item, the classes'
// kernels launched side by side on streams of their own
// (device/batch_class.hip, device/batch_kernel.hip).
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "sodecl_internal.hpp"

using namespace sodecl_amd;

struct sodecl_batch {
    std::string source;
    PluginFeatures features;
    int solver = 3;
    double dt = 0.0;
    int ksteps = 1, npar = 0;
    std::vector<int> class_neq;
    sodecl_options opts{};
    int device = 0;
    // per-orbit layout
    int orbits = 0;
    std::vector<int> cls, steps, order;
    std::vector<long long> yoff, ooff;
    size_t state_size = 0, output_size = 0;
    // per class: its work items (an orbit per slot of its wavefront, -1: none, longest
    // first; one workgroup each), its kernel, LDS size and stream; classes
    // are launched in order of their total cost, the most expensive first
    struct Class {
        BatchShape shape;
        std::vector<int> items;
        int nitems = 0;
        double cost = 0.0;
        hipFunction_t fn = nullptr;
        int* d_items = nullptr;
        size_t lds_bytes = 0;
        hipStream_t stream = nullptr;
        hipEvent_t done = nullptr;
    };
    std::vector<Class> classes;
    std::vector<int> launch_order;
    hipEvent_t fork = nullptr;
    // device
    std::vector<char> code;
    hipModule_t module = nullptr;
    int* d_steps = nullptr;
    long long *d_yoff = nullptr, *d_ooff = nullptr;
    bool ready = false;
    std::string last_error, program;
};

namespace {

int bfail(sodecl_batch* b, const std::string& m)
{
    if (b) b->last_error = m;
    return 0;
}

bool bhip(sodecl_batch* b, hipError_t e, const char* what)
{
    if (e == hipSuccess) return true;
    bfail(b, std::string(what) + ": " + hipGetErrorString(e));
    return false;
}

void free_batch(sodecl_batch* b)
{
    // work queued on the classes' streams ends before their memory goes
    for (auto& c : b->classes) {
        if (c.stream) {
            hipStreamSynchronize(c.stream);
            hipStreamDestroy(c.stream);
        }
        if (c.done) hipEventDestroy(c.done);
        hipFree(c.d_items);
    }
    b->classes.clear();
    b->launch_order.clear();
    if (b->fork) hipEventDestroy(b->fork);
    b->fork = nullptr;
    if (b->module) hipModuleUnload(b->module);
    hipFree(b->d_steps);
    hipFree(b->d_yoff);
    hipFree(b->d_ooff);
    b->module = nullptr;
    b->d_steps = nullptr;
    b->d_yoff = b->d_ooff = nullptr;
    b->ready = false;
}

ProgramKey batch_key(const sodecl_batch* b)
{
    ProgramKey k;
    k.solver = b->solver;
    k.npar = b->npar;
    k.orbits = b->orbits;
    k.ksteps = b->ksteps;
    k.dt = b->dt;
    k.newton_max_iter = b->opts.newton_max_iter > 0 ? b->opts.newton_max_iter : 1000;
    k.newton_tol = b->opts.newton_tol;
    k.fp_contract = b->opts.fp_contract;
    k.library_sin = b->opts.library_sin;
    k.library_exp = b->opts.library_exp;
    return k;
}

// Least power of two of lanes that hold neq rows, rows of them on each.
int lanes_for(int neq, int rows)
{
    int lanes = 1;
    while (lanes * rows < neq) lanes *= 2;
    return lanes;
}

// LDS bytes of a wavefront's parameters (device/batch_class.hip, SODECL_PLDS).
size_t param_lds(const sodecl_batch* b, const BatchShape& s)
{
    const size_t row = b->npar <= 8 ? 0 : s.window ? b->npar | 1 : b->npar;
    return row * s.slots() * sizeof(double);
}

// Lanes per orbit and form of every size class.
//
// Windowed form (up to 512 equations), by the wavefronts per SIMD of the whole
// batch:
//  * up to three with eight rows per lane, one wavefront at a time on a SIMD (each
//    asks for the whole register file): the classes' kernels run side by side and
//    the dispatcher would put two wavefronts on one SIMD while others idle, and a
//    SIMD works off its wavefronts, longest orbits first, faster one after another
//    than stacked.  The time is then the longest chains of Newton iterations, which
//    fewer rows per lane shorten: two rows, or four, if they keep the batch at two
//    wavefronts per SIMD, else eight.  450 orbits of 10, 74 and 200 equations to
//    convergence, us: 390 with two and four rows, 580 with eight, and 443 with four
//    if stacked.  Chains of 32, 128 and 512 equations, 50 to 200 steps, ms with two,
//    four and eight rows, and two rows stacked: 2000 orbits 0.64 0.64 0.62 0.79,
//    3000 orbits 0.82 0.67 0.76 0.90, 6000 orbits 1.47 1.18 1.10 1.26;
//    of 22, 66 and 140 equations: 2000 orbits 0.57 0.57 0.76 0.68, 6000 orbits 1.26
//    1.18 0.97 1.11, 8000 orbits 1.58 1.43 1.29 1.38;
//  * from three to four, four rows, stacked (8000 chains of 32, 128 and 512
//    equations with two, four and eight rows: 1.47 1.28 1.39, one at a time 1.88
//    1.50 1.40);
//  * from four on, eight rows, where instructions count (32768 orbits of 32, 128 and
//    512 equations: 7.6 ms, against 8.1 ms with four and 8.8 ms with two).
// A power of two of rows keeps the parity of a row's index known to the compiler.
// More than eight parameters are in LDS, a row per orbit: an orbit gets more
// lanes than its rows need where a wavefront's orbits would take more than 16
// KiB (which lets ten wavefronts onto a CU).
//
// Through LDS: 16 lanes up to 32 equations, 32 up to 128, else 64; the
// 128-equation class ran 2.5-3% faster on 32 lanes (four rows per lane, four
// wavefronts per SIMD) than on 16 (eight rows, two wavefronts per SIMD by
// registers), and up to eight rows on 64 lanes fit 168 registers (three
// wavefronts per SIMD).
std::vector<BatchShape> batch_shapes(const sodecl_batch* b)
{
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device) != hipSuccess || cus <= 0)
        cus = 256;
    const int reach = b->features.window_reach;   // 0: no windowed form
    std::vector<long> count(b->class_neq.size(), 0);
    for (int c : b->cls)
        if (c >= 0 && c < (int)count.size()) ++count[c];
    auto window = [&](int neq) { return reach >= 1 && reach <= 8 && lanes_for(neq, 8) <= 64; };
    auto shape = [&](int neq, int rows) {
        BatchShape s;
        s.neq = neq;
        s.window = window(neq);
        if (s.window) {
            s.rows = rows;
            while (s.rows < reach || lanes_for(neq, s.rows) > 64) s.rows *= 2;
            s.lanes = lanes_for(neq, s.rows);
            while (s.lanes < 64 && param_lds(b, s) > 16 * 1024) s.lanes *= 2;
            s.waves = 4;
        } else {
            s.lanes = neq <= 32 ? 16 : neq <= 128 ? 32 : 64;
            s.rows = (neq + s.lanes - 1) / s.lanes;
            s.waves = s.rows <= 2 || (s.lanes == 32 && s.rows <= 4) ? 4 : (s.lanes == 64 && s.rows <= 8) ? 3 : 2;
        }
        return s;
    };
    bool windows = true;
    auto per_simd = [&](int rows) {
        double waves = 0.0;
        for (size_t k = 0; k < count.size(); ++k) waves += (double)count[k] * shape(b->class_neq[k], rows).lanes / 64.0;
        return waves / (4.0 * cus);
    };
    for (int neq : b->class_neq) windows = windows && window(neq);
    int rows = 8;
    bool alone = false;
    if (!b->cls.empty() && per_simd(8) < 4.0) {
        rows = per_simd(8) > 3.0 ? 4 : per_simd(2) <= 2.0 ? 2 : per_simd(4) <= 2.0 ? 4 : 8;
        alone = per_simd(8) <= 3.0 && (windows || per_simd(rows) <= 1.0);
    }
    std::vector<BatchShape> shapes;
    for (int neq : b->class_neq) {
        shapes.push_back(shape(neq, rows));
        shapes.back().alone = alone;
    }
    return shapes;
}

}  // namespace

extern "C" {

int sodecl_batch_create(sodecl_batch** out, const char* system_source, int solver, double dt, int ksteps, int npar,
                        int nclasses, const int* class_neq)
{
    if (!out) return 0;
    auto* b = new sodecl_batch();
    *out = b;
    sodecl_default_options(&b->opts);
    b->source = system_source ? system_source : "";
    b->features = detect_features(b->source);
    b->solver = solver;
    b->dt = dt;
    b->ksteps = ksteps;
    b->npar = npar;
    if (solver != SODECL_IMPLICIT_EULER && solver != SODECL_IMPLICIT_MIDPOINT)
        return bfail(b, "the batched integrator runs the implicit Euler and implicit midpoint solvers");
    if (!(dt > 0) || ksteps <= 0 || npar < 0 || nclasses <= 0 || !class_neq)
        return bfail(b, "invalid dt, ksteps, npar or size classes");
    for (int c = 0; c < nclasses; ++c) {
        if (class_neq[c] <= 0) return bfail(b, "size classes must be positive");
        b->class_neq.push_back(class_neq[c]);
    }
    if (!b->features.component || !b->features.jacobian_band_i)
        return bfail(b, "the batched integrator needs sode_system_i and calc_jacobian_band_i in the system source");
    return 1;
}

void sodecl_batch_destroy(sodecl_batch* b)
{
    if (!b) return;
    free_batch(b);
    delete b;
}

int sodecl_batch_set_options(sodecl_batch* b, const sodecl_options* o)
{
    if (!b || !o) return 0;
    b->opts = *o;
    return 1;
}

int sodecl_batch_choose_device(sodecl_batch* b, uint32_t device)
{
    if (!b) return 0;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || (int)device >= n) return bfail(b, "device number out of bounds");
    b->device = (int)device;
    return 1;
}

size_t sodecl_batch_compile_only(sodecl_batch* b, const char* arch)
{
    if (!b) return 0;
    b->program = assemble_batch_program(b->source, batch_key(b), b->features, batch_shapes(b));
    std::vector<char> code;
    std::string log;
    if (!compile_program(b->program, arch ? arch : "gfx950", b->opts.fp_contract, code, log)) {
        bfail(b, "Failed to build program executable:\n" + log);
        return 0;
    }
    return code.size();
}

int sodecl_batch_setup(sodecl_batch* b, int orbits, const int* orbit_class, const int* orbit_steps)
{
    if (!b) return 0;
    if (orbits <= 0 || !orbit_class || !orbit_steps) return bfail(b, "invalid orbit description");
    free_batch(b);
    b->orbits = orbits;
    b->cls.assign(orbit_class, orbit_class + orbits);
    b->steps.assign(orbit_steps, orbit_steps + orbits);
    b->yoff.resize(orbits);
    b->ooff.resize(orbits);
    size_t ys = 0, os = 0;
    std::vector<double> cost(orbits);
    for (int o = 0; o < orbits; ++o) {
        const int c = b->cls[o];
        if (c < 0 || c >= (int)b->class_neq.size()) return bfail(b, "orbit size class out of range");
        if (b->steps[o] < 0 || b->steps[o] % b->ksteps != 0)
            return bfail(b, "per-orbit step counts must be non-negative multiples of ksteps");
        const int n = b->class_neq[c];
        b->yoff[o] = (long long)ys;
        b->ooff[o] = (long long)os;
        ys += n;
        os += (size_t)(b->steps[o] / b->ksteps + 1) * n;
        cost[o] = (double)n * (double)b->steps[o];
    }
    b->state_size = ys;
    b->output_size = os;
    // longest first: the queue hands the most expensive orbits out first
    b->order.resize(orbits);
    std::iota(b->order.begin(), b->order.end(), 0);
    std::stable_sort(b->order.begin(), b->order.end(), [&](int a, int c) { return cost[a] > cost[c]; });
    // work items of each class: as many consecutive orbits (similar costs) as
    // share a wavefront
    const int nclass = (int)b->class_neq.size();
    const std::vector<BatchShape> shapes = batch_shapes(b);
    b->classes.assign(nclass, sodecl_batch::Class{});
    for (int ci = 0; ci < nclass; ++ci) b->classes[ci].shape = shapes[ci];
    for (int o : b->order) {
        auto& c = b->classes[b->cls[o]];
        const int opw = c.shape.slots();
        if (c.nitems == 0 || c.items[(size_t)opw * c.nitems - 1] >= 0) {
            c.items.insert(c.items.end(), opw, -1);
            ++c.nitems;
        }
        int* slot = &c.items[(size_t)opw * (c.nitems - 1)];
        int k = 0;
        while (slot[k] >= 0) ++k;
        slot[k] = o;
        c.cost += cost[o];
    }
    b->launch_order.resize(nclass);
    std::iota(b->launch_order.begin(), b->launch_order.end(), 0);
    std::stable_sort(b->launch_order.begin(), b->launch_order.end(),
                     [&](int x, int y) { return b->classes[x].cost > b->classes[y].cost; });

    if (!bhip(b, hipSetDevice(b->device), "hipSetDevice")) return 0;
    b->program = assemble_batch_program(b->source, batch_key(b), b->features, shapes);
    std::string log;
    if (!compile_program(b->program, device_arch(b->device), b->opts.fp_contract, b->code, log))
        return bfail(b, "Failed to build program executable:\n" + log);
    if (!bhip(b, hipModuleLoadData(&b->module, b->code.data()), "hipModuleLoadData")) return 0;
    auto up = [&](void** dst, const void* src, size_t bytes, const char* what) {
        return bhip(b, hipMalloc(dst, bytes), what) &&
               bhip(b, hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice), what);
    };
    // (the device's limit for a block: 160 KiB)
    const size_t max_lds = 160 * 1024;
    for (int ci = 0; ci < nclass; ++ci) {
        auto& c = b->classes[ci];
        const std::string name = "sodecl_batch_" + std::to_string(ci);
        if (!bhip(b, hipModuleGetFunction(&c.fn, b->module, name.c_str()), "class kernel")) return 0;
        // LDS per wavefront: per orbit (more than 8) parameters, and in the
        // form through LDS four rows of the class's size (the evaluation point
        // shared with the right-hand side, three band rows), times the
        // orbits per wavefront (batch_class.hip)
        const long n = c.shape.neq;
        const long tlen = c.shape.rows >= 2 ? (n + 15) / 16 * 16 : n;
        c.lds_bytes = param_lds(b, c.shape) + (c.shape.window ? 0 : (size_t)(4 * tlen * c.shape.slots()) * sizeof(double));
        if (c.nitems > 0 && c.lds_bytes > max_lds)
            return bfail(b, "a size class needs " + std::to_string(c.lds_bytes) + " bytes of LDS per wavefront (" +
                                std::to_string(b->npar) + " parameters), more than a block can have");
        if (c.nitems > 0 &&
            !up((void**)&c.d_items, c.items.data(), c.items.size() * sizeof(int), "work items"))
            return 0;
        if (!bhip(b, hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking), "hipStreamCreate") ||
            !bhip(b, hipEventCreateWithFlags(&c.done, hipEventDisableTiming), "hipEventCreate"))
            return 0;
    }
    if (!bhip(b, hipEventCreateWithFlags(&b->fork, hipEventDisableTiming), "hipEventCreate")) return 0;
    if (!up((void**)&b->d_steps, b->steps.data(), orbits * sizeof(int), "steps")) return 0;
    if (!up((void**)&b->d_yoff, b->yoff.data(), orbits * sizeof(long long), "state offsets")) return 0;
    if (!up((void**)&b->d_ooff, b->ooff.data(), orbits * sizeof(long long), "output offsets")) return 0;
    b->ready = true;
    return 1;
}

size_t sodecl_batch_state_size(const sodecl_batch* b) { return b ? b->state_size : 0; }
size_t sodecl_batch_output_size(const sodecl_batch* b) { return b ? b->output_size : 0; }

int sodecl_batch_offsets(const sodecl_batch* b, long long* yoff, long long* ooff)
{
    if (!b || b->yoff.empty()) return 0;
    if (yoff) std::memcpy(yoff, b->yoff.data(), b->yoff.size() * sizeof(long long));
    if (ooff) std::memcpy(ooff, b->ooff.data(), b->ooff.size() * sizeof(long long));
    return 1;
}

int sodecl_batch_run_device(sodecl_batch* b, const double* y0, const double* params, double* out, long long* newton,
                            void* stream)
{
    if (!b) return 0;
    if (!b->ready) return bfail(b, "sodecl_batch_setup has not succeeded");
    if (!y0 || !out || !newton || (b->npar > 0 && !params)) return bfail(b, "null device pointer");
    if (!bhip(b, hipSetDevice(b->device), "hipSetDevice")) return 0;
    hipStream_t s = (hipStream_t)stream;
    // every class's kernel on its own stream after the work queued on the
    // caller's stream, then the caller's stream after all of them (its waits
    // are queued last: a class stream that shares a hardware queue with the
    // caller's would otherwise wait behind them)
    if (!bhip(b, hipEventRecord(b->fork, s), "hipEventRecord")) return 0;
    for (int ci : b->launch_order) {
        auto& c = b->classes[ci];
        if (c.nitems == 0) continue;
        void* args[] = {&c.d_items, &b->d_steps, &b->d_yoff, &b->d_ooff, (void*)&y0, (void*)&params, &out, &newton};
        if (!bhip(b, hipStreamWaitEvent(c.stream, b->fork, 0), "hipStreamWaitEvent") ||
            !bhip(b, hipModuleLaunchKernel(c.fn, (unsigned)c.nitems, 1, 1, 64, 1, 1, (unsigned)c.lds_bytes, c.stream,
                                           args, nullptr),
                  "hipModuleLaunchKernel(batch)") ||
            !bhip(b, hipEventRecord(c.done, c.stream), "hipEventRecord"))
            return 0;
    }
    for (int ci : b->launch_order)
        if (b->classes[ci].nitems > 0 && !bhip(b, hipStreamWaitEvent(s, b->classes[ci].done, 0), "hipStreamWaitEvent"))
            return 0;
    return 1;
}

const char* sodecl_batch_last_error(const sodecl_batch* b) { return b ? b->last_error.c_str() : "null batch"; }
const char* sodecl_batch_program_source(const sodecl_batch* b) { return b ? b->program.c_str() : ""; }

}  // extern "C"
