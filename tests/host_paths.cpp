// Host paths of csrc/plife.hip on a HIP runtime made of host memory, for what
// no run on a device shows: failed allocations, calls that must not wait, what
// the planner believes while the device is behind.  Compiled for the host
// alone; kernels are functions on their arguments, or nothing.
//   host_paths CASE   exit 0: as stated
#include "../particle-life-app_amd/csrc/plife.hip"

#include <functional>
#include <map>

namespace fake {
std::map<const void *, std::string> kernels;       // host stub -> mangled name
std::vector<std::string> launched;
int syncs = 0;                                      // waits for a stream
std::vector<int> syncs_at_record;                   // their count at each event record
long allocs_left = -1;                              // hipMalloc calls that succeed (-1: all)
bool capturing = false;
int attributes = 0, attributes_in_capture = 0;      // hipFuncSetAttribute calls
hipError_t attribute_result = hipSuccess;
std::function<void(const std::string &, void **)> device;

bool has(const std::string &name, const char *what) { return name.find(what) != std::string::npos; }
int count(const char *what)
{
    int n = 0;
    for (const std::string &s : launched) n += has(s, what);
    return n;
}

template <typename T>
T arg(void **args, int k) { return *static_cast<T *>(args[k]); }

// k_bin, k_set_positions and k_copy_u64 as far as the host sees them: the step's counters.
void counters(const std::string &name, void **a)
{
    if (has(name, "k_bin")) {
        auto *counters = arg<unsigned long long *>(a, 9);
        auto *out = arg<unsigned long long *>(a, 12);
        const int nc = arg<int>(a, 10);
        for (int t = 0; t <= nc; ++t) {
            if (out) out[t] = counters[t];
            counters[t] = t < nc ? 0ull : arg<unsigned long long>(a, 11);
        }
    } else if (has(name, "k_set_positions")) {
        if (arg<PresetArgs>(a, 0).tag) *arg<PresetArgs>(a, 0).tag = 0;
    } else if (has(name, "k_copy_u64")) {
        std::memcpy(arg<unsigned long long *>(a, 1), arg<const unsigned long long *>(a, 0), 8u * (size_t)arg<int>(a, 2));
    }
}

// The force kernels' record of their workgroups' pairs: table entry e had pairs_of(e).
void work(const std::string &name, void **args, const std::function<uint32_t(int)> &pairs_of)
{
    if (!has(name, "k_force")) return;
    const ForceArgs &a = *static_cast<ForceArgs *>(args[0]);
    for (int e = 0; e < a.nb_total; ++e) a.block_work[e] = pairs_of(e);
    a.block_work[a.nb_total] = a.work_tag;
}
}  // namespace fake

struct ihipStream_t {};
struct ihipEvent_t {};
struct ihipGraph {};
struct hipGraphExec {};

extern "C" {
char __hip_fatbin[1];
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    fake::kernels[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t)
{
    fake::launched.push_back(fake::kernels[f]);
    if (fake::device) fake::device(fake::kernels[f], args);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    if (fake::allocs_left == 0) return hipErrorOutOfMemory;
    if (fake::allocs_left > 0) --fake::allocs_left;
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) { *d = p; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 65536;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static void *scratch_mem = std::calloc(kNa.total, 1);
    *p = scratch_mem;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int)
{
    ++fake::attributes;
    fake::attributes_in_capture += fake::capturing;
    return fake::attribute_result;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = new ihipStream_t; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { ++fake::syncs; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { fake::capturing = true; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { fake::capturing = false; *g = new ihipGraph; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { fake::syncs_at_record.push_back(fake::syncs); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { delete g; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { *x = new hipGraphExec; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete x; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
}

namespace {

#define CHECK(cond)                                                                                       \
    do {                                                                                                  \
        if (!(cond)) {                                                                                    \
            std::printf("%s:%d: not so: %s (last error: %s)\n", __FILE__, __LINE__, #cond, plife_last_error()); \
            std::exit(1);                                                                                 \
        }                                                                                                 \
    } while (0)

const double kMatrix[4] = {0.5, -0.25, 0.125, 1.0};

plife_settings settings(int dim, double rmax) { return plife_settings{dim, 1, rmax, 0.8, 1.0, 0.01, 0.3}; }

plife_physics *engine(int dim, double rmax, int n, plife_tuning t = plife_tuning{})
{
    plife_physics *h = nullptr;
    const plife_settings s = settings(dim, rmax);
    CHECK(plife_create(0, &h) == PLIFE_OK);
    CHECK(plife_set_settings(h, &s, 2, kMatrix) == PLIFE_OK);
    CHECK(plife_set_tuning(h, &t) == PLIFE_OK);
    if (n > 0) CHECK(plife_generate_particles(h, n, 7) == PLIFE_OK);
    return h;
}

// A growth that fails at any allocation leaves a handle that steps what it
// holds or refuses to, and that a later growth mends.
void failed_growth()
{
    for (int batch = 0; batch < 2; ++batch)
        for (int fail_at = 0; fail_at < 21; ++fail_at) {
            plife_physics *h = nullptr;
            plife_batch *b = nullptr;
            const plife_settings s = settings(2, 0.05);
            int32_t id;
            if (batch) {
                CHECK(plife_batch_create(0, &b) == PLIFE_OK);
                h = b;
                CHECK(plife_batch_add_generated_world(b, &s, 2, kMatrix, 500, 1, &id) == PLIFE_OK);
            } else {
                h = engine(2, 0.05, 500);
            }
            auto update = [&]() { return batch ? plife_batch_update(b, 1) : plife_update(h, 1); };
            auto grow = [&](int n) {
                return batch ? plife_batch_add_generated_world(b, &s, 2, kMatrix, n, 2, &id) : plife_generate_particles(h, n, 2);
            };
            CHECK(update() == PLIFE_OK);
            fake::allocs_left = fail_at;
            CHECK(grow(5000) == PLIFE_ERR_MEMORY);
            fake::allocs_left = -1;
            fake::launched.clear();
            const int rc = update();
            if (h->n > 0 && !(h->keys0 && h->kA && h->skeys && h->perm && h->rec)) CHECK(rc != PLIFE_OK && fake::launched.empty());
            CHECK(grow(5000) == PLIFE_OK);
            CHECK(update() == PLIFE_OK);
            CHECK(h->n == (batch ? 5500 : 5000) && h->cap >= h->n && h->keys0 && h->kA && h->skeys && h->perm && h->rec);
            if (batch) plife_batch_destroy(b);
            else plife_destroy(h);
        }
}

// What measure_cells leaves in the counters is of no step: while the device is
// at the first step's binning, a 3D batch's neighbours are still unknown.
void measured_cells_are_no_step()
{
    plife_batch *b = nullptr;
    const plife_settings s = settings(3, 0.1);
    const plife_tuning t{0, 0, 1, 0.0, 0, 0, 1};        // direct launches, multi-launch path
    int32_t id;
    CHECK(plife_batch_create(0, &b) == PLIFE_OK && plife_batch_set_tuning(b, &t) == PLIFE_OK);
    CHECK(plife_batch_add_generated_world(b, &s, 2, kMatrix, 20000, 1, &id) == PLIFE_OK);
    int bins = 0;
    fake::device = [&](const std::string &name, void **a) {
        if (bins >= 2) return;
        bins += fake::has(name, "k_bin");
        fake::counters(name, a);
    };
    CHECK(plife_batch_update(b, 3) == PLIFE_OK);
    CHECK(fake::count("k_bin") == 4);                    // the measurement's and three steps'
    CHECK(plife_batch_update(b, 1) == PLIFE_OK);
    CHECK(b->worlds[0].nb < 0.0);
    plife_batch_destroy(b);
}

// A stop that arrives before an update's first step leaves the last step's
// exports, also where that step's counters have not reached the host yet.
void stopped_update_keeps_the_last_step()
{
    plife_physics *h = engine(3, 0.1, 20000, plife_tuning{0, 0, 1, 0.0, 0, 0, 1});
    CHECK(plife_update(h, 1) == PLIFE_OK);               // (the device has copied no counters)
    fake::device = [&](const std::string &name, void **) {
        if (fake::has(name, "k_bin")) CHECK(plife_force_update_stop(h) == PLIFE_OK);
    };
    int64_t steps = 0;
    CHECK(plife_update(h, 8) == PLIFE_STOPPED);
    CHECK(plife_get_steps(h, &steps) == PLIFE_OK && steps >= 1);
    int32_t ncells = 0;
    std::vector<int32_t> end(1000);
    CHECK(plife_get_grid(h, nullptr, &ncells) == PLIFE_OK && ncells == 1000);
    CHECK(plife_get_cells(h, nullptr, end.data(), nullptr, ncells) == PLIFE_OK);
    plife_destroy(h);
}

// Positions or particles made anew: the planner keeps neither the workgroups'
// measured work nor the neighbours of the state before, whatever the way in.  An
// uploaded state keeps the work, as estimates.
void new_state_forgets_measured_work()
{
    const plife_tuning t{256, 0, 1, 0.0, 1, 0, 1};
    for (int way = 0; way < 4; ++way) {
        plife_physics *h = nullptr;
        plife_batch *b = nullptr;
        int32_t id = 0;
        const plife_settings s = settings(2, 0.05);
        if (way == 2) {
            CHECK(plife_batch_create(0, &b) == PLIFE_OK && plife_batch_set_tuning(b, &t) == PLIFE_OK);
            CHECK(plife_batch_add_generated_world(b, &s, 2, kMatrix, 40000, 1, &id) == PLIFE_OK);
            h = b;
        } else {
            h = engine(2, 0.05, 40000, t);
        }
        auto update = [&]() { return b ? plife_batch_update(b, 1) : plife_update(h, 1); };
        bool recording = true;
        fake::device = [&](const std::string &name, void **a) {
            fake::counters(name, a);
            if (recording) fake::work(name, a, [&](int e) { return e == h->nb_total - 1 ? 1000000u : 1000u; });
            if (fake::has(name, "k_force")) h->d_pairs[2] = 4000000ull;       // 100 neighbours each
        };
        CHECK(update() == PLIFE_OK);
        recording = false;                  // the device's next record is not there yet
        if (way == 0) CHECK(plife_set_positions(h, 0, 5) == PLIFE_OK);
        if (way == 1) CHECK(plife_generate_particles(h, 40000, 5) == PLIFE_OK);
        if (way == 2) CHECK(plife_batch_set_world_positions(b, id, 0, 5) == PLIFE_OK);
        if (way == 3) {
            std::vector<double> x(3 * 40000, 0.5);
            std::vector<int32_t> types(40000, 1);
            CHECK(plife_set_particles(h, 40000, x.data(), x.data(), types.data()) == PLIFE_OK);
        }
        CHECK(prepare_step(h) == PLIFE_OK);
        CHECK(h->worlds[0].nb < 0.0 && (int)h->blocks.size() == 157);
        if (way == 3) {
            CHECK((int)h->blocks[0].y == 256 * 156 && h->block_est[0] == 1000000u);   // the heaviest, first
            plife_destroy(h);
            continue;
        }
        for (int i = 0; i < 157; ++i) {
            CHECK((int)h->blocks[i].y == 256 * i);                            // no order made from the old work
            if (i < 156) CHECK(h->block_est[i] == h->block_est[0]);
        }
        CHECK(do_step(h, nullptr) == PLIFE_OK);   // its binning hands on the counters of the state before
        fake::device = nullptr;
        refresh_occupancy(h);
        if (way != 1) CHECK(h->stat_host[2 + 1] != h->version + 1);
        if (b) plife_batch_destroy(b);
        else plife_destroy(h);
    }
}

// Forces and time steps so large that what clear_high leaves of a pair out of
// range could show take the literal path, as matrices that are not finite do.
void extreme_forces_take_the_literal_law()
{
    auto literal = [](double force, double dt, double entry) {
        WorldHost w;
        w.st = settings(2, 0.05);
        w.st.force = force;
        w.st.dt = dt;
        w.matrix = {entry};
        return world_dev(w, 0u, 0).all_global;
    };
    CHECK(!literal(0x1p400, 0.01, 1.0) && !literal(1.0, -0x1p400, 1.0) && !literal(1.0, 0.01, 1e290));
    CHECK(literal(0x1p401, 0.01, 1.0) && literal(-1e300, 0.01, 1.0) && literal(1.0, 1e121, 1.0) && literal(1.0, 0.01, 1e301));
}

// A no-alloc step of no particles hands no kernel the caller's matrix: it was
// never read for one.
void empty_noalloc_step_reads_no_matrix()
{
    const plife_settings s = settings(2, 0.05);
    bool seen = false;
    fake::device = [&](const std::string &name, void **a) {
        if (!fake::has(name, "k_na_setup")) return;
        seen = true;
        CHECK(fake::arg<const double *>(a, 1) == nullptr);
    };
    CHECK(plife_step_noalloc(&s, 2, kMatrix, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                             nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr) == PLIFE_OK);
    CHECK(seen);
}

// A launch of more than 64 KB of LDS raises the kernel's limit before any
// capture, once, and an update whose limit cannot be raised says so.
void lds_limit_is_raised_ahead()
{
    const plife_tuning t{0, 0, 0, 0.0, 1, 0, 1};
    for (const bool fails : {true, false}) {
        plife_physics *h = engine(3, 0.04, 130000, t);
        fake::attribute_result = fails ? hipErrorInvalidValue : hipSuccess;
        fake::launched.clear();
        fake::attributes = 0;
        const int rc = plife_update(h, 70);
        CHECK(h->plan.lds > 65536);
        if (fails) {
            CHECK(rc == PLIFE_ERR_DEVICE && fake::count("k_force") == 0);
        } else {
            CHECK(rc == PLIFE_OK && fake::attributes_in_capture == 0);
            const int before = fake::attributes;
            CHECK(before > 0 && plife_update(h, 3) == PLIFE_OK && fake::attributes == before);
        }
        plife_destroy(h);
    }
}

// The homes per workgroup measured for a layout go to no layout that the planner
// itself would give others: here two worlds of one density, either side of the
// particle count its rule for short rows changes at.
void kept_homes_follow_the_plan()
{
    const double rmax = 1.0 / 700.5;
    const plife_tuning t{0, 0, 0, 0.0, 1, 0, 1};
    plife_physics *h = engine(2, rmax, 99999, t);
    CHECK(plife_update(h, 40) == PLIFE_OK && h->bs_seen.size() == 1 && h->plan.bs == 128);
    CHECK(plife_generate_particles(h, 99998, 8) == PLIFE_OK && plife_update(h, 3) == PLIFE_OK);
    CHECK(h->bs_meas == h->version && h->plan.bs == 128);        // the same class: kept
    CHECK(plife_generate_particles(h, 100001, 8) == PLIFE_OK && plife_update(h, 3) == PLIFE_OK);
    CHECK(h->plan.bs == 256);
    plife_destroy(h);
}

// A timing of steps holds steps alone: the wait of a new state's first update
// for its first step lies before it.
void timed_steps_do_not_wait()
{
    for (const int dim : {2, 3}) {
        plife_physics *h = engine(dim, dim == 3 ? 0.1 : 0.02, 30000, plife_tuning{0, 0, 1, 0.0, 0, 0, 1});
        fake::device = [&](const std::string &name, void **a) {
            fake::counters(name, a);
            if (fake::has(name, "k_scan")) h->d_pairs[1] = 40000;            // sum of squares: uniform
        };
        double ms = 0.0;
        fake::syncs_at_record.clear();
        CHECK(plife_time_steps(h, 12, &ms) == PLIFE_OK);
        const std::vector<int> &s = fake::syncs_at_record;
        CHECK(s.size() >= 2 && s[s.size() - 2] == s.back());                 // the two events around the steps
        plife_destroy(h);
    }
}

}  // namespace

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> cases = {
        {"failed_growth", failed_growth},
        {"kept_homes_follow_the_plan", kept_homes_follow_the_plan},
        {"lds_limit_is_raised_ahead", lds_limit_is_raised_ahead},
        {"measured_cells_are_no_step", measured_cells_are_no_step},
        {"empty_noalloc_step_reads_no_matrix", empty_noalloc_step_reads_no_matrix},
        {"extreme_forces_take_the_literal_law", extreme_forces_take_the_literal_law},
        {"new_state_forgets_measured_work", new_state_forgets_measured_work},
        {"timed_steps_do_not_wait", timed_steps_do_not_wait},
        {"stopped_update_keeps_the_last_step", stopped_update_keeps_the_last_step},
    };
    const auto it = argc == 2 ? cases.find(argv[1]) : cases.end();
    if (it == cases.end()) return 2;
    it->second();
    return 0;
}
