// C-ABI of environments, state validity and motion validation.
#include <algorithm>
#include <cmath>
#include <functional>
#include <memory>
#include <vector>

#include "runtime.hpp"

using namespace ompl_amd;

namespace {

Env &env_of(ompl_amd_env e)
{
    OA_REQUIRE(e, OMPL_AMD_ERR_ARG, "null environment");
    return e->env;
}

// Word of the thread's pinned slot that an environment's build reports in.
constexpr int kEnvBaseAt = 520;

// Order of an obstacle list in the grid's table: increasing distance from the
// arm's base (the world origin) to the obstacle's nearest point, ties in the
// caller's order.  Every check result is "any obstacle hit", so the order leaves
// results unchanged; links near the base sweep the least volume, so the
// obstacles nearest to it are hit by the most configurations, and a state tested
// against all of them is done sooner.
std::vector<int> nearest_first(int n, const std::function<double(int)> &gap)
{
    std::vector<double> key(n);
    std::vector<int> order(n);
    for (int i = 0; i < n; ++i) {
        key[i] = gap(i);
        order[i] = i;
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return key[x] < key[y]; });
    return order;
}

} // namespace

// Batched DiscreteMotionValidator::checkMotion(s1, s2) over device arrays.
void ompl_amd::check_motions_tuned(const Tuning &t, const Env &env, const double *a, const double *b, int64_t n,
                                   double lvs, unsigned factor, uint8_t *out, int32_t *checked, hipStream_t s,
                                   Workspace *own)
{
    OA_REQUIRE(n >= 0, OMPL_AMD_ERR_ARG, "negative edge count");
    if (n == 0) return;
    OA_REQUIRE(a && b && out, OMPL_AMD_ERR_ARG, "null edge or output pointer");
    OA_REQUIRE(lvs > 0.0 && factor >= 1, OMPL_AMD_ERR_ARG, "longest valid segment must be > 0 and factor >= 1");
    OA_REQUIRE(n < (int64_t)1 << 31, OMPL_AMD_ERR_ARG, "at most 2^31-1 edges per call");
    MotionArgs A{};
    A.a = a;
    A.b = b;
    A.n = n;
    A.lvs = lvs;
    A.factor = factor;
    A.out = out;
    A.checked = checked;
    std::unique_lock<std::mutex> lk; // held until this batch's launches are enqueued
    Workspace &w = own ? *own : workspace(s, (size_t)n, lk);
    launch_grid_motions(env.grid, A, own ? grid_scratch(w) : stream_grid_scratch(w, s), t.motion_strategy == 2, s);
}

namespace {

void check_motions(const ompl_amd_env_s &e, const double *a, const double *b, int64_t n, double lvs, unsigned factor,
                   uint8_t *out, int32_t *checked, hipStream_t s)
{
    check_motions_tuned(tuning_for(e), e.env, a, b, n, lvs, factor, out, checked, s);
}

} // namespace

// A captured motion batch: the launches of one check_motions call recorded in
// HIP graphs (pointers, sizes and launch shape fixed at capture) with their own
// survivor workspace, so replays on any stream do not share state with eager
// calls.  No memset nodes: the strategies clear their counters with kernels.
// The batch is recorded twice, once per survivor counter set (each recording
// clears the other set for the next replay), and replays alternate between
// the two, as eager batches on one workspace do.
// A group of independent batches is recorded in one graph, batch 0 on the
// capturing stream and batch i > 0 on a side stream forked from it and joined
// back, so a replay runs the batches concurrently.
struct ompl_amd_motion_graph_s {
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    int next = 0; // the recording the next replay launches
    std::vector<std::unique_ptr<Workspace>> ws; // one per batch
    std::vector<hipStream_t> side;     // batches 1.. are recorded on these
    std::vector<hipEvent_t> fork_join; // fork, then one join per side stream
    ~ompl_amd_motion_graph_s()
    {
        for (int i = 0; i < 2; ++i) {
            if (exec[i]) hipGraphExecDestroy(exec[i]);
            if (graph[i]) hipGraphDestroy(graph[i]);
        }
        for (auto &w : ws) {
            free_workspace_arrays(*w);
            if (w->counters) hipFree(w->counters);
        }
        for (hipStream_t st : side) hipStreamDestroy(st);
        for (hipEvent_t ev : fork_join) hipEventDestroy(ev);
    }
};

namespace {

void graph_workspace(Workspace &w, int64_t n)
{
    const size_t cap = (size_t)n < 1024 ? 1024 : (size_t)n;
    OA_HIP(device_malloc(&w.counters, kWorkspaceCounters * sizeof(int32_t)));
    OA_HIP(hipMemset(w.counters, 0, kWorkspaceCounters * sizeof(int32_t)));
    alloc_workspace_arrays(w, cap);
}

// Records the group twice (once per survivor counter set of every batch's
// workspace) and instantiates both recordings.
void record_group(ompl_amd_motion_graph_s *g, const Env &env, const Tuning &t, int nb, const double *const *a,
                  const double *const *b, const int64_t *n, double lvs, unsigned factor, uint8_t *const *out,
                  int32_t *const *checked)
{
    for (int i = 0; i < nb; ++i) graph_workspace(*g->ws[(size_t)i], n[i]);
    for (int i = 1; i < nb; ++i) {
        hipStream_t st = nullptr;
        OA_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking)); // default priority
        g->side.push_back(st);
    }
    for (int i = 0; i < nb; ++i) {
        hipEvent_t ev = nullptr;
        OA_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        g->fork_join.push_back(ev);
    }
    OA_HIP(hipDeviceSynchronize());
    // capture on the calling thread's own stream (the null stream cannot capture)
    hipStream_t cs = thread_resources().stream;
    for (int r = 0; r < 2; ++r) {
        // recording r uses counter set r of each workspace when its batch
        // alternates sets (grid_scratch takes them in turn)
        OA_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        try {
            if (nb > 1) {
                OA_HIP(hipEventRecord(g->fork_join[0], cs));
                for (int i = 1; i < nb; ++i) OA_HIP(hipStreamWaitEvent(g->side[(size_t)i - 1], g->fork_join[0], 0));
            }
            for (int i = 0; i < nb; ++i) {
                hipStream_t st = i == 0 ? cs : g->side[(size_t)i - 1];
                check_motions_tuned(t, env, a[i], b[i], n[i], lvs, factor, out[i], checked ? checked[i] : nullptr, st,
                                    g->ws[(size_t)i].get());
            }
            for (int i = 1; i < nb; ++i) {
                OA_HIP(hipEventRecord(g->fork_join[(size_t)i], g->side[(size_t)i - 1]));
                OA_HIP(hipStreamWaitEvent(cs, g->fork_join[(size_t)i], 0));
            }
        } catch (...) {
            hipGraph_t dropped = nullptr;
            hipStreamEndCapture(cs, &dropped);
            if (dropped) hipGraphDestroy(dropped);
            throw;
        }
        OA_HIP(hipStreamEndCapture(cs, &g->graph[r]));
        OA_HIP(hipGraphInstantiate(&g->exec[r], g->graph[r], nullptr, nullptr, 0));
    }
}

} // namespace

extern "C" {

int ompl_amd_env_create(const float *spheres, int n_spheres, const float *boxes, int n_boxes, ompl_amd_env *out)
{
    return guarded([&] {
        OA_REQUIRE(out, OMPL_AMD_ERR_ARG, "null output handle");
        OA_REQUIRE(n_spheres >= 0 && n_boxes >= 0, OMPL_AMD_ERR_ARG, "negative obstacle count");
        OA_REQUIRE(n_spheres == 0 || spheres, OMPL_AMD_ERR_ARG, "null sphere array");
        OA_REQUIRE(n_boxes == 0 || boxes, OMPL_AMD_ERR_ARG, "null box array");
        OA_REQUIRE((int64_t)n_spheres + 2 * (int64_t)n_boxes <= kMaxEnvWords, OMPL_AMD_ERR_ARG,
                   "environment too large: spheres + 2*boxes must be <= %d", kMaxEnvWords);
        ensure_init();
        std::vector<float4> h((size_t)n_spheres + 2 * (size_t)n_boxes + 1);
        for (int i = 0; i < n_spheres; ++i) {
            const float *o = spheres + 4 * i;
            OA_REQUIRE(std::isfinite(o[0]) && std::isfinite(o[1]) && std::isfinite(o[2]) && std::isfinite(o[3]),
                       OMPL_AMD_ERR_ARG, "sphere obstacle %d: non-finite value", i);
            OA_REQUIRE(o[3] >= 0.0f, OMPL_AMD_ERR_ARG, "negative sphere radius");
            const float rs = o[3] + kRobotR;
            h[i] = make_float4(o[0], o[1], o[2], rs * rs);
        }
        for (int i = 0; i < n_boxes; ++i) {
            const float *o = boxes + 6 * i;
            OA_REQUIRE(std::isfinite(o[0]) && std::isfinite(o[1]) && std::isfinite(o[2]) && std::isfinite(o[3]) &&
                           std::isfinite(o[4]) && std::isfinite(o[5]),
                       OMPL_AMD_ERR_ARG, "box obstacle %d: non-finite value", i);
            OA_REQUIRE(o[3] >= 0.0f && o[4] >= 0.0f && o[5] >= 0.0f, OMPL_AMD_ERR_ARG, "negative box extent");
            h[n_spheres + 2 * i] = make_float4(o[0] - o[3], o[1] - o[4], o[2] - o[5], 0.0f);
            h[n_spheres + 2 * i + 1] = make_float4(o[0] + o[3], o[1] + o[4], o[2] + o[5], 0.0f);
        }
        const std::vector<int> so = nearest_first(n_spheres, [&](int i) {
            const float *o = spheres + 4 * i;
            return std::sqrt((double)o[0] * o[0] + (double)o[1] * o[1] + (double)o[2] * o[2]) - (double)o[3];
        });
        const std::vector<int> bo = nearest_first(n_boxes, [&](int i) {
            const float4 lo = h[n_spheres + 2 * i], hi = h[n_spheres + 2 * i + 1];
            const double dx = std::max({(double)lo.x, -(double)hi.x, 0.0});
            const double dy = std::max({(double)lo.y, -(double)hi.y, 0.0});
            const double dz = std::max({(double)lo.z, -(double)hi.z, 0.0});
            return std::sqrt(dx * dx + dy * dy + dz * dz);
        });
        // the grid's obstacle table: every obstacle as a box with a squared
        // contact distance (a sphere is the box lo = hi = centre)
        const int n_obs = n_spheres + n_boxes;
        std::vector<float4> tab;
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int i = 0; i < n_obs; ++i) {
            const bool sphere = i < n_spheres;
            const int at = sphere ? so[i] : n_spheres + 2 * bo[i - n_spheres];
            float4 l = h[at], u = sphere ? l : h[at + 1];
            if (!sphere) l.w = kRobotR * kRobotR;
            u.w = 0.0f;
            tab.push_back(l);
            tab.push_back(u);
            const double r = std::sqrt((double)l.w) * 1.00002 + 2e-4;
            const float a[3] = {l.x, l.y, l.z}, c[3] = {u.x, u.y, u.z};
            for (int k = 0; k < 3; ++k) {
                lo[k] = std::min(lo[k], (double)a[k] - r);
                hi[k] = std::max(hi[k], (double)c[k] + r);
            }
        }
        auto *e = new ompl_amd_env_s();
        Env &env = e->env;
        env.ns = n_spheres;
        env.nb = n_boxes;
        env.grid.n_obs = n_obs;
        grid_extent(env.grid, lo, hi, n_obs == 0);
        // one allocation: obstacles (the caller's order) and table, cells, lists, build counter
        auto up = [](size_t b) { return (b + 255) / 256 * 256; };
        const size_t n_words = h.size();
        h.insert(h.end(), tab.begin(), tab.end());
        const size_t obs_b = up(h.size() * sizeof(float4)), cells_b = grid_cells_bytes(env.grid),
                     lists_b = grid_lists_bytes(env.grid);
        env.bytes = obs_b + cells_b + lists_b + 256;
        char *mem = nullptr;
        const hipError_t err = device_malloc(&mem, env.bytes);
        if (err != hipSuccess) {
            delete e;
            fail(OMPL_AMD_ERR_NOMEM, "environment allocation failed: %s", hipGetErrorString(err));
        }
        env.obs = (float4 *)mem;
        try {
            uint32_t *cells = (uint32_t *)(mem + obs_b);
            uint16_t *lists = (uint16_t *)(mem + obs_b + cells_b);
            uint32_t *counter = (uint32_t *)(mem + obs_b + cells_b + lists_b);
            env.grid.tab = env.obs + n_words;
            env.grid.cells = cells;
            env.grid.lists = lists;
            ThreadResources &r = thread_resources();
            OA_HIP(hipMemcpyAsync(env.obs, h.data(), h.size() * sizeof(float4), hipMemcpyHostToDevice, r.stream));
            launch_grid_build(env.grid, cells, lists, counter, r.pinned_dev + kEnvBaseAt, r.stream);
            OA_HIP(hipStreamSynchronize(r.stream));
            env.grid.base_hit = r.pinned[kEnvBaseAt];
        } catch (...) {
            (void)hipFree(mem);
            delete e;
            throw;
        }
        *out = e;
    });
}

int ompl_amd_env_destroy(ompl_amd_env e)
{
    return guarded([&] {
        if (!e) return;
        const int users = e->server_users.load();
        OA_REQUIRE(users == 0, OMPL_AMD_ERR_ARG,
                   "environment still in use by %d queued or running server request(s); destroy it after they finish",
                   users);
        if (e->env.obs) OA_HIP(hipFree(e->env.obs));
        delete e;
    });
}

int ompl_amd_env_bytes(ompl_amd_env e, size_t *bytes)
{
    return guarded([&] {
        OA_REQUIRE(bytes, OMPL_AMD_ERR_ARG, "null output");
        *bytes = env_of(e).bytes;
    });
}

int ompl_amd_validate_states_dev(ompl_amd_env e, const float *q, int64_t n, uint8_t *out, void *stream)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n >= 0, OMPL_AMD_ERR_ARG, "negative state count");
        if (n == 0) return;
        OA_REQUIRE(q && out, OMPL_AMD_ERR_ARG, "null state or output pointer");
        launch_grid_validate<float>(env.grid, q, n, out, resolve_stream(stream));
    });
}

int ompl_amd_validate_states_f64_dev(ompl_amd_env e, const double *q, int64_t n, uint8_t *out, void *stream)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n >= 0, OMPL_AMD_ERR_ARG, "negative state count");
        if (n == 0) return;
        OA_REQUIRE(q && out, OMPL_AMD_ERR_ARG, "null state or output pointer");
        launch_grid_validate<double>(env.grid, q, n, out, resolve_stream(stream));
    });
}

int ompl_amd_is_valid(ompl_amd_env e, const double *q, int *valid)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(q && valid, OMPL_AMD_ERR_ARG, "null state or output pointer");
        ThreadResources &r = thread_resources();
        State1 st;
        for (int j = 0; j < kDof; ++j) st.q[j] = q[j];
        launch_validate_single(env.grid, st, r.pinned_dev, r.stream);
        OA_HIP(hipStreamSynchronize(r.stream));
        *valid = r.pinned[0];
    });
}

int ompl_amd_arm_spheres_dev(const float *q, int64_t n, float *out, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(n >= 0, OMPL_AMD_ERR_ARG, "negative state count");
        if (n == 0) return;
        OA_REQUIRE(q && out, OMPL_AMD_ERR_ARG, "null pointer");
        launch_arm_spheres(q, n, out, resolve_stream(stream));
    });
}

int ompl_amd_check_motions_dev(ompl_amd_env e, const double *a, const double *b, int64_t n, double lvs,
                               unsigned factor, uint8_t *out, int32_t *checked, void *stream)
{
    return guarded([&] {
        env_of(e);
        check_motions(*e, a, b, n, lvs, factor, out, checked, resolve_stream(stream));
    });
}

int ompl_amd_check_motions_last_valid_dev(ompl_amd_env e, const double *a, const double *b, int64_t n, double lvs,
                                          unsigned factor, uint8_t *out, double *last_t, void *stream)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n >= 0, OMPL_AMD_ERR_ARG, "negative edge count");
        if (n == 0) return;
        OA_REQUIRE(a && b && out && last_t, OMPL_AMD_ERR_ARG, "null pointer");
        OA_REQUIRE(lvs > 0.0 && factor >= 1, OMPL_AMD_ERR_ARG, "longest valid segment must be > 0 and factor >= 1");
        OA_REQUIRE(n < (int64_t)1 << 31, OMPL_AMD_ERR_ARG, "at most 2^31-1 edges per call");
        MotionArgs A{};
        A.a = a;
        A.b = b;
        A.n = n;
        A.lvs = lvs;
        A.factor = factor;
        A.out = out;
        const hipStream_t st = resolve_stream(stream);
        std::unique_lock<std::mutex> lk; // held until the launches are enqueued
        Workspace &w = workspace(st, (size_t)n, lk);
        launch_grid_last_valid(env.grid, A, last_t, stream_grid_scratch(w, st), st);
    });
}

int ompl_amd_check_motion(ompl_amd_env e, const double *a, const double *b, double lvs, unsigned factor, int *valid)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(a && b && valid, OMPL_AMD_ERR_ARG, "null pointer");
        OA_REQUIRE(lvs > 0.0 && factor >= 1, OMPL_AMD_ERR_ARG, "longest valid segment must be > 0 and factor >= 1");
        ThreadResources &r = thread_resources();
        Edge1 E;
        for (int j = 0; j < kDof; ++j) {
            E.a[j] = a[j];
            E.b[j] = b[j];
        }
        launch_motion_single(env.grid, E, lvs, factor, r.pinned_dev, r.stream);
        OA_HIP(hipStreamSynchronize(r.stream));
        *valid = r.pinned[0];
    });
}

int ompl_amd_check_state_lists_dev(ompl_amd_env e, const double *q_soa, int64_t n_states, const int64_t *offsets,
                                   int64_t n_lists, uint8_t *out, int32_t *first_invalid, void *stream)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n_states >= 0 && n_lists >= 0, OMPL_AMD_ERR_ARG, "negative sizes");
        if (n_lists == 0) return;
        OA_REQUIRE(offsets && out && (n_states == 0 || q_soa), OMPL_AMD_ERR_ARG, "null pointer");
        OA_REQUIRE(n_lists < (int64_t)1 << 31 && n_states < (int64_t)1 << 31, OMPL_AMD_ERR_ARG,
                   "at most 2^31-1 lists and states per call");
        const hipStream_t st = resolve_stream(stream);
        std::unique_lock<std::mutex> lk; // held until the launches are enqueued
        Workspace &w = workspace(st, (size_t)n_lists, lk);
        launch_grid_state_lists(env.grid, q_soa, n_states, offsets, n_lists, out, first_invalid,
                                stream_grid_scratch(w, st), st);
    });
}

int ompl_amd_check_states(ompl_amd_env e, const double *states, int count, int *valid, int *first_invalid)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(count >= 0 && valid && (count == 0 || states), OMPL_AMD_ERR_ARG, "bad arguments");
        ThreadResources &r = thread_resources();
        // staging: offsets [2] int64, result u8 + i32, then the states dof-major
        const size_t head = 64;
        stage_reserve(r, head + (size_t)count * kDof * sizeof(double));
        int64_t *off = reinterpret_cast<int64_t *>(r.stage);
        off[0] = 0;
        off[1] = count;
        double *q = reinterpret_cast<double *>(r.stage + head);
        for (int i = 0; i < count; ++i)
            for (int j = 0; j < kDof; ++j) q[(size_t)j * count + i] = states[(size_t)i * kDof + j];
        {
            std::unique_lock<std::mutex> lk; // held until the launches are enqueued
            Workspace &w = workspace(r.stream, 1, lk);
            launch_grid_state_lists(env.grid, reinterpret_cast<const double *>(r.stage_dev + head), count,
                                    reinterpret_cast<const int64_t *>(r.stage_dev), 1,
                                    reinterpret_cast<uint8_t *>(r.stage_dev + 16),
                                    reinterpret_cast<int32_t *>(r.stage_dev + 32), grid_scratch(w), r.stream);
        }
        OA_HIP(hipStreamSynchronize(r.stream));
        *valid = reinterpret_cast<uint8_t *>(r.stage)[16];
        if (first_invalid && !*valid) *first_invalid = *reinterpret_cast<int32_t *>(r.stage + 32);
    });
}

int ompl_amd_check_motion_last_valid(ompl_amd_env e, const double *a, const double *b, double lvs, unsigned factor,
                                     int *valid, double *last_t)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(a && b && valid && last_t, OMPL_AMD_ERR_ARG, "null pointer");
        OA_REQUIRE(lvs > 0.0 && factor >= 1, OMPL_AMD_ERR_ARG, "longest valid segment must be > 0 and factor >= 1");
        ThreadResources &r = thread_resources();
        // endpoints staged through the pinned slot: [a(7), b(7), last_t] doubles
        double *pd = reinterpret_cast<double *>(r.pinned + 16);
        for (int j = 0; j < kDof; ++j) {
            pd[j] = a[j];
            pd[kDof + j] = b[j];
        }
        pd[2 * kDof] = *last_t;
        // the kernel reads dof-major [7][1] arrays: identical to a flat vector
        double *dev_pd = reinterpret_cast<double *>(r.pinned_dev + 16);
        uint8_t *dev_out = reinterpret_cast<uint8_t *>(r.pinned_dev);
        MotionArgs A{};
        A.a = dev_pd;
        A.b = dev_pd + kDof;
        A.n = 1;
        A.lvs = lvs;
        A.factor = factor;
        A.out = dev_out;
        {
            std::unique_lock<std::mutex> lk; // held until the launches are enqueued
            Workspace &w = workspace(r.stream, 1, lk);
            launch_grid_last_valid(env.grid, A, dev_pd + 2 * kDof, grid_scratch(w), r.stream);
        }
        OA_HIP(hipStreamSynchronize(r.stream));
        *valid = reinterpret_cast<uint8_t *>(r.pinned)[0];
        *last_t = pd[2 * kDof];
    });
}

} // extern "C"

extern "C" int ompl_amd_env_set_tuning(ompl_amd_env e, const ompl_amd_tuning *t)
{
    return guarded([&] {
        env_of(e);
        if (t) check_tuning(tuning_from_c(*t));
        std::lock_guard<std::mutex> lk(e->tuning_mutex);
        e->has_tuning = t != nullptr;
        if (t) e->tuning = tuning_from_c(*t);
    });
}

extern "C" int ompl_amd_env_get_tuning(ompl_amd_env e, ompl_amd_tuning *t, int *own)
{
    return guarded([&] {
        env_of(e);
        OA_REQUIRE(t, OMPL_AMD_ERR_ARG, "null tuning");
        bool has = false;
        {
            std::lock_guard<std::mutex> lk(e->tuning_mutex);
            has = e->has_tuning;
        }
        *t = tuning_to_c(tuning_for(*e));
        if (own) *own = has ? 1 : 0;
    });
}

extern "C" int ompl_amd_autotune_motions(ompl_amd_env e, const double *a, const double *b, int64_t n, double lvs,
                                         unsigned factor, int reps, ompl_amd_tuning *best, double *best_us)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n > 0 && a && b && reps >= 1, OMPL_AMD_ERR_ARG, "bad autotune arguments");
        ThreadResources &r = thread_resources();
        hipStream_t s = r.stream;
        uint8_t *out = nullptr;
        OA_HIP(device_malloc(&out, (size_t)n));
        hipEvent_t e0, e1;
        OA_HIP(hipEventCreate(&e0));
        OA_HIP(hipEventCreate(&e1));
        // every shape runs the same kernels: one is timed and installed
        const Tuning win{8, 2, 256, 8, 1, 256, 8, 3, 0};
        for (int w = 0; w < 2; ++w) check_motions_tuned(win, env, a, b, n, lvs, factor, out, nullptr, s);
        OA_HIP(hipEventRecord(e0, s));
        for (int i = 0; i < reps; ++i) check_motions_tuned(win, env, a, b, n, lvs, factor, out, nullptr, s);
        OA_HIP(hipEventRecord(e1, s));
        OA_HIP(hipEventSynchronize(e1));
        float win_ms = 0.0f;
        OA_HIP(hipEventElapsedTime(&win_ms, e0, e1));
        OA_HIP(hipEventDestroy(e0));
        OA_HIP(hipEventDestroy(e1));
        OA_HIP(hipFree(out));
        set_tuning(win);
        if (best) {
            *best = tuning_to_c(win);
        }
        if (best_us) *best_us = 1e3 * (double)win_ms / reps;
    });
}

namespace {

// Device buffers and events of one stream-pipeline autotune, released on
// every exit.
struct PipelineScratch {
    uint8_t *out = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    std::vector<hipEvent_t> join;
    ~PipelineScratch()
    {
        if (out) (void)hipFree(out);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        for (hipEvent_t e : join) (void)hipEventDestroy(e);
    }
};

} // namespace

extern "C" int ompl_amd_autotune_motions_streams(ompl_amd_env e, const double *a, const double *b, int64_t n,
                                                 double lvs, unsigned factor, void *const *streams, int n_streams,
                                                 int steps, ompl_amd_tuning *best, double *best_us)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(n > 0 && a && b && steps >= 1, OMPL_AMD_ERR_ARG, "bad autotune arguments");
        OA_REQUIRE(streams && n_streams >= 1 && n_streams <= 16, OMPL_AMD_ERR_ARG, "1 to 16 streams");
        {
            std::lock_guard<std::mutex> lk(e->tuning_mutex);
            OA_REQUIRE(!e->has_tuning, OMPL_AMD_ERR_ARG,
                       "the environment has its own launch shapes, which take the place of the library's");
        }
        std::vector<hipStream_t> st((size_t)n_streams);
        for (int j = 0; j < n_streams; ++j) st[(size_t)j] = resolve_stream(streams[j]);
        PipelineScratch S;
        OA_HIP(device_malloc(&S.out, (size_t)n * (size_t)n_streams));
        OA_HIP(hipEventCreate(&S.e0));
        OA_HIP(hipEventCreate(&S.e1));
        for (int j = 0; j < n_streams; ++j) {
            hipEvent_t ev = nullptr;
            OA_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
            S.join.push_back(ev);
        }
        // k batches round-robin on the streams, between events on the first,
        // which waits for the others at the end; microseconds per batch
        auto per_batch = [&](const Tuning &t, int k) {
            for (int i = 0; i < 2 * n_streams; ++i) { // warm: workspaces sized, kernels loaded
                const int j = i % n_streams;
                check_motions_tuned(t, env, a, b, n, lvs, factor, S.out + (size_t)j * (size_t)n, nullptr,
                                    st[(size_t)j]);
            }
            for (hipStream_t s : st) OA_HIP(hipStreamSynchronize(s));
            OA_HIP(hipEventRecord(S.e0, st[0]));
            for (int j = 1; j < n_streams; ++j) OA_HIP(hipStreamWaitEvent(st[(size_t)j], S.e0, 0));
            for (int i = 0; i < k; ++i) {
                const int j = i % n_streams;
                check_motions_tuned(t, env, a, b, n, lvs, factor, S.out + (size_t)j * (size_t)n, nullptr,
                                    st[(size_t)j]);
            }
            for (int j = 1; j < n_streams; ++j) {
                OA_HIP(hipEventRecord(S.join[(size_t)j], st[(size_t)j]));
                OA_HIP(hipStreamWaitEvent(st[0], S.join[(size_t)j], 0));
            }
            OA_HIP(hipEventRecord(S.e1, st[0]));
            OA_HIP(hipEventSynchronize(S.e1));
            float ms = 0.0f;
            OA_HIP(hipEventElapsedTime(&ms, S.e0, S.e1));
            return 1e3 * (double)ms / k;
        };
        // every shape runs the same kernels: one of those a tuning for streams
        // names (eight lanes a state throughout) is timed and installed
        Tuning win = get_tuning();
        win.validity_lanes_per_state = win.motion_lanes_per_state = win.motion_waves_per_cu = 8;
        win.validity_obstacle_parts = 4;
        win.motion_obstacle_parts = 8;
        win.motion_strategy = 3;
        win.validity_shared_fk = 0;
        const double win_us = per_batch(win, steps);
        set_tuning(win);
        if (best) *best = tuning_to_c(win);
        if (best_us) *best_us = win_us;
    });
}

extern "C" {

int ompl_amd_motion_graph_create(ompl_amd_env e, const double *a, const double *b, int64_t n, double lvs,
                                 unsigned factor, uint8_t *out, int32_t *checked, ompl_amd_motion_graph *graph)
{
    return ompl_amd_motion_graph_create_group(e, 1, &a, &b, &n, lvs, factor, &out, checked ? &checked : nullptr,
                                              graph);
}

int ompl_amd_motion_graph_create_group(ompl_amd_env e, int n_batches, const double *const *a, const double *const *b,
                                       const int64_t *n, double lvs, unsigned factor, uint8_t *const *out,
                                       int32_t *const *checked, ompl_amd_motion_graph *graph)
{
    return guarded([&] {
        const Env &env = env_of(e);
        OA_REQUIRE(graph, OMPL_AMD_ERR_ARG, "null graph handle");
        OA_REQUIRE(n_batches >= 1 && n_batches <= 16, OMPL_AMD_ERR_ARG, "a captured group holds 1 to 16 batches");
        OA_REQUIRE(a && b && n && out, OMPL_AMD_ERR_ARG, "null batch arrays");
        for (int i = 0; i < n_batches; ++i) {
            OA_REQUIRE(n[i] >= 1, OMPL_AMD_ERR_ARG, "a captured batch needs at least one edge");
            OA_REQUIRE(a[i] && b[i] && out[i], OMPL_AMD_ERR_ARG, "null pointer in batch %d", i);
        }
        auto *g = new ompl_amd_motion_graph_s();
        for (int i = 0; i < n_batches; ++i) g->ws.push_back(std::make_unique<Workspace>());
        try {
            record_group(g, env, tuning_for(*e), n_batches, a, b, n, lvs, factor, out, checked);
        } catch (...) {
            delete g;
            throw;
        }
        *graph = g;
    });
}

int ompl_amd_motion_graph_launch(ompl_amd_motion_graph graph, void *stream)
{
    return guarded([&] {
        OA_REQUIRE(graph && graph->exec[0] && graph->exec[1], OMPL_AMD_ERR_ARG, "null graph");
        OA_HIP(hipGraphLaunch(graph->exec[graph->next], resolve_stream(stream)));
        graph->next ^= 1;
    });
}

int ompl_amd_motion_graph_destroy(ompl_amd_motion_graph graph)
{
    return guarded([&] {
        if (graph) OA_HIP(hipDeviceSynchronize());
        delete graph;
    });
}

} // extern "C"
