// Host checks of the library's device buffers (vv_ctx.hpp, vv_api.cpp,
// vv_batch.cpp) against a device memory of a set size: hipMalloc and hipFree
// are counted here instead of calling the runtime, and the kernels' launchers
// check that what they are given lies in a live buffer.  Prints one line per
// failed check; the exit code is their number.
#include "vv_api.cpp"
#include "vv_batch.cpp"

#include <iterator>
#include <map>

using namespace vv_host;

static size_t g_limit = 0, g_held = 0;
static int g_mallocs = 0, g_frees = 0, g_failed = 0;
static std::map<void*, size_t> g_blocks;
static int g_graph, g_pair_passes = 0, g_frames = 0, g_pair_frames = 0;
static char* g_next = (char*)(1ull << 40);
static hipStreamCaptureStatus g_capture = hipStreamCaptureStatusNone;
static hipError_t g_query = hipSuccess, g_last = hipSuccess;

extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    if (g_capture != hipStreamCaptureStatusNone) return g_last = hipErrorStreamCaptureUnsupported;
    if (g_held + n > g_limit) return g_last = hipErrorOutOfMemory;
    ++g_mallocs;
    *p = g_next;  // addresses alone: nothing is read or written
    g_next += (n + 4095) / 4096 * 4096 + 4096;
    g_blocks[*p] = n;
    g_held += n;
    return hipSuccess;
}

extern "C" hipError_t hipFree(void* p)
{
    ++g_frees;
    g_held -= g_blocks.at(p);
    g_blocks.erase(p);
    return hipSuccess;
}

extern "C" hipError_t hipGetLastError(void)
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}

extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
    *s = g_capture;
    return g_query == hipSuccess ? hipSuccess : (g_last = g_query);
}

#define CHECK(x)                                             \
    do {                                                     \
        if (!(x)) {                                          \
            std::printf("line %d: %s\n", __LINE__, #x);      \
            ++g_failed;                                      \
        }                                                    \
    } while (0)

extern "C" {
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)&g_graph, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return *e = (hipGraphExec_t)&g_graph, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
}

namespace vv_host {
vv_status ensure_illum_luts(vv_ctx*) { return VV_OK; }
}  // namespace vv_host

extern "C" void vv_default_line_material(vv_line_material*) {}

// the kernels: whether each buffer that is given holds what they touch
static bool live(const void* p, size_t n)
{
    const auto b = g_blocks.upper_bound((char*)p);
    if (b == g_blocks.begin()) return false;
    const auto& [base, size] = *std::prev(b);
    return (char*)p + n <= (char*)base + size;
}

static size_t field_size(const int* d, int type) { return field_texel_bytes(type) * (size_t)clamp_elems(d); }

static hipError_t check_lic(const LicLaunch& L)
{
    CHECK(live(L.field.p, field_size(L.field.n, L.field_type)));
    CHECK(live(L.noise.p, L.nc * (size_t)repeat_elems(L.noise.n)));
    if (L.gate) CHECK(live(L.scalar.p, (size_t)clamp_elems(L.scalar.n)));
    return hipSuccess;
}

static hipError_t check_frame(const RenderLaunch& R)
{
    CHECK(live(R.field.p, field_size(R.field.n, R.field_type)));
    if (R.lic.p) CHECK(live(R.lic.p, sizeof(float) * R.lc * (size_t)repeat_elems(R.lic.n)));
    ++g_frames;
    g_pair_frames += R.pair != nullptr;
    if (R.pair) CHECK(live(R.pair, pair_bytes(R.lc, R.lic.n)));
    if (R.sigma.p) CHECK(live(R.sigma.p, sizeof(float) * (size_t)clamp_elems(R.sigma.n)));
    CHECK(live(R.image, (size_t)4 * R.view.width * R.view.height));
    return hipSuccess;
}

namespace vv {
hipError_t noalloc_scratch(int, void** p) { return *p = nullptr, hipSuccess; }
hipError_t launch_fill_u32(uint32_t*, uint32_t, long long, hipStream_t) { return hipSuccess; }
hipError_t launch_fill_i64(long long*, long long, long long, hipStream_t) { return hipSuccess; }
hipError_t launch_field_maxlen(const float*, const float*, float, long long, uint32_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_field_encode(const float*, const float*, float, const int d[3], const uint32_t*, void* f, int type,
                               hipStream_t, int)
{
    CHECK(live(f, field_size(d, type)));
    return hipSuccess;
}
hipError_t launch_noise_gen(uint64_t, int, uint64_t, const int*, uint8_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_noise_tex(const uint8_t*, const uint8_t*, const int d[3], void* tex, int nc, hipStream_t)
{
    CHECK(live(tex, nc * (size_t)repeat_elems(d)));
    return hipSuccess;
}
hipError_t launch_noise_grad_tex(const uint8_t*, const int d[3], const float*, void* tex, hipStream_t)
{
    CHECK(live(tex, 4 * (size_t)repeat_elems(d)));
    return hipSuccess;
}
hipError_t launch_pack_lic_field(const void*, int type, const uint8_t*, const int d[3], void* out, hipStream_t)
{
    CHECK(live(out, field_size(d, type)));
    return hipSuccess;
}
hipError_t launch_pack_lic_field4(const void*, const void*, const int d[3], void* out, hipStream_t)
{
    CHECK(live(out, field_size(d, 0)));
    return hipSuccess;
}
hipError_t launch_pad_clamp_u8(const uint8_t*, const int*, uint8_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_pad_clamp_f32(const float*, const int*, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_pad_repeat_f32(const float*, int, const int*, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_sample_pair(const void* f, int type, int, const float* lic, const int d[3], float* pair, hipStream_t)
{
    ++g_pair_passes;
    CHECK(live(f, field_size(d, type)));
    CHECK(live(lic, sizeof(float) * (size_t)repeat_elems(d)));
    CHECK(live(pair, pair_bytes(1, d)));
    return hipSuccess;
}
hipError_t launch_sample_plane(const void*, int, int, const int*, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_lic(const LicLaunch& L, hipStream_t)
{
    CHECK(live(L.out.p, sizeof(float) * L.nc * (size_t)repeat_elems(L.out.n)));
    return check_lic(L);
}
hipError_t launch_render(const RenderLaunch& R, hipStream_t) { return check_frame(R); }
hipError_t launch_render_rg(const RenderLaunch& R, int, hipStream_t) { return check_frame(R); }
hipError_t launch_render_fused(const RenderLaunch& R, const LicLaunch& L, hipStream_t) { return (void)check_lic(L), check_frame(R); }
hipError_t launch_render_group(const RenderLaunch& R, const LicLaunch& L, const SliceSetup&, int, int, hipStream_t)
{
    return (void)check_lic(L), check_frame(R);
}
size_t lic_args_size() { return 64; }
hipError_t lic_args_fill(const LicLaunch& L, void* args, int* ntiles)
{
    std::memset(args, 0, 64);
    return *ntiles = 1, check_lic(L);
}
hipError_t launch_lic_batch(const LicBatchLaunch&, hipStream_t) { return hipSuccess; }
hipError_t launch_render_batch(const RenderBatchLaunch&, hipStream_t) { return hipSuccess; }
hipError_t launch_stamp(unsigned long long*, hipStream_t) { return hipSuccess; }
int render_batch_blocks_per_cu(int, int, int, int, int) { return 1; }
hipError_t launch_adjoint_forward(const AdjointLaunch& A, hipStream_t) { return check_frame(A.r); }
}  // namespace vv

static const int kDims[3] = {30, 31, 32};

static size_t lic_size(int channels) { return sizeof(float) * channels * (size_t)repeat_elems(kDims); }

// a context whose memory holds `room` bytes beyond its scalar LIC volume of kDims
struct Scene {
    vv_ctx c;
    explicit Scene(size_t room, int channels = 1)
    {
        g_capture = hipStreamCaptureStatusNone;
        g_query = g_last = hipSuccess;
        g_limit = 1ull << 40;
        CHECK(c.field.ensure(field_size(kDims, c.storage)) == hipSuccess);
        g_limit = g_held + lic_size(channels) + room;
        g_mallocs = g_frees = 0;
        c.has_field = true;
        for (int a = 0; a < 3; ++a) c.fdims[a] = kDims[a];
        c.lch = channels;
    }
    ~Scene()
    {
        for (DevBuf* b : c.required()) b->release();
        for (DevBuf* b : *c.optional) b->release();
    }
    hipError_t lic(int channels = 1)
    {
        const hipError_t e = lic_buffer(&c, channels, kDims);
        if (e != hipSuccess) return e;
        c.has_lic = true;
        c.lch = channels;
        for (int a = 0; a < 3; ++a) c.ldims[a] = kDims[a];
        return pair_buffer(&c);
    }
    // whether a frame large enough to be worth it samples through the sample volume
    bool frame()
    {
        RenderLaunch R;
        std::memset(&R, 0, sizeof(R));
        R.view.width = R.view.height = 1024;
        R.step = 1.0f / 256.0f;
        for (int a = 0; a < 3; ++a) R.view.tex_max[a] = 1.0f;
        R.tf_ch = 2;
        CHECK(ensure_pair(&c, R) == VV_OK);
        return R.pair != nullptr;
    }
};

static size_t free_memory(size_t n) { return g_limit = g_held + n; }

// the library's entry points on a context with a field, noise and LIC volume of kDims
struct Api {
    vv_ctx* c = nullptr;
    float* data = (float*)(1ull << 20);  // inputs and images: device pointers
    explicit Api(int with_gradients = 0)
    {
        g_capture = hipStreamCaptureStatusNone;
        g_limit = 1ull << 40;
        CHECK(vv_create(&c, 0) == VV_OK);
        CHECK(vv_upload_field(c, data, nullptr, 0.0f, kDims, nullptr, VV_STORE_FP32, 1) == VV_OK);
        CHECK(vv_generate_noise(c, 1, VV_NOISE_UNIFORM, 0.0, kDims, with_gradients) == VV_OK);
        CHECK(vv_compute_lic(c) == VV_OK);
    }
    ~Api() { CHECK(vv_destroy(c) == VV_OK && g_blocks.empty()); }
};

static void lic_buffer_stays()
{
    // room for both: the second LIC volume allocates nothing
    Scene a(1u << 20);
    CHECK(a.lic() == hipSuccess && a.frame());
    const void* p = a.c.lic.p;
    const int m = g_mallocs;
    CHECK(a.lic() == hipSuccess && a.c.lic.p == p && g_mallocs == m && g_frees == 0);
    CHECK(a.frame());

    // room for the LIC volume alone: it is not moved for the other's sake,
    // nor once there is memory again
    Scene b(0);
    CHECK(b.lic() == hipSuccess && !b.frame());
    p = b.c.lic.p;
    for (int k = 0; k < 2; ++k) {
        const int n = g_mallocs, f = g_frees;
        CHECK(b.lic() == hipSuccess && b.c.lic.p == p && g_mallocs == n && g_frees == f);
        CHECK(!b.frame() && hipGetLastError() == hipSuccess);
        g_limit += 1u << 20;
    }
}

static void capture_allocates_nothing()
{
    Scene a(0);
    CHECK(a.lic() == hipSuccess);
    const void* p = a.c.lic.p;
    g_capture = hipStreamCaptureStatusActive;
    const int n = g_mallocs, f = g_frees;
    CHECK(a.lic() == hipSuccess && a.c.lic.p == p && g_mallocs == n && g_frees == f);
    CHECK(!a.frame() && hipGetLastError() == hipSuccess);
    g_capture = hipStreamCaptureStatusNone;
    CHECK(a.lic() == hipSuccess && a.c.lic.p == p && g_mallocs == n && g_frees == f);

    // no captured frame reads the sample volume; a captured LIC volume changes
    // unseen, so no later frame does either
    Scene b(1u << 20);
    CHECK(b.lic() == hipSuccess && b.frame());
    g_capture = hipStreamCaptureStatusActive;
    CHECK(!b.frame());
    g_capture = hipStreamCaptureStatusNone;
    CHECK(b.frame());
    g_capture = hipStreamCaptureStatusActive;
    CHECK(b.lic() == hipSuccess && !b.frame());
    g_capture = hipStreamCaptureStatusNone;
    CHECK(!b.frame());

    // until the caller says that none is replayed any more
    int on = -1;
    CHECK(vv_get_tuning(&b.c, "render.sample_volume", &on) == VV_OK && on == 0);
    CHECK(vv_set_tuning(&b.c, "render.sample_volume", 1) == VV_OK && !b.c.pair.p && !b.frame());
    CHECK(b.lic() == hipSuccess && b.frame());
}

// "render.sample_volume" 0: no memory for it
static void switched_off()
{
    Scene a(1u << 20);
    CHECK(vv_set_tuning(&a.c, "render.sample_volume", 2) == VV_EINVAL);
    CHECK(vv_set_tuning(&a.c, "render.sample_volume", 0) == VV_OK);
    CHECK(a.lic() == hipSuccess && !a.frame() && !a.c.pair.p);
    CHECK(vv_set_tuning(&a.c, "render.sample_volume", 1) == VV_OK && a.lic() == hipSuccess && a.frame());
    CHECK(vv_set_tuning(&a.c, "render.sample_volume", 0) == VV_OK && !a.c.pair.p && !a.frame());
}

// a failed query costs the call its sample volume, not the context, and leaves
// no error behind
static void failed_capture_query()
{
    for (int channels : {1, 4}) {
        Scene a(1u << 20, channels);
        CHECK(a.lic(channels) == hipSuccess && a.frame());
        g_query = hipErrorUnknown;
        CHECK(!a.frame() && hipGetLastError() == hipSuccess);
        g_query = hipSuccess;
        CHECK(a.frame());
    }
    Api b(1);
    g_query = hipErrorUnknown;
    CHECK(vv_compute_lic(b.c) == VV_OK && hipGetLastError() == hipSuccess);
    g_query = hipSuccess;
}

static void refused_lic_volume_is_gone()
{
    Scene a(0);
    CHECK(a.lic() == hipSuccess && a.c.has_lic);
    CHECK(a.lic(4) == hipErrorOutOfMemory);
    CHECK(!a.c.has_lic);
}

// what does not fit beside the sample volume takes its memory, for good
static void sample_volume_gives_way()
{
    Scene a(1u << 20);
    CHECK(a.lic() == hipSuccess && a.frame());
    const void* p = a.c.lic.p;
    CHECK(a.c.adj_ckpt.ensure(900u << 10) == hipSuccess && hipGetLastError() == hipSuccess);
    CHECK(!a.frame());
    const int n = g_mallocs, f = g_frees;
    CHECK(a.lic() == hipSuccess && a.c.lic.p == p && !a.frame() && g_mallocs == n && g_frees == f);
    CHECK(a.c.image.ensure(900u << 10) == hipErrorOutOfMemory);

    // a larger LIC volume does too
    Scene b(1u << 20);
    CHECK(b.lic() == hipSuccess && b.frame());
    g_limit = g_held - b.c.lic.bytes - b.c.pair.bytes + lic_size(4);
    CHECK(b.lic(4) == hipSuccess && !b.frame());
}

// no kernel runs on a volume whose buffer could not grow
static void refused_volumes_are_gone()
{
    const int big[3] = {40, 40, 40};
    for (int kind = 0; kind < 3; ++kind) {
        Api a;
        vv_ctx* c = a.c;
        CHECK(vv_upload_scalar(c, (const uint8_t*)a.data, kDims, 1) == VV_OK);
        c->params.gate_enable = 1;
        CHECK(vv_compute_lic(c) == VV_OK);
        CHECK(c->stage.ensure((size_t)nvox(big)) == hipSuccess);
        c->pair.release();
        free_memory(0);
        if (kind == 0)
            CHECK(vv_upload_field(c, a.data, nullptr, 0.0f, big, nullptr, VV_STORE_FP32, 1) == VV_ENOMEM);
        else if (kind == 1)
            CHECK(vv_generate_noise(c, 1, VV_NOISE_UNIFORM, 0.0, big, 0) == VV_ENOMEM);
        else
            CHECK(vv_upload_scalar(c, (const uint8_t*)a.data, big, 1) == VV_ENOMEM);
        CHECK(vv_compute_lic(c) == VV_ESTATE);
        // the refusal is reported once, and the next volume is taken
        CHECK(hipGetLastError() == hipSuccess);
        free_memory(1u << 22);
        CHECK(vv_upload_field(c, a.data, nullptr, 0.0f, kDims, nullptr, VV_STORE_FP32, 1) == VV_OK);
        CHECK(vv_generate_noise(c, 1, VV_NOISE_UNIFORM, 0.0, kDims, 0) == VV_OK);
        CHECK(vv_upload_scalar(c, (const uint8_t*)a.data, kDims, 1) == VV_OK);
        CHECK(vv_compute_lic(c) == VV_OK);
    }
}

// RGBA noise on an FP32 field: the LIC copy gives way too, also in the middle
// of the call that would have read it
static void rgba_copy_gives_way()
{
    Api a(1);
    vv_ctx* c = a.c;
    vv_camera cam;
    CHECK(vv_default_camera(&cam, 64, 48, nullptr) == VV_OK);
    std::vector<float> image(4 * 64 * 48);
    std::vector<uint8_t> bytes(4 * 64 * 48);
    for (int call = 0; call < 3; ++call) {
        CHECK(vv_upload_noise(c, (const uint8_t*)a.data, kDims, 1, nullptr, 1) == VV_OK);
        g_limit = 1ull << 40;
        for (DevBuf* b : *c->optional) b->denied = 0;
        CHECK(vv_compute_lic(c) == VV_OK && vv_render_fused(c, &cam, image.data(), 0, nullptr) == VV_OK);
        (call == 0 ? c->lic : c->image).release();
        c->pair.release();
        free_memory(0);
        if (call == 0)
            CHECK(vv_compute_lic(c) == VV_OK);
        else if (call == 1)
            CHECK(vv_render_fused(c, &cam, image.data(), 0, nullptr) == VV_OK);
        else
            CHECK(vv_render_slices_blend(c, &cam, bytes.data(), 0, nullptr) == VV_OK);
        CHECK(vv_compute_lic(c) == VV_OK);
    }
}

// a batch step's sample volume comes with the views that are worth it, serves
// run and autotune alike, and gives way to another step
static void batch_sample_volumes()
{
    Api a;
    vv_batch* b = nullptr;
    CHECK(vv_batch_create(a.c, &b) == VV_OK);
    auto add_step = [&] {
        return vv_batch_add_timestep(b, a.data, kDims, nullptr, VV_STORE_FP32, 1, VV_NOISE_UNIFORM, 0.0, 1);
    };
    void* image = nullptr;
    CHECK(hipMalloc(&image, 16 << 20) == hipSuccess);
    auto add_view = [&](int step, int width) {
        vv_camera cam;
        CHECK(vv_default_camera(&cam, width, width, nullptr) == VV_OK);
        return vv_batch_add_view(b, step, &cam, (float*)image);
    };
    // every view that a run shows reads live memory; their number through a sample volume
    auto run = [&] {
        CHECK(vv_batch_run(b) == VV_OK);
        const int frames = g_pair_frames;
        for (const RenderLaunch& R : b->host_views) CHECK(check_frame(R) == hipSuccess);
        return g_pair_frames - frames;
    };
    auto autotune = [&] {
        const int frames = g_pair_frames;
        CHECK(vv_batch_autotune(b) == VV_OK);
        return g_pair_frames - frames;
    };
    CHECK(add_step() == VV_OK && add_view(0, 8) == VV_OK);
    CHECK(!b->steps[0]->pair.p && run() == 0 && autotune() == 0);
    CHECK(add_view(0, 512) == VV_OK);
    CHECK(b->steps[0]->pair.p && run() == 2 && autotune() > 0);
    int passes = g_pair_passes;
    CHECK(run() == 2 && g_pair_passes == passes + 1);  // autotune drops the graph

    // the line modes read both volumes
    a.c->params.illum_mode = VV_ILLUM_MALLO;
    CHECK(run() == 0);
    a.c->params.illum_mode = VV_ILLUM_LIC;
    CHECK(run() == 2);

    // few samples: neither is worth the pass
    a.c->params.step_size_vol = 10.0f;
    CHECK(run() == 0 && autotune() == 0);
    a.c->params.step_size_vol = 1.0f / 128.0f;
    CHECK(run() == 2 && autotune() > 0);

    // a step that does not fit beside it, with the context's own still there
    const size_t step = 2 * 16 * (size_t)clamp_elems(kDims) + 5 * (size_t)repeat_elems(kDims);
    a.c->pair.denied = 0;
    CHECK(vv_compute_lic(a.c) == VV_OK && a.c->pair.p);
    free_memory(step - (1u << 16));
    CHECK(add_step() == VV_OK && add_view(1, 512) == VV_OK);
    CHECK(!b->steps[0]->pair.p && !a.c->pair.p && b->steps[1]->pair.p);
    free_memory(1u << 30);
    CHECK(run() == 1);

    CHECK(vv_batch_destroy(b) == VV_OK);
    CHECK(hipFree(image) == hipSuccess);
    CHECK(vv_compute_lic(a.c) == VV_OK && a.c->optional->size() == 2);
}

// lanes per ray: the measured best of each size, or what is within 5 % of it
static void lanes_per_ray()
{
    Api a;
    RenderLaunch R;
    std::memset(&R, 0, sizeof(R));
    auto view = [&](int n, int width, int illum, int lc, bool pair) {
        R.view.width = R.view.height = width;
        R.step = 1.0f / (float)n;
        R.illum = illum;
        R.lc = lc;
        R.pair = pair ? (const float*)&R : nullptr;
    };
    const struct { int n, width, illum, lc, pair, lo, hi; } frames[] = {
        {128, 256, 0, 1, 1, 8, 8},   {256, 256, 0, 1, 1, 16, 16}, {256, 1024, 0, 1, 1, 2, 4}, {128, 1448, 0, 1, 1, 1, 1},
        {128, 256, 2, 1, 0, 16, 16}, {128, 512, 2, 1, 0, 4, 4},   {128, 768, 3, 1, 0, 4, 4},  {128, 1448, 3, 1, 0, 2, 4},
        {256, 256, 3, 1, 0, 16, 16}, {256, 512, 3, 1, 0, 8, 8},   {256, 1024, 2, 1, 0, 4, 4}, {256, 1448, 2, 1, 0, 2, 4}};
    for (const auto& f : frames) {
        view(f.n, f.width, f.illum, f.lc, f.pair);
        const int G = volume_group_for(a.c, R);
        CHECK(G >= f.lo && G <= f.hi);
    }
    const struct { int n, width, illum, lc, pair, lo, hi; } records[] = {
        {128, 512, 0, 1, 1, 2, 4},  {128, 768, 0, 1, 1, 1, 2},  {128, 1024, 0, 1, 1, 1, 1}, {256, 640, 0, 1, 1, 4, 4},
        {256, 768, 0, 1, 1, 2, 2},  {256, 1024, 0, 1, 1, 2, 2}, {256, 1448, 0, 1, 1, 1, 1}, {512, 768, 0, 1, 1, 4, 4},
        {512, 1448, 0, 1, 1, 2, 2}, {512, 2048, 0, 1, 1, 1, 2}, {128, 768, 1, 4, 1, 2, 2},  {128, 1448, 1, 4, 1, 1, 2},
        {256, 768, 1, 4, 1, 4, 4},  {256, 1448, 1, 4, 1, 2, 2}, {256, 2048, 1, 4, 1, 1, 2}, {128, 1024, 0, 1, 0, 2, 2},
        {128, 2048, 0, 1, 0, 1, 1}, {256, 768, 0, 1, 0, 4, 4},  {256, 1024, 0, 1, 0, 4, 4}, {256, 1448, 1, 4, 0, 2, 2},
        {512, 1024, 0, 1, 0, 4, 4}, {128, 640, 2, 1, 0, 4, 4},  {128, 1448, 3, 1, 0, 2, 2}, {256, 768, 3, 1, 0, 4, 4},
        {256, 1024, 2, 1, 0, 4, 4}, {256, 1448, 2, 1, 0, 2, 4}, {512, 1024, 2, 1, 0, 4, 4}, {512, 1448, 3, 1, 0, 4, 4}};
    for (const auto& f : records) {
        view(f.n, f.width, f.illum, f.lc, f.pair);
        const int G = record_group_for(a.c, R, 4);
        CHECK(G >= f.lo && G <= f.hi);
        CHECK(record_group_for(a.c, R, 2) <= 2);
        a.c->volume_group = 1;
        CHECK(record_group_for(a.c, R, 1) == 1 && volume_group_for(a.c, R) == 1);
        a.c->volume_group = 0;
    }
}

int main()
{
    lanes_per_ray();
    batch_sample_volumes();
    rgba_copy_gives_way();
    refused_volumes_are_gone();
    sample_volume_gives_way();
    lic_buffer_stays();
    capture_allocates_nothing();
    switched_off();
    failed_capture_query();
    refused_lic_volume_is_gone();
    return g_failed;
}
