// Host checks of the context's buffers (vv_ctx.hpp) against a device memory of
// a set size: hipMalloc and hipFree are counted here instead of calling the
// runtime.  Prints one line per failed check; the exit code is their number.
#include "vv_ctx.hpp"

#include <cstdlib>
#include <map>

using namespace vv_host;

static size_t g_limit = 0, g_held = 0;
static int g_mallocs = 0, g_frees = 0, g_failed = 0;
static std::map<void*, size_t> g_blocks;
static hipStreamCaptureStatus g_capture = hipStreamCaptureStatusNone;
static hipError_t g_query = hipSuccess, g_last = hipSuccess;

extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    if (g_capture != hipStreamCaptureStatusNone) return g_last = hipErrorStreamCaptureUnsupported;
    if (g_held + n > g_limit) return g_last = hipErrorOutOfMemory;
    ++g_mallocs;
    *p = std::malloc(1);
    g_blocks[*p] = n;
    g_held += n;
    return hipSuccess;
}

extern "C" hipError_t hipFree(void* p)
{
    ++g_frees;
    g_held -= g_blocks.at(p);
    g_blocks.erase(p);
    std::free(p);
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
    return g_last = g_query;
}

extern "C" const char* hipGetErrorString(hipError_t) { return "error"; }

namespace vv {
hipError_t launch_sample_pair(const void*, int, int, const float*, const int*, float*, hipStream_t) { return hipSuccess; }
hipError_t launch_sample_plane(const void*, int, int, const int*, float*, hipStream_t) { return hipSuccess; }
}  // namespace vv

#define CHECK(x)                                             \
    do {                                                     \
        if (!(x)) {                                          \
            std::printf("line %d: %s\n", __LINE__, #x);      \
            ++g_failed;                                      \
        }                                                    \
    } while (0)

static const int kDims[3] = {30, 31, 32};

static size_t lic_size(int channels) { return sizeof(float) * channels * (size_t)repeat_elems(kDims); }

// a context whose memory holds `room` bytes beyond its scalar LIC volume of kDims
struct Scene {
    vv_ctx c;
    explicit Scene(size_t room, int channels = 1)
    {
        g_limit = lic_size(channels) + 256 + room;
        g_held = 0;
        g_mallocs = g_frees = 0;
        g_capture = hipStreamCaptureStatusNone;
        g_query = g_last = hipSuccess;
        g_blocks.clear();
        c.has_field = true;
        for (int a = 0; a < 3; ++a) c.fdims[a] = kDims[a];
        c.lch = channels;
    }
    hipError_t lic(int channels = 1)
    {
        const hipError_t e = lic_buffer(&c, channels, kDims);
        if (e == hipSuccess) {
            c.has_lic = true;
            c.lch = channels;
            for (int a = 0; a < 3; ++a) c.ldims[a] = kDims[a];
        }
        return e;
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

    // a graph replays without the context's flags: no sample volume after it
    Scene b(1u << 20);
    CHECK(b.lic() == hipSuccess && b.frame());
    g_capture = hipStreamCaptureStatusActive;
    CHECK(b.lic() == hipSuccess && !b.frame());
    g_capture = hipStreamCaptureStatusNone;
    CHECK(!b.frame());
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
    g_limit = lic_size(4) + 256;
    CHECK(b.lic(4) == hipSuccess && !b.frame());
}

int main()
{
    sample_volume_gives_way();
    lic_buffer_stays();
    capture_allocates_nothing();
    refused_lic_volume_is_gone();
    return g_failed;
}
