/* Host side of the dense calls (csrc/qmsg_api.cpp) against a small stand-in for the HIP runtime and
 * the launchers: which buffer each launch is given, and whether it outlives the graph that holds it.
 * The stand-in keeps the runtime's rules the calls depend on: a failed call's error stays the
 * thread's last error until hipGetLastError reads it, launchers return that error, and a
 * synchronisation or free on a capturing stream fails.
 *
 *     dense_call_host SCENARIO        exit 0, or a line on stderr and exit 1 */
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <vector>

#include "../include/qmsg.h"
#include "../large_model_amd/csrc/qmsg_internal.h"

namespace {

std::set<void *> live;
size_t malloc_limit = ~(size_t)0;      /* larger allocations fail */
int mallocs = 0;
hipError_t last = hipSuccess;
bool capturing = false;

hipError_t ret(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}

struct Launch {
    bool exact, records;
    int T, type;
    uint8_t *xqk;
};
std::vector<Launch> launches;

}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    mallocs++;
    if (n > malloc_limit) return ret(hipErrorOutOfMemory);
    *p = malloc(64);                   /* addresses only */
    live.insert(*p);
    return hipSuccess;
}
/* freed blocks stay reserved, so that an address is never handed out twice */
hipError_t hipFree(void *p) { live.erase(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? ret(hipErrorStreamCaptureUnsupported) : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
}

namespace qmsg {
thread_local const LaunchTimer *g_launch_timer = nullptr;
hipError_t launch_dense(const DenseArgs &a, int type, uint8_t *xqk, uint64_t, bool *records, hipStream_t)
{
    launches.push_back({ false, records != nullptr, a.T, type, xqk });
    return hipGetLastError();
}
hipError_t launch_dense_exact(const DenseArgs &a, int type, hipStream_t)
{
    launches.push_back({ true, false, a.T, type, nullptr });
    return hipGetLastError();
}
}  // namespace qmsg

#define CHECK(c)                                                                     \
    do {                                                                             \
        if (!(c)) { fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #c, qmsg_last_error(ctx)); exit(1); } \
    } while (0)

static qmsg_ctx *ctx;

static int mat(int type, int64_t rows, int64_t cols)
{
    static uint8_t data[16];
    const uint64_t rb = type == QMSG_T_Q4_0 ? (uint64_t)cols / 32 * 18
                        : type == QMSG_T_Q4_1 ? (uint64_t)cols / 32 * 20
                        : type == QMSG_T_Q8_0 ? (uint64_t)cols / 32 * 34
                        : type == QMSG_T_Q6_K ? (uint64_t)cols / 256 * 210 : (uint64_t)cols * 4;
    const qmsg_mat m = { type, rows, cols, rb, data };
    int id = -1;
    CHECK(qmsg_mat_upload(ctx, &m, &id) == QMSG_OK);
    return id;
}

static int call(int id, int T)
{
    float *const x = (float *)4096;
    float *const y[1] = { (float *)8192 };
    return qmsg_matmul_n_device(ctx, &id, 1, x, T, y);
}

/* the buffers that the launches recorded so far would use when replayed */
static bool launches_safe(size_t first, size_t end)
{
    for (size_t i = first; i < end; i++) {
        const Launch &l = launches[i];
        const bool uses = !l.exact && (l.records || l.T >= qmsg::kDenseQuantT);
        if (uses && l.xqk && !live.count(l.xqk)) return false;
    }
    return true;
}

/* a captured call of 5-7 rows on a large matrix, after a call that left the buffer large enough */
static void capture_small()
{
    const int big = mat(QMSG_T_Q4_0, 8192, 4096);
    for (int T = 5; T < qmsg::kDenseQuantT; T++) {
        CHECK(call(big, 8 * T) == QMSG_OK);
        capturing = true;
        const size_t n = launches.size();
        CHECK(call(big, T) == QMSG_OK);
        capturing = false;
        CHECK(launches.size() == n + 1 && !launches[n].records);
        CHECK(call(big, 64 * T) == QMSG_OK);        /* replaces the buffer */
        CHECK(launches_safe(n, n + 1));
        CHECK(call(big, T) == QMSG_OK && launches.back().records);
    }
    /* rows that only the MFMA kernels take: the buffer that is there, kept */
    const int wide = mat(QMSG_T_Q4_0, 1024, 32768);
    CHECK(call(wide, 6) == QMSG_OK && launches.back().records);
    capturing = true;
    const size_t n = launches.size();
    CHECK(call(wide, 6) == QMSG_OK && launches[n].records);
    capturing = false;
    CHECK(call(wide, 64) == QMSG_OK && launches_safe(n, n + 1));
}

/* captured calls of 8 and more rows, on MFMA and on pair records, and larger calls after them */
static void capture_large()
{
    const int big = mat(QMSG_T_Q4_0, 8192, 4096), few = mat(QMSG_T_Q4_0, 64, 4096);
    std::vector<size_t> held;
    for (int T : { 8, 16, 64 })
        for (int id : { big, few }) {
            CHECK(call(id, T) == QMSG_OK);
            capturing = true;
            held.push_back(launches.size());
            CHECK(call(id, T) == QMSG_OK && launches.back().xqk);
            capturing = false;
            CHECK(call(big, 2 * T) == QMSG_OK);         /* replaces the buffer */
            for (size_t n : held) CHECK(launches_safe(n, n + 1));
        }
}

/* no memory for the record buffer: 5-7 rows fall to the row kernels, 8 and more to the smaller pair
 * records, and with none for those either the call says so; nothing of it reaches the next call */
static void no_memory()
{
    const int C = 4096, big = mat(QMSG_T_Q4_0, 8192, C), f32 = mat(QMSG_T_F32, 8, C);
    malloc_limit = 4096;
    for (int T = 5; T < qmsg::kDenseQuantT; T++) {
        CHECK(call(big, T) == QMSG_OK && !launches.back().records);
        CHECK(call(f32, 1) == QMSG_OK);
    }
    CHECK(call(big, 16) == QMSG_E_NOMEM);
    CHECK(call(f32, 1) == QMSG_OK);
    malloc_limit = 16 * (C / 64) * qmsg::kPairBytes + 256;
    CHECK(call(big, 16) == QMSG_OK && !launches.back().records && launches.back().xqk);
    CHECK(call(big, 16) == QMSG_OK && !launches.back().records);
    CHECK(qmsg_device_alloc(ctx, (size_t)1 << 40) == nullptr);
    CHECK(call(f32, 1) == QMSG_OK);
    malloc_limit = ~(size_t)0;
    CHECK(call(big, 16) == QMSG_OK && launches.back().records);
    /* a captured call that would have to replace the buffer is refused, the next one runs */
    capturing = true;
    CHECK(call(big, 512) == QMSG_E_DEVICE);
    capturing = false;
    CHECK(call(f32, 1) == QMSG_OK);
}

/* calls whose launches read no record buffer allocate none: fp32 chains, F32 rows, widths of the
 * direct-read kernel, and at 5-7 rows matrices too small for the MFMA kernels; 8 and more rows on
 * the row kernels allocate the pair records only */
static void no_buffer()
{
    const int q8 = mat(QMSG_T_Q8_0, 8192, 4096), f32 = mat(QMSG_T_F32, 8192, 4096), big = mat(QMSG_T_Q4_0, 8192, 4096);
    const int off = mat(QMSG_T_Q4_0, 8192, 4128), small = mat(QMSG_T_Q4_0, 256, 256), few = mat(QMSG_T_Q4_0, 64, 4096);
    const int n = mallocs;
    for (int T : { 1, 4, 5, 7, 8, 64 }) {
        CHECK(call(q8, T) == QMSG_OK && call(f32, T) == QMSG_OK && call(off, T) == QMSG_OK);
        if (T < qmsg::kDenseQuantT) CHECK(call(small, T) == QMSG_OK && call(few, T) == QMSG_OK);
        CHECK(qmsg_set_path(ctx, QMSG_PATH_FP32) == QMSG_OK);
        CHECK(call(big, T) == QMSG_OK);
        CHECK(qmsg_set_path(ctx, QMSG_PATH_AUTO) == QMSG_OK);
    }
    CHECK(mallocs == n);
    malloc_limit = 64 * (4096 / 64) * qmsg::kPairBytes + 256;
    CHECK(call(few, 64) == QMSG_OK && mallocs == n + 1);
}

/* a captured call that pair records suffice for uses those there are */
static void capture_pairs()
{
    const int big = mat(QMSG_T_Q4_0, 8192, 4096);
    malloc_limit = 16 * (4096 / 64) * qmsg::kPairBytes + 256;
    CHECK(call(big, 16) == QMSG_OK && !launches.back().records);
    capturing = true;
    CHECK(call(big, 16) == QMSG_OK && !launches.back().records && live.count(launches.back().xqk));
    capturing = false;
}

/* at 5-8 tokens matrices that the row kernels' blocks cover in one pass over the CUs stay with them */
static void few_rows()
{
    const struct { int type; int64_t rows, C; bool mfma; } m[] = {
        { QMSG_T_Q6_K, 4096, 4096, false }, { QMSG_T_Q6_K, 4096, 8192, false }, { QMSG_T_Q6_K, 8192, 2048, false },
        { QMSG_T_Q4_0, 4096, 8192, false }, { QMSG_T_Q4_0, 6144, 1024, false }, { QMSG_T_Q4_0, 8192, 2048, true },
        { QMSG_T_Q6_K, 9216, 4096, true },  { QMSG_T_Q6_K, 151936, 2048, true },
        /* rows too long for the row kernels' LDS at several tokens */
        { QMSG_T_Q4_0, 1024, 32768, true }, { QMSG_T_Q4_1, 256, 65536, true }, { QMSG_T_Q6_K, 704, 24576, true },
    };
    for (const auto &k : m)
        for (int T = 5; T <= 8; T++) CHECK(call(mat(k.type, k.rows, k.C), T) == QMSG_OK && launches.back().records == k.mfma);
    CHECK(call(mat(QMSG_T_Q6_K, 128, 512), 9) == QMSG_OK && launches.back().records);
}

/* down rows of an odd number of Q6_K super-blocks: short ones take the MFMA kernels from 64 slots */
static void odd_down()
{
    CHECK(!qmsg::mx_auto_down(5, 8, 768, 14) && !qmsg::mx_auto_down(7, 8, 256, 14) && qmsg::mx_auto_down(8, 8, 768, 14));
    CHECK(qmsg::mx_auto_down(4, 8, 1280, 14) && qmsg::mx_auto_down(4, 8, 1536, 14) && qmsg::mx_auto_down(4, 8, 512, 14));
    CHECK(!qmsg::mx_auto_down(3, 8, 1280, 14) && !qmsg::mx_auto_down(7, 8, 768, 2) && qmsg::mx_auto_down(8, 8, 768, 2));
}

/* rows so long that a block's byte offsets (32 bits, the top one a flag) would not hold them stay off
 * the MFMA kernels */
static void wide_rows()
{
    for (int type : { QMSG_T_Q4_0, QMSG_T_Q4_1, QMSG_T_Q6_K })
        for (int64_t C : { (int64_t)4096, (int64_t)1 << 22, (int64_t)1 << 24, (int64_t)1 << 26, (int64_t)1 << 30 }) {
            qmsg::DenseArgs a{};
            a.rb = (uint64_t)(type == QMSG_T_Q4_0 ? C / 32 * 18 : type == QMSG_T_Q4_1 ? C / 32 * 20 : C / 256 * 210);
            a.C = (int)C;
            a.T = 16;
            a.nm = 1;
            a.m[0].rows = 128;
            CHECK(!qmsg::dense_mx_takes(a, type) || 128 * a.rb < (uint64_t)1 << 31);
            CHECK(C > 4096 || qmsg::dense_mx_takes(a, type));
        }
}

/* the chain kernels' reads of input rows staged whole, the block read ahead included, stay inside
 * the LDS their launch asks for */
static void chain_lds()
{
    for (int T = 1; T <= 16; T++)
        for (int C = 32; T * C <= 16384; C += 32) {
            const int end = (T - 1) * qmsg::chain_row_floats(C) + qmsg::chain_row_read(C / 32, 3, 1) + 4;
            CHECK((size_t)end * 4 <= qmsg::chain_rows_lds(T, C));
        }
}

int main(int argc, char **argv)
{
    const qmsg_cfg cfg = { 256, 16, 4, 128 };
    if (argc != 2 || qmsg_create(&ctx, 0, &cfg, 1, 1) != QMSG_OK) return 2;
    const std::string s = argv[1];
    if (s == "capture_small") capture_small();
    else if (s == "capture_large") capture_large();
    else if (s == "no_memory") no_memory();
    else if (s == "no_buffer") no_buffer();
    else if (s == "capture_pairs") capture_pairs();
    else if (s == "few_rows") few_rows();
    else if (s == "odd_down") odd_down();
    else if (s == "wide_rows") wide_rows();
    else if (s == "chain_lds") chain_lds();
    else return 2;
    qmsg_destroy(ctx);
    if (!live.empty()) {
        fprintf(stderr, "%zu allocations outlive the context\n", live.size());
        return 1;
    }
    return 0;
}
