// model.cpp -- a CPU model of the device for the host layer (et_host.cpp).
//
// Linked with et_host.cpp in place of the HIP runtime and the kernels.  Device
// memory is host memory of known blocks; a launch checks that everything its
// arguments name lies inside live blocks, and then records what it leaves
// there as a tag: a hash of the tags of what it read.  Two results with equal
// tags were formed by the same launches from the same contents, so a result
// that used something stale differs from a fresh plan's.  Allocations can be
// limited, launches made to fail, and a stream captured and replayed.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "et_internal.h"

typedef unsigned long long u64;

namespace {

struct Block {
    size_t bytes;
    std::map<size_t, u64> tags;             // by offset: what was written from there on
    std::set<const void *> used;            // streams whose launches use it and were not waited for
};
std::map<const char *, Block> blocks;       // live device blocks by address
size_t used_bytes = 0, limit_bytes = ~(size_t)0;
std::string violations;                     // one per line
std::vector<std::string> log_;              // executed launches
std::vector<std::vector<std::function<void()>>> graphs;
const void *capturing = nullptr;            // the captured stream
std::string fail_name;
int fail_at = 0;
int sweep_blocks = 0, sweep_planes = 0;     // of the last row-lane sweep: its grid, planes per block

void violation(const std::string &s) { violations += s + "\n"; }

u64 mix(u64 a, u64 b)
{
    u64 h = a * 0x9e3779b97f4a7c15ull + b;
    h ^= h >> 32;
    h *= 0xd6e8feb86659fd93ull;
    h ^= h >> 32;
    return h;
}
u64 mix_all(std::initializer_list<u64> v)
{
    u64 h = 17;
    for (u64 x : v) h = mix(h, x);
    return h;
}

Block *block_of(const void *p, size_t &off)
{
    const char *c = static_cast<const char *>(p);
    auto it = blocks.upper_bound(c);
    if (it == blocks.begin()) return nullptr;
    --it;
    if (c >= it->first + it->second.bytes) return nullptr;
    off = c - it->first;
    return &it->second;
}

// [p, p + n floats) inside one live block.
bool need(const void *p, size_t n, const char *what)
{
    size_t off = 0;
    Block *b = p ? block_of(p, off) : nullptr;
    if (b && off + n * sizeof(float) <= b->bytes) return true;
    violation(std::string(what) + (b ? ": past the end of its buffer" : ": not a live buffer"));
    return false;
}
u64 tag(const void *p)
{
    size_t off = 0;
    Block *b = p ? block_of(p, off) : nullptr;
    if (!b) return 0;
    auto it = b->tags.upper_bound(off);
    if (it == b->tags.begin()) return 1;  // never written
    --it;
    return it->first == off ? it->second : mix(it->second, off - it->first);
}
void set_tag(const void *p, u64 t)
{
    size_t off = 0;
    if (Block *b = block_of(p, off)) b->tags[off] = t;
}

// One launch: fails, is recorded, or runs; uses: the buffers it works on.
int launch(const char *name, et_stream_t st, std::vector<const void *> uses, std::function<void()> run)
{
    if (!fail_name.empty() && fail_name == name && --fail_at == 0) {
        fail_name.clear();
        return (int)hipErrorLaunchFailure;
    }
    const std::string n = name;
    auto all = [=]() {
        log_.push_back(n);
        for (const void *p : uses) {
            size_t off;
            if (Block *b = p ? block_of(p, off) : nullptr) b->used.insert(st);
        }
        run();
    };
    if (capturing && st == capturing)
        graphs.back().push_back(all);
    else
        all();
    return 0;
}

// What a sweep over `a` reads: every buffer checked, one tag.
u64 sweep_reads(const EtSweepArgs &a, bool act, bool mu, size_t att_elems, size_t sino_elems)
{
    const size_t yf = (size_t)a.yp * a.xp * (a.nz + 2);
    u64 t = mix_all({(u64)a.D, (u64)a.zlen, (u64)a.V, (u64)a.truncate});
    const size_t n_rec = a.rec_stride ? (size_t)a.V * a.rec_stride : ET_VIEW_REC;
    if (need(a.views, n_rec, "view records")) t = mix(t, tag(a.views));
    if (act && need(a.act, yf + (a.V - 1) * a.act_vs, "activity")) t = mix(t, tag(a.act));
    if (mu && need(a.mu, yf + (a.V - 1) * a.mu_vs, "attenuation")) t = mix(t, tag(a.mu));
    if (a.psf && need(a.psf, (size_t)a.nz * 2 * a.K, "PSF")) t = mix(t, tag(a.psf));
    if (att_elems && need(a.att, att_elems, "factors")) t = mix(t, tag(a.att));
    if (sino_elems && need(a.sino, sino_elems, "sinogram")) t = mix(t, tag(a.sino));
    return t;
}

size_t yl_att(const EtSweepArgs &a) { return a.att ? (a.V - 1) * a.att_vs + (size_t)a.nz * a.nx * a.yu : 0; }

u64 pull_reads(const EtPullArgs &a)
{
    u64 t = mix_all({(u64)a.V, (u64)a.adjoint, (u64)a.epilogue, (u64)a.truncate});
    unsigned f;
    std::memcpy(&f, &a.floor, 4);
    t = mix(t, f);
    if (need(a.views, (size_t)a.V * ET_VIEW_REC, "view records")) t = mix(t, tag(a.views));
    if (need(a.u, (size_t)a.V * a.ustride, "rotated-frame volumes")) t = mix(t, tag(a.u));
    return t;
}
void pull(const EtPullArgs &a)
{
    u64 t = pull_reads(a);
    const size_t yf = (size_t)a.yp * a.xp * (a.nz + 2);
    if (a.epilogue == ET_EPI_OSEM) {
        if (need(a.x, yf, "iterate") && need(a.sens, yf, "sensitivity"))
            set_tag(a.x, mix_all({tag(a.x), tag(a.sens), t}));
        return;
    }
    const size_t n = a.epilogue == ET_EPI_ABI_STORE ? (size_t)a.nx * a.ny * a.nz : yf;
    if (a.epilogue == ET_EPI_ABI_STORE ? need(a.out, (size_t)a.nx * a.nz, "image") : need(a.out, n, "accumulator"))
        set_tag(a.out, a.accumulate ? mix(tag(a.out), t) : t);
}

}  // namespace

// ---- the runtime ---------------------------------------------------------------------
extern "C" {

hipError_t hipMalloc(void **p, size_t n)
{
    if (capturing) return hipErrorStreamCaptureUnsupported;
    if (used_bytes + n > limit_bytes) return hipErrorOutOfMemory;
    void *q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return hipErrorOutOfMemory;
    std::memset(q, 0xa5, std::min<size_t>(n, 65536));  // (what was there before)
    blocks[static_cast<char *>(q)] = {n, {}, {}};
    used_bytes += n;
    *p = q;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    auto it = blocks.find(static_cast<char *>(p));
    if (it == blocks.end()) {
        violation("hipFree: not a live block");
        return hipErrorInvalidValue;
    }
    for (auto &b : blocks) b.second.used.clear();  // it waits for the device
    used_bytes -= it->second.bytes;
    munmap(p, it->second.bytes);
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_, size_t *total)
{
    *total = (size_t)288 << 30;
    *free_ = limit_bytes == ~(size_t)0 ? *total - used_bytes : (limit_bytes > used_bytes ? limit_bytes - used_bytes : 0);
    return hipSuccess;
}
static u64 bytes_tag(const void *p, size_t n)
{
    u64 h = n;
    for (size_t i = 0; i + 4 <= n; i += 4) {
        unsigned v;
        std::memcpy(&v, static_cast<const char *>(p) + i, 4);
        h = mix(h, v);
    }
    return h;
}
static hipError_t copy(void *d, const void *s, size_t n, hipMemcpyKind k, const void *st)
{
    size_t off;
    if (k == hipMemcpyHostToDevice || k == hipMemcpyDeviceToDevice) {
        if (!need(d, n / 4, "copy")) return hipErrorInvalidValue;
        for (const void *q : block_of(d, off)->used)
            if (q != st) violation("a copy overwrites a buffer that another stream's launches still use");
    }
    if (k == hipMemcpyHostToDevice) {
        std::memcpy(d, s, n);
        set_tag(d, bytes_tag(s, n));
    } else if (k == hipMemcpyDeviceToDevice) {
        set_tag(d, tag(s));
    } else if (need(s, n / 4, "copy")) {
        std::memcpy(d, s, n);
    }
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k, nullptr); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    if (capturing && (const void *)st == capturing) {
        violation("a copy from or to pageable memory under capture");
        return hipErrorStreamCaptureUnsupported;
    }
    return copy(d, s, n, k, st);
}
hipError_t hipStreamSynchronize(hipStream_t st)
{
    if (capturing) return hipErrorStreamCaptureUnsupported;
    for (auto &b : blocks) b.second.used.erase(st);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    for (auto &b : blocks) b.second.used.clear();
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus *s)
{
    *s = capturing && (const void *)st == capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
static size_t n_streams = 0;
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(0x1000 + 16 * ++n_streams);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = reinterpret_cast<hipEvent_t>(16);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;  // (the first candidate of a timed choice is kept)
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *, int) { return hipErrorNotSupported; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorNotSupported; }

// ---- the test's side -------------------------------------------------------------------
void model_limit(size_t bytes) { limit_bytes = bytes; }
size_t model_used() { return used_bytes; }
void *model_volume(size_t floats, u64 t)
{
    void *p = nullptr;
    if (hipMalloc(&p, floats * sizeof(float)) != hipSuccess) return nullptr;
    set_tag(p, t);
    return p;
}
void model_set(void *p, u64 t) { set_tag(p, t); }
u64 model_tag(const void *p) { return tag(p); }
void model_fail(const char *name, int nth)
{
    fail_name = name;
    fail_at = nth;
}
const char *model_violations() { return violations.c_str(); }
void model_clear()
{
    violations.clear();
    log_.clear();
}
int model_count(const char *name)
{
    int n = 0;
    for (const std::string &s : log_) n += s == name;
    return n;
}
int model_sweep_blocks() { return sweep_blocks; }
int model_sweep_planes() { return sweep_planes; }
void model_begin(void *stream)
{
    capturing = stream;
    graphs.emplace_back();
}
int model_end()
{
    capturing = nullptr;
    return (int)graphs.size() - 1;
}
void model_replay(int g)
{
    for (auto &f : graphs[g]) f();
}
}

// ---- the launches --------------------------------------------------------------------------
void et_offer_launch_events(et_event_t, et_event_t) {}
bool et_withdraw_launch_events() { return false; }
int et_sweep_slab_rows(int, int) { return 16; }
int et_fingerprint_blocks(size_t) { return 1; }
int et_pack_keys_blocks(int, int, int) { return 2; }

int et_launch_fill(float *buf, size_t n, float value, et_stream_t st)
{
    return launch("fill", st, {buf}, [=]() {
        if (!need(buf, n, "fill")) return;
        if (value == 0.f && n <= 16384) std::memset(buf, 0, n * sizeof(float));
        unsigned v;
        std::memcpy(&v, &value, 4);
        set_tag(buf, mix(3, v));
    });
}
int et_launch_store(void *dst, const void *src, size_t bytes, et_stream_t st)
{
    const std::string b(static_cast<const char *>(src), bytes);
    return launch("store", st, {dst}, [=]() {
        if (need(dst, bytes / 4, "table")) std::memcpy(dst, b.data(), bytes);
    });
}
int et_launch_fingerprint(const float *p, size_t n, u64 *parts, et_stream_t st)
{
    return launch("fingerprint", st, {p, parts}, [=]() {
        if (need(p, n, "map") && need(parts, 2, "fingerprint")) *parts = tag(p);
    });
}
int et_launch_pack_yf(const float *abi, float *yf, int nx, int ny, int nz, int yp, int, et_stream_t st)
{
    return launch("pack", st, {abi, yf}, [=]() {
        if (need(abi, (size_t)nx * ny * nz, "volume") && need(yf, (size_t)yp * (nx + 2) * (nz + 2), "YF copy"))
            set_tag(yf, tag(abi));
    });
}
int et_launch_unpack_yf(const float *yf, float *abi, int nx, int ny, int nz, int yp, int, et_stream_t st)
{
    return launch("unpack", st, {abi, yf}, [=]() {
        if (need(abi, (size_t)nx * ny * nz, "volume") && need(yf, (size_t)yp * (nx + 2) * (nz + 2), "YF copy"))
            set_tag(abi, tag(yf));
    });
}
int et_launch_pack_keys(const EtPackArgs &a, int n, et_stream_t st)
{
    return launch("pack_keys", st, {a.src[0], a.src[1], a.dst[0], a.dst[1]}, [=]() {
        if (a.st && need(a.st, 2 * ET_KEY_WORDS, "keys")) std::copy(a.st, a.st + ET_KEY_LAST, a.st + ET_KEY_LAST);
        for (int k = 0; k < n; k++) {
            if (!need(a.src[k], (size_t)a.nx * a.ny * a.nz, "volume") ||
                !need(a.dst[k], (size_t)a.yp * (a.nx + 2) * (a.nz + 2), "YF copy"))
                continue;
            set_tag(a.dst[k], tag(a.src[k]));
            if (a.parts && need(a.parts + 2 * k, 4, "keys")) {
                a.parts[2 * k] = tag(a.src[k]);
                a.parts[2 * k + 1] = 0;
            }
        }
    });
}
int et_launch_yl_factors(int, bool, const EtSweepArgs &a, const EtKeys &k, et_stream_t st)
{
    return launch("factors", st, {a.att, a.mu, a.views, k.st}, [=]() {
        const u64 t = sweep_reads(a, false, true, 0, 0);
        if (!need(a.att, yl_att(a), "factors") || !need(k.st, 2 * ET_KEY_WORDS, "keys")) return;
        const u64 km = k.mu[0] + k.mu[1], ka = k.act ? k.act[0] + k.act[1] : 0;
        const u64 *last = k.st + ET_KEY_LAST;
        const bool keep = et_keys_keep_factors(k, last, km);
        et_keys_end(k, last, km, ka);
        if (keep) return;
        log_.push_back("factors built");
        set_tag(a.att, t);
    });
}
int et_launch_yl_sweep(int kind, int R, int RPL, int NR, int nthr, size_t lds, const EtSweepArgs *args, const void *tab,
                       int n, int blocks, et_stream_t st)
{
    return launch("yl_sweep", st, {args}, [=]() {
        if (!need(args, n * sizeof(EtSweepArgs) / 4, "table") || !need(tab, 4 * (size_t)n, "table")) return;
        const int *t4 = static_cast<const int *>(tab);
        for (int j = 0; j < n; j++) {
            const EtSweepArgs a = args[j];
            sweep_blocks = t4[4 * j + 1] * t4[4 * j + 2];
            sweep_planes = a.zlen;
            const int end = j + 1 < n ? t4[4 * (j + 1)] : blocks, k = kind % ET_YL_COND;
            if (t4[4 * j] + t4[4 * j + 1] * t4[4 * j + 2] > end) violation("table: more blocks than the grid has");
            const bool grad = k == 3 || k == 4 || k == 5 || k == 8, bpu = k == 1 || k == 7;
            for (const void *p : {(const void *)a.act, (const void *)a.att, (const void *)a.sino, (const void *)a.u,
                                  (const void *)a.part, (const void *)a.views}) {
                size_t off;
                if (Block *b = p ? block_of(p, off) : nullptr) b->used.insert(st);
            }
            const size_t pl = (size_t)a.nx * a.yu;
            u64 t = sweep_reads(a, !bpu, false, yl_att(a), grad || (bpu && a.src == ET_SRC_SINO) ? a.V * pl : 0);
            t = mix_all({t, (u64)k, (u64)R, (u64)RPL, (u64)NR, (u64)nthr, (u64)lds, (u64)a.src});
            // partial sums: of the activity, the factors and the view, not of the batch
            const u64 sums = mix_all({tag(a.act), a.att ? tag(a.att) : 0, (u64)a.D, (u64)a.zlen});
            if (kind >= ET_YL_COND && need(a.skip, 1, "skip flag") && *a.skip) {
                log_.push_back("sums kept");
                continue;
            }
            if (!bpu && !(grad && a.D == 1) && need(a.part, ((a.D - 1) * (size_t)a.part_V + a.V) * pl, "partial sums")) {
                if (!grad) {
                    set_tag(a.part, mix(sums, k == 5 ? 1 : 0));
                    log_.push_back("sums formed");
                } else {
                    t = mix(t, tag(a.part));
                }
            }
            if ((grad || bpu) && need(a.u, (size_t)a.V * a.ustride, "rotated-frame volumes")) set_tag(a.u, t);
        }
    });
}
int et_launch_yl_pull(int, int, const EtPullArgs *args, const void *tab, int n, int, et_stream_t st)
{
    return launch("yl_pull", st, {args}, [=]() {
        if (need(args, n * sizeof(EtPullArgs) / 4, "table") && need(tab, 4 * (size_t)n, "table"))
            for (int j = 0; j < n; j++) pull(args[j]);
    });
}
int et_launch_yl_pull_adj(int RPL, const EtPullArgs *args, const void *tab, int n, int blocks, et_stream_t st)
{
    return et_launch_yl_pull(0, RPL, args, tab, n, blocks, st);
}
int et_launch_ratio_group(const EtRatioArgs *args, const void *tab, int n, int, et_stream_t st)
{
    return launch("ratio_group", st, {args}, [=]() {
        if (!need(args, n * sizeof(EtRatioArgs) / 4, "table") || !need(tab, 4 * (size_t)n, "table")) return;
        for (int j = 0; j < n; j++) {
            const EtRatioArgs &a = args[j];
            unsigned e;
            std::memcpy(&e, &a.eps, 4);
            if (need(a.meas, a.VP, "counts") && need(a.part, a.D * a.VP, "partial sums") && need(a.out, a.VP, "ratio"))
                set_tag(a.out, mix_all({tag(a.meas), tag(a.part), (u64)a.D, e}));
        }
    });
}
int et_launch_gather_planes_t(float *dst, const float *src, const int *order, int V, int nx, int ny, int rows,
                              et_stream_t st)
{
    return launch("planes_t", st, {dst, src, order}, [=]() {
        if (need(dst, (size_t)V * nx * rows, "planes") && need(src, (size_t)V * nx * ny, "sinogram") &&
            (!order || need(order, V, "order")))
            set_tag(dst, mix(tag(src), order ? tag(order) : 0));
    });
}
int et_launch_yl_parts_to_sino(const float *part, int D, int V, int nx, int ny, int rows, int truncate, float *sino,
                               et_stream_t st)
{
    return launch("parts_to_sino", st, {part, sino}, [=]() {
        if (need(part, (size_t)D * V * nx * rows, "partial sums") && need(sino, (size_t)V * nx * ny, "sinogram"))
            set_tag(sino, mix_all({tag(part), (u64)D, (u64)truncate}));
    });
}
// the sweep kernels and the general path
int et_launch_sweep(int mode, int R, int has_mu, int has_act, const EtSweepArgs &a, et_stream_t st)
{
    const size_t P = (size_t)a.nx * a.ny, nthr = (a.nx + 63) / 64 * 64;
    if ((size_t)a.V * a.D > 65535) return (int)hipErrorInvalidConfiguration;
    return launch("sweep", st, {a.act, a.mu, a.views, a.part, a.u, a.sino, a.att}, [=]() {
        u64 t = sweep_reads(a, mode != ET_MODE_BPU && mode != ET_MODE_MUSUM && has_act, has_mu == 1,
                            has_mu == 3 ? (size_t)a.V * a.nz * a.yu * nthr : 0,
                            mode != ET_MODE_PROJECT && mode != ET_MODE_MUSUM && a.src == ET_SRC_SINO ? a.V * P : 0);
        t = mix_all({t, (u64)mode, (u64)R, (u64)has_mu});
        if (mode == ET_MODE_PROJECT || mode == ET_MODE_MUSUM) {
            if (need(a.part, (size_t)a.D * a.V * P, "partial sums")) set_tag(a.part, t);
        } else if (need(a.u, (size_t)a.V * a.ustride, "rotated-frame volumes")) {
            set_tag(a.u, t);
        }
    });
}
int et_launch_att_factors(const EtSweepArgs &a, et_stream_t st)
{
    const size_t nthr = (a.nx + 63) / 64 * 64;
    return launch("att_factors", st, {a.att, a.mu, a.views}, [=]() {
        const u64 t = sweep_reads(a, false, true, 0, 0);
        if (need(a.att, (size_t)a.V * a.nz * a.yu * nthr, "factors")) set_tag(a.att, t);
    });
}
int et_launch_pull(const EtPullArgs &a, et_stream_t st)
{
    return launch("pull", st, {a.u, a.out, a.x, a.views}, [=]() { pull(a); });
}
int et_launch_pull_general(const EtPullArgs &a, et_stream_t st)
{
    return launch("pull_general", st, {a.u, a.out, a.views}, [=]() { pull(a); });
}
int et_launch_resample_general(const float *src, int nx, int ny, int nz, const float *M, float, float *dst, int, int,
                               int, int nv, size_t vs, et_stream_t st)
{
    if (nv <= 0 || nv > 65535) return (int)hipErrorInvalidValue;
    return launch("resample", st, {src, M, dst}, [=]() {
        if (need(src, (size_t)nx * ny * nz, "volume") && need(M, nv > 1 ? (size_t)nv * ET_VIEW_REC : 12, "records") &&
            need(dst, (nv - 1) * vs + (size_t)nx * ny * nz, "rotated copies"))
            set_tag(dst, mix(tag(src), tag(M)));
    });
}
int et_launch_rotate_yf(const float *s0, const float *s1, int nx, int, int nz, const float *recs, int yp, int,
                        float *d0, float *d1, size_t vs, int nv, et_stream_t st)
{
    if (!s0 || !d0 || (s1 && !d1) || nv <= 0 || nv > 65535 || nz > 65535) return (int)hipErrorInvalidValue;
    return launch("rotate_yf", st, {s0, s1, recs, d0, d1}, [=]() {
        const size_t yf = (size_t)yp * (nx + 2) * (nz + 2);
        if (!need(recs, (size_t)nv * ET_VIEW_REC, "records")) return;
        if (need(s0, yf, "volume") && need(d0, (nv - 1) * vs + yf, "rotated copies")) set_tag(d0, mix(tag(s0), tag(recs)));
        if (s1 && need(s1, yf, "volume") && need(d1, (nv - 1) * vs + yf, "rotated copies"))
            set_tag(d1, mix(tag(s1), tag(recs)));
    });
}
int et_launch_conv_axis(const float *src, float *dst, int nx, int ny, int nz, long, long, long, long, int axis,
                        const float *sep, int K, int flip, int nv, size_t vs, et_stream_t st)
{
    if (nv <= 0 || nv > 65535) return (int)hipErrorInvalidValue;
    return launch("conv_axis", st, {src, dst, sep}, [=]() {
        const size_t n = (nv - 1) * vs + (size_t)nx * ny * nz;
        if (need(src, n, "volume") && need(dst, n, "volume") && need(sep, (size_t)nz * 2 * K, "PSF"))
            set_tag(dst, mix_all({tag(src), tag(sep), (u64)axis, (u64)flip}));
    });
}
int et_launch_chunk_scan(const float *csum, const float *lo, float *astart, float *atot, float *atot_lo, int V, int D,
                         int P, et_stream_t st)
{
    return launch("chunk_scan", st, {csum, lo, astart, atot, atot_lo}, [=]() {
        const size_t n = (size_t)V * P;
        if (!need(csum, n * D, "chunk sums") || !need(lo, n * D, "chunk sums")) return;
        if (astart && need(astart, n * D, "prefixes")) set_tag(astart, tag(csum));
        if (atot && need(atot, n, "totals") && need(atot_lo, n, "totals")) set_tag(atot, tag(csum));
    });
}
int et_launch_reduce_parts(const float *part, int D, int V, int P, float *sino, int truncate, et_stream_t st)
{
    return launch("reduce_parts", st, {part, sino}, [=]() {
        if (need(part, (size_t)D * V * P, "partial sums") && need(sino, (size_t)V * P, "sinogram"))
            set_tag(sino, mix_all({tag(part), (u64)D, (u64)truncate}));
    });
}
int et_launch_bg_only(const float *atot, const float *lo, float, int n, float *sino, int, et_stream_t st)
{
    return launch("bg_only", st, {atot, lo, sino}, [=]() {
        if (need(atot, n, "totals") && need(lo, n, "totals") && need(sino, n, "sinogram")) set_tag(sino, tag(atot));
    });
}
int et_launch_truncate(float *p, size_t n, et_stream_t st)
{
    return launch("truncate", st, {p}, [=]() { need(p, n, "truncate"); });
}
int et_launch_clamp_min(float *p, size_t n, float, et_stream_t st)
{
    return launch("clamp_min", st, {p}, [=]() { need(p, n, "clamp"); });
}
int et_launch_yf_clamp_min(float *p, int nx, int, int nz, int yp, int, float, et_stream_t st)
{
    return launch("yf_clamp", st, {p}, [=]() { need(p, (size_t)yp * (nx + 2) * (nz + 2), "sensitivity"); });
}
int et_launch_em_update_flat(float *x, const float *b, const float *s, size_t n, et_stream_t st)
{
    return launch("em_update", st, {x, b, s}, [=]() {
        if (need(x, n, "iterate") && need(b, n, "image") && need(s, n, "image"))
            set_tag(x, mix_all({tag(x), tag(b), tag(s)}));
    });
}
int et_launch_gather_planes(float *dst, const float *src, const int *order, int V, size_t P, et_stream_t st)
{
    return launch("planes", st, {dst, src, order}, [=]() {
        if (need(dst, V * P, "planes") && need(order, V, "order")) set_tag(dst, mix(tag(src), tag(order)));
    });
}
int et_launch_ratio_parts(const float *meas, const float *part, int D, size_t VP, float eps, float *out, et_stream_t st)
{
    unsigned e;
    std::memcpy(&e, &eps, 4);
    return launch("ratio_parts", st, {meas, part, out}, [=]() {
        if (need(meas, VP, "counts") && need(part, D * VP, "partial sums") && need(out, VP, "ratio"))
            set_tag(out, mix_all({tag(meas), tag(part), (u64)D, e}));
    });
}
int et_launch_ratio(const float *meas, const float *proj, float *out, size_t n, float, et_stream_t st)
{
    return launch("ratio", st, {meas, proj, out}, [=]() {
        if (need(meas, n, "counts") && need(proj, n, "projection") && need(out, n, "ratio"))
            set_tag(out, mix(tag(meas), tag(proj)));
    });
}
int et_launch_sweep_group(int, int, int, int, const EtSweepArgs *, const void *, int, int, et_stream_t)
{
    return (int)hipErrorNotSupported;  // (batches are not modelled)
}
int et_launch_pull_group(int, const EtPullArgs *, const void *, int, int, et_stream_t)
{
    return (int)hipErrorNotSupported;
}
int et_launch_partial_line(const float *, const float *, const float *, float, int, int, int, float *, float *,
                           et_stream_t)
{
    return (int)hipErrorNotSupported;
}
int et_launch_fisher_pairs(const EtFisherArgs &, et_stream_t) { return (int)hipErrorNotSupported; }
