// ibh_runtime.hip -- device/stream/error runtime of libibhip and the
// host-pointer dispatch-table entries (ib_init_kernels_hip).
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "ibh_common.h"

// ── errors (same convention as src/error.c:7-21 of the reference) ─────────
static thread_local char g_err[512];
static thread_local int g_err_set = 0;

extern "C" void ibh_set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    g_err_set = 1;
}

extern "C" const char* ibh_last_error(void) {
    if (!g_err_set) return nullptr;
    g_err_set = 0;
    return g_err;
}

extern "C" int ibh_device_errors(int clear) {
    if (hipDeviceSynchronize() != hipSuccess) {
        ibh_set_error("ibh_device_errors: device synchronisation failed");
        return IBH_ERROR_INTERNAL;
    }
    const int a = ibh_tile_errors(clear != 0), b = ibh_pq_errors(clear != 0);
    if (a < 0 || b < 0) {
        ibh_set_error("ibh_device_errors: cannot read the device error words");
        return IBH_ERROR_INTERNAL;
    }
    return a | b;
}

extern "C" const char* ibh_version(void) { return "libinferbit_amd 0.1.0 (gfx950)"; }

// ── per-device state ───────────────────────────────────────────────────────
namespace {
constexpr int kMaxDev = 16;
struct DevState {
    bool ready = false;
    void* ws = nullptr;          // library workspace (activation operand staging)
    size_t ws_bytes = 0;
};
constexpr size_t kDefaultWorkspace = 4u << 20;
DevState g_dev[kMaxDev];
std::mutex g_mu;

int current_device() {
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess) return -1;
    return d;
}
}  // namespace

int ibh_noalloc_setup(int device);   // ibh_gemv.hip
int ibh_launch_matvec_exact(float* y, const void* w, const void* sc, int kind, const float* x, int M, int N, int bits,
                            const uint8_t* mask, hipStream_t st);   // ibh_exact.hip
int ibh_launch_int8_batch_exact(const ibh::MatDesc* d, int n, int kind, const float* x, int N, int B, bool avx,
                                hipStream_t st, int M_stride = 0);

extern "C" int ibh_init(int device) {
    std::lock_guard<std::mutex> lk(g_mu);
    int n = 0;
    IBH_HIP(hipGetDeviceCount(&n), "ibh_init: hipGetDeviceCount");
    if (device < 0 || device >= n || device >= kMaxDev) {
        ibh_set_error("ibh_init: device %d out of range (%d visible)", device, n);
        return IBH_ERROR_PARAM;
    }
    IBH_HIP(hipSetDevice(device), "ibh_init: hipSetDevice");
    DevState& s = g_dev[device];
    if (!s.ready) {
        if (hipMalloc(&s.ws, kDefaultWorkspace) != hipSuccess) {
            ibh_set_error("ibh_init: cannot allocate the %zu-byte workspace", kDefaultWorkspace);
            return IBH_ERROR_MEMORY;
        }
        s.ws_bytes = kDefaultWorkspace;
        const int rc = ibh_noalloc_setup(device);
        if (rc != IBH_OK) return rc;
        s.ready = true;
    }
    return IBH_OK;
}

// Per-device workspace allocated by ibh_init (fixed size, so calls can be
// captured in HIP graphs).  Shared by every call on the device: calls that
// use it must not overlap in time (one stream, or stream-ordered).
void* ibh_workspace(size_t bytes) {
    const int d = current_device();
    if (d < 0 || d >= kMaxDev) return nullptr;
    if (!g_dev[d].ready && ibh_init(d) != IBH_OK) return nullptr;
    return bytes <= g_dev[d].ws_bytes ? g_dev[d].ws : nullptr;
}

// NULL selects the device's null stream, which is ordered with every
// blocking stream of the process (torch's default stream included).
hipStream_t ibh_resolve_stream(void* s) {
    if (s) return (hipStream_t)s;
    const int d = current_device();
    if (d >= 0 && d < kMaxDev && !g_dev[d].ready) ibh_init(d);
    return nullptr;
}

extern "C" void* ibh_default_stream(void) { return (void*)ibh_resolve_stream(nullptr); }

extern "C" int ibh_synchronize(void* stream) {
    IBH_HIP(hipStreamSynchronize(ibh_resolve_stream(stream)), "ibh_synchronize");
    return IBH_OK;
}

extern "C" int ibh_device_malloc(void** dptr, size_t bytes) {
    if (!dptr) {
        ibh_set_error("ibh_device_malloc: null out-pointer");
        return IBH_ERROR_PARAM;
    }
    if (hipMalloc(dptr, bytes ? bytes : 1) != hipSuccess) {
        ibh_set_error("ibh_device_malloc: out of device memory (%zu bytes)", bytes);
        *dptr = nullptr;
        return IBH_ERROR_MEMORY;
    }
    return IBH_OK;
}

extern "C" int ibh_device_free(void* dptr) {
    if (dptr) IBH_HIP(hipFree(dptr), "ibh_device_free");
    return IBH_OK;
}

static int copy(void* dst, const void* src, size_t n, hipMemcpyKind k, void* stream, const char* who) {
    if (!n) return IBH_OK;
    hipStream_t st = ibh_resolve_stream(stream);
    IBH_HIP(hipMemcpyAsync(dst, src, n, k, st), who);
    if (k == hipMemcpyDeviceToHost) IBH_HIP(hipStreamSynchronize(st), who);
    return IBH_OK;
}
extern "C" int ibh_memcpy_h2d(void* d, const void* s, size_t n, void* st) {
    return copy(d, s, n, hipMemcpyHostToDevice, st, "ibh_memcpy_h2d");
}
extern "C" int ibh_memcpy_d2h(void* d, const void* s, size_t n, void* st) {
    return copy(d, s, n, hipMemcpyDeviceToHost, st, "ibh_memcpy_d2h");
}
extern "C" int ibh_memcpy_d2d(void* d, const void* s, size_t n, void* st) {
    return copy(d, s, n, hipMemcpyDeviceToDevice, st, "ibh_memcpy_d2d");
}

// ── host-pointer dispatch table ────────────────────────────────────────────
//
// The reference calls its table from CPU code with host pointers
// (src/threading.c:220-258).  Registered weight regions are uploaded once;
// activations, scales and outputs are staged through a grow-only device
// workspace.  Table entries return void like the reference's; a failure is
// reported on stderr and through ibh_last_error(), and the output is left
// NaN-filled so it cannot pass for a result.
namespace {
struct Region {
    const uint8_t* host;
    size_t bytes;
    uint8_t* dev;
};
std::vector<Region> g_regions;
std::mutex g_tab_mu;
uint8_t* g_ws = nullptr;
size_t g_ws_bytes = 0;

const uint8_t* lookup(const void* hp, size_t need) {
    const uint8_t* p = (const uint8_t*)hp;
    for (const Region& r : g_regions)
        if (p >= r.host && p + need <= r.host + r.bytes) return r.dev + (p - r.host);
    return nullptr;
}

uint8_t* workspace(size_t bytes) {
    if (bytes <= g_ws_bytes) return g_ws;
    if (g_ws) (void)hipFree(g_ws);
    g_ws = nullptr;
    g_ws_bytes = 0;
    size_t want = bytes + (bytes >> 2) + 4096;
    if (hipMalloc((void**)&g_ws, want) != hipSuccess) return nullptr;
    g_ws_bytes = want;
    return g_ws;
}

size_t al256(size_t n) { return (n + 255) & ~(size_t)255; }

void fail(float* out, size_t n, const char* who) {
    const char* e = ibh_last_error();
    fprintf(stderr, "libinferbit_amd: %s failed: %s\n", who, e ? e : "unknown error");
    ibh_set_error("%s failed: %s", who, e ? e : "unknown error");
    for (size_t i = 0; i < n; i++) out[i] = __builtin_nanf("");
}

// Stage host operands, run `launch(device pointers...)`, copy `out` back.
struct Staged {
    uint8_t* base = nullptr;
    size_t off = 0;
    uint8_t* put(const void* h, size_t n, hipStream_t st) {
        uint8_t* d = base + off;
        off += al256(n);
        if (h && n) (void)hipMemcpyAsync(d, h, n, hipMemcpyHostToDevice, st);
        return d;
    }
};

int tab_weight(const void* w, size_t wbytes, Staged& S, hipStream_t st, const uint8_t** dw) {
    *dw = lookup(w, wbytes);
    if (!*dw) *dw = S.put(w, wbytes, st);
    return IBH_OK;
}

size_t wbytes_of(int bits, int M, int N) {
    return (size_t)M * (bits == 8 ? (size_t)N : (bits == 4 ? (size_t)N / 2 : (size_t)N / 4));
}

void tab_matmul(float* out, const void* w, const float* sc, const float* x, int M, int N, int bits) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    hipStream_t st = ibh_resolve_stream(nullptr);
    const size_t wb = wbytes_of(bits, M, N);
    const bool resident = lookup(w, wb) != nullptr;
    Staged S;
    S.base = workspace(al256(4 * (size_t)M) * 2 + al256(4 * (size_t)N) + (resident ? 0 : al256(wb)));
    if (!S.base) { ibh_set_error("out of device memory"); fail(out, M, "matmul table entry"); return; }
    const uint8_t* dw;
    tab_weight(w, wb, S, st, &dw);
    float* dsc = (float*)S.put(sc, 4 * (size_t)M, st);
    float* dx = (float*)S.put(x, 4 * (size_t)N, st);
    float* dout = (float*)S.put(nullptr, 4 * (size_t)M, st);
    // The x86 table's operation order (matvec_exact), so a reference build
    // that swaps its table keeps its logits bit for bit; rows longer than the
    // exact kernel's LDS tile (N > 15360 at 8/4 bits) take the tolerance kernel.
    int rc = ibh_launch_matvec_exact(dout, dw, dsc, IBH_SCALE_F32, dx, M, N, bits, nullptr, st);
    if (rc == IBH_ERROR_PARAM) {
        (void)ibh_last_error();
        rc = ibh_matmul(dout, dw, dsc, IBH_SCALE_F32, dx, M, N, bits, st);
    }
    if (rc == IBH_OK && hipMemcpyAsync(out, dout, 4 * (size_t)M, hipMemcpyDeviceToHost, st) == hipSuccess &&
        hipStreamSynchronize(st) == hipSuccess)
        return;
    if (rc == IBH_OK) ibh_set_error("device copy failed");
    fail(out, M, "matmul table entry");
}

void hip_int8(float* o, const void* w, const float* s, const float* x, int M, int N) { tab_matmul(o, w, s, x, M, N, 8); }
void hip_int4(float* o, const void* w, const float* s, const float* x, int M, int N) { tab_matmul(o, w, s, x, M, N, 4); }
void hip_int2(float* o, const void* w, const float* s, const float* x, int M, int N) { tab_matmul(o, w, s, x, M, N, 2); }

void tab_w4a8(float* out, const void* w, const float* sw, const int8_t* qx, const float* sa, int M, int N,
              int B, int M_stride, bool fused) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    hipStream_t st = ibh_resolve_stream(nullptr);
    const size_t wb = (size_t)M * (N / 2);
    const bool resident = lookup(w, wb) != nullptr;
    const int G = (N + 127) / 128;
    // The output keeps rows this slice does not own (M_stride > M): copy the
    // whole strided region in and out so they are preserved.
    const size_t ob = 4 * ((size_t)(B - 1) * M_stride + M);
    Staged S;
    S.base = workspace(al256(4 * (size_t)M) + al256((size_t)B * N) + al256(4 * (size_t)B * G) + al256(ob) +
                       (resident ? 0 : al256(wb)));
    if (!S.base) { ibh_set_error("out of device memory"); fail(out, ob / 4, "w4a8 table entry"); return; }
    const uint8_t* dw;
    tab_weight(w, wb, S, st, &dw);
    float* dsw = (float*)S.put(sw, 4 * (size_t)M, st);
    int8_t* dq = (int8_t*)S.put(qx, (size_t)B * N, st);
    float* dsa = (float*)S.put(sa, 4 * (size_t)B * G, st);
    float* dout = (float*)S.put(out, ob, st);
    int rc = fused ? ibh_matmul_w4a8(dout, dw, dsw, IBH_SCALE_F32, dq, dsa, M, N, st)
                   : ibh_matmul_w4a8_batch(dout, dw, dsw, IBH_SCALE_F32, dq, dsa, M, N, B,
                                                             M_stride, st);
    if (rc == IBH_OK && hipMemcpyAsync(out, dout, ob, hipMemcpyDeviceToHost, st) == hipSuccess &&
        hipStreamSynchronize(st) == hipSuccess)
        return;
    if (rc == IBH_OK) ibh_set_error("device copy failed");
    fail(out, ob / 4, "w4a8 table entry");
}

// The single-row W4A8 entry is the x86 AVX2 kernel (fused fold); the batched
// entry is the scalar kernel (unfused fold), also at B == 1.
void hip_w4a8(float* out, const void* w, const float* sw, const int8_t* qx, const float* sa, int M, int N) {
    tab_w4a8(out, w, sw, qx, sa, M, N, 1, M, true);
}
void hip_w4a8_batch(float* out, const void* w, const float* sw, const int8_t* qx, const float* sa, int M,
                    int N, int B, int M_stride) {
    tab_w4a8(out, w, sw, qx, sa, M, N, B, M_stride, false);
}

void hip_int8_batch(float* out, const void* w, const float* sw, const float* x, int M, int N, int B,
                    int M_stride) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    hipStream_t st = ibh_resolve_stream(nullptr);
    const size_t wb = (size_t)M * N;
    const bool resident = lookup(w, wb) != nullptr;
    const size_t ob = 4 * ((size_t)(B - 1) * M_stride + M);
    Staged S;
    S.base = workspace(al256(4 * (size_t)M) + al256(4 * (size_t)B * N) + al256(ob) + (resident ? 0 : al256(wb)));
    if (!S.base) { ibh_set_error("out of device memory"); fail(out, ob / 4, "int8 batch table entry"); return; }
    const uint8_t* dw;
    tab_weight(w, wb, S, st, &dw);
    float* dsw = (float*)S.put(sw, 4 * (size_t)M, st);
    float* dx = (float*)S.put(x, 4 * (size_t)B * N, st);
    float* dout = (float*)S.put(out, ob, st);
    // scalar.c:70-84 (the x86 table's batched INT8 entry): serial sums
    const ibh::MatDesc d{dout, dw, dsw, M};
    int rc = ibh_launch_int8_batch_exact(&d, 1, IBH_SCALE_F32, dx, N, B, false, st, M_stride);
    if (rc == IBH_OK && hipMemcpyAsync(out, dout, ob, hipMemcpyDeviceToHost, st) == hipSuccess &&
        hipStreamSynchronize(st) == hipSuccess)
        return;
    if (rc == IBH_OK) ibh_set_error("device copy failed");
    fail(out, ob / 4, "int8 batch table entry");
}
}  // namespace

extern "C" void ib_init_kernels_hip(ibh_kernels* k) {
    if (!k) return;
    k->matmul_int8 = hip_int8;
    k->matmul_int4 = hip_int4;
    k->matmul_int2 = hip_int2;
    k->matmul_w4a8 = hip_w4a8;
    k->matmul_w4a8_batch = hip_w4a8_batch;
    k->matmul_int8_batch = hip_int8_batch;
}

extern "C" int ibh_register_host_weights(const void* host_base, size_t bytes, void** dev_base) {
    if (!host_base || !bytes) {
        ibh_set_error("ibh_register_host_weights: empty region");
        return IBH_ERROR_PARAM;
    }
    std::lock_guard<std::mutex> lk(g_tab_mu);
    for (const Region& r : g_regions)
        if (r.host == host_base && r.bytes == bytes) {
            if (dev_base) *dev_base = r.dev;
            return IBH_OK;
        }
    uint8_t* d = nullptr;
    if (hipMalloc((void**)&d, bytes) != hipSuccess) {
        ibh_set_error("ibh_register_host_weights: out of device memory (%zu bytes)", bytes);
        return IBH_ERROR_MEMORY;
    }
    if (hipMemcpy(d, host_base, bytes, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d);
        ibh_set_error("ibh_register_host_weights: upload failed");
        return IBH_ERROR_INTERNAL;
    }
    g_regions.push_back({(const uint8_t*)host_base, bytes, d});
    if (dev_base) *dev_base = d;
    return IBH_OK;
}

extern "C" void ibh_unregister_host_weights(const void* host_base) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    for (size_t i = 0; i < g_regions.size(); i++)
        if (g_regions[i].host == host_base) {
            (void)hipFree(g_regions[i].dev);
            g_regions.erase(g_regions.begin() + (long)i);
            return;
        }
}

// ── attention hook on host pointers (forward.c's head loop) ─────────────────
// The reference keeps its KV cache in host memory (ib_kv_cache,
// src/inferbit_internal.h:101-109) and writes it with kv_cache_write
// (src/forward.c:352-413) right before the head loop at every position.  The
// hook keeps a device mirror per host cache: rows the device lacks (positions
// from its length up to pos) are uploaded as the host stored them, then every
// head runs on the device in the x86 order (attn_scores_exact +
// attn_out_exact), so the head outputs are the reference's bit for bit.  A
// rewind (inferbit_kv_truncate / _clear) needs no call: the next position the
// host writes is below the mirror's length, which then drops to it.
namespace {
struct KvMirror {
    const void* key;
    int capacity, kv_bits, n_kv, head_dim;
    uint8_t* k;
    uint8_t* v;
    float* ks;
    float* vs;
    int len;
};
std::vector<KvMirror> g_kv;

size_t kv_row_bytes(int bits, int kv_dim) {
    return bits >= 16 ? 4 * (size_t)kv_dim : bits == 8 ? (size_t)kv_dim : (size_t)(kv_dim + 1) / 2;
}

void kv_mirror_free(KvMirror& mm) {
    (void)hipFree(mm.k);
    (void)hipFree(mm.v);
    (void)hipFree(mm.ks);
    (void)hipFree(mm.vs);
    mm.k = mm.v = nullptr;
    mm.ks = mm.vs = nullptr;
}
}  // namespace

size_t ibh_attn_exact_scratch(int n_heads, int max_pos);   // ibh_exact.hip
int ibh_launch_attn_exact(float* out, const float* q, const void* kdata, const void* vdata, const float* ks,
                          const float* vs, const int* dpos, int max_pos, int n_heads, int n_kv, int hd, int kv_bits,
                          float* att, hipStream_t st);

extern "C" int ibh_host_attn(const void* cache, const void* kdata, const void* vdata, const float* kscales,
                             const float* vscales, int capacity, int pos, int kv_bits, const float* q, float* out,
                             int n_heads, int n_kv, int head_dim) {
    if (!cache || !kdata || !vdata || !q || !out || pos < 0 || pos >= capacity || n_kv <= 0 || n_heads % n_kv ||
        (kv_bits <= 8 && (!kscales || !vscales))) {
        ibh_set_error("ibh_host_attn: invalid arguments (pos %d, capacity %d)", pos, capacity);
        return IBH_ERROR_PARAM;
    }
    std::lock_guard<std::mutex> lk(g_tab_mu);
    hipStream_t st = ibh_resolve_stream(nullptr);
    const int kv_dim = n_kv * head_dim;
    const size_t rbytes = kv_row_bytes(kv_bits, kv_dim);
    KvMirror* mm = nullptr;
    for (KvMirror& e : g_kv)
        if (e.key == cache) mm = &e;
    if (mm && (mm->capacity != capacity || mm->kv_bits != kv_bits || mm->n_kv != n_kv || mm->head_dim != head_dim)) {
        kv_mirror_free(*mm);                       // the host cache was re-shaped (a dynamic cache grew)
        mm->len = 0;
    }
    if (!mm) {
        g_kv.push_back({cache, capacity, kv_bits, n_kv, head_dim, nullptr, nullptr, nullptr, nullptr, 0});
        mm = &g_kv.back();
    }
    if (!mm->k) {
        mm->capacity = capacity;
        mm->kv_bits = kv_bits;
        mm->n_kv = n_kv;
        mm->head_dim = head_dim;
        const size_t sb = kv_bits <= 8 ? 4 * (size_t)capacity * n_kv : 0;
        if (hipMalloc((void**)&mm->k, rbytes * capacity) != hipSuccess ||
            hipMalloc((void**)&mm->v, rbytes * capacity) != hipSuccess ||
            (sb && (hipMalloc((void**)&mm->ks, sb) != hipSuccess || hipMalloc((void**)&mm->vs, sb) != hipSuccess))) {
            kv_mirror_free(*mm);
            ibh_set_error("ibh_host_attn: out of device memory for the KV mirror");
            return IBH_ERROR_MEMORY;
        }
        mm->len = 0;
    }
    // rows [len, pos] as the host stored them (a rewound position re-uploads)
    const int from = std::min(mm->len, pos);
    const size_t nrow = (size_t)(pos + 1 - from);
    IBH_HIP(hipMemcpyAsync(mm->k + from * rbytes, (const uint8_t*)kdata + from * rbytes, nrow * rbytes,
                           hipMemcpyHostToDevice, st), "ibh_host_attn: K upload");
    IBH_HIP(hipMemcpyAsync(mm->v + from * rbytes, (const uint8_t*)vdata + from * rbytes, nrow * rbytes,
                           hipMemcpyHostToDevice, st), "ibh_host_attn: V upload");
    if (kv_bits <= 8) {
        const size_t sr = 4 * (size_t)n_kv;
        IBH_HIP(hipMemcpyAsync((uint8_t*)mm->ks + from * sr, (const uint8_t*)kscales + from * sr, nrow * sr,
                               hipMemcpyHostToDevice, st), "ibh_host_attn: K scales upload");
        IBH_HIP(hipMemcpyAsync((uint8_t*)mm->vs + from * sr, (const uint8_t*)vscales + from * sr, nrow * sr,
                               hipMemcpyHostToDevice, st), "ibh_host_attn: V scales upload");
    }
    mm->len = pos + 1;
    const size_t qb = 4 * (size_t)n_heads * head_dim;
    Staged S;
    S.base = workspace(al256(qb) * 2 + al256(16) + al256(ibh_attn_exact_scratch(n_heads, pos)));
    if (!S.base) {
        ibh_set_error("ibh_host_attn: out of device memory");
        return IBH_ERROR_MEMORY;
    }
    float* dq = (float*)S.put(q, qb, st);
    int* dpos = (int*)S.put(&pos, sizeof(int), st);
    float* dout = (float*)S.put(nullptr, qb, st);
    float* att = (float*)S.put(nullptr, ibh_attn_exact_scratch(n_heads, pos), st);
    int rc = ibh_launch_attn_exact(dout, dq, mm->k, mm->v, mm->ks, mm->vs, dpos, pos, n_heads, n_kv, head_dim,
                                   kv_bits, att, st);
    if (rc != IBH_OK) return rc;
    IBH_HIP(hipMemcpyAsync(out, dout, qb, hipMemcpyDeviceToHost, st), "ibh_host_attn: output copy");
    IBH_HIP(hipStreamSynchronize(st), "ibh_host_attn: synchronize");
    return IBH_OK;
}

extern "C" void ibh_host_kv_release(const void* cache) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    for (size_t i = 0; i < g_kv.size(); i++)
        if (g_kv[i].key == cache) {
            kv_mirror_free(g_kv[i]);
            g_kv.erase(g_kv.begin() + (long)i);
            return;
        }
}

// ── PQ matvec on a host ib_pq_tensor (ib_pq_matmul_fp32's twin) ─────────────
// The reference's PQ entries take an ib_pq_tensor whose arrays are host
// memory (an arena from the fread loaders or the file mmap,
// src/pq_decode.c:391-555, 685-744).  The first call on a tensor builds its
// device description: arrays inside a region registered with
// ibh_register_host_weights map to that device copy, the others are uploaded
// once into an allocation of the entry; inner_cols and a stamped PQ workspace
// come with it.  Entries are keyed by the tensor's array addresses and
// checked against a fingerprint of its shape and of the first and last bytes
// of every array, so a tensor freed and another loaded at the same addresses
// is uploaded anew; ibh_pq_host_release (from ib_pq_free) frees an entry.
namespace {
struct PqHostEntry {
    const void* key;          // codebook_l1_l
    const void* key2;         // indices_l1_l
    uint64_t fp;
    uint8_t* blob;            // uploaded arrays + inner_cols
    void* ws;                 // stamped PQ workspace
    size_t ws_bytes;
    ibh_pq_tensor d;          // device description
};
std::vector<PqHostEntry> g_pqh;

struct PqArr {
    const void* h;
    size_t n;
};

// The reference tensor's arrays with their byte sizes (src/pq_decode.c:470-489).
int pq_host_arrays(const ibh_ref_pq_tensor* t, PqArr* a) {
    const int K2 = t->K_l2 > 0 ? t->K_l2 : t->K;
    const int hf = t->G / 2;
    const size_t l2s = K2 == 16 ? (size_t)(t->C + 1) / 2 : (size_t)t->C * (t->l2_idx_bytes == 2 ? 2 : 1);
    const size_t M = (size_t)t->M, no = (size_t)(t->n_outlier > 0 ? t->n_outlier : 0);
    const bool two = t->n_levels == 2;
    a[0] = {t->codebook_l1_l, (size_t)t->K * hf * 2};
    a[1] = {t->codebook_l1_r, (size_t)t->K * hf * 2};
    a[2] = {two ? t->codebook_l2_l : nullptr, two ? (size_t)K2 * hf * 2 : 0};
    a[3] = {two ? t->codebook_l2_r : nullptr, two ? (size_t)K2 * hf * 2 : 0};
    a[4] = {t->indices_l1_l, M * t->C};
    a[5] = {t->indices_l1_r, M * t->C};
    a[6] = {two ? t->indices_l2_l : nullptr, two ? M * l2s : 0};
    a[7] = {two ? t->indices_l2_r : nullptr, two ? M * l2s : 0};
    a[8] = {t->row_scale, M * 2};
    a[9] = {no ? t->outlier_cols : nullptr, no * 4};
    a[10] = {no ? t->outlier_sidecar : nullptr, M * no};
    a[11] = {no ? t->outlier_scale : nullptr, no * 2};
    return 12;
}

uint64_t fnv(uint64_t h, const void* p, size_t n) {
    const uint8_t* b = (const uint8_t*)p;
    for (size_t i = 0; i < n; i++) h = (h ^ b[i]) * 0x100000001b3ull;
    return h;
}

uint64_t pq_host_fp(const ibh_ref_pq_tensor* t, const PqArr* a, int na) {
    const int dims[] = {t->M, t->N, t->G, t->K, t->K_l2, t->n_levels, t->n_outlier, t->format, t->C, t->l2_idx_bytes};
    uint64_t h = fnv(0xcbf29ce484222325ull, dims, sizeof(dims));
    for (int i = 0; i < na; i++) {
        if (!a[i].h) continue;
        const size_t k = std::min<size_t>(a[i].n, 512);
        h = fnv(h, a[i].h, k);
        h = fnv(h, (const uint8_t*)a[i].h + a[i].n - k, k);
    }
    return h;
}

void pq_host_free(PqHostEntry& e) {
    (void)hipFree(e.blob);
    (void)hipFree(e.ws);
    e.blob = nullptr;
    e.ws = nullptr;
}

int pq_host_entry(const ibh_ref_pq_tensor* t, PqHostEntry** out) {
    PqArr a[12];
    const int na = pq_host_arrays(t, a);
    const uint64_t fp = pq_host_fp(t, a, na);
    for (PqHostEntry& e : g_pqh)
        if (e.key == t->codebook_l1_l && e.key2 == t->indices_l1_l) {
            if (e.fp == fp) {
                *out = &e;
                return IBH_OK;
            }
            pq_host_free(e);          // another tensor at the same addresses
            e = g_pqh.back();
            g_pqh.pop_back();
            break;
        }
    // arrays not resident in a registered region go to one allocation
    const uint8_t* dev[12];
    size_t up = 0;
    for (int i = 0; i < na; i++) {
        dev[i] = a[i].h ? lookup(a[i].h, a[i].n) : nullptr;
        if (a[i].h && !dev[i]) up += al256(a[i].n);
    }
    const int ninner = t->N - t->n_outlier;
    std::vector<int32_t> inner;
    if (t->n_outlier > 0) {
        std::vector<char> is_out((size_t)t->N, 0);
        for (int j = 0; j < t->n_outlier; j++) {
            const int c = t->outlier_cols[j];
            if (c < 0 || c >= t->N) {
                ibh_set_error("ibh_pq_matmul_fp32_host: outlier column %d outside [0, %d)", c, t->N);
                return IBH_ERROR_PARAM;
            }
            is_out[(size_t)c] = 1;
        }
        for (int c = 0; c < t->N; c++)
            if (!is_out[(size_t)c]) inner.push_back(c);
        if ((int)inner.size() != ninner) {
            ibh_set_error("ibh_pq_matmul_fp32_host: repeated outlier columns");
            return IBH_ERROR_PARAM;
        }
        up += al256(inner.size() * 4);
    }
    PqHostEntry e{};
    e.key = t->codebook_l1_l;
    e.key2 = t->indices_l1_l;
    e.fp = fp;
    if (up && hipMalloc((void**)&e.blob, up) != hipSuccess) {
        ibh_set_error("ibh_pq_matmul_fp32_host: out of device memory (%zu bytes)", up);
        return IBH_ERROR_MEMORY;
    }
    size_t off = 0;
    for (int i = 0; i < na; i++) {
        if (!a[i].h || dev[i]) continue;
        if (hipMemcpy(e.blob + off, a[i].h, a[i].n, hipMemcpyHostToDevice) != hipSuccess) {
            pq_host_free(e);
            ibh_set_error("ibh_pq_matmul_fp32_host: upload failed");
            return IBH_ERROR_INTERNAL;
        }
        dev[i] = e.blob + off;
        off += al256(a[i].n);
    }
    const int32_t* dinner = nullptr;
    if (!inner.empty()) {
        if (hipMemcpy(e.blob + off, inner.data(), inner.size() * 4, hipMemcpyHostToDevice) != hipSuccess) {
            pq_host_free(e);
            ibh_set_error("ibh_pq_matmul_fp32_host: upload failed");
            return IBH_ERROR_INTERNAL;
        }
        dinner = (const int32_t*)(e.blob + off);
    }
    ibh_pq_tensor& d = e.d;
    d.M = t->M; d.N = t->N; d.G = t->G; d.K = t->K; d.K_l2 = t->K_l2; d.n_levels = t->n_levels;
    d.n_outlier = t->n_outlier; d.C = t->C; d.l2_idx_bytes = t->l2_idx_bytes; d.format = t->format;
    d.codebook_l1_l = (const uint16_t*)dev[0]; d.codebook_l1_r = (const uint16_t*)dev[1];
    d.codebook_l2_l = (const uint16_t*)dev[2]; d.codebook_l2_r = (const uint16_t*)dev[3];
    d.indices_l1_l = dev[4]; d.indices_l1_r = dev[5]; d.indices_l2_l = dev[6]; d.indices_l2_r = dev[7];
    d.row_scale = (const uint16_t*)dev[8];
    d.outlier_cols = (const int32_t*)dev[9]; d.outlier_sidecar = (const int8_t*)dev[10];
    d.outlier_scale = (const uint16_t*)dev[11];
    d.inner_cols = dinner;
    e.ws_bytes = ibh_pq_workspace_bytes(&d);
    if (!e.ws_bytes) {
        pq_host_free(e);
        ibh_set_error("ibh_pq_matmul_fp32_host: unsupported tensor geometry");
        return IBH_ERROR_PARAM;
    }
    if (hipMalloc(&e.ws, e.ws_bytes) != hipSuccess) {
        pq_host_free(e);
        ibh_set_error("ibh_pq_matmul_fp32_host: out of device memory for the workspace");
        return IBH_ERROR_MEMORY;
    }
    const int rc = ibh_pq_workspace_init(e.ws, e.ws_bytes, nullptr);
    if (rc != IBH_OK) {
        pq_host_free(e);
        return rc;
    }
    g_pqh.push_back(e);
    *out = &g_pqh.back();
    return IBH_OK;
}
}  // namespace

// policy: NULL = ib_pq_matmul_fp32 (matmul_impl), else the session's dispatch
static int pq_host_run(const ibh_ref_pq_tensor* t, const ibh_pq_policy* policy, const float* x, float* out,
                       const char* who) {
    if (!t || !x || !out || t->M <= 0 || t->N <= 0 || t->C <= 0 || t->G <= 0 || t->K <= 0 || !t->codebook_l1_l ||
        !t->indices_l1_l) {
        ibh_set_error("%s: invalid arguments", who);
        return -1;
    }
    std::lock_guard<std::mutex> lk(g_tab_mu);
    PqHostEntry* e = nullptr;
    if (pq_host_entry(t, &e) != IBH_OK) return -1;
    hipStream_t st = ibh_resolve_stream(nullptr);
    Staged S;
    S.base = workspace(al256(4 * (size_t)t->N) + al256(4 * (size_t)t->M));
    if (!S.base) {
        ibh_set_error("%s: out of device memory", who);
        return -1;
    }
    float* dx = (float*)S.put(x, 4 * (size_t)t->N, st);
    float* dout = (float*)S.put(nullptr, 4 * (size_t)t->M, st);
    const int rc = policy ? ibh_pq_matmul_policy(&e->d, dx, dout, policy, e->ws, e->ws_bytes, st)
                          : ibh_pq_matmul(&e->d, dx, dout, e->ws, e->ws_bytes, st);
    if (rc != IBH_OK) return -1;
    if (hipMemcpyAsync(out, dout, 4 * (size_t)t->M, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
        ibh_set_error("%s: device copy failed", who);
        return -1;
    }
    return 0;
}

extern "C" int ibh_pq_matmul_fp32_host(const ibh_ref_pq_tensor* t, const float* x, float* out) {
    return pq_host_run(t, nullptr, x, out, "ibh_pq_matmul_fp32_host");
}

extern "C" int ibh_pq_matmul_policy_host(const ibh_ref_pq_tensor* t, const ibh_pq_policy* p, const float* x,
                                         float* out) {
    if (!p) {
        ibh_set_error("ibh_pq_matmul_policy_host: null policy");
        return -1;
    }
    return pq_host_run(t, p, x, out, "ibh_pq_matmul_policy_host");
}

extern "C" void ibh_pq_host_release(const ibh_ref_pq_tensor* t) {
    if (!t) return;
    std::lock_guard<std::mutex> lk(g_tab_mu);
    for (size_t i = 0; i < g_pqh.size(); i++)
        if (g_pqh[i].key == t->codebook_l1_l && g_pqh[i].key2 == t->indices_l1_l) {
            pq_host_free(g_pqh[i]);
            g_pqh.erase(g_pqh.begin() + (long)i);
            return;
        }
}

// ── INT4 group-scale matvec on a host ib_int4_tensor (the session's branch) ──
// The PQ session's INT4 tensors (struct ib_int4_tensor, src/pq_decode.c:
// 3474-3482) point into the session's mmap or arena.  As for PQ tensors, the
// first call builds a device copy (registered regions used in place), keyed
// by the q array and checked by a fingerprint; x goes in raw (the AWQ
// pre-scale and the outliers run on the device).
namespace {
struct I4HostEntry {
    const void* key;
    uint64_t fp;
    uint8_t* blob;
    void* ws;
    size_t ws_bytes;
    ibh_int4g_tensor d;       // inv_act: the device copy of ia_host (or null)
    const float* ia_host;     // the host AWQ vector last uploaded
    uint64_t fp_ia;
    float* ia_dev;
};
std::vector<I4HostEntry> g_i4h;

float act_sparse_rel_env() {
    // read once, as build_skip_mask does (src/pq_decode.c:3855-3863)
    static float rel = -2.0f;
    if (rel < -1.0f) {
        const char* e = getenv("IB_ACT_SPARSE_REL");
        rel = (e && atof(e) >= 0.0) ? (float)atof(e) : 0.0f;
    }
    return rel;
}

void i4_host_free(I4HostEntry& e) {
    (void)hipFree(e.blob);
    (void)hipFree(e.ws);
    (void)hipFree(e.ia_dev);
    e.blob = nullptr;
    e.ws = nullptr;
    e.ia_dev = nullptr;
}

// The call's AWQ vector on the device (re-uploaded when the host pointer or
// its first and last bytes change); d.inv_act follows the call.
int i4_host_act(I4HostEntry& e, const ibh_ref_int4_tensor* t) {
    if (!t->inv_act) {
        e.d.inv_act = nullptr;
        return IBH_OK;
    }
    const size_t n = (size_t)t->N * 4, k = std::min<size_t>(n, 512);
    const uint64_t fp = fnv(fnv(0xcbf29ce484222325ull, t->inv_act, k), (const uint8_t*)t->inv_act + n - k, k);
    const uint8_t* res = lookup(t->inv_act, n);
    if (res) {
        e.d.inv_act = (const float*)res;
        return IBH_OK;
    }
    if (!e.ia_dev || e.ia_host != t->inv_act || e.fp_ia != fp) {
        if (!e.ia_dev && hipMalloc((void**)&e.ia_dev, n) != hipSuccess) {
            ibh_set_error("ibh_int4g_matmul_host: out of device memory");
            return IBH_ERROR_MEMORY;
        }
        if (hipMemcpy(e.ia_dev, t->inv_act, n, hipMemcpyHostToDevice) != hipSuccess) {
            ibh_set_error("ibh_int4g_matmul_host: upload failed");
            return IBH_ERROR_INTERNAL;
        }
        e.ia_host = t->inv_act;
        e.fp_ia = fp;
    }
    e.d.inv_act = e.ia_dev;
    return IBH_OK;
}

int i4_host_entry(const ibh_ref_int4_tensor* t, I4HostEntry** out) {
    // the AWQ vector is not part of the entry's identity: a caller may pass
    // the tensor with and without it (the session applies it only when the
    // row fits its scratch, src/pq_decode.c:4444); it is uploaded on demand
    const size_t M = (size_t)t->M, N = (size_t)t->N, ko = (size_t)(t->K_out > 0 ? t->K_out : 0);
    const PqArr a[5] = {{t->q, M * (N / 2)},
                        {t->s, M * (N / (size_t)t->G) * 2},
                        {nullptr, 0},
                        {ko ? t->outl_idx : nullptr, M * ko * 2},
                        {ko ? t->outl_val : nullptr, M * ko * 2}};
    const int dims[] = {t->M, t->N, t->G, t->K_out};
    uint64_t fp = fnv(0xcbf29ce484222325ull, dims, sizeof(dims));
    for (const PqArr& r : a) {
        if (!r.h || !r.n) continue;
        const size_t k = std::min<size_t>(r.n, 512);
        fp = fnv(fnv(fp, r.h, k), (const uint8_t*)r.h + r.n - k, k);
    }
    for (I4HostEntry& e : g_i4h)
        if (e.key == t->q) {
            if (e.fp == fp) {
                *out = &e;
                return i4_host_act(e, t);
            }
            i4_host_free(e);
            e = g_i4h.back();
            g_i4h.pop_back();
            break;
        }
    const uint8_t* dev[5];
    size_t up = 0;
    for (int i = 0; i < 5; i++) {
        dev[i] = a[i].h && a[i].n ? lookup(a[i].h, a[i].n) : nullptr;
        if (a[i].h && a[i].n && !dev[i]) up += al256(a[i].n);
    }
    I4HostEntry e{};
    e.key = t->q;
    e.fp = fp;
    if (up && hipMalloc((void**)&e.blob, up) != hipSuccess) {
        ibh_set_error("ibh_int4g_matmul_host: out of device memory (%zu bytes)", up);
        return IBH_ERROR_MEMORY;
    }
    size_t off = 0;
    for (int i = 0; i < 5; i++) {
        if (!a[i].h || !a[i].n || dev[i]) continue;
        if (hipMemcpy(e.blob + off, a[i].h, a[i].n, hipMemcpyHostToDevice) != hipSuccess) {
            i4_host_free(e);
            ibh_set_error("ibh_int4g_matmul_host: upload failed");
            return IBH_ERROR_INTERNAL;
        }
        dev[i] = e.blob + off;
        off += al256(a[i].n);
    }
    e.d.q = dev[0];
    e.d.s = (const uint16_t*)dev[1];
    e.d.inv_act = nullptr;
    e.d.outl_idx = (const uint16_t*)dev[3];
    e.d.outl_val = (const uint16_t*)dev[4];
    e.d.M = t->M; e.d.N = t->N; e.d.G = t->G; e.d.K_out = (int)ko;
    e.ws_bytes = ibh_int4g_workspace_bytes(&e.d);
    if (e.ws_bytes && hipMalloc(&e.ws, e.ws_bytes) != hipSuccess) {
        i4_host_free(e);
        ibh_set_error("ibh_int4g_matmul_host: out of device memory for the workspace");
        return IBH_ERROR_MEMORY;
    }
    g_i4h.push_back(e);
    *out = &g_i4h.back();
    return i4_host_act(**out, t);
}
}  // namespace

extern "C" int ibh_int4g_matmul_host(const ibh_ref_int4_tensor* t, const float* x, float* out) {
    if (!t || !x || !out || !t->q || !t->s || t->M <= 0 || t->N <= 0 || t->G <= 0 || t->N % t->G ||
        (t->K_out > 0 && (!t->outl_idx || !t->outl_val))) {
        ibh_set_error("ibh_int4g_matmul_host: invalid arguments");
        return -1;
    }
    std::lock_guard<std::mutex> lk(g_tab_mu);
    I4HostEntry* e = nullptr;
    if (i4_host_entry(t, &e) != IBH_OK) return -1;
    hipStream_t st = ibh_resolve_stream(nullptr);
    Staged S;
    S.base = workspace(al256(4 * (size_t)t->N) + al256(4 * (size_t)t->M));
    if (!S.base) {
        ibh_set_error("ibh_int4g_matmul_host: out of device memory");
        return -1;
    }
    float* dx = (float*)S.put(x, 4 * (size_t)t->N, st);
    float* dout = (float*)S.put(nullptr, 4 * (size_t)t->M, st);
    if (ibh_int4g_matmul(&e->d, dx, dout, act_sparse_rel_env(), e->ws, e->ws_bytes, st) != IBH_OK) return -1;
    if (hipMemcpyAsync(out, dout, 4 * (size_t)t->M, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
        ibh_set_error("ibh_int4g_matmul_host: device copy failed");
        return -1;
    }
    return 0;
}

extern "C" void ibh_int4g_host_release(const ibh_ref_int4_tensor* t) {
    if (!t) return;
    std::lock_guard<std::mutex> lk(g_tab_mu);
    for (size_t i = 0; i < g_i4h.size(); i++)
        if (g_i4h[i].key == t->q) {
            i4_host_free(g_i4h[i]);
            g_i4h.erase(g_i4h.begin() + (long)i);
            return;
        }
}
