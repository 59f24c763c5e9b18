// Engine<T>: context set-up, caller-buffer staging and the batched per-field
// transforms of the shtns.f90 API (spectogrd, grdtospec, getuv,
// getvrtdivspec, getgrad) on the device.
#include <cstring>
#include <mutex>

#include "engine.h"

namespace gfsdc {

// ---------------------------------------------------------------------------
// Scratch of the no-allocation synthesis (gfsdc_spectogrd_noalloc): one
// file-scope device array per GPU, held until the process ends, holding the
// synthesis descriptors, the extended spectral columns and the Fourier buffer
// that gfsdc_spectogrd keeps in the context's lazily allocated work buffers.
// Its device address is looked up once per device at context creation, with
// that device current; host code uses only that address, never the symbol.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[MAX_DEVICES] = {};

static int scratch_setup(int device) {
    if (device < 0 || device >= MAX_DEVICES) {
        set_error("device ordinal out of range for the no-allocation scratch");
        return GFSDC_EINVAL;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return 0;
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        return GFSDC_EHIP;
    }
    g_scratch_ptr[device] = ptr;
    return 0;
}

static void *scratch_ptr(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return (device >= 0 && device < MAX_DEVICES) ? g_scratch_ptr[device] : nullptr;
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

template <typename Tin, typename Tout>
__global__ void k_convert(const Tin *__restrict__ a, Tout *__restrict__ b, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) b[i] = (Tout)a[i];
}

template <typename Tin, typename Tout> static void convert(const Tin *a, Tout *b, size_t n, hipStream_t s) {
    if (n == 0) return;
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL((k_convert<Tin, Tout>), dim3((unsigned)blocks), dim3(256), 0, s, a, b, n);
}

template <typename T> int Engine<T>::init(const gfsdc_cfg &c) {
    cfg = c;
    if (c.nlev > 0) {
        if (!c.ak || !c.bk) {
            set_error("cfg.ak / cfg.bk required when nlev > 0");
            return GFSDC_EINVAL;
        }
        ak.assign(c.ak, c.ak + c.nlev + 1);
        bk.assign(c.bk, c.bk + c.nlev + 1);
    }
    cfg.ak = ak.empty() ? nullptr : ak.data();
    cfg.bk = bk.empty() ? nullptr : bk.data();
    if (cfg.nmem <= 0) cfg.nmem = 1;
    GFSDC_CHECK(hipSetDevice(c.device));
    hipDeviceProp_t prop;
    GFSDC_CHECK(hipGetDeviceProperties(&prop, c.device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        set_error(std::string("gfsdc is built for gfx950; device is ") + prop.gcnArchName);
        return GFSDC_ENODEV;
    }
    GFSDC_CHECK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    int rc = scratch_setup(c.device);
    if (rc) return rc;
    rc = plan_create(plan, c.nlon, c.nlat, c.ntrunc, stream);
    plan.leg_bf16x3 = (c.precision == GFSDC_BF16X3) ? 1 : 0;
    if (rc) return rc;
    if (c.nlev > 0) {
        rc = dyn_init();
        if (rc) return rc;
    }
    return 0;
}

template <typename T> void Engine<T>::destroy() {
    if (stream) (void)hipStreamSynchronize(stream);
    dyn_destroy();
    work_free(work);
    plan_destroy(plan);
    for (int i = 0; i < 4; i++)
        if (stage[i]) (void)hipFree(stage[i]);
    if (pinned) (void)hipHostFree(pinned);
    if (d_sdesc) (void)hipFree(d_sdesc);
    if (d_rflag) (void)hipFree(d_rflag);
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
}

template <typename T> int Engine<T>::ensure_stage(int i, size_t bytes) {
    if (bytes <= stage_sz[i]) return 0;
    GFSDC_CHECK(hipStreamSynchronize(stream));
    if (stage[i]) GFSDC_CHECK(hipFree(stage[i]));
    stage[i] = nullptr;
    stage_sz[i] = 0;
    GFSDC_CHECK(hipMalloc(&stage[i], bytes));
    stage_sz[i] = bytes;
    return 0;
}

template <typename T>
int Engine<T>::upload_descs(const std::vector<SynthDesc> &sd, const std::vector<unsigned char> &rf) {
    const int need = (int)std::max(sd.size(), rf.size());
    if (need > desc_cap) {
        if (d_sdesc) GFSDC_CHECK(hipFree(d_sdesc));
        if (d_rflag) GFSDC_CHECK(hipFree(d_rflag));
        GFSDC_CHECK(hipMalloc((void **)&d_sdesc, sizeof(SynthDesc) * need));
        GFSDC_CHECK(hipMalloc((void **)&d_rflag, need));
        desc_cap = need;
    }
    h_sdesc = sd;
    h_rflag = rf;
    if (!sd.empty())
        GFSDC_CHECK(hipMemcpyAsync(d_sdesc, h_sdesc.data(), sizeof(SynthDesc) * sd.size(), hipMemcpyHostToDevice,
                                   stream));
    if (!rf.empty())
        GFSDC_CHECK(hipMemcpyAsync(d_rflag, h_rflag.data(), rf.size(), hipMemcpyHostToDevice, stream));
    return 0;
}

template <typename T> int Engine<T>::input(const void *p, size_t n, int dtype, int loc, int slot, const T **out) {
    if (!p) {
        set_error("null buffer");
        return GFSDC_EINVAL;
    }
    if (dtype != GFSDC_DT_F64 && dtype != GFSDC_DT_F32) {
        set_error("bad dtype");
        return GFSDC_EINVAL;
    }
    size_t esz = dtype == GFSDC_DT_F64 ? 8 : 4;
    bool same = (esz == sizeof(T));
    if (loc == GFSDC_DEVICE && same) {
        *out = (const T *)p;
        return 0;
    }
    int rc = ensure_stage(slot, n * (esz + sizeof(T)));
    if (rc) return rc;
    char *raw = (char *)stage[slot];
    T *conv = (T *)(raw + n * esz);
    const void *src = p;
    if (loc == GFSDC_HOST) {
        GFSDC_CHECK(hipMemcpyAsync(raw, p, n * esz, hipMemcpyHostToDevice, stream));
        src = raw;
        if (same) {
            *out = (const T *)raw;
            return 0;
        }
    }
    if (dtype == GFSDC_DT_F64)
        convert((const double *)src, conv, n, stream);
    else
        convert((const float *)src, conv, n, stream);
    GFSDC_CHECK(hipGetLastError());
    *out = conv;
    return 0;
}

template <typename T> int Engine<T>::output(const T *d, void *p, size_t n, int dtype, int loc, int slot) {
    if (!p) {
        set_error("null buffer");
        return GFSDC_EINVAL;
    }
    size_t esz = dtype == GFSDC_DT_F64 ? 8 : 4;
    bool same = (esz == sizeof(T));
    if (loc == GFSDC_DEVICE) {
        if (same)
            GFSDC_CHECK(hipMemcpyAsync(p, d, n * esz, hipMemcpyDeviceToDevice, stream));
        else if (dtype == GFSDC_DT_F64)
            convert(d, (double *)p, n, stream);
        else
            convert(d, (float *)p, n, stream);
        GFSDC_CHECK(hipGetLastError());
        return 0;
    }
    const void *src = d;
    if (!same) {
        int rc = ensure_stage(slot, n * esz);
        if (rc) return rc;
        if (dtype == GFSDC_DT_F64)
            convert(d, (double *)stage[slot], n, stream);
        else
            convert(d, (float *)stage[slot], n, stream);
        src = stage[slot];
    }
    GFSDC_CHECK(hipMemcpyAsync(p, src, n * esz, hipMemcpyDeviceToHost, stream));
    GFSDC_CHECK(hipStreamSynchronize(stream));
    return 0;
}

// Host fields up to this size (in the context's element type) are copied by the host
// into pinned memory that the first kernel reads and the last one writes over the bus,
// instead of by two queued copies of a pageable buffer, each longer than such a kernel.
// T42 FP64, synthesis and analysis: one field (64 KB) 38 and 43 -> 28 and 26 us; T126 one
// field (0.6 MB) 71 and 69 -> 55 and 53 us; T170 one (1 MB, the limit) 110 and 103 -> 91
// and 88 us. The line bounds what a context holds of such memory, 4 MB: larger fields would
// gain as well, T254 one (2.3 MB) 197 and 167 -> 166 and 147 us, two 348 and 247 -> 304 and
// 237 us, until at four (9 MB, 648 and 423 -> 569 and 442 us) the analysis loses.
constexpr size_t HOST_SMALL = 1 << 20;

// pinned buffer i (0, 1: inputs, 2, 3: outputs) for n values of a caller's field, or null:
// the field is not in host memory, of another type or larger, or there is no memory for it
template <typename T> T *Engine<T>::host_small(const void *p, size_t n, int dtype, int loc, int i) {
    if (!p || loc != GFSDC_HOST || dtype != (sizeof(T) == 8 ? GFSDC_DT_F64 : GFSDC_DT_F32) || n * sizeof(T) > HOST_SMALL)
        return nullptr;
    if (!pinned && hipHostMalloc((void **)&pinned, 4 * HOST_SMALL, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        pinned = nullptr;
        return nullptr;
    }
    return (T *)(pinned + i * HOST_SMALL);
}

// The last transform that read or wrote pinned memory has ended (finish), so the host
// may write it.
template <typename T>
int Engine<T>::field_in(const void *p, size_t n, int dtype, int loc, int i, const T **out) {
    T *h = host_small(p, n, dtype, loc, i);
    if (!h) return input(p, n, dtype, loc, 2 * i, out);
    std::memcpy(h, p, n * sizeof(T));
    *out = h;
    return 0;
}

// Where the last kernel of a transform writes a caller's field itself: a device buffer of
// the context's element type, or pinned memory for a small host field; else null (it
// writes the workspace, and output() converts or copies). Grids take 16-byte stores.
template <typename T> T *Engine<T>::field_out(void *p, size_t n, int dtype, int loc, int i, bool grid) {
    if (!p) return nullptr;
    if (is_direct<T>(dtype, loc)) return grid && ((uintptr_t)p & 15) ? nullptr : (T *)p;
    return host_small(p, n, dtype, loc, 2 + i);
}

// The end of a transform whose np fields went to d: to the caller's buffers p where they
// are not there yet.
template <typename T>
int Engine<T>::finish(T *const *d, void *const *p, int np, size_t n, int dtype, int loc) {
    GFSDC_CHECK(hipGetLastError());
    bool waited = false;
    for (int i = 0; i < np; i++) {
        if ((void *)d[i] == p[i]) continue;
        if (pinned && (char *)d[i] == pinned + (2 + i) * HOST_SMALL) {
            if (!waited) GFSDC_CHECK(hipStreamSynchronize(stream));
            waited = true;
            std::memcpy(p[i], d[i], n * sizeof(T));
            continue;
        }
        const int rc = output(d[i], p[i], n, dtype, loc, 1);
        if (rc) return rc;
    }
    return 0;
}

template <typename T> int Engine<T>::spectogrd(const void *spec, void *grid, int nf, int dtype, int loc) {
    if (nf <= 0) return nf == 0 ? 0 : GFSDC_EINVAL;
    int rc = work_alloc(work, plan, nf);
    if (rc) return rc;
    const T *in;
    const size_t n = (size_t)nf * plan.nlat * plan.nlon;
    if ((rc = field_in(spec, (size_t)nf * plan.nlm * 2, dtype, loc, 0, &in))) return rc;
    T *out = field_out(grid, n, dtype, loc, 0, true);
    if (!out) out = work.grid;
    launch_gather_ref(plan, (const cplx<T> *)in, nf, work.sx, work.ldc, stream);
    launch_leg_synth(plan, work.sx, work.ldc, work.fs, work.ldc, 2 * nf, stream);
    launch_fft_synth(plan, work.fs, work.ldc, out, (long)plan.nlat * plan.nlon, nf, nullptr, stream);
    return finish(&out, &grid, 1, n, dtype, loc);
}

// spectogrd on device buffers of the context's element type with every
// intermediate in the per-device scratch: no allocation, no host copy, no
// synchronisation (work is queued on the context stream).
template <typename T> int Engine<T>::spectogrd_noalloc(const void *spec, void *grid, int nf) {
    if (nf == 0) return 0;
    if (nf < 0 || !spec || !grid) {
        set_error("spectogrd_noalloc: need nfield >= 0 and device buffers");
        return GFSDC_EINVAL;
    }
    char *base = (char *)scratch_ptr(cfg.device);
    if (!base) {
        set_error("spectogrd_noalloc: no scratch address for this device");
        return GFSDC_ESTATE;
    }
    const int ldc = round_up(2 * nf, COL_PAD) + COL_SKEW;
    const size_t o_fs = align256(sizeof(T) * (size_t)plan.nlme * ldc);
    const size_t need = o_fs + sizeof(T) * (size_t)(plan.ntrunc + 1) * plan.nlat * ldc;
    if (need > NOALLOC_SCRATCH_BYTES) {
        set_error("spectogrd_noalloc: " + std::to_string(nf) + " fields at T" + std::to_string(plan.ntrunc) + " (" +
                  std::to_string(plan.nlon) + "x" + std::to_string(plan.nlat) + ") need " + std::to_string(need >> 20) +
                  " MiB of scratch; the maximum is " + std::to_string(NOALLOC_SCRATCH_BYTES >> 20) +
                  " MiB (use gfsdc_spectogrd, or fewer fields per call)");
        return GFSDC_EINVAL;
    }
    T *sx = (T *)base, *fs = (T *)(base + o_fs);
    launch_gather_ref(plan, (const cplx<T> *)spec, nf, sx, ldc, stream);
    launch_leg_synth(plan, sx, ldc, fs, ldc, 2 * nf, stream);
    launch_fft_synth(plan, fs, ldc, (T *)grid, (long)plan.nlat * plan.nlon, nf, nullptr, stream);
    GFSDC_CHECK(hipGetLastError());
    return 0;
}

template <typename T> int Engine<T>::grdtospec(const void *grid, void *spec, int nf, int dtype, int loc) {
    if (nf <= 0) return nf == 0 ? 0 : GFSDC_EINVAL;
    int rc = work_alloc(work, plan, nf);
    if (rc) return rc;
    const T *in;
    const size_t ng = (size_t)plan.nlat * plan.nlon, n = (size_t)nf * plan.nlm * 2;
    if ((rc = field_in(grid, (size_t)nf * ng, dtype, loc, 0, &in))) return rc;
    launch_fft_anal(plan, in, (long)ng, nf, nullptr, work.fa, work.ldc, stream);
    launch_leg_anal(plan, work.fa, work.ldc, work.sx, work.ldc, 2 * nf, stream);
    T *out = field_out(spec, n, dtype, loc, 0, false);
    if (!out) out = work.grid;  // reuse as spectral output buffer (nf * nlm complex <= nf * ng)
    launch_scatter_ref(plan, work.sx, work.ldc, (cplx<T> *)out, nf, stream);
    return finish(&out, &spec, 1, n, dtype, loc);
}

// Transform microbenchmark with device-resident buffers: per iteration a
// spectogrd + grdtospec round trip of ns scalar fields and a getuv of nv
// vector pairs through the same entry points as callers (loc = device).
template <typename T> __global__ void k_fill_spec(cplx<T> *s, long n, int nlm) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int k = (int)(i % nlm);
    T a = T(1) / (T(1) + T(k % 97));
    s[i] = cplx<T>{a, (k % 7) ? a : T(0)};
}

template <typename T> int Engine<T>::bench_transforms(int ns, int nv, int reps, double *ms) {
    if (ns < 1 || nv < 0 || reps < 1) {
        set_error("bench_transforms: ns >= 1, nv >= 0, reps >= 1");
        return GFSDC_EINVAL;
    }
    const size_t ng = (size_t)plan.nlat * plan.nlon, nlm = plan.nlm;
    const int dt = sizeof(T) == 8 ? GFSDC_DT_F64 : GFSDC_DT_F32;
    T *spec = nullptr, *grid = nullptr, *spec2 = nullptr, *uv = nullptr;
    GFSDC_CHECK(hipMalloc((void **)&spec, sizeof(cplx<T>) * nlm * (ns + 2 * nv)));
    GFSDC_CHECK(hipMalloc((void **)&spec2, sizeof(cplx<T>) * nlm * ns));
    GFSDC_CHECK(hipMalloc((void **)&grid, sizeof(T) * ng * ns));
    GFSDC_CHECK(hipMalloc((void **)&uv, sizeof(T) * ng * 2 * (nv > 0 ? nv : 1)));
    const long nsp = (long)nlm * (ns + 2 * nv);
    hipLaunchKernelGGL(k_fill_spec<T>, dim3((unsigned)((nsp + 255) / 256)), dim3(256), 0, stream, (cplx<T> *)spec,
                       nsp, (int)nlm);
    const T *vrt = spec + 2 * nlm * ns, *div = vrt + 2 * nlm * nv;
    auto iter = [&]() -> int {
        int rc = spectogrd(spec, grid, ns, dt, GFSDC_DEVICE);
        if (!rc) rc = grdtospec(grid, spec2, ns, dt, GFSDC_DEVICE);
        if (!rc && nv > 0)
            rc = sphtor_to_spat(vrt, div, uv, uv + ng * nv, nv, 6.3712e6, 1, 6.3712e6, 1, dt, GFSDC_DEVICE);
        return rc;
    };
    int rc = iter();
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (!rc) {
        GFSDC_CHECK(hipStreamSynchronize(stream));
        GFSDC_CHECK(hipEventCreate(&e0));
        GFSDC_CHECK(hipEventCreate(&e1));
        GFSDC_CHECK(hipEventRecord(e0, stream));
        for (int r = 0; r < reps && !rc; r++) rc = iter();
        GFSDC_CHECK(hipEventRecord(e1, stream));
        GFSDC_CHECK(hipEventSynchronize(e1));
        float t = 0.f;
        GFSDC_CHECK(hipEventElapsedTime(&t, e0, e1));
        if (ms) *ms = t / reps;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(spec);
    (void)hipFree(spec2);
    (void)hipFree(grid);
    (void)hipFree(uv);
    return rc;
}

// plain 16-byte-vector copy, grid-stride
__global__ void k_copy_bytes(float4 *__restrict__ dst, const float4 *__restrict__ src, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

template <typename T> int Engine<T>::bench_copy(long nbytes, int reps, double *ms) {
    if (nbytes < 16 || nbytes % 16 || reps < 1) {
        set_error("bench_copy: nbytes a positive multiple of 16, reps >= 1");
        return GFSDC_EINVAL;
    }
    void *a = nullptr, *b = nullptr;
    GFSDC_CHECK(hipMalloc(&a, nbytes));
    if (hipMalloc(&b, nbytes) != hipSuccess) {
        (void)hipFree(a);
        set_error("bench_copy: device allocation failed");
        return GFSDC_ENOMEM;
    }
    const long n = nbytes / 16;
    GFSDC_CHECK(hipMemsetAsync(a, 0, nbytes, stream));
    hipEvent_t e0, e1;
    GFSDC_CHECK(hipEventCreate(&e0));
    GFSDC_CHECK(hipEventCreate(&e1));
    GFSDC_CHECK(hipEventRecord(e0, stream));
    for (int r = 0; r < reps; r++)
        hipLaunchKernelGGL(k_copy_bytes, dim3(4096), dim3(256), 0, stream, (float4 *)b, (const float4 *)a, n);
    GFSDC_CHECK(hipEventRecord(e1, stream));
    GFSDC_CHECK(hipEventSynchronize(e1));
    float t = 0.f;
    GFSDC_CHECK(hipEventElapsedTime(&t, e0, e1));
    if (ms) *ms = t / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    return 0;
}

// (S, T) -> (Vt, Vp) of SHTns sphtor_to_spat with S = sscale [invlap] s, T = tscale [invlap] t;
// s may be null (zero spheroidal part, as getgrad).
template <typename T>
int Engine<T>::sphtor_to_spat(const void *s, const void *t, void *u, void *v, int nf, double sscale, int sinv,
                              double tscale, int tinv, int dtype, int loc) {
    if (nf <= 0) return nf == 0 ? 0 : GFSDC_EINVAL;
    int rc = work_alloc(work, plan, 2 * nf);
    if (rc) return rc;
    const size_t ns = (size_t)nf * plan.nlm * 2, ng = (size_t)plan.nlat * plan.nlon;
    const T *is = nullptr, *it;
    if (s && (rc = field_in(s, ns, dtype, loc, 0, &is))) return rc;
    if ((rc = field_in(t, ns, dtype, loc, 1, &it))) return rc;
    // the Fourier synthesis writes the caller's two grids, or both into the workspace
    T *d[2] = {field_out(u, nf * ng, dtype, loc, 0, true), field_out(v, nf * ng, dtype, loc, 1, true)};
    if (!d[0] || !d[1]) {
        d[0] = work.grid;
        d[1] = work.grid + nf * ng;
    }
    launch_gather_ref_vec(plan, (const cplx<T> *)is, (const cplx<T> *)it, nf, work.sx, work.ldc, sscale, sinv, tscale,
                          tinv, stream);
    launch_leg_synth(plan, work.sx, work.ldc, work.fs, work.ldc, 4 * nf, stream);
    launch_fft_synth(plan, work.fs, work.ldc, d[0], (long)ng, 2 * nf, nullptr, stream, (const T *)nullptr, nullptr, 0,
                     nullptr, nullptr, 0.0, FftOpt<T>{d[1], nf, 1});
    void *const p[2] = {u, v};
    return finish(d, p, 2, nf * ng, dtype, loc);
}

// (Vt, Vp) -> vorticity / divergence (lap/rsphere S, lap/rsphere T), or SHTns (S, T) when inv = 1.
template <typename T>
int Engine<T>::spat_to_sphtor(const void *u, const void *v, void *s, void *t, int nf, double rsphere, int inv,
                              int dtype, int loc) {
    if (nf <= 0) return nf == 0 ? 0 : GFSDC_EINVAL;
    int rc = work_alloc(work, plan, 2 * nf);
    if (rc) return rc;
    const size_t ng = (size_t)plan.nlat * plan.nlon, ns = (size_t)nf * plan.nlm * 2;
    const T *iu, *iv;
    if ((rc = field_in(u, nf * ng, dtype, loc, 0, &iu))) return rc;
    if ((rc = field_in(v, nf * ng, dtype, loc, 1, &iv))) return rc;
    launch_fft_anal(plan, iu, (long)ng, 2 * nf, nullptr, work.fa, work.ldc, stream, nullptr,
                    FftOpt<const T>{iv, nf, 1});
    launch_leg_anal(plan, work.fa, work.ldc, work.sx, work.ldc, 4 * nf, stream);
    T *d[2] = {field_out(s, ns, dtype, loc, 0, false), field_out(t, ns, dtype, loc, 1, false)};
    if (!d[0] || !d[1]) {
        d[0] = work.grid;
        d[1] = work.grid + ns;
    }
    launch_scatter_ref_vec(plan, work.sx, work.ldc, (cplx<T> *)d[0], (cplx<T> *)d[1], nf, rsphere, inv, stream);
    void *const p[2] = {s, t};
    return finish(d, p, 2, ns, dtype, loc);
}

template struct Engine<float>;
template struct Engine<double>;

}  // namespace gfsdc
