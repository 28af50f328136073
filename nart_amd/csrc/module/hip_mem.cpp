// hip_mem_tp: the memory type of the `hip` workspace — a device buffer plus a pinned host mirror, kept
// coherent on demand.  Implements the mem_tp vtable of art/include/art/mem.h:48-64.
#include <immintrin.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "hip_module.h"

// The streams of the live `hip` workspaces.  A memory remembers the stream that last used its device side and the one
// that last read its host mirror, and may outlive the workspace that owned it: a stream that has been retired was
// synchronised when its workspace went away, so there is nothing left to wait for (and nothing valid to wait on).
static std::vector<hipStream_t> &live_streams()
{
    static std::vector<hipStream_t> v;
    return v;
}

void hip_stream_register(hipStream_t st) { live_streams().push_back(st); }

void hip_stream_retire(hipStream_t st)
{
    HIPM_HIP(hipStreamSynchronize(st));
    auto &v = live_streams();
    v.erase(std::remove(v.begin(), v.end(), st), v.end());
}

void hip_stream_forget(hipStream_t st)
{
    auto &v = live_streams();
    v.erase(std::remove(v.begin(), v.end(), st), v.end());
}

// wait for the work queued on st - and only on st: another workspace's kernels keep running.  A stream this module no
// longer knows (its workspace is gone, or it was a caller's stream that has been replaced) cannot be named any more:
// then the whole device is waited for, as the runtime's other GPU modules always do.
static void wait_stream(hipStream_t st)
{
    auto &v = live_streams();
    if (st == nullptr || std::find(v.begin(), v.end(), st) != v.end())
        HIPM_HIP(hipStreamSynchronize(st));
    else
        HIPM_HIP(hipDeviceSynchronize());
}

static void grow_dev(void **p, size_t *cap, size_t need)
{
    if (*cap >= need)
        return;
    if (*p)
        HIPM_HIP(hipFree(*p));
    HIPM_HIP(hipMalloc(p, need));
    *cap = need;
}

static size_t dev_bytes(const hip_mem_t *m)
{
    return m->layout == HIP_LAYOUT_NHWC_U8 ? (size_t)m->N * m->H * m->W * m->cs : m->size;
}

static mem_t *hm_new(void)
{
    constexpr size_t bytes = (sizeof(hip_mem_t) + 63) / 64 * 64;
    void *m = aligned_alloc(64, bytes); // whole cache lines
    HIPM_CHECK(m != nullptr);
    memset(m, 0, bytes);
    return &static_cast<hip_mem_t *>(m)->m;
}

static void hm_free(mem_t *mm)
{
    hip_mem_t *m = as_hip(mm);
    if (m->host)
        HIPM_HIP(hipHostFree(m->host));
    if (m->dev)
        HIPM_HIP(hipFree(m->dev));
    if (m->stage)
        HIPM_HIP(hipFree(m->stage));
    if (m->qhost)
        HIPM_HIP(hipHostFree(m->qhost));
    if (m->qdev)
        HIPM_HIP(hipFree(m->qdev));
    m->qhost = m->qdev = nullptr;
    m->qhost_cap = m->qdev_cap = 0;
    m->q_valid = m->down_issued = m->host_read = false;
    m->host = m->dev = m->stage = nullptr;
    m->host_cap = m->dev_cap = m->stage_cap = m->size = 0;
    m->host_valid = m->dev_valid = false;
    m->up_pending = false;
    m->pending = nullptr;
}

static void hm_delete(mem_t *mm)
{
    hm_free(mm);
    free(mm);
}

// grow-only, like every mem_tp of the runtime (art/src/mem.c:45-55); buffers appear lazily
static bool hm_alloc(mem_t *mm, size_t sz)
{
    hip_mem_t *m = as_hip(mm);
    if (sz > m->size)
        m->size = sz;
    return true;
}

static size_t hm_size(mem_t *mm) { return as_hip(mm)->size; }

static void ensure_host(hip_mem_t *m)
{
    if (m->host_cap >= m->size && m->host)
        return;
    void *p = nullptr;
    HIPM_HIP(hipHostMalloc(&p, m->size ? m->size : 1, hipHostMallocDefault));
    memset(p, 0, m->size);
    if (m->host) {
        if (m->up_pending) { // an upload may still read the old mirror
            wait_stream(m->up_stream);
            m->up_pending = false;
        }
        memcpy(p, m->host, m->host_cap);
        HIPM_HIP(hipHostFree(m->host));
    }
    m->host = p;
    m->host_cap = m->size;
}

static bool stream_known(hipStream_t st)
{
    auto &v = live_streams();
    return st != nullptr && std::find(v.begin(), v.end(), st) != v.end();
}

// device -> host (dense NCHW), queued behind the work that wrote the device side
void hip_mem_start_download(hip_mem_t *m)
{
    ensure_host(m);
    const hipStream_t st = stream_known(m->prod_stream) ? m->prod_stream : nullptr;
    if (st == nullptr)
        wait_stream(m->prod_stream);
    if (m->layout == HIP_LAYOUT_NHWC_U8 && m->size <= kHostDirect) {
        HIPM_HIPQ(hipq_nhwc_to_nchw_u8(m->dev, m->host, m->N, m->C, m->H, m->W, m->cs, st));
    } else if (m->layout == HIP_LAYOUT_NHWC_U8) {
        grow_dev(&m->stage, &m->stage_cap, m->size);
        HIPM_HIPQ(hipq_nhwc_to_nchw_u8(m->dev, m->stage, m->N, m->C, m->H, m->W, m->cs, st));
        HIPM_HIP(hipMemcpyAsync(m->host, m->stage, m->size, hipMemcpyDeviceToHost, st));
    } else {
        HIPM_HIP(hipMemcpyAsync(m->host, m->dev, m->size, hipMemcpyDeviceToHost, st));
    }
    m->down_issued = true;
}

// the same, finished
static void download(hip_mem_t *m)
{
    if (!m->down_issued)
        hip_mem_start_download(m);
    wait_stream(m->prod_stream);
    m->down_issued = false;
    m->host_valid = m->host_read = true;
}

bool hip_mem_uploads_direct(const hip_mem_t *m) { return m->layout == HIP_LAYOUT_NHWC_U8 && m->size <= kHostDirect; }

// the pinned memory is about to be handed out for writing: what still reads it must finish first
static void finish_upload(hip_mem_t *m)
{
    if (m->up_pending) {
        wait_stream(m->up_stream);
        m->up_pending = false;
    }
}

void hip_mem_read_on(hip_mem_t *m, hipStream_t st)
{
    if (m->up_stream != st)
        finish_upload(m); // one stream is remembered: the one before has finished
}

void hip_mem_use_on(hip_mem_t *m, hipStream_t st)
{
    if (m->prod_stream == st)
        return;
    if (m->dev)
        wait_stream(m->prod_stream);
    m->prod_stream = st;
}

static void upload(hip_mem_t *m, hipStream_t st)
{
    hip_mem_read_on(m, st);
    hip_mem_use_on(m, st);
    grow_dev(&m->dev, &m->dev_cap, dev_bytes(m));
    if (hip_mem_uploads_direct(m)) {
        HIPM_HIPQ(hipq_nchw_to_nhwc_u8(m->host, m->dev, m->N, m->C, m->H, m->W, m->cs, st));
    } else if (m->layout == HIP_LAYOUT_NHWC_U8) {
        grow_dev(&m->stage, &m->stage_cap, m->size);
        HIPM_HIP(hipMemcpyAsync(m->stage, m->host, m->size, hipMemcpyHostToDevice, st));
        HIPM_HIPQ(hipq_nchw_to_nhwc_u8(m->stage, m->dev, m->N, m->C, m->H, m->W, m->cs, st));
    } else {
        HIPM_HIP(hipMemcpyAsync(m->dev, m->host, m->size, hipMemcpyHostToDevice, st));
    }
    m->dev_valid = true;
    m->up_pending = true; // the copy still reads the mirror
    m->up_stream = st;
    m->down_issued = false;
}

// mem_cpu_data(): the caller may read or WRITE through the pointer (the runtime fills inputs and weights this
// way, art/src/serialize_v1.c:239-241), so afterwards the host side is the master copy.
static void *hm_cpu_data(const mem_t *mm)
{
    hip_mem_t *m = as_hip(const_cast<mem_t *>(mm));
    hip_mem_settle(m);
    if (m->dev_valid && !m->host_valid)
        download(m); // waits for the workspace whose kernels wrote it; other workspaces are not waited for
    ensure_host(m);
    finish_upload(m);
    m->host_valid = true;
    m->dev_valid = m->q_valid = false;
    ++m->fills;
    return m->host;
}

const void *hip_mem_host_in(mem_t *mm)
{
    hip_mem_t *m = as_hip(mm);
    hip_mem_settle(m);
    if (m->dev_valid && !m->host_valid)
        download(m);
    ensure_host(m);
    m->host_valid = true; // read-only: the device copy stays valid
    return m->host;
}

const void *hip_mem_dev_in(mem_t *mm, hipStream_t st)
{
    hip_mem_t *m = as_hip(mm);
    hip_mem_settle(m);
    if (!m->dev_valid) {
        ensure_host(m); // never-written memory reads as zeros
        m->host_valid = true;
        upload(m, st);
    } else {
        hip_mem_use_on(m, st);
    }
    return m->dev;
}

void *hip_mem_dev_out(mem_t *mm, hipStream_t st)
{
    hip_mem_t *m = as_hip(mm);
    m->pending = nullptr; // about to be overwritten: a deferred producer's result is dead
    hip_mem_use_on(m, st);
    grow_dev(&m->dev, &m->dev_cap, dev_bytes(m));
    m->dev_valid = true;
    m->host_valid = m->down_issued = m->q_valid = false;
    ++m->fills;
    return m->dev;
}

// mem_data(): device pointer for callers outside the module; they may read or write it
static void *hm_data(const mem_t *mm)
{
    mem_t *m = const_cast<mem_t *>(mm);
    const void *p = hip_mem_dev_in(m, nullptr);
    // the caller is foreign code with streams of its own: every producer of this memory (kernels on a workspace
    // stream, a settled convolution, the upload on the null stream) must have finished
    HIPM_HIP(hipDeviceSynchronize());
    as_hip(m)->up_pending = false;
    as_hip(m)->host_valid = as_hip(m)->down_issued = as_hip(m)->q_valid = false;
    ++as_hip(m)->fills;
    return const_cast<void *>(p);
}

// ---- a caller's array into the memory --------------------------------------------------------------------------------------
// What `memcpy(mem_cpu_data(m), src, bytes)` followed by the upload at the next run does, as one pass over the array that
// overlaps with the way to the device.  One core copies 27 - 45 GB/s and the host link takes 57: 38.5 MB were 1.4 ms of copying
// before 0.68 ms of upload.  Here the array is cut into pieces that a few threads copy with streaming stores (four threads
// 160 GB/s, eight 220), and the copy engine starts on what they have finished.  Its copies cost 9 us each beside their bytes,
// so they grow: 1 MB, 2 MB, 4 MB and so on, each covering the copying of the next.  Values that are going to be quantized
// are quantized here (the reference's arithmetic, quantize.c:145-157) and travel as bytes; the mirror still gets the values.
namespace {

typedef long long v2ll __attribute__((vector_size(16)));
typedef v2ll v2ll_a1 __attribute__((aligned(1)));

// streaming stores: the destination is read by the copy engine, not by this core
void copy_stream(void *dst, const void *src, size_t n)
{
    uint8_t *d = static_cast<uint8_t *>(dst);
    const uint8_t *s = static_cast<const uint8_t *>(src);
    const size_t head = std::min(n, (size_t)(-reinterpret_cast<uintptr_t>(d) & 15));
    memcpy(d, s, head);
    d += head, s += head, n -= head;
    for (; n >= 64; n -= 64, d += 64, s += 64)
        for (int i = 0; i < 4; ++i)
            __builtin_ia32_movntdq(reinterpret_cast<v2ll *>(d) + i, reinterpret_cast<const v2ll_a1 *>(s)[i]);
    memcpy(d, s, n);
}

// op_quantize_run_u8 (quantize.c:145-157): fp32 subtract and divide, the 0.5 added in double and truncated - here the integer
// part plus one where the fraction (exact in fp32) is a half or more.  A NaN ends as 0.
__attribute__((always_inline)) inline void quantize_values(const float *__restrict__ x, uint8_t *__restrict__ y, size_t n, float alpha,
                                                           float beta, float hi)
{
    for (size_t i = 0; i < n; ++i) {
        float q = (x[i] - beta) / alpha;
        q = q > hi ? hi : q;
        q = q > 0.f ? q : 0.f;
        const int r = (int)q;
        y[i] = (uint8_t)(r + (q - (float)r >= 0.5f ? 1 : 0));
    }
}

#define QUANTIZE_SPAN(NAME, ...)                                                                                      \
    __attribute__((__VA_ARGS__ optimize("O3,no-trapping-math"))) void NAME(const float *x, uint8_t *y, size_t n, float alpha, float beta, float hi) \
    {                                                                                                                  \
        quantize_values(x, y, n, alpha, beta, hi);                                                                     \
    }
QUANTIZE_SPAN(quantize_span_sse2)
QUANTIZE_SPAN(quantize_span_avx2, target("avx2"), )
#undef QUANTIZE_SPAN

void quantize_span(const float *x, uint8_t *y, size_t n, float alpha, float beta, float hi)
{
    static const auto f = __builtin_cpu_supports("avx2") ? quantize_span_avx2 : quantize_span_sse2;
    f(x, y, n, alpha, beta, hi);
}

// Both in one pass over registers, whole blocks of 64 values; returns how many values it took.  (One thread: 38.5 MB in 0.87 ms,
// what the copy alone takes, against 1.7 ms as two passes; eight threads: 0.22 against 0.31.)
__attribute__((target("avx512f,avx512bw,avx512dq,avx512vl")))
size_t quantize_and_copy_avx512(const float *x, float *copy, uint8_t *y, size_t n, float alpha, float beta, float hi)
{
    const __m512 va = _mm512_set1_ps(alpha), vb = _mm512_set1_ps(beta), vh = _mm512_set1_ps(hi), half = _mm512_set1_ps(0.5f);
    size_t i = 0;
    for (; i + 64 <= n; i += 64) {
        __m128i part[4];
        for (int k = 0; k < 4; ++k) {
            const __m512 v = _mm512_loadu_ps(x + i + 16 * k);
            _mm512_stream_ps(copy + i + 16 * k, v);
            __m512 q = _mm512_div_ps(_mm512_sub_ps(v, vb), va);
            q = _mm512_max_ps(_mm512_min_ps(vh, q), _mm512_setzero_ps()); // a NaN passes the first and ends as the second's 0
            const __m512i r = _mm512_cvttps_epi32(q);
            const __mmask16 up = _mm512_cmp_ps_mask(_mm512_sub_ps(q, _mm512_cvtepi32_ps(r)), half, _CMP_GE_OQ);
            part[k] = _mm512_cvtepi32_epi8(_mm512_mask_add_epi32(r, up, r, _mm512_set1_epi32(1)));
        }
        __m512i out = _mm512_castsi128_si512(part[0]);
        out = _mm512_inserti32x4(out, part[1], 1);
        out = _mm512_inserti32x4(out, part[2], 2);
        out = _mm512_inserti32x4(out, part[3], 3);
        _mm512_stream_si512(reinterpret_cast<__m512i *>(y + i), out);
    }
    return i;
}

bool has_avx512()
{
    static const bool yes = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512dq")
        && __builtin_cpu_supports("avx512vl");
    return yes;
}

constexpr size_t kHelpFrom = 1 << 20; // waking the helpers takes about what copying a megabyte takes

struct WriteJob {
    const uint8_t *src;
    uint8_t *dst; // the mirror
    uint8_t *q;   // the quantized bytes, or null
    size_t bytes, piece, npieces;
    float alpha, beta, hi;
    std::atomic<size_t> next{0};
    std::atomic<size_t> done_upto[64]; // pieces finished per copy to the device
    size_t first[65];                  // first piece of every copy to the device
    size_t ncopies;

    bool take() // one piece; false: none left
    {
        const size_t k = next.fetch_add(1, std::memory_order_relaxed);
        if (k >= npieces)
            return false;
        const size_t o = k * piece, n = std::min(piece, bytes - o);
        constexpr size_t kSpan = 16 << 10; // stays in the first-level cache between the two passes
        size_t u = 0;
        if (q && has_avx512())
            u = 4 * quantize_and_copy_avx512(reinterpret_cast<const float *>(src + o), reinterpret_cast<float *>(dst + o), q + o / 4, n / 4,
                                             alpha, beta, hi);
        for (; u < n; u += kSpan) {
            const size_t len = std::min(kSpan, n - u);
            if (q)
                quantize_span(reinterpret_cast<const float *>(src + o + u), q + (o + u) / 4, len / 4, alpha, beta, hi);
            copy_stream(dst + o + u, src + o + u, len);
        }
        __builtin_ia32_sfence();
        size_t c = 0;
        while (k >= first[c + 1])
            ++c;
        done_upto[c].fetch_add(1, std::memory_order_release);
        return true;
    }
};

// The helpers sleep until a job is posted; the caller never depends on them: it takes pieces itself and waits only for
// pieces that a helper has taken.
class WritePool {
  public:
    static WritePool &get()
    {
        static WritePool *p = new WritePool; // never destroyed: its threads end with the process
        return *p;
    }
    // true: the helpers join `j` until leave(); false: another thread's job has them
    bool post(WriteJob *j)
    {
        std::lock_guard<std::mutex> l(m_);
        if (job_ != nullptr)
            return false;
        if (threads_ == 0) {
            const unsigned cores = std::thread::hardware_concurrency();
            const int want = cores >= 4 ? (int)std::min(7u, cores / 2 - 1) : 0;
            for (; threads_ < want; ++threads_)
                std::thread([this] { loop(); }).detach();
        }
        job_ = j;
        ++serial_;
        cv_.notify_all();
        return true;
    }
    void leave() // returns when no helper looks at the job any more
    {
        std::unique_lock<std::mutex> l(m_);
        job_ = nullptr;
        idle_.wait(l, [this] { return busy_ == 0; });
    }

  private:
    void loop()
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> l(m_);
        for (;;) {
            cv_.wait(l, [&] { return job_ != nullptr && serial_ != seen; });
            seen = serial_;
            WriteJob *j = job_;
            ++busy_;
            l.unlock();
            while (j->take()) {
            }
            l.lock();
            if (--busy_ == 0)
                idle_.notify_all();
        }
    }
    std::mutex m_;
    std::condition_variable cv_, idle_;
    WriteJob *job_ = nullptr;
    uint64_t serial_ = 0;
    int threads_ = 0, busy_ = 0;
};

} // namespace

extern "C" __attribute__((visibility("default"))) bool hip_mem_write(mem_t *mm, const void *src, size_t bytes)
{
    if (mm == nullptr || !is_hip_mem(mm) || bytes != as_hip(mm)->size || bytes == 0)
        return false;
    hip_mem_t *m = as_hip(mm);
    m->pending = nullptr; // about to be overwritten, all of it
    ++m->fills;
    if (m->down_issued) { // the device is still writing the mirror
        wait_stream(m->prod_stream);
        m->down_issued = false;
    }
    ensure_host(m);
    finish_upload(m);
    const bool known = stream_known(m->up_stream);
    const bool quant = m->q_op != nullptr && m->layout == HIP_LAYOUT_RAW && bytes % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 4 == 0
        && (known || bytes / 4 <= kHostDirect);
    if (quant && m->qhost_cap < bytes / 4) {
        if (m->qhost)
            HIPM_HIP(hipHostFree(m->qhost));
        HIPM_HIP(hipHostMalloc(reinterpret_cast<void **>(&m->qhost), bytes / 4, hipHostMallocDefault));
        m->qhost_cap = bytes / 4;
    }
    WriteJob j;
    j.src = static_cast<const uint8_t *>(src), j.dst = static_cast<uint8_t *>(m->host), j.q = quant ? m->qhost : nullptr;
    j.bytes = bytes, j.piece = 256 << 10, j.npieces = (bytes + j.piece - 1) / j.piece;
    j.alpha = m->q_alpha, j.beta = -(m->q_alpha * (float)m->q_zp), j.hi = (float)((1 << m->q_bits) - 1);
    // what goes to the device, and from where: pieces map to one contiguous range of it
    const size_t share = quant ? 4 : 1, dbytes = bytes / share;
    uint8_t *to = nullptr;
    const uint8_t *from = quant ? m->qhost : static_cast<const uint8_t *>(m->host);
    if (known && dbytes > kHostDirect) {
        if (!quant)
            hip_mem_use_on(m, m->up_stream);
        if (quant) {
            grow_dev(reinterpret_cast<void **>(&m->qdev), &m->qdev_cap, dbytes);
            to = m->qdev;
        } else if (m->layout == HIP_LAYOUT_NHWC_U8) {
            grow_dev(&m->dev, &m->dev_cap, dev_bytes(m));
            grow_dev(&m->stage, &m->stage_cap, m->size);
            to = static_cast<uint8_t *>(m->stage);
        } else {
            grow_dev(&m->dev, &m->dev_cap, dev_bytes(m));
            to = static_cast<uint8_t *>(m->dev);
        }
    }
    j.ncopies = 0, j.first[0] = 0;
    for (size_t at = 0, len = std::max<size_t>(1, (1 << 20) / (j.piece / share)); at < j.npieces; ++j.ncopies) {
        at = std::min(at + len, j.npieces);
        if (j.ncopies == 62)
            at = j.npieces;
        j.first[j.ncopies + 1] = at;
        len = quant ? std::max(len, j.npieces / 6) : 2 * len; // quantizing is the slower side: equal shares
    }
    for (size_t c = 0; c < j.ncopies; ++c)
        j.done_upto[c].store(0, std::memory_order_relaxed);
    const bool helped = bytes > kHelpFrom && WritePool::get().post(&j);
    for (size_t c = 0; c < j.ncopies;) {
        if (j.done_upto[c].load(std::memory_order_acquire) < j.first[c + 1] - j.first[c]) {
            if (!j.take())
                __builtin_ia32_pause(); // a helper is at work on it
            continue;
        }
        if (to) {
            const size_t o = j.first[c] * j.piece / share, e = std::min(j.first[c + 1] * j.piece / share, dbytes);
            HIPM_HIP(hipMemcpyAsync(to + o, from + o, e - o, hipMemcpyHostToDevice, m->up_stream));
        }
        ++c;
    }
    if (helped)
        WritePool::get().leave();
    m->host_valid = true;
    m->dev_valid = m->down_issued = false;
    m->q_valid = quant;
    if (to) {
        if (!quant) {
            if (m->layout == HIP_LAYOUT_NHWC_U8)
                HIPM_HIPQ(hipq_nchw_to_nhwc_u8(m->stage, m->dev, m->N, m->C, m->H, m->W, m->cs, m->up_stream));
            m->dev_valid = true;
        }
        m->up_pending = true;
    }
    return true;
}

static void *hm_copy_from_cpu(void *to, const void *from, size_t sz)
{
    HIPM_HIP(hipMemcpy(to, from, sz, hipMemcpyHostToDevice));
    return to;
}

static void *hm_copy_to_cpu(void *to, const void *from, size_t sz)
{
    HIPM_HIP(hipMemcpy(to, from, sz, hipMemcpyDeviceToHost));
    return to;
}

const mem_tp hip_mem_tp_st = {
    "hip_mem", hm_new, hm_delete, hm_alloc, hm_free, hm_data, hm_cpu_data, hm_size, hm_copy_from_cpu, hm_copy_to_cpu,
    nullptr,
};

void hip_mem_tag(tensor_t *t)
{
    if (!is_hip_mem(t->mem))
        return;
    hip_mem_t *m = as_hip(t->mem);
    const size_t count = shape_count(&t->shape);
    if (m->layout == HIP_LAYOUT_NHWC_U8 && (size_t)m->N * m->C * m->H * m->W == count && m->size == count)
        return; // a view (reshape) of a tagged tensor keeps the producer's geometry
    const int nd = t->shape.dim_size;
    hip_layout_t layout = HIP_LAYOUT_RAW;
    int N = 0, C = 0, H = 1, W = 1;
    if ((t->dtype == dtUINT8 || t->dtype == dtINT8) && (nd == 4 || nd == 2)) { // one byte per element either way
        layout = HIP_LAYOUT_NHWC_U8;
        N = (int)t->shape.dim[0], C = (int)t->shape.dim[1];
        if (nd == 4)
            H = (int)t->shape.dim[2], W = (int)t->shape.dim[3];
    }
    if (layout != m->layout || N != m->N || C != m->C || H != m->H || W != m->W) {
        // geometry changed (first use, or a batch reshape): what the device holds is no longer addressable
        if (m->pending) { // a convolution that never launched: there is nothing to keep
            m->pending = nullptr;
            m->dev_valid = false;
        }
        if (m->dev_valid && !m->host_valid && m->dev)
            download(m);
        m->dev_valid = m->down_issued = m->q_valid = false;
        m->layout = layout;
        m->N = N, m->C = C, m->H = H, m->W = W;
        m->cs = layout == HIP_LAYOUT_NHWC_U8 ? hipq_channel_stride(C) : 0;
    }
}
