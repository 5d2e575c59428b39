/*
 * The host side of janas_attn_run_dev over a made-up HIP runtime: a program
 * that takes calls from its standard input and prints, a line a call, what the
 * call launched and what it did to the runtime. No GPU and no kernel: the
 * launches are recorded, device memory is never touched, and a stream that is
 * "captured" refuses what HIP's stream capture refuses (an allocation, a
 * synchronization, a wait for an event recorded outside the capture).
 *
 *   new H KV HD WINDOW N_CTX        a new instance (the one before is gone)
 *   first KV EXACT N POS0           row block, tile and whether the halves take it
 *   call ENTRY KV STREAM CAPTURED N POS0 [N POS0 ...]
 *       ENTRY dev, noalloc, split or kernels1 .. kernels3
 *
 * A call's line: rc, allocations, frees, refused calls of a captured stream,
 * waits for another stream's event, and per launch its name, workgroups,
 * whether it has partials, the halves, and each sequence's key segments.
 */
#include "../janas_amd/csrc/attn_api.cpp"

#include <iostream>
#include <sstream>

namespace {
struct Runtime {
    int allocs = 0, frees = 0, refused = 0, waits = 0;
    bool captured = false;            /* the call's stream */
    hipStream_t stream = nullptr;
    std::vector<std::string> launches;
} R;
char memory[1 << 16];                 /* addresses only */
uint64_t next_mem = 1;

std::string seqs_of(const SeqDesc *s, uint32_t n, bool split)
{
    std::string r;
    for (uint32_t i = 0; i < n; i++)
        r += (i ? "," : "") + std::to_string(split ? s[i].span : s[i].nseg);
    return r;
}
void record(const char *what, uint32_t wg, bool parts, int halves, const std::string &seqs)
{
    R.launches.push_back(std::string(what) + ":" + std::to_string(wg) + ":" +
                         std::to_string(parts) + ":" + std::to_string(halves) + ":" + seqs);
}
hipError_t refuse()
{
    R.refused++;
    return hipErrorStreamCaptureUnsupported;
}
bool in_capture(hipStream_t s) { return R.captured && s == R.stream; }
}  // namespace

/* ---- the runtime ---- */
extern "C" {
hipError_t hipMalloc(void **p, size_t)
{
    if (R.captured)
        return refuse();
    R.allocs++;
    *p = (void *)(next_mem++ << 32);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (p)
        R.frees++;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t, unsigned) { return hipMalloc(p, 0); }
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t)(memory + 1000);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return in_capture(s) ? refuse() : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c)
{
    *c = in_capture(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned)
{
    R.waits++;
    return in_capture(s) ? refuse() : hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = (hipEvent_t)memory;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *, int) { return hipErrorInvalidDevice; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *)
{
    return hipErrorInvalidValue;
}
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t)
{
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind,
                            hipStream_t)
{
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetD32Async(hipDeviceptr_t, int, size_t, hipStream_t) { return hipSuccess; }
}

/* ---- the launches ---- */
namespace janas {
hipError_t launch_split(int, const SplitArgs &a, hipStream_t)
{
    record("split", a.n_wg, a.part_ml != nullptr, 0, seqs_of(a.seq, a.n_seqs, true));
    return hipSuccess;
}
hipError_t launch_merge(const SplitArgs &a, uint32_t n, hipStream_t)
{
    record("merge", n, a.part_ml != nullptr, 0, seqs_of(a.seq, a.n_seqs, true));
    return hipSuccess;
}
hipError_t launch_prefill(int, const PrefillArgs &a, hipStream_t)
{
    record("prefill", a.n_wg, a.part_ml != nullptr, a.halves, seqs_of(a.seq, a.n_seqs, false));
    return hipSuccess;
}
hipError_t launch_prefill_merge(const PrefillArgs &a, uint32_t n, hipStream_t)
{
    record("pmerge", n, a.part_ml != nullptr, a.halves, seqs_of(a.seq, a.n_seqs, false));
    return hipSuccess;
}
hipError_t launch_xcopy(int, const XcopyArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_q8k(const Q8kArgs &, hipStream_t) { return hipSuccess; }
hipError_t launch_refresh(const RefreshArgs &, hipStream_t) { return hipSuccess; }
int scratch_init(int) { return 0; }
void *scratch_ptr(int) { return (void *)(1ull << 60); }
}  // namespace janas

int main()
{
    janas_attn *a = nullptr;
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string what;
        in >> what;
        R = Runtime();
        if (what == "new") {
            uint32_t h, kv, hd, window, n_ctx;
            in >> h >> kv >> hd >> window >> n_ctx;
            janas_attn_destroy(a);
            R = Runtime();
            a = janas_attn_create(h, kv, hd, n_ctx, 1, JANAS_ATTN_FLOAT);
            if (!a)
                return 1;
            janas_attn_set_window(a, window);
            std::cout << a->part_rows << " " << R.allocs << std::endl;
        } else if (what == "first") {
            int kv, ex;
            uint32_t n;
            in >> kv >> ex >> n;
            for (int hv = 0; hv < 2; hv++)
                std::cout << prefill_row_blocks(n, a->group, a->hd, hv, ex) << " "
                          << prefill_tile(a->hd, hv, ex) << " ";
            std::cout << prefill_halves_supported(kv, a->hd) << std::endl;
        } else {
            std::string entry;
            int kv, stream, captured;
            in >> entry >> kv >> stream >> captured;
            std::vector<janas_attn_seq> seqs;
            uint32_t n, pos0;
            while (in >> n >> pos0) {
                janas_attn_seq s;
                memset(&s, 0, sizeof s);
                s.k = s.v = memory;
                s.ks = s.vs = (const float *)memory;
                s.q = (const float *)memory;
                s.out = (float *)memory;
                s.cap = pos0 + n;
                s.n = n;
                s.pos0 = pos0;
                seqs.push_back(s);
            }
            R.captured = captured != 0;
            R.stream = (hipStream_t)(memory + 1 + stream);
            const uint32_t m = (uint32_t)seqs.size();
            int rc;
            if (entry == "noalloc")
                rc = janas_attn_run_dev_noalloc(a, kv, kGateNone, seqs.data(), m, R.stream);
            else if (entry == "split")
                rc = janas_attn_run_dev_split(a, kv, kGateNone, seqs.data(), m, R.stream);
            else if (entry.compare(0, 7, "kernels") == 0)
                rc = janas_attn_run_dev_kernels(a, kv, kGateNone, seqs.data(), m, R.stream,
                                                entry[7] - '0');
            else
                rc = janas_attn_run_dev(a, kv, kGateNone, seqs.data(), m, R.stream);
            std::cout << rc << " " << R.allocs << " " << R.frees << " " << R.refused << " "
                      << R.waits;
            for (const std::string &l : R.launches)
                std::cout << " " << l;
            std::cout << std::endl;
        }
    }
    return 0;
}
