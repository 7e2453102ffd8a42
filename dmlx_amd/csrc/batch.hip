// batch_builder.build on the device (batch_builder.zig:90-214): the scheduler's requests arrive as one
// concatenated token array plus per-request (length, base position); positions, the token -> request map and
// the [T,T] block-diagonal causal mask are produced by kernels. The reference fills the mask on the host
// (O(T^2) floats, 268 MB at T = 8192) and copies it over; here it is written once at HBM speed.
//
// At the sizes of a serving step (a few thousand tokens) the call is bound by the host's way to the device, not by the
// kernels (3 + 7 us at 2080 tokens). So the host lists take no copy of their own: they are laid out in a slot of pinned
// memory, and the first kernel reads them there, over the bus, while it writes the per-token arrays. A slot is used again
// two calls later, behind an event: only a caller that is two calls ahead of the device waits for it. (Three copies from pageable memory and a
// synchronisation before: 2080 tokens 150 us per call, of which the lists' conversion in the caller's language is not this
// file's.)
#include <string.h>

#include "common.h"

namespace dmoe {

constexpr int kBatchBlock = 256; // tokens per workgroup of the first kernel
constexpr size_t kStagingTokens = 8192; // batches of up to so many tokens never allocate (128 KiB of pinned memory per slot)

// Slot layout (32-bit words): first[n_blocks] = index of the non-empty request that holds the first token of each block of
// tokens; then, per non-empty request, offset[m], base position[m], request index[m]; then tokens[T] if wanted.
struct BatchView {
    const int32_t *first, *offset, *base, *index;
    const uint32_t *tokens;
};

// one thread per token; the block's requests (at most one per token, and the one the next block starts with) come to LDS
__global__ __launch_bounds__(kBatchBlock) void batch_tokens_kernel(uint32_t *__restrict__ out_tokens, int32_t *__restrict__ pos,
                                                                   uint32_t *__restrict__ req_of_token,
                                                                   int32_t *__restrict__ seg_start, BatchView v, int n_blocks,
                                                                   int m, int T) {
    __shared__ int32_t off[kBatchBlock + 1], base[kBatchBlock + 1], index[kBatchBlock + 1];
    const int tid = (int)threadIdx.x, b = (int)blockIdx.x, t = b * kBatchBlock + tid;
    uint32_t tok = 0;
    if (out_tokens && t < T) tok = v.tokens[t];
    const int lo = v.first[b], hi = b + 1 < n_blocks ? v.first[b + 1] : m - 1, n = hi - lo + 1; // 1 .. kBatchBlock + 1
    for (int i = tid; i < n; i += kBatchBlock) {
        off[i] = v.offset[lo + i];
        base[i] = v.base[lo + i];
        index[i] = v.index[lo + i];
    }
    __syncthreads();
    if (t >= T) return;
    int a = 0, z = n - 1; // last request whose offset is <= t
    while (a < z) {
        const int mid = (a + z + 1) >> 1;
        if (off[mid] <= t) a = mid;
        else z = mid - 1;
    }
    if (out_tokens) out_tokens[t] = tok;
    if (pos) pos[t] = base[a] + (t - off[a]);
    if (req_of_token) req_of_token[t] = (uint32_t)index[a];
    if (seg_start) seg_start[t] = off[a];
}

// mask[r][c] = 0 when r and c belong to the same request and c <= r, else -inf (batch_builder.zig:140-177): the zeros of a
// row are the run from its request's first token to itself. One workgroup per row, 16-byte stores; rows that do not start
// on a 16-byte boundary (T not a multiple of 4) store up to three values apart at either end.
__global__ __launch_bounds__(256) void batch_mask_kernel(float *__restrict__ mask, const int32_t *__restrict__ seg_start, int T) {
    const int r = (int)blockIdx.x, start = seg_start[r];
    const size_t row0 = (size_t)r * (size_t)T;
    float *const row = mask + row0;
    auto value = [&](int c) { return c >= start && c <= r ? 0.0f : -__builtin_inff(); };
    const int lead = (int)((4 - (row0 & 3)) & 3), head = lead < T ? lead : T, n4 = (T - head) >> 2;
    float4 *const body = (float4 *)(row + head);
    for (int i = (int)threadIdx.x; i < n4; i += 256) {
        const int c = head + 4 * i;
        body[i] = make_float4(value(c), value(c + 1), value(c + 2), value(c + 3));
    }
    const int tail = head + 4 * n4, i = (int)threadIdx.x;
    if (i < head) row[i] = value(i);
    else if (i - head < T - tail) row[tail + i - head] = value(tail + i - head);
}

static int staging_grow(StagingSlot &s, size_t words) {
    if (s.host) DMOE_HIP(hipHostFree(s.host));
    s.host = nullptr;
    s.words = 0;
    DMOE_HIP(hipHostMalloc((void **)&s.host, words * sizeof(uint32_t), hipHostMallocDefault));
    s.words = words;
    return DMOE_OK;
}

// Slots and events are made with the workspace, so that no call up to the size below allocates: 4 T + T / 256 words hold a
// batch of T tokens however it is cut into requests.
int staging_create(Workspace *w) {
    for (StagingSlot &s : w->staging) {
        DMOE_HIP(hipEventCreateWithFlags(&s.read, hipEventDisableTiming));
        DMOE_TRY(staging_grow(s, 4 * kStagingTokens + kStagingTokens / kBatchBlock));
    }
    return DMOE_OK;
}

// the next slot of the workspace's pinned staging memory, at least `words` long and no longer read by an earlier call
static int staging_slot(Workspace *w, size_t words, StagingSlot **out) {
    StagingSlot &s = w->staging[w->staging_next];
    w->staging_next = (w->staging_next + 1) % kStagingSlots;
    DMOE_HIP(hipEventSynchronize(s.read)); // passed long ago unless the caller is kStagingSlots calls ahead of the device
    if (s.words < words) DMOE_TRY(staging_grow(s, words + words / 4));
    *out = &s;
    return DMOE_OK;
}

void staging_clear(Workspace *w) {
    for (StagingSlot &s : w->staging) {
        if (s.read) {
            (void)hipEventSynchronize(s.read);
            (void)hipEventDestroy(s.read);
        }
        if (s.host) (void)hipHostFree(s.host);
        s = StagingSlot();
    }
}

} // namespace dmoe

using namespace dmoe;

extern "C" int dmoe_batch_build(uint32_t *d_out_tokens, int32_t *d_out_positions, float *d_out_mask,
                                uint32_t *d_out_request_of_token, const uint32_t *h_tokens, const int32_t *h_seq_lens,
                                const int32_t *h_base_pos, int n_requests, int T, dmoe_workspace ws, dmoe_stream s) {
    DMOE_REQUIRE(n_requests >= 0 && T >= 0, "batch_build: negative size");
    if (T == 0) return DMOE_OK; // emptyBatch (batch_builder.zig:92-94, :129-131)
    DMOE_REQUIRE(n_requests >= 1 && h_seq_lens && h_base_pos, "batch_build: tokens without requests");
    long long sum = 0;
    int m = 0; // non-empty requests
    for (int i = 0; i < n_requests; ++i) {
        DMOE_REQUIRE(h_seq_lens[i] >= 0 && h_base_pos[i] >= 0, "batch_build: request %d has a negative length or position", i);
        sum += h_seq_lens[i];
        m += h_seq_lens[i] > 0 ? 1 : 0;
    }
    DMOE_REQUIRE(sum == T, "batch_build: request lengths sum to %lld, T is %d", sum, T);
    DMOE_REQUIRE(T <= 65535 || d_out_mask == nullptr, "batch_build: a [T,T] mask is limited to T <= 65535");
    DMOE_REQUIRE(((uintptr_t)d_out_mask % 16) == 0, "batch_build: mask must be 16-byte aligned");
    DMOE_REQUIRE(!d_out_tokens || h_tokens != nullptr, "batch_build: token output requested without tokens");
    hipStream_t st = to_hip(s);
    // a captured launch would read the staging slot again at every replay, when later calls have long refilled it
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &capture) != hipSuccess) (void)hipGetLastError();
    DMOE_REQUIRE(capture == hipStreamCaptureStatusNone, "batch_build: host lists cannot be read by a captured graph");
    Bump b;
    const size_t o_start = b.take(d_out_mask ? sizeof(int32_t) * (size_t)T : 0);
    Workspace *w = nullptr;
    DMOE_TRY(workspace_reserve(ws, b.off, &w));
    const int n_blocks = ceil_div(T, kBatchBlock);
    const size_t words = (size_t)n_blocks + 3 * (size_t)m + (d_out_tokens ? (size_t)T : 0);
    StagingSlot *slot = nullptr;
    DMOE_TRY(staging_slot(w, words, &slot));
    int32_t *const first = (int32_t *)slot->host, *const offset = first + n_blocks, *const base = offset + m, *const index = base + m;
    uint32_t *const tokens = (uint32_t *)(index + m);
    int run = 0, k = 0, next_block = 0;
    for (int i = 0; i < n_requests; ++i) {
        if (h_seq_lens[i] == 0) continue; // no token belongs to it
        offset[k] = run;
        base[k] = h_base_pos[i];
        index[k] = i;
        run += h_seq_lens[i];
        for (; (long long)next_block * kBatchBlock < run; ++next_block) first[next_block] = k;
        ++k;
    }
    if (d_out_tokens) memcpy(tokens, h_tokens, sizeof(uint32_t) * (size_t)T);
    void *dev = nullptr;
    DMOE_HIP(hipHostGetDevicePointer(&dev, slot->host, 0));
    const int32_t *const d = (const int32_t *)dev;
    BatchView v;
    v.first = d, v.offset = d + n_blocks, v.base = v.offset + m, v.index = v.base + m;
    v.tokens = (const uint32_t *)(v.index + m);
    int32_t *const seg_start = d_out_mask ? at<int32_t>(w, o_start) : nullptr;
    hipLaunchKernelGGL(batch_tokens_kernel, dim3((unsigned)n_blocks), dim3(kBatchBlock), 0, st, d_out_tokens, d_out_positions,
                       d_out_request_of_token, seg_start, v, n_blocks, m, T);
    DMOE_LAUNCH_CHECK();
    DMOE_HIP(hipEventRecord(slot->read, st));
    if (d_out_mask) {
        hipLaunchKernelGGL(batch_mask_kernel, dim3((unsigned)T), dim3(256), 0, st, d_out_mask, seg_start, T);
        DMOE_LAUNCH_CHECK();
    }
    return DMOE_OK;
}
