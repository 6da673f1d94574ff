// Bit-parallel Boolean NFA-64 kernels for gfx950 (wave64).
//
// One lane walks one string. The state is a 64-bit mask (bit j = NFA state j
// active); one step is the union of the successor masks of the active states,
// the bit-parallel step of the reference's V4 kernel
// (cuda/nfa_tc_evolution.cu:683-745), which tests 64 rows per step and only
// handles two symbols. Here any symbol alphabet is handled with
// nibble-sliced successor tables in LDS:
//
//     N[c][p][v] = union of succ[c][4p + i] over the bits i of v   (uint64)
//
// so a step is 16 independent LDS lookups, one per nibble p of the state:
//     s' = OR_p N[c][p][(s >> 4p) & 15]
// The lookups depend on the state only through their index; all 16 are
// issued together.
//
// Byte -> class: `cls[byte]` names the table of that byte. Tables are built
// on the host for every symbol plus two extra classes, "reject" (all zero:
// the empty set, absorbing) and "skip" (the identity). In the window kernel,
// every byte outside one aligned 32-byte window [base, base+32) rejects and
// every byte inside it is its own class (byte & 31); a byte outside the
// window is only recorded (two bit operations per word) and forces the
// empty set at the end, exactly as if it had been stepped.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

#define TREX_NFA_BLOCK 512

namespace {

using namespace trexdev;

template <bool WINDOW>
__device__ __forceinline__ void nfa_kernel(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin,
                                           const int64_t* __restrict__ endp, int64_t n_strings,
                                           const uint64_t* __restrict__ tabg, int n_classes,
                                           const uint8_t* __restrict__ clsg, uint32_t win4, uint64_t start,
                                           uint64_t accept, uint64_t* __restrict__ out_mask,
                                           uint8_t* __restrict__ out_accept)
{
    extern __shared__ __attribute__((aligned(16))) uint64_t lds64[];
    uint64_t* tab = lds64;                                        // [n_classes][256]
    uint8_t* cls = reinterpret_cast<uint8_t*>(lds64 + (size_t)n_classes * 256);   // [256]
    {
        const uint4* s4 = reinterpret_cast<const uint4*>(tabg);
        uint4* d4 = reinterpret_cast<uint4*>(tab);
        for (int i = threadIdx.x; i < n_classes * 128; i += blockDim.x) d4[i] = s4[i];
        if (threadIdx.x < 256) cls[threadIdx.x] = clsg[threadIdx.x];
    }
    __syncthreads();

    const int64_t sid = (int64_t)blockIdx.x * TREX_NFA_BLOCK + threadIdx.x;
    if (sid >= n_strings) return;
    int64_t p = begin[sid];
    const int64_t end = endp[sid];
    uint64_t s = start;

    const int64_t head_end = min(end, p + (int64_t)((16u - ((uint32_t)(uintptr_t)(bytes + p) & 15u)) & 15u));
    for (; p < head_end; ++p) s = nfa_step(tab, cls[bytes[p]], s);

    WinCheck w;
    w.init();
    const int64_t nvec = (end - p) >> 4;
    const uint4* v = reinterpret_cast<const uint4*>(bytes + p);
    auto word = [&](uint32_t x) {
        if constexpr (WINDOW) {
            w.add(x);
            s = nfa_step(tab, x & 31u, s);
            s = nfa_step(tab, (x >> 8) & 31u, s);
            s = nfa_step(tab, (x >> 16) & 31u, s);
            s = nfa_step(tab, (x >> 24) & 31u, s);
        } else {
            s = nfa_step(tab, cls[x & 255u], s);
            s = nfa_step(tab, cls[(x >> 8) & 255u], s);
            s = nfa_step(tab, cls[(x >> 16) & 255u], s);
            s = nfa_step(tab, cls[x >> 24], s);
        }
    };
    int64_t i = 0;
    if (nvec >= 2) {
        uint4 a = v[0];
        for (i = 1; i < nvec; ++i) {
            const uint4 b = v[i];
            word(a.x); word(a.y); word(a.z); word(a.w);
            a = b;
        }
        word(a.x); word(a.y); word(a.z); word(a.w);
    } else if (nvec == 1) {
        const uint4 a = v[0];
        word(a.x); word(a.y); word(a.z); word(a.w);
        i = 1;
    }
    p += nvec << 4;
    for (; p < end; ++p) s = nfa_step(tab, cls[bytes[p]], s);
    if constexpr (WINDOW) {
        if (w.outside(win4)) s = 0;
    }
    out_mask[sid] = s;
    out_accept[sid] = (s & accept) != 0 ? 1 : 0;
}

#define TREX_NFA5_BLOCK 1024

__device__ __forceinline__ void nfa_slice5_kernel(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin,
                                            const int64_t* __restrict__ endp, int64_t n_strings,
                                            const uint8_t* __restrict__ tabg, uint32_t win4, uint64_t start,
                                            uint64_t accept, uint64_t* __restrict__ out_mask,
                                            uint8_t* __restrict__ out_accept)
{
    __shared__ __attribute__((aligned(16))) char tb[kTab5Bytes];
    stage_table_far(reinterpret_cast<uint8_t*>(tb), tabg, (int)kTab5Bytes);
    auto step = [&](uint32_t k, uint64_t x) { return nfa5_step(tb, k, x); };
    __syncthreads();

    const int64_t sid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (sid >= n_strings) return;
    int64_t p = begin[sid];
    const int64_t end = endp[sid];
    uint64_t s = start;
    WinCheck w;
    w.init();
    auto byte = [&](uint32_t b) {
        w.add(b * 0x01010101u);
        s = step(b & 31u, s);
    };
    const int64_t head_end = min(end, p + head_len(bytes, p));
    for (; p < head_end; ++p) byte(bytes[p]);
    const int64_t nvec = (end - p) >> 4;
    auto word = [&](uint32_t x) {
        w.add(x);
        s = step(x & 31u, s);
        s = step((x >> 8) & 31u, s);
        s = step((x >> 16) & 31u, s);
        s = step((x >> 24) & 31u, s);
    };
    stream_body<2>(reinterpret_cast<const uint4*>(bytes + p), nvec,
                   [&](uint4 v) { word(v.x); word(v.y); word(v.z); word(v.w); });
    p += nvec << 4;
    for (; p < end; ++p) byte(bytes[p]);
    if (w.outside(win4)) s = 0;
    out_mask[sid] = s;
    out_accept[sid] = (s & accept) != 0 ? 1 : 0;
}

// The 6/5-bit slice kernels: one lane a string, or two or four
// (nfa6_step_shared) for batches that leave SIMDs idle with one; the lanes of a
// group read the same vectors. Strings are read by aligned vectors (Span), and
// with one lane a string each workgroup orders its strings by length.
// Measured (64 states, 32 symbols; the 1,024-thread workgroups of before put
// 40,000 strings on 40 CUs): 40,000 x 2,048 B 744 us before, 258 / 240 / 278
// us with one / two / four lanes; 10,000: 247 / 180 / 154 us; 100,000 x
// 1,024 B: 203 / 272 / 435 us.
template <int LANES>
__device__ __forceinline__ void nfa_slice6_kernel(const uint8_t* __restrict__ bytes,
                                                  const int64_t* __restrict__ begin,
                                                  const int64_t* __restrict__ endp, int64_t n_strings,
                                                  const uint8_t* __restrict__ tabg, uint32_t win4, uint64_t start,
                                                  uint64_t accept, uint64_t* __restrict__ out_mask,
                                                  uint8_t* __restrict__ out_accept)
{
    __shared__ __attribute__((aligned(16))) char tb[kTab6Bytes + (LANES == 1 ? order_bytes(TREX_NFA5_BLOCK) : 0u)];
    const uint32_t q = threadIdx.x % LANES;
    int64_t sid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
    stage_table_far(reinterpret_cast<uint8_t*>(tb), tabg, (int)kTab6Bytes);
    if constexpr (LANES == 1) {
        const int64_t first = (int64_t)blockIdx.x * blockDim.x;
        const uint32_t n_here = (uint32_t)min<int64_t>(n_strings - first, blockDim.x);
        const int64_t mine = min(sid, n_strings - 1);
        const int64_t len = endp[mine] - begin[mine];
        uint32_t* count = reinterpret_cast<uint32_t*>(tb + kTab6Bytes);
        if (threadIdx.x < 64u) count[threadIdx.x] = 0u;
        __syncthreads();
        sid = first + order_by_length(count, n_here, len);
    } else {
        __syncthreads();
    }
    if (sid >= n_strings) return;
    const uint32_t part = q * (4096u / LANES);
    const Span sp(bytes, begin[sid], endp[sid]);
    const uint4 first = sp.first(), last = sp.last();
    uint64_t s = start;
    uint32_t bad = 0;
    auto step = [&](uint32_t b) {
        if constexpr (LANES == 1) s = nfa6_step(tb, b & 31u, s);
        else s = nfa6_step_shared<LANES>(tb, b & 31u, s, part);
    };
    auto word = [&](uint32_t x) {
        bad |= (x ^ win4) & 0xe0e0e0e0u;
        step(x);
        step(x >> 8);
        step(x >> 16);
        step(x >> 24);
    };
    auto some = [&](const uint4& v, uint32_t lo, uint32_t n) {   // bytes lo .. lo + n - 1
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (uint32_t i = 0; i < 16u; ++i) {
            if (i - lo < n) {
                const uint32_t b = (x[i >> 2] >> (8u * (i & 3u))) & 255u;
                bad |= (b ^ win4) & 0xe0u;
                step(b);
            }
        }
    };
    auto vec = [&](const uint4& v) { word(v.x); word(v.y); word(v.z); word(v.w); };
    if (sp.n_first) some(first, sp.lo, sp.n_first);
    stream_span<2>(sp.body, sp.full, [&](const uint4 (&a)[2]) { vec(a[0]); vec(a[1]); }, vec);
    if (sp.n_last) some(last, 0u, sp.n_last);
    if (bad) s = 0;
    if (q == 0) {
        out_mask[sid] = s;
        out_accept[sid] = (s & accept) != 0 ? 1 : 0;
    }
}

}  // namespace

// tabg: 32 window classes of 5-bit slice tables, class k at byte k * 3336
// (13 rows of 32 uint64 entries, 8 bytes of padding); kTab5Bytes in total.
extern "C" __global__ void __launch_bounds__(TREX_NFA5_BLOCK)
nfa64_window5(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin, const int64_t* __restrict__ end,
              int64_t n_strings, const uint8_t* __restrict__ tabg, uint32_t win4, uint64_t start, uint64_t accept,
              uint64_t* __restrict__ out_mask, uint8_t* __restrict__ out_accept)
{
    nfa_slice5_kernel(bytes, begin, end, n_strings, tabg, win4, start, accept, out_mask, out_accept);
}

// tabg: 32 window classes of 6/5-bit slice tables, class k at byte k * 4104
// (12 rows: 64, 32, 32 uint64 entries per quarter; 8 bytes of padding);
// kTab6Bytes in total. _x2, _x4: lanes a string.
#define TREX_NFA_SLICE6_KERNEL(NAME, LANES)                                                                    \
    extern "C" __global__ void __launch_bounds__(TREX_NFA5_BLOCK)                                              \
    NAME(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin, const int64_t* __restrict__ end, \
         int64_t n_strings, const uint8_t* __restrict__ tabg, uint32_t win4, uint64_t start, uint64_t accept,  \
         uint64_t* __restrict__ out_mask, uint8_t* __restrict__ out_accept) {                                  \
        nfa_slice6_kernel<LANES>(bytes, begin, end, n_strings, tabg, win4, start, accept, out_mask, out_accept); \
    }

TREX_NFA_SLICE6_KERNEL(nfa64_window6, 1)
TREX_NFA_SLICE6_KERNEL(nfa64_window6_x2, 2)
TREX_NFA_SLICE6_KERNEL(nfa64_window6_x4, 4)

// tabg: [n_classes][16][16] uint64 nibble tables; clsg: [256] class of every
// byte. Window kernel: classes 0..31 are the window bytes base + k (n_classes
// >= 32); the byte map is used for the unaligned head and tail bytes only.
// Dynamic LDS: n_classes * 2048 + 256 bytes.
extern "C" __global__ void __launch_bounds__(TREX_NFA_BLOCK)
nfa64_window(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin, const int64_t* __restrict__ end,
             int64_t n_strings, const uint64_t* __restrict__ tabg, int n_classes, const uint8_t* __restrict__ clsg,
             uint32_t win4, uint64_t start, uint64_t accept, uint64_t* __restrict__ out_mask,
             uint8_t* __restrict__ out_accept)
{
    nfa_kernel<true>(bytes, begin, end, n_strings, tabg, n_classes, clsg, win4, start, accept, out_mask, out_accept);
}

extern "C" __global__ void __launch_bounds__(TREX_NFA_BLOCK)
nfa64_bytes(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin, const int64_t* __restrict__ end,
            int64_t n_strings, const uint64_t* __restrict__ tabg, int n_classes, const uint8_t* __restrict__ clsg,
            uint32_t win4, uint64_t start, uint64_t accept, uint64_t* __restrict__ out_mask,
            uint8_t* __restrict__ out_accept)
{
    nfa_kernel<false>(bytes, begin, end, n_strings, tabg, n_classes, clsg, win4, start, accept, out_mask, out_accept);
}
