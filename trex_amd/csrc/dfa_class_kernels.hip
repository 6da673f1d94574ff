// DFA walks over byte classes (gfx950, wave64): contiguous strings of any
// alignment, any alphabet.
//
// Bytes with equal table columns form one class; a pattern rarely has more
// than 31. One LDS read maps a byte to its class, and one more per byte pair
// fetches what the pair does to the state, whatever bytes the pattern uses:
//
//  * dfa16_cls_n10 / _n15 / _n16 (at most that many states): the pair's whole
//    function as one 64-bit word, so the reads do not wait for the state, and a
//    step is one, two or three instructions (Width).
//  * dfa_cls_pair (17 to 256 states): the successor bytes of a pair, read at the
//    state;
//  * dfa_cls_rows, where the pairs' table would not fit: the successor bytes of
//    every byte, without classes.
//
// Every string is read as the aligned 16-byte vectors that hold its bytes (Span),
// so up to 15 bytes on either side of it are read and not used: no byte loop but
// _rows' two ends, and no load that could leave a page that the string is on.
// Missing bytes of the first and last vector take the identity class.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

// Arguments of every kernel (same layout in dfa_class.cpp).
struct ClassArgs {
    const uint8_t* bytes;
    const int64_t* begin;
    const int64_t* end;
    int64_t n_strings;
    const uint8_t* tab;
    uint32_t tab_bytes;
    uint32_t classes;        // identity class included (at most 16 states); _rows: bytes from row to row
    uint32_t accept;         // bit s: state s accepts (at most 16 states)
    uint32_t start;
    const uint8_t* acc;      // accept byte of every state
    const uint64_t* masks;   // _mask: what each state stands for
    uint8_t* out_state;
    uint64_t* out_mask;      // _mask
    uint8_t* out_accept;
};

namespace {

using namespace trexdev;

constexpr int kClsBytes = 256;    // byte -> class * 8
constexpr int kMapBytes = 1040;   // map[257] of the pair form, padded
constexpr int kPF = 4;            // vectors in flight ahead of the block being walked

// Function words by number of states: the field of state s holds its successor,
// and the walk keeps its state as the shift amount of its field, so that a step
// is as few dependent instructions as the width allows.
//   W10: ten 6-bit fields of 6 * successor. word >> amount is the next amount
//        (the hardware reads the low six bits of an amount).
//   W15: fifteen 4-bit fields from bit 2 on: word >> amount has 4 * successor in
//        bits 2 to 5, and the field below's top bits to mask off under them.
//   W16: sixteen 4-bit fields: a mask and a shift.
enum Width { W10, W15, W16 };

template <Width W>
__device__ __forceinline__ uint32_t fn_step(uint64_t f, uint32_t amount) {
    const uint32_t x = (uint32_t)(f >> (amount & 63u));
    return W == W10 ? x : W == W15 ? x & 60u : (x & 15u) << 2;
}

template <Width W>
struct ClassWalk {
    const uint8_t* cls;   // [256] class * 8
    const char* f2;       // pair functions
    uint32_t stride;      // entries from one second class to the next
    uint32_t ident;       // identity class * 8
    uint32_t s;           // the state as its field's shift amount (W10: in the low six bits)

    __device__ __forceinline__ uint64_t fn(uint32_t c0, uint32_t c1) const {
        return *reinterpret_cast<const uint64_t*>(f2 + (__umul24(c1, stride) + c0));
    }
    __device__ __forceinline__ void vector(const uint4& v) {
        uint32_t c[16];
        uint64_t f[8];
        classes(v, c);
        functions(c, f);
#pragma unroll
        for (int i = 0; i < 8; ++i) s = fn_step<W>(f[i], s);
    }
    __device__ __forceinline__ void classes(const uint4& v, uint32_t (&c)[16]) const {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 16; ++i) c[i] = cls[(x[i >> 2] >> (8 * (i & 3))) & 255u];
    }
    __device__ __forceinline__ void functions(const uint32_t (&c)[16], uint64_t (&f)[8]) const {
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = fn(c[2 * i], c[2 * i + 1]);
    }
    // A block of vectors as a pipeline of three stages: the class reads of
    // vector k + 2 and the function reads of vector k + 1 go out ahead of
    // vector k's chain of steps, so neither read's latency is waited for
    // vector by vector (an empty asm ties each vector's words to the state, or
    // the compiler issues the whole block's reads at once and runs out of
    // registers).
    template <int PF>
    __device__ __forceinline__ void block(const uint4 (&a)[PF]) {
        uint32_t c[16];
        uint64_t f[8];
        classes(a[0], c);
        functions(c, f);
        classes(a[1], c);
#pragma unroll
        for (int k = 0; k < PF; ++k) {
            uint64_t g[8];
            if (k + 1 < PF) functions(c, g);
            if (k + 2 < PF) {
                uint4 x = a[k + 2];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w) : "v"(s));
                classes(x, c);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) s = fn_step<W>(f[i], s);
            if (k + 1 < PF) {
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i] = g[i];
            }
        }
    }
    // bytes lo .. lo + n - 1 of a vector
    __device__ __forceinline__ void masked(const uint4& v, uint32_t lo, uint32_t n) {
        uint32_t c[16];
        uint64_t f[8];
        classes(v, c);
#pragma unroll
        for (uint32_t i = 0; i < 16u; ++i) c[i] = i - lo < n ? c[i] : ident;
        functions(c, f);
#pragma unroll
        for (int i = 0; i < 8; ++i) s = fn_step<W>(f[i], s);
    }
    __device__ __forceinline__ uint32_t state() const { return W == W10 ? (s & 63u) / 6u : s >> 2; }
};

// LEAVE: workgroups whose strings are alike are left to the rotated kernel.
// MASK: results are the states' masks.
template <Width W, bool LEAVE, bool MASK>
__device__ __forceinline__ void class_kernel(const ClassArgs& A)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    if constexpr (LEAVE) {
        if (strings_alike(reinterpret_cast<uint32_t*>(lds), A.begin, A.end, A.n_strings)) return;
    }
    const int64_t sid = stage_and_pick(lds, A.tab, A.tab_bytes, A.begin, A.end, A.n_strings);
    if (sid < 0) return;
    const Span sp(A.bytes, A.begin[sid], A.end[sid]);
    const uint4 first = sp.first(), last = sp.last();
    ClassWalk<W> w{lds, reinterpret_cast<const char*>(lds) + kClsBytes, A.classes | 1u, (A.classes - 1u) * 8u,
                   A.start * (W == W10 ? 6u : 4u)};
    if (sp.n_first) w.masked(first, sp.lo, sp.n_first);
    // the slower steps let half-read cache lines be evicted: whole lines there
    // (13 states, 262,144 x 4 KiB: 304 us by fours, 254 us by eights; ten
    // states and less: 250 us either way, and short strings run 10 to 20 %
    // faster with the registers of four)
    constexpr int PF = W == W10 ? kPF : 8;
    stream_span<PF>(sp.body, sp.full, [&](const uint4 (&a)[PF]) { w.block(a); }, [&](const uint4& v) { w.vector(v); });
    if (sp.n_last) w.masked(last, 0u, sp.n_last);
    const uint32_t s = w.state();
    if constexpr (MASK) A.out_mask[sid] = A.masks[s];
    else A.out_state[sid] = (uint8_t)s;
    A.out_accept[sid] = (uint8_t)((A.accept >> s) & 1u);
}

// 17 to 256 states, pairs of classes. map[byte] holds the byte's class times the
// strides of the two positions of a pair: low half for the first byte, high half
// for the second; map[256] is the identity class. A step reads succ[row + s].
struct PairWalk {
    static constexpr int kPF = 4;
    const uint32_t* map;    // [257]
    const uint8_t* succ;
    uint32_t s;

    __device__ __forceinline__ PairWalk(const uint8_t* lds, const ClassArgs& A)
        : map(reinterpret_cast<const uint32_t*>(lds)), succ(lds + kMapBytes), s(A.start) {}
    __device__ __forceinline__ void step2(uint32_t m0, uint32_t m1) { s = succ[(m0 & 0xffffu) + (m1 >> 16) + s]; }
    __device__ __forceinline__ void word(uint32_t x) {
        const uint32_t m0 = map[x & 255u], m1 = map[(x >> 8) & 255u], m2 = map[(x >> 16) & 255u], m3 = map[x >> 24];
        step2(m0, m1);
        step2(m2, m3);
    }
    __device__ __forceinline__ void vector(const uint4& v) { word(v.x); word(v.y); word(v.z); word(v.w); }
    __device__ __forceinline__ void maps(const uint4& v, uint32_t (&m)[16]) const {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 16; ++i) m[i] = map[(x[i >> 2] >> (8 * (i & 3))) & 255u];
    }
    // the next vector's map reads go out ahead of a vector's chain of steps
    template <int PF>
    __device__ __forceinline__ void block(const uint4 (&a)[PF]) {
        uint32_t m[16];
        maps(a[0], m);
#pragma unroll
        for (int k = 0; k < PF; ++k) {
            uint32_t n[16];
            if (k + 1 < PF) {
                uint4 x = a[k + 1];
                asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w) : "v"(s));
                maps(x, n);
            }
#pragma unroll
            for (int i = 0; i < 16; i += 2) step2(m[i], m[i + 1]);
            if (k + 1 < PF) {
#pragma unroll
                for (int i = 0; i < 16; ++i) m[i] = n[i];
            }
        }
    }
    __device__ __forceinline__ void masked(const uint4& v, uint32_t lo, uint32_t n) {
        uint32_t m[16];
        maps(v, m);
        const uint32_t ident = map[256];
#pragma unroll
        for (uint32_t i = 0; i < 16u; ++i) m[i] = i - lo < n ? m[i] : ident;
#pragma unroll
        for (int i = 0; i < 16; i += 2) step2(m[i], m[i + 1]);
    }
};

// 17 to 256 states where the pairs' table would not fit: a row of successors for
// every byte value. Rows by class need a second read a byte for the class, which
// fills the LDS pipe: 100 states and classes, 100,000 strings of 1 to 2 KB: 94 us
// by class, 74 us so; 262,144 x 4 KiB: 421 us, 268 us; 400,000 of 20 to 400
// bytes: 55 us, 51 us. (The pairs' rows halve the chain of reads: 20,000 x 4 KiB
// take 93 us, 131 us so.)
struct RowWalk {
    static constexpr int kPF = 8;
    const uint8_t* succ;
    uint32_t stride;
    uint32_t s;

    __device__ __forceinline__ RowWalk(const uint8_t* lds, const ClassArgs& A) : succ(lds), stride(A.classes), s(A.start) {}
    __device__ __forceinline__ uint32_t next(uint32_t b) const { return succ[__umul24(b, stride) + s]; }
    __device__ __forceinline__ void vector(const uint4& v) {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 16; ++i) s = next((x[i >> 2] >> (8 * (i & 3))) & 255u);
    }
    template <int PF>
    __device__ __forceinline__ void block(const uint4 (&a)[PF]) {
#pragma unroll
        for (int k = 0; k < PF; ++k) vector(a[k]);
    }
    __device__ __forceinline__ void masked(const uint4& v, uint32_t lo, uint32_t n) {
        each_byte(v, lo, n, [&](uint32_t b) { s = next(b); });
    }
};

template <class Walk, bool MASK>
__device__ __forceinline__ void wide_kernel(const ClassArgs& A)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int64_t sid = stage_and_pick(lds, A.tab, A.tab_bytes, A.begin, A.end, A.n_strings);
    if (sid < 0) return;
    const Span sp(A.bytes, A.begin[sid], A.end[sid]);
    const uint4 first = sp.first(), last = sp.last();
    Walk w(lds, A);
    constexpr int kPF = Walk::kPF;
    if (sp.n_first) w.masked(first, sp.lo, sp.n_first);
    stream_span<kPF>(sp.body, sp.full, [&](const uint4 (&a)[kPF]) { w.block(a); }, [&](const uint4& v) { w.vector(v); });
    if (sp.n_last) w.masked(last, 0u, sp.n_last);
    if constexpr (MASK) A.out_mask[sid] = A.masks[w.s];
    else A.out_state[sid] = (uint8_t)w.s;
    A.out_accept[sid] = A.acc[w.s];
}

}  // namespace

// tab: 256 bytes (byte -> class * 8), then the functions of the class pairs,
// pair (c0, c1) at entry c0 + c1 * (classes | 1): an odd stride spreads pairs
// that share their first class over the LDS banks (a power of two puts them
// all into one). The last class is the identity. Dynamic LDS: tab_bytes (a
// multiple of 16), 768 bytes more in workgroups of 256 threads.
// No kernel here has LDS of fixed size: the tables' copies then start at byte 0
// and every offset into them is an immediate (behind 256 bytes of it, 250 us
// of 262,144 x 4 KiB became 300 us).
// _left: workgroups of alike strings are left to the rotated kernel; _mask: the
// results are the states' masks.
#define TREX_CLASS_KERNEL(NAME, ...) \
    extern "C" __global__ void __launch_bounds__(256) NAME(ClassArgs A) { class_kernel<__VA_ARGS__>(A); }
#define TREX_CLASS_KERNELS(W, TAG)                               \
    TREX_CLASS_KERNEL(dfa16_cls_##TAG, W, false, false)          \
    TREX_CLASS_KERNEL(dfa16_cls_##TAG##_left, W, true, false)    \
    TREX_CLASS_KERNEL(dfa16_cls_##TAG##_mask, W, false, true)

TREX_CLASS_KERNELS(W10, n10)
TREX_CLASS_KERNELS(W15, n15)
TREX_CLASS_KERNELS(W16, n16)

// _pair: tab is map[257] (uint32, padded to 1,040 bytes), then the successor
// rows of the class pairs, padded to 16 states; _rows: the successor rows of the
// 256 bytes (`classes` is their stride). Dynamic LDS as above.
#define TREX_WIDE_KERNEL(NAME, ...) \
    extern "C" __global__ void __launch_bounds__(256) NAME(ClassArgs A) { wide_kernel<__VA_ARGS__>(A); }

TREX_WIDE_KERNEL(dfa_cls_pair, PairWalk, false)
TREX_WIDE_KERNEL(dfa_cls_pair_mask, PairWalk, true)
TREX_WIDE_KERNEL(dfa_cls_rows, RowWalk, false)
TREX_WIDE_KERNEL(dfa_cls_rows_mask, RowWalk, true)
