// Multi-pattern DFA-16 walk with compact pair tables (gfx950).
//
// The multi-pattern kernels (dfa_multi_kernels.hip) read one 8-byte pair
// function per pattern and byte pair, and are bound by those LDS reads. A
// pattern of at most 4 states needs 2 bits per state: its pair function fits
// one byte, so eight such patterns share one 8-byte word. Here a launch holds
// NF patterns with full functions (16 nibbles, one word each) and NB
// patterns of at most 4 states (one byte each, eight per word); entry x of
// the launch's table is NW = NF + ceil(NB / 8) words, stored word pair by word
// pair: table j (j < NW / 2) holds words 2j, 2j+1 of every entry as 16 bytes,
// so each step reads NW / 2 16-byte entries at stride 16 (random entries
// spread over all 16 bank quads), plus one 8-byte entry when NW is odd.
//
// Full pattern k:  s = (w_k >> 4s) & 15
// Byte pattern i:  s = bits [8 (i % 8) + 2s, +2) of w_{NF + i/8} (one bit-field
//                  extract from the word's half that holds the byte)
//
// Behind the 1,024 pairs, entry 1024 + c is symbol c alone and entry 1056 is
// the identity, for bytes without a partner and for missing ones. The window
// check and the outputs are those of the other multi-pattern kernels; launch
// pattern k writes row slot[k] of the pattern-major outputs (the host orders a
// launch's patterns full ones first).
//
// Contiguous strings (compact_strings) are the form of every launch whose form
// the caller left open. Two things bound them: the LDS reads where the chip is
// full, and where it is not (less than about four waves a CU) a wave's own
// chain of steps. So the reads go out a word ahead of the steps, a workgroup's
// strings are ordered by length, their ends are whole aligned vectors with the
// missing bytes set to the identity, and a full pattern of at most eight states
// besides its dead one steps in one byte permute (_n8): its word holds a byte
// for each live state, the successor's number or 0xff for the dead state, and
// v_perm_b32 selects the byte that the state numbers (and 0xff by 0xff, so the
// dead state needs no byte). A 64-bit shift costs four times that.
// 8 patterns, 50,000 strings of 200 to 3,000 bytes: 130 us before, 85 us now;
// 10,000 of 100 to 1,500: 80 us, 48 us; 262,144 x 4 KiB (LDS reads): 531 us,
// 514 us.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "device_common.h"

#define TREX_COMPACT_BLOCK 256

namespace {

using namespace trexdev;

constexpr int kCompactMax = 8;   // patterns per launch
constexpr int kIlGroup = 64;     // strings per group of the interleaved layout

}  // namespace

// Per-pattern scalars of one launch, in launch order.
struct CompactParams {
    uint32_t win4[kCompactMax];
    uint32_t start[kCompactMax];
    uint32_t dead[kCompactMax];
    uint32_t accept[kCompactMax];   // bit s set = state s accepts
    uint32_t slot[kCompactMax];     // output row of the pattern
};

namespace {

constexpr int kEntries = 1058;      // 1,024 pairs, 32 single symbols, the identity, padding
constexpr uint32_t kSingle = 1024u, kIdentity = 1056u;

// The tables of a launch in LDS and the states of one string.
template <int NF, int NB, bool N8>
struct CompactWalk {
    static constexpr int P = NF + NB;
    static constexpr int NW = NF + (NB + 7) / 8;
    static constexpr int kPairTables = NW / 2;
    static constexpr int kBytes = kEntries * NW * 8;
    const uint8_t* tw;
    uint32_t s[P];   // full: the shift amount of the state's field (N8: the state's byte, in the low byte), byte patterns: the state

    __device__ __forceinline__ void start(const CompactParams& prm) {
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const uint32_t q = prm.start[k];
            s[k] = k >= NF ? q : !N8 ? q << 2 : q == prm.dead[k] ? 0xffu : q - (q > prm.dead[k] ? 1u : 0u);
        }
    }
    __device__ __forceinline__ uint32_t state(int k, uint32_t dead) const {
        if (k >= NF) return s[k];
        if (!N8) return s[k] >> 2;
        const uint32_t b = s[k] & 0xffu;
        return b > 7u ? dead : b + (b >= dead ? 1u : 0u);
    }

    __device__ __forceinline__ void fetch(uint32_t x, uint64_t (&W)[NW]) const {
#pragma unroll
        for (int j = 0; j < kPairTables; ++j) {
            const uint4 v = reinterpret_cast<const uint4*>(tw + j * (kEntries * 16))[x];
            W[2 * j] = (uint64_t)v.x | ((uint64_t)v.y << 32);
            W[2 * j + 1] = (uint64_t)v.z | ((uint64_t)v.w << 32);
        }
        if constexpr (NW & 1) W[NW - 1] = reinterpret_cast<const uint64_t*>(tw + kPairTables * (kEntries * 16))[x];
    }
    __device__ __forceinline__ void step(const uint64_t (&W)[NW]) {
#pragma unroll
        for (int k = 0; k < NF; ++k) {
            if constexpr (N8) s[k] = __builtin_amdgcn_perm((uint32_t)(W[k] >> 32), (uint32_t)W[k], s[k]);
            else s[k] = ((uint32_t)(W[k] >> s[k]) & 15u) << 2;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            // the byte's dword, then one bit-field extract (offset 8 (i % 4) + 2s)
            const uint64_t wv = W[NF + i / 8];
            const uint32_t dw = (i % 8) < 4 ? (uint32_t)wv : (uint32_t)(wv >> 32);
            s[NF + i] = __builtin_amdgcn_ubfe(dw, 8u * (i % 4) + (s[NF + i] << 1), 2u);
        }
    }
    __device__ __forceinline__ void fetch_step(uint32_t x) {
        uint64_t W[NW];
        fetch(x, W);
        step(W);
    }
    // a word's reads go out once the previous word's steps are done (an empty
    // asm ties it to a state): one word ahead at most, or the compiler hoists
    // a whole block's reads and runs out of registers
    __device__ __forceinline__ void tie(uint32_t& x) const { asm volatile("" : "+v"(x) : "v"(s[0])); }

    __device__ __forceinline__ void finish(const WinCheck& w, const CompactParams& prm, int64_t n_strings, int64_t sid,
                                           uint8_t* __restrict__ out_state, uint8_t* __restrict__ out_accept) const {
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const uint32_t q = w.outside(prm.win4[k]) ? prm.dead[k] : state(k, prm.dead[k]);
            const int64_t row = (int64_t)prm.slot[k] * n_strings + sid;
            out_state[row] = (uint8_t)q;
            out_accept[row] = (uint8_t)((prm.accept[k] >> q) & 1u);
        }
    }
};

// Interleaved layout.
template <int NF, int NB>
__device__ __forceinline__ void compact_groups(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin,
                                               const int64_t* __restrict__ endp, int64_t n_strings,
                                               const uint8_t* __restrict__ wordsg, const CompactParams& prm,
                                               uint8_t* __restrict__ out_state, uint8_t* __restrict__ out_accept)
{
    typedef CompactWalk<NF, NB, false> Walk;
    __shared__ __attribute__((aligned(16))) uint8_t tw[Walk::kBytes];
    stage_table(tw, wordsg, Walk::kBytes);
    __syncthreads();

    const int64_t sid = (int64_t)blockIdx.x * TREX_COMPACT_BLOCK + threadIdx.x;
    if (sid >= n_strings) return;
    const int64_t p = begin[sid], len = endp[sid] - p;
    Walk walk{tw, {}};
    walk.start(prm);
    WinCheck w; w.init();
    auto word = [&](uint32_t x) {
        w.add(x);
        walk.tie(x);
        walk.fetch_step(pair_lo(x));
        walk.fetch_step(pair_hi(x));
    };
    const int64_t nvec = len >> 4;
    stream_body_nt<8, kIlGroup>(reinterpret_cast<const uint4*>(bytes + p), nvec, [&](uint4 v) {
        word(v.x); word(v.y); word(v.z); word(v.w);
    });
    const uint8_t* tail = bytes + p + nvec * (16 * kIlGroup);
    for (int t = 0; t < (int)(len & 15); ++t) {
        const uint32_t b = tail[t];
        w.add(b * 0x01010101u);
        walk.fetch_step(kSingle + (b & 31u));
    }
    walk.finish(w, prm, n_strings, sid, out_state, out_accept);
}

// Words whose reads are in flight ahead of the steps (4 * NW registers each).
template <int NW>
constexpr int kAhead = NW <= 3 ? 2 : 1;

// Contiguous strings.
template <int NF, int NB, bool N8>
__device__ __forceinline__ void compact_strings(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin,
                                                const int64_t* __restrict__ endp, int64_t n_strings,
                                                const uint8_t* __restrict__ wordsg, const CompactParams& prm,
                                                uint8_t* __restrict__ out_state, uint8_t* __restrict__ out_accept)
{
    typedef CompactWalk<NF, NB, N8> Walk;
    constexpr int NW = Walk::NW, PF = NW <= 2 ? 8 : 4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[Walk::kBytes + order_bytes(TREX_COMPACT_BLOCK)];
    const int64_t sid = stage_and_pick(lds, wordsg, Walk::kBytes, begin, endp, n_strings);
    if (sid < 0) return;
    const Span sp(bytes, begin[sid], endp[sid]);
    const uint4 first = sp.first(), last = sp.last();
    Walk walk{lds, {}};
    walk.start(prm);
    WinCheck w; w.init();

    // the reads of word k + D go out ahead of the steps of word k
    auto words = [&](const uint4* a, auto count_tag) {
        constexpr int N = decltype(count_tag)::value;
        constexpr int D = kAhead<NW> < 4 * N - 1 ? kAhead<NW> : 4 * N - 1;
        uint64_t lo[D + 1][NW], hi[D + 1][NW];
        auto word = [&](int k) { const uint4& v = a[k / 4]; return k % 4 == 0 ? v.x : k % 4 == 1 ? v.y : k % 4 == 2 ? v.z : v.w; };
        auto fetch = [&](int k, uint32_t x) {
            walk.fetch(pair_lo(x), lo[k % (D + 1)]);
            walk.fetch(pair_hi(x), hi[k % (D + 1)]);
        };
#pragma unroll
        for (int k = 0; k < D; ++k) fetch(k, word(k));
#pragma unroll
        for (int k = 0; k < 4 * N; ++k) {
            if (k + D < 4 * N) {
                uint32_t x = word(k + D);
                walk.tie(x);
                fetch(k + D, x);
            }
            w.add(word(k));
            walk.step(lo[k % (D + 1)]);
            walk.step(hi[k % (D + 1)]);
        }
    };
    // bytes at, ..., at + n - 1 of a vector
    auto masked = [&](const uint4& v, uint32_t at, uint32_t n) {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t pair = (x[k >> 1] >> (16 * (k & 1))) & 0xffffu;
            const bool in0 = 2 * k - at < n, in1 = 2 * k + 1 - at < n;
            const uint32_t m = (in0 ? 0xffu : 0u) | (in1 ? 0xff00u : 0u);
            w.any_hi |= pair & m & 0xe0e0u;
            w.all &= pair | ~m;
            const uint32_t c0 = pair & 31u, c1 = (pair >> 8) & 31u;
            walk.fetch_step(in0 ? (in1 ? c0 | c1 << 5 : kSingle + c0) : in1 ? kSingle + c1 : kIdentity);
        }
    };

    if (sp.n_first) masked(first, sp.lo, sp.n_first);
    stream_span<PF>(sp.body, sp.full, [&](const uint4 (&a)[PF]) { words(a, std::integral_constant<int, PF>{}); },
                    [&](const uint4& v) { words(&v, std::integral_constant<int, 1>{}); });
    if (sp.n_last) masked(last, 0u, sp.n_last);
    walk.finish(w, prm, n_strings, sid, out_state, out_accept);
}

// Waves per SIMD the LDS footprint allows (160 KB per CU), at most 4 (3 for
// the one split whose code spills to scratch at 128 registers).
template <int NF, int NB>
constexpr int compact_waves() {
    constexpr int NW = NF + (NB + 7) / 8;
    constexpr int cap = (NF == 2 && NB == 3) ? 3 : 4;
    const int blocks = (160 * 1024) / (kEntries * NW * 8 + order_bytes(TREX_COMPACT_BLOCK));
    return blocks < 1 ? 1 : (blocks > cap ? cap : blocks);
}

}  // namespace

// wordsg: the launch's compact tables of 1,058 entries (NW / 2 tables of 16
// bytes an entry, then one of 8 bytes when NW is odd), in the kernel's width
#define TREX_COMPACT_KERNEL(NF, NB, SUFFIX, ...)                                                                \
    extern "C" __global__ void __launch_bounds__(TREX_COMPACT_BLOCK)                                            \
    __attribute__((amdgpu_waves_per_eu(compact_waves<NF, NB>())))                                                \
    dfa16_multi_k2fc_f##NF##_b##NB##SUFFIX(const uint8_t* __restrict__ bytes, const int64_t* __restrict__ begin, \
                                          const int64_t* __restrict__ end, int64_t n_strings,                   \
                                          const uint8_t* __restrict__ wordsg, CompactParams prm,                \
                                          uint8_t* __restrict__ out_state, uint8_t* __restrict__ out_accept) {  \
        __VA_ARGS__(bytes, begin, end, n_strings, wordsg, prm, out_state, out_accept);                          \
    }

// _il: interleaved layout; _n8: the full patterns have at most eight live states
#define TREX_COMPACT_BYTES(NF, NB)                                           \
    TREX_COMPACT_KERNEL(NF, NB, , compact_strings<NF, NB, false>)            \
    TREX_COMPACT_KERNEL(NF, NB, _il, compact_groups<NF, NB>)
#define TREX_COMPACT_BOTH(NF, NB)                                            \
    TREX_COMPACT_KERNEL(NF, NB, _n8, compact_strings<NF, NB, true>)         \
    TREX_COMPACT_BYTES(NF, NB)

// every split of 1..8 patterns into full and byte patterns
TREX_COMPACT_BYTES(0, 1) TREX_COMPACT_BYTES(0, 2) TREX_COMPACT_BYTES(0, 3) TREX_COMPACT_BYTES(0, 4)
TREX_COMPACT_BYTES(0, 5) TREX_COMPACT_BYTES(0, 6) TREX_COMPACT_BYTES(0, 7) TREX_COMPACT_BYTES(0, 8)
TREX_COMPACT_BOTH(1, 0) TREX_COMPACT_BOTH(1, 1) TREX_COMPACT_BOTH(1, 2) TREX_COMPACT_BOTH(1, 3)
TREX_COMPACT_BOTH(1, 4) TREX_COMPACT_BOTH(1, 5) TREX_COMPACT_BOTH(1, 6) TREX_COMPACT_BOTH(1, 7)
TREX_COMPACT_BOTH(2, 0) TREX_COMPACT_BOTH(2, 1) TREX_COMPACT_BOTH(2, 2) TREX_COMPACT_BOTH(2, 3)
TREX_COMPACT_BOTH(2, 4) TREX_COMPACT_BOTH(2, 5) TREX_COMPACT_BOTH(2, 6)
TREX_COMPACT_BOTH(3, 0) TREX_COMPACT_BOTH(3, 1) TREX_COMPACT_BOTH(3, 2) TREX_COMPACT_BOTH(3, 3)
TREX_COMPACT_BOTH(3, 4) TREX_COMPACT_BOTH(3, 5)
TREX_COMPACT_BOTH(4, 0) TREX_COMPACT_BOTH(4, 1) TREX_COMPACT_BOTH(4, 2) TREX_COMPACT_BOTH(4, 3)
TREX_COMPACT_BOTH(4, 4)
TREX_COMPACT_BOTH(5, 0) TREX_COMPACT_BOTH(5, 1) TREX_COMPACT_BOTH(5, 2) TREX_COMPACT_BOTH(5, 3)
TREX_COMPACT_BOTH(6, 0) TREX_COMPACT_BOTH(6, 1) TREX_COMPACT_BOTH(6, 2)
TREX_COMPACT_BOTH(7, 0) TREX_COMPACT_BOTH(7, 1)
TREX_COMPACT_BOTH(8, 0)
