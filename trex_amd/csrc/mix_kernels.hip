// One persistent launch over a mixed batch of DFA-16 and Boolean NFA-64
// patterns and strings of uneven length (gfx950, wave64).
//
// The host (mix.cpp) turns the batch into a queue of work batches. A work
// batch holds up to kMixBlock lane items of ONE pattern and one role, so the
// workgroup that claims it stages that pattern's tables in LDS once (skipped
// when the previous batch had the same pattern). Workgroups claim batches from
// an atomic ticket until the queue is empty. Roles:
//
//   DFA_WHOLE  a string walked from the start state: pair-function table f2
//              (two bytes per LDS lookup) with the 32-byte symbol window check
//   DFA_CHUNK  one chunk of a long string, chained by the decoupled look-back
//              over 16-state functions (the scheme of scan_kernels.hip)
//   NFA_WHOLE  a string walked by the bit-parallel NFA-64 step
//   NFA_SPEC   one chunk of a long string: the first chunk of the string is
//              walked from the start set; every other chunk is walked from
//              the pattern's guess set `warm` bytes ahead of it, which makes a
//              guess of the set it is entered with, and on to its end (some
//              patterns have a second guess: NFA handle). Its end is known when
//              the chunk before it ends in that set (taken from the
//              neighbouring lane, or published by the wave before) and was
//              entered with the right set itself, up to sticky sets
//              (known_end(): text that was found before stays found). Long chunks also record their set every kCk bytes (checkpoints)
//   NFA_FIXUP  one per long string, after all its NFA_SPEC chunks are done:
//              when every chunk's guess was right, the last end and the sticky
//              sets found on the way are the string's. Otherwise it goes over
//              the chunks: where the guesses make a chunk's end known, that is
//              taken; any other chunk is walked again from the set it is
//              entered with, with checkpoints only until the set recorded at
//              the same position makes the end known. The result is exact
//              either way. Many strings take a lane each, few a wave each
//
// Forward progress: the queue puts every batch that is waited on before the
// batches that wait on it (DFA chunks after their predecessors, fix-ups after
// all NFA_SPEC batches), so every waited-on item has been claimed by a running
// workgroup, which publishes it before it waits itself. A DFA chunk never waits
// on a chunk of its own wave (those come by shuffle). Waits are bounded by a
// poll count (max_spins) and by wall-clock ticks (max_ticks); on expiry the
// error word is set and the wave moves on. Fix-ups of a wave each stand behind
// the whole strings, since each holds a workgroup while it waits.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

#define MIX_BLOCK 512
#define MIX_BLOCK_SLICE 1024

namespace {

using namespace trexdev;

constexpr uint32_t kRoleDfaWhole = 0, kRoleDfaChunk = 1, kRoleNfaWhole = 2, kRoleNfaSpec = 3, kRoleNfaFixup = 4;
constexpr uint32_t kStatusAggregate = 1u, kStatusPrefix = 2u;
constexpr int kNfaClasses = 34;   // window bytes 0..31, reject, skip
constexpr int kFixupBlock = 4;    // chunks a fix-up of one lane reads at once

constexpr int kSticky = 4;

struct Sticky {
    uint64_t state;   // a state outside the start set that every symbol keeps (a mask; 0: unused)
    uint64_t set;     // what it leads to, closed under every symbol
};

// Pattern descriptor (host layout in mix.cpp).
struct MixPattern {
    uint32_t kind;        // 0 DFA, 1 NFA
    uint32_t win4;        // window base byte x 0x01010101
    uint32_t start;       // DFA start state
    uint32_t dead;        // DFA dead state
    uint32_t nstates;     // DFA state count (<= 16)
    uint32_t reserved;
    uint64_t nstart;      // NFA start set
    uint64_t naccept;     // NFA accept set
    uint64_t nguess;      // NFA set a chunk's guess is walked from
    uint64_t nsecond;     // and its second guess, 0: none
    Sticky sticky[kSticky];   // of NFAs whose guesses are walked from the start set
    const uint8_t* t1;    // DFA byte table [256][16]
    const uint8_t* t2;    // DFA pair rows [1024][16]
    const uint8_t* f2;    // DFA pair functions [1024] x uint64
    const uint8_t* acc;   // DFA accept [16]
    const uint8_t* ntab;  // NFA window tables: [34][256] x uint64 (bank-swizzled) or 6/5-bit slices
    const uint8_t* ncls;  // NFA byte -> class [256]
};

struct MixArgs {
    const uint8_t* bytes;
    const MixPattern* patterns;
    const int32_t* bfirst;    // batch: first item
    const int32_t* bcount;    // batch: item count
    const int32_t* bpattern;  // batch: pattern
    const int32_t* brole;     // batch: role
    int32_t n_batches;
    int32_t ck;               // NFA checkpoint spacing in bytes (multiple of 16)
    const int64_t* ibeg;      // item: byte range (FIXUP: first NFA_SPEC item)
    const int64_t* iend;      //       (FIXUP: one past the last NFA_SPEC item)
    const int32_t* ia;        // item: DFA_CHUNK predecessor item / NFA string slot
    const int32_t* ib;        // item: output string, -1 if none
    const int32_t* ic;        // item: NFA_SPEC checkpoint ordinal
    const uint32_t* iflags;   // item: bit 0 first chunk of its string
    int32_t n_ck;             // checkpoints per NFA_SPEC item, 0: none recorded
    int32_t warm;             // bytes walked ahead of a NFA_SPEC chunk for its guess (at most a chunk)
    uint32_t* ticket;
    uint32_t* status;         // per item (DFA_CHUNK; NFA_SPEC: 1 once its end is published)
    uint64_t* agg;            // two words per item (DFA_CHUNK: function, item to go on from; NFA_SPEC: both guesses)
    uint32_t* done;           // per NFA string slot: finished NFA_SPEC chunks
    uint32_t* unmet;          // per NFA string slot: chunks whose guess is wrong after their predecessor's end
    uint64_t* found;          // per NFA string slot: sticky sets reached in some chunk, missing from the next one's guess
    uint64_t* ckpt;           // [n_spec][n_ck]
    uint64_t* spec_exit;      // [n_spec][2], of both guesses
    uint32_t* error;
    uint32_t* converged;      // chunks whose end the fix-ups took as recorded
    uint32_t max_spins;       // wait bound in polls (0: none)
    uint32_t reserved;
    uint64_t max_ticks;       // wait bound in wall-clock ticks
    uint64_t* out_mask;       // per string: DFA final state / NFA final set
    uint8_t* out_accept;      // per string
};

// ---------------------------------------------------------------------------
// DFA roles
// ---------------------------------------------------------------------------

struct DfaLds {
    const uint8_t* t1;     // [256][16]
    const uint8_t* t2;     // [1024][16]
    const uint64_t* f2;    // [1024]
    const uint8_t* acc;    // [16]
};

__device__ __forceinline__ uint32_t k2f_word(const uint64_t* __restrict__ f2, uint32_t s, uint32_t x) {
    const uint64_t a = f2[pair_lo(x)];
    const uint64_t b = f2[pair_hi(x)];
    s = (uint32_t)(a >> (s << 2)) & 15u;
    return (uint32_t)(b >> (s << 2)) & 15u;
}

__device__ __forceinline__ uint32_t dfa_walk(const uint8_t* __restrict__ bytes, int64_t p, int64_t end, const DfaLds& L,
                             const MixPattern& P) {
    uint32_t s = P.start;
    const Span sp(bytes, p, end);
    const uint4 first = sp.first(), last = sp.last();
    auto byte = [&](uint32_t b) { s = L.t1[(b << 4) | s]; };
    each_byte(first, sp.lo, sp.n_first, byte);
    WinCheck w;
    w.init();
    stream_body<8>(sp.body, sp.full, [&](uint4 v) {
        w.add(v.x); w.add(v.y); w.add(v.z); w.add(v.w);
        s = k2f_word(L.f2, s, v.x);
        s = k2f_word(L.f2, s, v.y);
        s = k2f_word(L.f2, s, v.z);
        s = k2f_word(L.f2, s, v.w);
    });
    each_byte(last, 0u, sp.n_last, byte);
    if (w.outside(P.win4)) s = P.dead;
    return s;
}

// Walk one state or compose the function of a chunk (window pair rows).
struct ChunkScanner {
    const DfaLds* L;
    bool walking;
    uint32_t s;
    Fn16 f;
    WinCheck w;
    __device__ __forceinline__ void byte(uint32_t b) {
        if (walking) s = L->t1[(b << 4) | s];
        else f = fn_then(f, load_row(L->t1, b));
    }
    __device__ __forceinline__ void word(uint32_t x) {
        w.add(x);
        if (walking) {
            s = k2f_word(L->f2, s, x);
        } else {
            f = fn_then(f, load_row(L->t2, pair_lo(x)));
            f = fn_then(f, load_row(L->t2, pair_hi(x)));
        }
    }
    __device__ __forceinline__ void settle() {
        if (!walking && fn_is_const(f)) {
            walking = true;
            s = f.d[0] & 0xffu;
        }
    }
    // One 16-byte vector, walked or composed as decided once for the whole
    // wave: when every active lane walks, the branch-free path issues the
    // vector's pair-function reads together (a per-lane test around each
    // word made every word wait for its own reads).
    __device__ __forceinline__ void vector(const uint4& a) {
        if (__ballot(!walking) == 0ull) {
            w.add(a.x); w.add(a.y); w.add(a.z); w.add(a.w);
            s = k2f_word(L->f2, s, a.x);
            s = k2f_word(L->f2, s, a.y);
            s = k2f_word(L->f2, s, a.z);
            s = k2f_word(L->f2, s, a.w);
        } else {
            word(a.x); word(a.y); word(a.z); word(a.w);
            settle();
        }
    }
};

// One chunk per lane; every lane of the workgroup calls it (inactive lanes
// take part in the wave's shuffles). Always inlined into the persistent loop.
__device__ __forceinline__ void dfa_chunk(const MixArgs& A, const MixPattern& P, const DfaLds& L, int64_t item,
                                          bool active) {
    ChunkScanner sc;
    sc.L = &L;
    sc.w.init();
    int32_t pred = -1;
    int64_t p = 0, end = 0;
    if (active) {
        pred = (A.iflags[item] & 1u) ? -1 : A.ia[item];
        p = A.ibeg[item];
        end = A.iend[item];
    }
    sc.walking = pred < 0;
    sc.s = P.start;
    sc.f = fn_identity_on(P.nstates);
    const Span sp(A.bytes, p, end);
    const uint4 first = sp.first(), last = sp.last();
    auto byte = [&](uint32_t b) { sc.byte(b); };
    each_byte(first, sp.lo, sp.n_first, byte);
    stream_body<4>(sp.body, sp.full, [&](const uint4& a) { sc.vector(a); });
    each_byte(last, 0u, sp.n_last, byte);
    sc.settle();
    if (sc.w.outside(P.win4)) { sc.walking = true; sc.s = P.dead; }

    // In-wave chains in registers (as in scan_kernels.hip): a lane whose
    // predecessor item lies in its own wave takes that lane's function by
    // shuffle; pointer jumping leaves in g the composition from the chain's
    // root lane up to this one. Only roots look back through memory, and a
    // root's predecessor belongs to another wave (of this workgroup or of an
    // earlier batch), which publishes without waiting on this one.
    const uint32_t lane = threadIdx.x & 63u;
    const int64_t wave_first = item - (int64_t)lane;
    const bool own_known = pred < 0 || sc.walking;
    Fn16 g = own_known ? fn_const(sc.s) : sc.f;
    const bool inwave = active && (int64_t)pred >= wave_first;
    uint32_t root = inwave ? (uint32_t)((int64_t)pred - wave_first) : lane;
    bool closed = !inwave;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        Fn16 up;
        up.d[0] = __shfl(g.d[0], (int)root, 64);
        up.d[1] = __shfl(g.d[1], (int)root, 64);
        up.d[2] = __shfl(g.d[2], (int)root, 64);
        up.d[3] = __shfl(g.d[3], (int)root, 64);
        const bool up_closed = __shfl((int)closed, (int)root, 64) != 0;
        const uint32_t up_root = (uint32_t)__shfl((int)root, (int)root, 64);
        if (!closed) {
            g = fn_then(up, g);   // the earlier lanes' chunks apply first
            closed = up_closed;
            root = up_root;
        }
    }

    // A chunk whose chain function is constant knows its final state and
    // publishes PREFIX at once; any other publishes the function of its chain
    // up to here and the predecessor of the chain's root, where a look-back
    // that meets it goes on (one step per wave of a string's chunks).
    const int32_t root_pred = __shfl(pred, (int)root, 64);
    const bool known = fn_is_const(g);
    const uint32_t kstate = g.d[0] & 0xffu;
    if (active) {
        if (known) {
            store_relaxed(&A.status[item], kStatusPrefix | (kstate << 8));   // the word says it all
        } else {
            A.agg[2 * item] = fn_pack(g);
            A.agg[2 * item + 1] = (uint64_t)(int64_t)root_pred;
            store_release(&A.status[item], kStatusAggregate);   // agg first
        }
    }
    uint32_t incoming = 0;
    if (active && !known && root == lane) {
        uint64_t acc_fn = 0xfedcba9876543210ull;   // identity
        int32_t j = pred;
        BoundedWait wait(A.max_spins, A.max_ticks);
        while (true) {
            const uint32_t st = load_relaxed(&A.status[j]);
            if (st == 0u) {
                if (wait.expired()) {
                    atomicOr(A.error, 1u);
                    incoming = P.dead;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
                continue;
            }
            if ((st & 0xffu) == kStatusPrefix) {   // the word holds the state
                incoming = nib(acc_fn, (st >> 8) & 15u);
                break;
            }
            fence_acquire();   // agg[j] was written before status[j] was released
            acc_fn = nib_then(A.agg[2 * (int64_t)j], acc_fn);   // the earlier chunks apply first
            j = (int32_t)(int64_t)A.agg[2 * (int64_t)j + 1];
            if (j < 0) {   // cannot happen: a string's first chunk publishes a prefix
                atomicOr(A.error, 2u);
                incoming = P.dead;
                break;
            }
        }
    }
    incoming = __shfl(incoming, (int)root, 64);
    const uint32_t state = known ? kstate : fn_apply(g, incoming);
    if (active && !known) store_relaxed(&A.status[item], kStatusPrefix | (state << 8));
    if (active && A.ib[item] >= 0) {
        A.out_mask[A.ib[item]] = state;
        A.out_accept[A.ib[item]] = L.acc[state];
    }
}

// ---------------------------------------------------------------------------
// NFA roles
// ---------------------------------------------------------------------------

// The NFA step over the tables of the launch's form: nibble tables (34
// classes, reject and skip included, bank-swizzled) with a byte -> class map,
// or 6/5-bit slice tables of the 32 window classes, where every byte enters the
// window check and steps with class byte & 31.
template <bool SLICE>
struct NfaWalker {
    const void* tab;
    const uint8_t* cls;
    uint64_t s;
    WinCheck w;
    __device__ __forceinline__ uint64_t step(uint32_t k, uint64_t x) const {
        if constexpr (SLICE) return nfa6_step(static_cast<const char*>(tab), k, x);
        else return nfa_step(static_cast<const uint64_t*>(tab), k, x);
    }
    __device__ __forceinline__ void byte(uint32_t b) {
        if constexpr (SLICE) {
            w.add(b * 0x01010101u);
            s = step(b & 31u, s);
        } else {
            s = step(cls[b], s);
        }
    }
    __device__ __forceinline__ void word(uint32_t x) {
        w.add(x);
        s = step(x & 31u, s);
        s = step((x >> 8) & 31u, s);
        s = step((x >> 16) & 31u, s);
        s = step((x >> 24) & 31u, s);
    }
    __device__ __forceinline__ void vec(uint4 v) { word(v.x); word(v.y); word(v.z); word(v.w); }
    // A byte outside the window rejects: once seen, the set is empty for good.
    // Applied before every set that is compared or stored, so both forms give
    // the same sets there.
    __device__ __forceinline__ void settle(uint32_t win4) {
        if (w.outside(win4)) s = 0;
        w.init();
    }
};

// f(vector) for the n vectors from v on, two in flight ahead of the one being
// walked, until f returns false. One copy of f: sixteen NFA steps are 15 KB of
// code, and two workgroups of a CU with different roles share 64 KB of
// instruction cache with a second CU. (Blocks of two vectors, unrolled, made 185 KB
// of the kernel, 95 KB now: 1,024 strings of up to 1 MiB 240 us, 234 us; 218 of up
// to 140 KB 123 us, 117 us.)
template <class F>
__device__ __forceinline__ void each_vector(const uint4* __restrict__ v, int64_t n, F&& f) {
    uint4 n0 = make_uint4(0u, 0u, 0u, 0u), n1 = n0;
    if (n > 0) n0 = v[0];
    if (n > 1) n1 = v[1];
#pragma unroll 1
    for (int64_t i = 0; i < n; ++i) {
        const uint4 x = n0;
        n0 = n1;
        if (i + 2 < n) n1 = v[i + 2];
        if (!f(x)) return;
    }
}

template <bool SLICE>
__device__ __forceinline__ uint64_t nfa_walk(const uint8_t* __restrict__ bytes, int64_t p, int64_t end, uint64_t s,
                             const void* tab, const uint8_t* cls, uint32_t win4) {
    NfaWalker<SLICE> nw{tab, cls, s, {}};
    nw.w.init();
    const Span sp(bytes, p, end);
    const uint4 first = sp.first(), last = sp.last();
    auto byte = [&](uint32_t b) { nw.byte(b); };
    each_byte(first, sp.lo, sp.n_first, byte);
    each_vector(sp.body, sp.full, [&](const uint4& x) { nw.vec(x); return true; });
    nw.settle(win4);
    each_byte(last, 0u, sp.n_last, byte);
    nw.settle(win4);
    return nw.s;
}

// Walks [p, end) from set s and stores the set at every absolute position that
// is a multiple of ck (ck a multiple of 16) into ck_out[0..n_ck); n_ck = 0
// stores none.
template <bool SLICE>
__device__ __forceinline__ uint64_t nfa_walk_record(const uint8_t* __restrict__ bytes, int64_t p, int64_t end, uint64_t s,
                                    const void* tab, const uint8_t* cls, uint32_t win4, int32_t ck,
                                    uint64_t* __restrict__ ck_out, int32_t n_ck) {
    NfaWalker<SLICE> nw{tab, cls, s, {}};
    nw.w.init();
    const Span sp(bytes, p, end);
    const uint4 first = sp.first(), last = sp.last();
    auto byte = [&](uint32_t b) { nw.byte(b); };
    each_byte(first, sp.lo, sp.n_first, byte);
    p += sp.n_first;
    // vectors to the first multiple of ck after p (positions off the vectors'
    // grid meet none), then ck / 16 at a time; no division per vector
    const int64_t to_ck = (p + 16 + ck - 1) / ck * ck - p;
    int32_t left = n_ck > 0 && (to_ck & 15) == 0 ? (int32_t)(to_ck >> 4) : 0;
    int32_t idx = 0;
    each_vector(sp.body, sp.full, [&](const uint4& x) {
        nw.vec(x);
        if (--left == 0) {
            left = ck >> 4;
            if (idx < n_ck) {
                nw.settle(win4);
                ck_out[idx++] = nw.s;
            }
        }
        return true;
    });
    nw.settle(win4);
    each_byte(last, 0u, sp.n_last, byte);
    nw.settle(win4);
    return nw.s;
}

// The sticky sets that a set of states has reached.
__device__ __forceinline__ uint64_t sticky_of(const MixPattern& P, uint64_t t) {
    uint64_t u = 0;
#pragma unroll 1   // (unrolled, the nibble kernel goes over 128 VGPRs)
    for (int k = 0; k < kSticky && P.sticky[k].state != 0ull; ++k)
        u |= (t & P.sticky[k].state) != 0ull ? P.sticky[k].set : 0ull;
    return u;
}

// The end of a walk from `t` when a walk over the same bytes from g, which ends
// in e, makes it known. A step is linear in the set: a walk from g | sticky ends
// in e and the sticky sets, which stay as they are unless a byte rejects and
// empties everything. (g holds a start state that every symbol keeps unless it
// is empty itself: e is empty only then.)
__device__ __forceinline__ bool known_end(const MixPattern& P, uint64_t t, uint64_t g, uint64_t e, uint64_t& out) {
    if (t == g) {
        out = e;
        return true;
    }
    const uint64_t sticky = sticky_of(P, t);
    if (g == 0ull || t != (g | sticky)) return false;
    out = e != 0ull ? e | sticky : 0ull;
    return true;
}

// The same with a second guess, whose set and end are g1 and e1 (in memory:
// written, and needed, for few patterns).
__device__ __forceinline__ bool known_end(const MixPattern& P, uint64_t t, uint64_t g, uint64_t e,
                                          const uint64_t* __restrict__ g1, const uint64_t* __restrict__ e1,
                                          uint64_t& out) {
    if (known_end(P, t, g, e, out)) return true;
    return P.nsecond != 0ull && g != 0ull &&
           known_end(P, t, g | load_through(g1), e != 0ull ? e | load_through(e1) : 0ull, out);
}

// Walks [p, end) from set s, up to the first multiple of ck where the set
// recorded there (ck_in, by nfa_walk_record; `stop` is that walk's end) makes
// the end known: reported through `met`.
template <bool SLICE>
__device__ __forceinline__ uint64_t nfa_walk_meet(const uint8_t* __restrict__ bytes, int64_t p, int64_t end, uint64_t s,
                                  const void* tab, const uint8_t* cls, const MixPattern& P, int32_t ck,
                                  const uint64_t* __restrict__ ck_in, int32_t n_ck, uint64_t stop, bool& met) {
    const uint32_t win4 = P.win4;
    NfaWalker<SLICE> nw{tab, cls, s, {}};
    nw.w.init();
    met = false;
    const Span sp(bytes, p, end);
    const uint4 first = sp.first(), last = sp.last();
    auto byte = [&](uint32_t b) { nw.byte(b); };
    each_byte(first, sp.lo, sp.n_first, byte);
    p += sp.n_first;
    int32_t idx = 0;
    int64_t next_ck = (p + 16 + ck - 1) / ck * ck;
    uint64_t out = 0;
    each_vector(sp.body, sp.full, [&](const uint4& x) {
        nw.vec(x);
        p += 16;
        if (p != next_ck) return true;
        next_ck += ck;
        if (idx < n_ck) {
            nw.settle(win4);
            met = known_end(P, nw.s, ck_in[idx++], stop, out);
        }
        return !met;
    });
    if (met) return out;
    nw.settle(win4);
    each_byte(last, 0u, sp.n_last, byte);
    nw.settle(win4);
    return nw.s;
}

// Waits for the chunks of a fix-up's string. True when its end is known, false
// when some guess was wrong; s is then the end of the first chunk.
__device__ __forceinline__ bool fixup_known(const MixArgs& A, int64_t item, uint64_t& s, uint32_t& converged) {
    const int64_t c0 = A.ibeg[item], c1 = A.iend[item];
    const uint32_t need = (uint32_t)(c1 - c0);
    const int32_t slot = A.ia[item];
    const int64_t o0 = A.ic[c0];
    s = 0;
    converged = 0;
    BoundedWait wait(A.max_spins, A.max_ticks);
    while (load_relaxed(&A.done[slot]) < need) {
        if (wait.expired()) {
            atomicOr(A.error, 4u);
            return true;
        }
        __builtin_amdgcn_s_sleep(8);
    }
    // guesses and ends were written through before each chunk counted itself
    if (A.n_ck) fence_acquire();
    const uint64_t first = load_through(&A.spec_exit[2 * o0]), last = load_through(&A.spec_exit[2 * (o0 + need - 1)]);
    const uint64_t found = load_through(&A.found[slot]);
    const bool known = load_relaxed(&A.unmet[slot]) == 0u;
    s = !known ? first : last != 0ull ? last | found : 0ull;   // (the first chunk was walked from the start set)
    if (known) converged = need - 1u;
    return known;
}

__device__ __forceinline__ void fixup_result(const MixArgs& A, const MixPattern& P, int64_t item, uint64_t s,
                                             uint32_t converged) {
    if (converged != 0u) atomicAdd(A.converged, converged);
    A.out_mask[A.ib[item]] = s;
    A.out_accept[A.ib[item]] = (s & P.naccept) != 0 ? 1 : 0;
}

// A string's fix-up by one lane, chunk after chunk.
template <bool SLICE>
__device__ __forceinline__ void fixup_lane(const MixArgs& A, const MixPattern& P, const void* ntab,
                                           const uint8_t* ncls, int64_t item) {
    uint64_t s;
    uint32_t converged;
    if (!fixup_known(A, item, s, converged)) {
        const int64_t c0 = A.ibeg[item], c1 = A.iend[item], o0 = A.ic[c0];
        // the empty set is absorbing: once the true set is empty, so are all later exits
        for (int64_t c = c0 + 1; c < c1 && s != 0; c += kFixupBlock) {
            // guesses and ends of the next chunks (items and ordinals of a string are
            // consecutive), read together
            uint64_t ends[kFixupBlock], guesses[kFixupBlock];
#pragma unroll
            for (int k = 0; k < kFixupBlock; ++k) {
                const int64_t j = min(c + k, c1 - 1);
                ends[k] = load_through(&A.spec_exit[2 * (o0 + (j - c0))]);
                guesses[k] = load_through(&A.agg[2 * j]);
            }
            bool known = true;
            uint64_t t = s;
#pragma unroll
            for (int k = 0; k < kFixupBlock; ++k) {
                const int64_t j = c + k;
                if (j < c1)
                    known = known && known_end(P, t, guesses[k], ends[k], &A.agg[2 * j + 1],
                                               &A.spec_exit[2 * (o0 + (j - c0)) + 1], t);
            }
            if (known) {
                s = t;
                converged += (uint32_t)min<int64_t>(kFixupBlock, c1 - c);
                continue;
            }
            for (int64_t j = c; j < min(c + kFixupBlock, c1) && s != 0; ++j) {
                const int64_t o = o0 + (j - c0);
                const uint64_t stop = load_through(&A.spec_exit[2 * o]);
                bool met = known_end(P, s, load_through(&A.agg[2 * j]), stop, &A.agg[2 * j + 1],
                                     &A.spec_exit[2 * o + 1], s);
                if (!met)
                    s = nfa_walk_meet<SLICE>(A.bytes, A.ibeg[j], A.iend[j], s, ntab, ncls, P, A.ck,
                                             A.ckpt + o * A.n_ck, A.n_ck, stop, met);
                converged += met ? 1u : 0u;
            }
        }
    }
    fixup_result(A, P, item, s, converged);
}

// A string's fix-up by a whole wave, 64 chunks at a time: lane k has chunk k
// enter with what chunk k - 1 ends in as far as it is known, and walks it again
// where the guesses do not give its end for that set, until no entry set changes
// any more. The first chunk's entry set is the true one, so each round makes at
// least one more chunk final: where sets coincide somewhere in a chunk, one or
// two rounds do, where they never do it takes as long as one lane. Walks that
// coincide at a letter every 50 / 100 / 200 / 500 bytes, 16 strings of 1 MiB in
// 512 byte chunks: 179 / 185 / 182 / 184 ms by a lane, 3.7 / 4.1 / 7.2 / 16.5 ms
// by a wave; at no letter 185 and 220 ms.
template <bool SLICE>
__device__ __forceinline__ void fixup_wave(const MixArgs& A, const MixPattern& P, const void* ntab,
                                           const uint8_t* ncls, int64_t item, uint64_t t) {
    const uint32_t lane = threadIdx.x & 63u;
    const int64_t c0 = A.ibeg[item], c1 = A.iend[item], o0 = A.ic[c0];
    uint32_t converged = 0;
    auto lane_of = [](uint64_t x, int from) {
        return (uint64_t)(uint32_t)__shfl((int)(uint32_t)x, from, 64) |
               ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(x >> 32), from, 64) << 32);
    };
    for (int64_t c = c0 + 1; c < c1 && t != 0ull; c += 64) {   // t: the true set so far, the same in every lane
        const int64_t j = min(c + lane, c1 - 1), o = o0 + (j - c0);
        const bool have = c + lane < c1;
        const uint64_t g = load_through(&A.agg[2 * j]), e = load_through(&A.spec_exit[2 * o]);
        auto entry = [&](uint64_t outs) {
            const uint64_t up = lane_of(outs, (int)max(lane, 1u) - 1);
            return lane > 0u ? up : t;
        };
        uint64_t in = entry(e), out = 0, walked_in = 0, walked_out = 0;   // (an empty set stays empty)
        bool known, met = false;
        while (true) {
            known = known_end(P, in, g, e, &A.agg[2 * j + 1], &A.spec_exit[2 * o + 1], out);
            if (!known) {
                if (have && in != walked_in) {
                    walked_in = in;
                    walked_out = nfa_walk_meet<SLICE>(A.bytes, A.ibeg[j], A.iend[j], in, ntab, ncls, P, A.ck,
                                                      A.ckpt + o * A.n_ck, A.n_ck, e, met);
                }
                out = walked_out;
            }
            const uint64_t next = entry(out);
            if (__ballot(have && next != in) == 0ull) break;
            in = next;
        }
        converged += (uint32_t)__popcll(__ballot(have && (known || met)));
        t = lane_of(out, (int)min<int64_t>(c1 - 1 - c, 63));
    }
    if (lane == 0u) fixup_result(A, P, item, t, converged);
}

// Puts a pattern's tables in LDS unless they are there (layout in mix_loop).
template <bool SLICE>
__device__ __forceinline__ void stage_pattern(uint8_t* lds, const MixPattern& P, int32_t pat, int32_t& loaded) {
    if (pat == loaded) return;
    if (P.kind == 0) {
        stage_table(lds, P.t1, 4096);
        stage_table(lds + 4096, P.t2, 16384);
        stage_table(lds + 20480, P.f2, 8192);
        stage_table(lds + 28672, P.acc, 16);
    } else if constexpr (SLICE) {
        stage_table_far(lds, P.ntab, (int)kTab6Bytes);
    } else {
        stage_table_far(lds, P.ntab, kNfaClasses * 2048);
        stage_table(lds + kNfaClasses * 2048, P.ncls, 256);
    }
    __syncthreads();
    if (threadIdx.x == 0) loaded = pat;
}

// One persistent workgroup's loop. Dynamic LDS: the NFA tables of the form
// (nibble: kNfaClasses * 2048 + 256 bytes; 6/5-bit slices: kTab6Bytes); the
// DFA tables use the first 29 KB of the same space.
template <bool SLICE, bool WAVES>
__device__ __forceinline__ void mix_loop(const MixArgs& A)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ int32_t s_batch;
    __shared__ int32_t s_loaded;
    __shared__ int32_t s_walk;
    if (threadIdx.x == 0) s_loaded = -1;

    DfaLds dl;
    dl.t1 = lds;                                              // 4 KB
    dl.t2 = lds + 4096;                                       // 16 KB
    dl.f2 = reinterpret_cast<const uint64_t*>(lds + 20480);   // 8 KB
    dl.acc = lds + 28672;                                     // 16 B
    const void* ntab = lds;
    const uint8_t* ncls = SLICE ? nullptr : lds + kNfaClasses * 2048;

    while (true) {
        __syncthreads();   // the previous batch is finished with LDS and s_batch
        if (threadIdx.x == 0) s_batch = (int32_t)atomicAdd(A.ticket, 1u);
        __syncthreads();
        const int32_t b = __builtin_amdgcn_readfirstlane(s_batch);   // uniform: the pattern is read by scalar loads
        if (b >= A.n_batches) break;
        const int32_t pat = A.bpattern[b];
        const uint32_t role = (uint32_t)A.brole[b];
        const MixPattern& P = A.patterns[pat];
        const int32_t count = A.bcount[b];
        const bool active = (int32_t)threadIdx.x < count;
        const int64_t item = (int64_t)A.bfirst[b] + threadIdx.x;

        if (WAVES && role == kRoleNfaFixup) {   // one string, the first wave; tables only if it walks
            uint64_t s = 0;
            uint32_t converged;
            if (threadIdx.x < 64u) {
                const bool known = fixup_known(A, A.bfirst[b], s, converged);
                if (threadIdx.x == 0u) s_walk = known ? 0 : 1;
                if (threadIdx.x == 0u && known) fixup_result(A, P, A.bfirst[b], s, converged);
            }
            __syncthreads();
            if (s_walk == 0) continue;
            stage_pattern<SLICE>(lds, P, pat, s_loaded);
            if (threadIdx.x < 64u) fixup_wave<SLICE>(A, P, ntab, ncls, A.bfirst[b], s);
            continue;
        }
        stage_pattern<SLICE>(lds, P, pat, s_loaded);
        if (role == kRoleDfaChunk) {
            // every lane takes part: the look-back publishes before it waits
            dfa_chunk(A, P, dl, item, active);
            continue;
        }
        if (!active) continue;
        if (role == kRoleDfaWhole) {
            const uint32_t s = dfa_walk(A.bytes, A.ibeg[item], A.iend[item], dl, P);
            A.out_mask[A.ib[item]] = s;
            A.out_accept[A.ib[item]] = dl.acc[s];
        } else if (role == kRoleNfaWhole) {
            const uint64_t s = nfa_walk<SLICE>(A.bytes, A.ibeg[item], A.iend[item], P.nstart, ntab, ncls, P.win4);
            A.out_mask[A.ib[item]] = s;
            A.out_accept[A.ib[item]] = (s & P.naccept) != 0 ? 1 : 0;
        } else if (role == kRoleNfaSpec) {
            const bool first = (A.iflags[item] & 1u) != 0;
            const int32_t o = A.ic[item];
            const int64_t p = A.ibeg[item], end = A.iend[item];
            uint64_t guess = 0, s = 0, exit = 0;   // of the first guess
            const int parts = P.nsecond != 0ull && !first ? 4 : 2;
#pragma unroll 1
            for (int part = 0; part < parts; ++part) {   // the bytes ahead, then the chunk: one copy of the walk
                const bool ahead = (part & 1) == 0;
                if (ahead) s = first ? P.nstart : part == 0 ? P.nguess : P.nsecond;
                else store_through(&A.agg[2 * item + (part >> 1)], s);
                const int64_t from = ahead && !first ? p - A.warm : p;
                if (part == 1) guess = s;
                s = nfa_walk_record<SLICE>(A.bytes, from, ahead ? p : end, s, ntab, ncls, P.win4, A.ck,
                                           A.ckpt + (int64_t)o * A.n_ck, part == 1 ? A.n_ck : 0);
                if (!ahead) store_through(&A.spec_exit[2 * (int64_t)o + (part >> 1)], s);
                if (part == 1) exit = s;
            }
            // the chunk before this one is the item before it: the lane below,
            // or the last lane of the wave before (of this batch or an earlier
            // one), which publishes before it waits itself
            const uint32_t lane = threadIdx.x & 63u;
            if (A.n_ck) __threadfence();   // checkpoints are ordinary stores
            wait_stores();
            if (lane == 63u || (int32_t)threadIdx.x == count - 1) store_relaxed(&A.status[item], 1u);
            uint64_t before = (uint64_t)(uint32_t)__shfl_up((int)(uint32_t)exit, 1, 64) |
                              ((uint64_t)(uint32_t)__shfl_up((int)(uint32_t)(exit >> 32), 1, 64) << 32);
            bool met = first || lane > 0u;
            if (!met) {
                BoundedWait wait(A.max_spins, A.max_ticks);
                while (!(met = load_relaxed(&A.status[item - 1]) != 0u) && !wait.expired())
                    __builtin_amdgcn_s_sleep(2);
                before = load_through(&A.spec_exit[2 * (int64_t)(o - 1)]);
                if (!met) atomicOr(A.error, 4u);
            }
            const int32_t slot = A.ia[item];
            if (!first && before != guess) {
                const uint64_t sticky = sticky_of(P, before);
                met = met && guess != 0ull && before == (guess | sticky);   // as in known_end
                // (once a string and sticky set, as a rule: later chunks find it there)
                if (met && (sticky & ~load_through(&A.found[slot])) != 0ull)
                    atomicOr(reinterpret_cast<unsigned long long*>(&A.found[slot]), (unsigned long long)sticky);
            }
            // one atomic per string and wave (they are served one after another,
            // about 70 ns each: one per chunk of a long string adds up)
            wait_stores();
            bool left = true;
            for (uint64_t todo; (todo = __ballot(left)) != 0ull;) {
                const int32_t of = __shfl(slot, (int)__builtin_ctzll(todo), 64);
                const uint64_t mine = __ballot(left && slot == of), un = __ballot(left && slot == of && !met);
                if (left && slot == of) {
                    if (lane == (uint32_t)__builtin_ctzll(mine)) {
                        if (un) {
                            atomicAdd(&A.unmet[of], (uint32_t)__popcll(un));
                            wait_stores();
                        }
                        atomicAdd(&A.done[of], (uint32_t)__popcll(mine));
                    }
                    left = false;
                }
            }
        } else if constexpr (!WAVES) {
            fixup_lane<SLICE>(A, P, ntab, ncls, item);
        }
    }
}

}  // namespace

// Nibble NFA tables: two 512-thread workgroups per CU (70 KB of LDS each). _waves:
// a fix-up is one string to a batch and a wave, otherwise one to a lane.
#define MIX_KERNEL(NAME, BLOCK, ...)                                                                       \
    extern "C" __global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) NAME(MixArgs A) { \
        mix_loop<__VA_ARGS__>(A);                                                                          \
    }
MIX_KERNEL(mix_persistent, MIX_BLOCK, false, false)
MIX_KERNEL(mix_persistent_waves, MIX_BLOCK, false, true)

// 6/5-bit slice NFA tables (12 reads per byte instead of 16): one
// 1024-thread workgroup per CU (128 KB of LDS).
MIX_KERNEL(mix_persistent_slice, MIX_BLOCK_SLICE, true, false)
MIX_KERNEL(mix_persistent_slice_waves, MIX_BLOCK_SLICE, true, true)
