// Byte-class form of a DFA byte table: the tables of dfa_class_kernels.hip, built
// from a full byte table, and the launch of its kernels over contiguous strings.

#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <vector>

#include "runtime_internal.h"

namespace trex {

namespace {

// Classes of bytes with equal columns of delta, numbered by first byte;
// returns their count.
int byte_classes(const uint8_t* delta, int n, uint8_t (&cls)[256]) {
    std::map<std::vector<uint8_t>, int> seen;
    std::vector<uint8_t> column((size_t)n);
    for (int b = 0; b < 256; ++b) {
        for (int s = 0; s < n; ++s) column[s] = delta[s * 256 + b];
        cls[b] = (uint8_t)seen.emplace(column, (int)seen.size()).first->second;
    }
    return (int)seen.size();
}

// Largest pair table of a wide DFA's class form: with the map it leaves four
// workgroups a CU.
constexpr int kWidePairBytes = 36 << 10;

// Arguments of the class kernels (same layout in dfa_class_kernels.hip).
struct ClassArgs {
    const uint8_t* bytes;
    const int64_t* begin;
    const int64_t* end;
    int64_t n_strings;
    const uint8_t* tab;
    uint32_t tab_bytes;
    uint32_t classes;
    uint32_t accept;
    uint32_t start;
    const uint8_t* acc;
    const uint64_t* masks;
    uint8_t* out_state;
    uint64_t* out_mask;
    uint8_t* out_accept;
};

// Launch shape of the class kernels: from kClassBlockFrom strings on, 256
// threads a workgroup, which orders its strings by length (kOrderBytes of LDS);
// below, one wave a workgroup, so that the waves spread over the CUs, while the
// LDS holds the tables of all of them at once (60,000 strings and rows of 200
// states, 50 KB: 1 to 2 KB a string 132 us by waves, 69 us by workgroups of 256;
// 8 to 30 bytes: 10.9 and 6.4 us).
constexpr int64_t kClassBlockFrom = 65536;
constexpr int kLdsBytes = 160 << 10;   // of a compute unit
constexpr unsigned kOrderBytes = 64 * 4 + 256 * 2;   // order_bytes(256) of device_common.h

// Byte-class tables of the class kernels (layouts in dfa_class_kernels.hip)
// and the kernel they are for; an empty result when the table has too many
// classes for either form.
std::vector<uint8_t> class_tables(const uint8_t* delta, int n, const char** kernel, int* classes) {
    uint8_t cls[256];
    const int count = byte_classes(delta, n, cls);
    std::vector<uint8_t> out;
    std::vector<int> byte_of(count, 0);   // one byte of each class
    for (int b = 255; b >= 0; --b) byte_of[cls[b]] = b;
    auto next = [&](int s, int c) { return c == count ? s : (int)delta[s * 256 + byte_of[c]]; };
    if (n <= 16) {
        if (count > 31) return out;   // class * 8 fits a byte, the identity class included
        const int all = count + 1, odd = all | 1;
        // field width, what a field holds per successor state, first bit (Width in dfa_class_kernels.hip)
        const int w = n <= 10 ? 6 : 4, mul = n <= 10 ? 6 : 1, first = n > 10 && n <= 15 ? 2 : 0;
        *kernel = n <= 10 ? "dfa16_cls_n10" : n <= 15 ? "dfa16_cls_n15" : "dfa16_cls_n16";
        std::vector<uint64_t> f2((size_t)(all * odd + 1) & ~(size_t)1, 0);
        for (int c1 = 0; c1 < all; ++c1)
            for (int c0 = 0; c0 < all; ++c0)
                for (int s = 0; s < n; ++s)
                    f2[c0 + c1 * odd] |= (uint64_t)(mul * next(next(s, c0), c1)) << (w * s + first);
        out.resize(256 + f2.size() * 8);
        for (int b = 0; b < 256; ++b) out[b] = (uint8_t)(8 * cls[b]);
        memcpy(out.data() + 256, f2.data(), f2.size() * 8);
        *classes = all;
        return out;
    }
    const int all = count + 1, stride = (n + 15) / 16 * 16;
    if (all * all * stride > kWidePairBytes) {
        *kernel = "dfa_cls_rows";
        *classes = stride;
        out.resize((size_t)256 * stride, 0);
        for (int b = 0; b < 256; ++b)
            for (int s = 0; s < n; ++s) out[(size_t)b * stride + s] = delta[s * 256 + b];
        return out;
    }
    *kernel = "dfa_cls_pair";
    out.resize(1040 + (size_t)all * all * stride, 0);
    uint32_t* map = reinterpret_cast<uint32_t*>(out.data());
    for (int b = 0; b < 257; ++b) {
        const uint32_t c = b < 256 ? cls[b] : (uint32_t)count;
        map[b] = (c * all * stride) | (c * stride) << 16;
    }
    for (int r = 0; r < all * all; ++r)
        for (int s = 0; s < n; ++s) out[1040 + (size_t)r * stride + s] = (uint8_t)next(next(s, r / all), r % all);
    return out;
}

}  // namespace

int make_class_form(const uint8_t* delta, const uint8_t* accept, const uint64_t* masks, int n, int start,
                    ClassForm* out) {
    std::vector<uint8_t> tab = class_tables(delta, n, &out->kernel, &out->classes);
    if (tab.empty()) return TREX_OK;
    out->tab_bytes = (int)tab.size();
    out->start = start;
    for (int s = 0; s < n && s < 32; ++s) out->accept |= accept[s] ? 1u << s : 0u;
    // one upload: the tables, the accept bytes, the masks
    out->acc_at = (tab.size() + 15) & ~(size_t)15;
    out->masks_at = (out->acc_at + n + 15) & ~(size_t)15;
    tab.resize(out->masks_at + (masks ? (size_t)n * 8 : 0), 0);
    for (int s = 0; s < n; ++s) tab[out->acc_at + s] = accept[s] ? 1 : 0;
    if (masks) memcpy(tab.data() + out->masks_at, masks, (size_t)n * 8);
    return upload((void**)&out->d_tab, tab.data(), tab.size());
}

int launch_class_form(const ClassForm& f, const uint8_t* d_bytes, const int64_t* d_begin, const int64_t* d_end,
                      int64_t n_strings, bool leave_alike, uint8_t* d_state, uint64_t* d_mask, uint8_t* d_accept,
                      hipStream_t stream) {
    const int64_t resident = (int64_t)device_cu_count() * (kLdsBytes / f.tab_bytes);   // tables
    const unsigned block = n_strings < kClassBlockFrom && n_strings <= 64 * resident ? 64u : kBlock;
    const int64_t blocks = (n_strings + block - 1) / block;
    if (blocks > 0x7fffffff) return fail(TREX_ERR_CAPACITY, "too many strings");
    const unsigned lds = (unsigned)f.tab_bytes + (block == kBlock ? kOrderBytes : 0u);
    ClassArgs A = {d_bytes, d_begin, d_end, n_strings, f.d_tab, (uint32_t)f.tab_bytes, (uint32_t)f.classes, f.accept,
                   (uint32_t)f.start, f.d_tab + f.acc_at, reinterpret_cast<const uint64_t*>(f.d_tab + f.masks_at),
                   d_state, d_mask, d_accept};
    void* args[] = {&A};
    char name[48];
    std::snprintf(name, sizeof(name), "%s%s", f.kernel, d_mask ? "_mask" : leave_alike ? "_left" : "");
    return launch(name, (unsigned)blocks, block, lds, stream, args);
}

}  // namespace trex
