// Device helpers and host checks shared by the w64 kernels (GEMV, decode,
// matrix product): the LDS table and staged tile block, the per-state decode
// step, the escape side table, and the geometry checks of the entry points.
// Everything sits in an anonymous namespace: each .hip file is a translation
// unit of its own.  The stream format is documented in include/vramc_rans.h.
#ifndef VRAMC_RANS_DEVICE_H
#define VRAMC_RANS_DEVICE_H

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "../../include/vramc_rans.h"

namespace {

constexpr uint32_t kProbM = 4096;
constexpr uint32_t kRansL = 1u << 16;
// Table entry in LDS, in one of two layouts:
//   - 8 bytes {freq | code<<24, slot - cum} (T4 = false): one mad consumes
//     both words and the code is the sign-extended top byte;
//   - 4 bytes freq | (slot - cum)<<12 | code<<24 (T4 = true): half the LDS
//     and half the bytes per random table read, for two more VALU
//     instructions per symbol (a mask and a field extract, one of them on
//     the state's dependency chain).  It pays on batch-1 launches with more
//     workgroups than the chip holds at once: the 16 KB saved per
//     workgroup lets more of them share a CU.
template <bool T4>
using TabEntry = std::conditional_t<T4, uint32_t, uint2>;

constexpr int kLdsMax = 160 * 1024;
constexpr int kBufWord3 = 0x00020000;  // buffer resource word 3 for gfx9 raw loads

// 32-bit LDS addresses (address space 3), so a word read is one ds_read with
// no base arithmetic.
using lds_cu16 = const __attribute__((address_space(3))) uint16_t;
using lds_void = __attribute__((address_space(3))) void;
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ uint32_t lds_read_u16(uint32_t a) {
    return *(lds_cu16*)(uintptr_t)a;
}

// Per-wave LDS region, in 16-bit words: the staged tile block plus one
// read-ahead word past its end.
struct WaveLayout {
    int raw_words;   // multiple of 8
    int wave_words;  // = raw_words
};

// freq*(st>>12) + bias (rans_gemv.cu:34): freq < 2^12 and st>>12 < 2^20
// both fit the 24-bit multiplier, whose operand ignores the code byte.
__device__ __forceinline__ uint32_t entry_next_state(uint2 e, uint32_t st) {
    return __umul24(e.x, st >> 12) + e.y;
}

__device__ __forceinline__ int32_t entry_code(uint2 e) { return (int32_t)e.x >> 24; }

// The 4-byte entry: freq is masked out (the multiplier would take the bias
// bits above it) and the bias extracted from bits 12..23.
__device__ __forceinline__ uint32_t entry_next_state(uint32_t e, uint32_t st) {
    return __umul24(e & 0xFFFu, st >> 12) + __builtin_amdgcn_ubfe(e, 12, 12);
}

__device__ __forceinline__ int32_t entry_code(uint32_t e) { return (int32_t)e >> 24; }

// Direct global->LDS copy (global_load_lds_dwordx4): lane i's 16 bytes land
// at the wave-uniform LDS address base + 16*i.  The copy is complete when
// the wave's vector-memory counter has drained (wait_vm).
__device__ __forceinline__ void copy16_to_lds(const uint4* src_lane, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds(src_lane, (lds_void*)lds_wave_base, 16, 0, 0);
}

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima), as a builtin
// so the compiler's own wait tracking knows every vector load is complete.
__device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The table image (32 KB of 8-byte or 16 KB of 4-byte entries, laid out as
// in LDS): chunks of 64 x 16 bytes, wave w of W copying chunks w, w+W, ...
// Issued after the tile block's copy: the table comes from L2 (every
// workgroup reads it), the block from HBM, so the block's copy is the one
// to start first.
template <class E>
__device__ __forceinline__ void stage_table(E* tab, const uint4* __restrict__ img, int wave, int W,
                                            int lane) {
    constexpr int nchunks = (int)(sizeof(E) * kProbM / 1024);
    for (int c = wave; c < nchunks; c += W)
        copy16_to_lds(img + c * 64 + lane, reinterpret_cast<uint4*>(tab) + c * 64);
}

// Extent of tile t's block: tile_off[t], tile_off[t+1] (loaded by every
// lane; the wave-uniform values are taken by tile_extent, as late as
// possible, so the loads issued in between are not waited for).
struct TileOff {
    uint32_t lo, hi;
};
__device__ __forceinline__ TileOff load_tile_off(const uint32_t* __restrict__ tile_off, int t) {
    return {tile_off[t], tile_off[t + 1]};
}

// Start (in words) and length (in 16-byte units, at most the region) of the
// block, as scalars; n16 is 0 for an inactive wave.
__device__ __forceinline__ void tile_extent(TileOff to, bool active, int raw_words, uint32_t& o0,
                                            uint32_t& n16) {
    uint32_t nw = to.hi - to.lo;
    if (nw > (uint32_t)raw_words) nw = (uint32_t)raw_words;
    o0 = __builtin_amdgcn_readfirstlane(to.lo);
    n16 = active ? __builtin_amdgcn_readfirstlane(nw >> 3) : 0u;
}

// The wave's tile block (n16 x 16 bytes at words + 8*o16) into its LDS region.
__device__ __forceinline__ void stage_tile(uint16_t* raw, const uint16_t* __restrict__ words,
                                           uint32_t o0, uint32_t n16, int lane) {
    const uint4* src = reinterpret_cast<const uint4*>(words + o0);
    for (uint32_t c = 0; c < n16; c += 64)
        if (c + lane < n16) copy16_to_lds(src + c + lane, reinterpret_cast<uint4*>(raw) + c);
}

__device__ __forceinline__ uint32_t load_x_bits(const void* x, int64_t i, bool bf16) {
    if (bf16) return reinterpret_cast<const uint16_t*>(x)[i];
    return reinterpret_cast<const uint32_t*>(x)[i];
}

__device__ __forceinline__ float bits_to_x(uint32_t v, bool bf16) {
    return __uint_as_float(bf16 ? v << 16 : v);
}

template <typename T>
__device__ __forceinline__ T raw_load(__amdgpu_buffer_rsrc_t r, int off) {
    if constexpr (std::is_same_v<T, __bf16>)
        return __builtin_bit_cast(__bf16, __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
    else
        return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}

__device__ __forceinline__ float raw_to_x(__bf16 v) { return (float)v; }
__device__ __forceinline__ float raw_to_x(uint32_t v) { return __uint_as_float(v); }

__device__ __forceinline__ float load_x(const void* x, int64_t i, bool bf16) {
    return bits_to_x(load_x_bits(x, i, bf16), bf16);
}

// v from lane (dpp CTRL) for the rows in ROWS; 0 in the other rows.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, false));
}

// Sum over the 64 lanes with DPP moves (no LDS round trips); the total is
// valid in lane 63.  Fixed order, so the result is deterministic.
__device__ __forceinline__ float wave_sum63(float v) {
    v += dpp<0xB1>(v);        // quad_perm [1,0,3,2]
    v += dpp<0x4E>(v);        // quad_perm [2,3,0,1]: quad sums
    v += dpp<0x141>(v);       // row_half_mirror: sums of 8
    v += dpp<0x140>(v);       // row_mirror: row (16-lane) sums
    v += dpp<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
    v += dpp<0x143, 0xC>(v);  // row_bcast:31 into rows 2, 3
    return v;
}

// Sums each of N values (a power of two up to 64) over the 64 lanes with
// about 2.2*N instructions instead of 6*N.  Stage j (j = 0..5) pairs the
// lanes that differ in lane-id bit 5-j.  While a lane holds n > 1 values it
// keeps the half selected by that bit and adds its partner's copy of the
// same half, so the value count halves; once n = 1 a stage is a plain pair
// sum.  Partners: v_permlane32_swap / v_permlane16_swap exchange the halves
// directly for bits 5 and 4; DPP row_mirror, row_half_mirror and quad_perm
// reach them for bits 3..0 (a mirror pairs lanes differing in that bit, and
// lanes that share the bits already summed hold disjoint lane sets).  Every
// lane ends with the complete total of value index lane >> (6 - log2 N).
template <int J, int N>
__device__ __forceinline__ void wave_transpose_stage(float* w, int lane) {
    if constexpr (J < 6) {
        constexpr int bit = 5 - J;
        constexpr int CTRL = J == 2 ? 0x140 : J == 3 ? 0x141 : J == 4 ? 0x4E : 0xB1;
        constexpr int h = N > 1 ? N / 2 : 1;
        const bool hi = (lane >> bit) & 1;
#pragma unroll
        for (int i = 0; i < h; i++) {
            const float a = w[i], b = N > 1 ? w[i + h] : w[i];
            if constexpr (J == 0) {
                const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                                false, false);
                w[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
            } else if constexpr (J == 1) {
                const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
                                                                false, false);
                w[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
            } else if constexpr (N > 1) {
                w[i] = (hi ? b : a) + dpp<CTRL>(hi ? a : b);
            } else {
                w[i] = a + dpp<CTRL>(a);
            }
        }
        wave_transpose_stage<J + 1, h>(w, lane);
    }
}

template <int N>
__device__ __forceinline__ float wave_transpose_sum(float (&v)[N], int lane) {
    static_assert(N >= 1 && N <= 64 && (N & (N - 1)) == 0, "N must be a power of two <= 64");
    wave_transpose_stage<0, N>(v, lane);
    return v[0];
}

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

// Sums each of the N values w[OFF..OFF+N) over the 64 lanes into
// out[OFF..OFF+N), for any N: power-of-two chunks of at most 64 values,
// largest first (35 = 32 + 2 + 1), each through wave_transpose_sum.
template <int OFF, int N, int NT>
__device__ __forceinline__ void transpose_sum_store(const float (&w)[NT], float* out, int lane) {
    if constexpr (N > 0) {
        constexpr int C = N >= 64 ? 64 : 1 << ilog2(N);
        float v[C];
#pragma unroll
        for (int i = 0; i < C; i++) v[i] = w[OFF + i];
        const float t = wave_transpose_sum<C>(v, lane);
        constexpr int sh = 6 - ilog2(C);
        if ((lane & ((1 << sh) - 1)) == 0) out[OFF + (lane >> sh)] = t;
        transpose_sum_store<OFF + C, N - C, NT>(w, out, lane);
    }
}

// Inclusive prefix sum over the 64 lanes: within each 16-lane row with
// row_shr 1, 2, 4, 8 (a lane without a source in its row adds 0), then the
// row totals carried into the rows above with row_bcast 15 and 31.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 to rows 1, 3
    v += __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 to rows 2, 3
    return v;
}

// Where each of the lane's S states lives in the tile block, from its
// length byte lb (length - base | exponent << 4) and the tile's meta word
// (base | blob words << 16): off, the word offset of its stream (the
// streams follow the blob in state order, j = s*64 + lane), and bit, the
// bit offset of its initial state's mantissa in the blob (16 + e bits per
// state, in state order).  Both sums go through one scan, packed in the two
// halves of a word (a wave's lengths stay below 2^16 words and its
// mantissas below 2^11 bits).
template <int S>
__device__ __forceinline__ void stream_layout(const uint32_t (&lb)[S], uint32_t meta,
                                              uint32_t (&off)[S], uint32_t (&bit)[S]) {
    const uint32_t base = meta & 0xFFu;
    uint32_t ocarry = meta >> 16, bcarry = 0;
#pragma unroll
    for (int s = 0; s < S; s++) {
        const uint32_t v = (base + (lb[s] & 15u)) | (16u + (lb[s] >> 4)) << 16;
        const uint32_t inc = wave_scan(v);
        const uint32_t ex = inc - v;
        off[s] = ocarry + (ex & 0xFFFFu);
        bit[s] = bcarry + (ex >> 16);
        const uint32_t tot = __builtin_amdgcn_readlane(inc, 63);
        ocarry += tot & 0xFFFFu;
        bcarry += tot >> 16;
    }
}

// A state's initial value from the staged blob: the 16 + e bits at bit
// offset `bit` below an implicit leading one.
__device__ __forceinline__ uint32_t initial_state(const uint16_t* raw, uint32_t bit, uint32_t lb) {
    const uint32_t* r32 = reinterpret_cast<const uint32_t*>(raw);
    const uint32_t lo = r32[bit >> 5], hi = r32[(bit >> 5) + 1];
    const uint32_t nb = 16u + (lb >> 4);
    return __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(hi, lo, bit & 31u), 0, nb) | (1u << nb);
}

// Per-lane decoder state of S interleaved rANS states, with the table entry
// of each state's next symbol already read (software pipelined: the read for
// symbol i+1 is issued before the GEMV work of symbol i).
template <int S, class E>
struct Lanes {
    uint32_t st[S];  // rANS states
    uint32_t a[S];   // LDS byte address of the next unread word of each state
    uint32_t w[S];   // that word (read ahead)
    E e[S];          // table entry for the next symbol of each state
};

// Staged-block setup: each state's read pointer, its first word and the
// table entry of its first symbol.  Call after the staging barrier.
template <int S, class E>
__device__ __forceinline__ void init_lanes(Lanes<S, E>& L, const E* tab, const uint16_t* raw,
                                           const uint32_t (&st0)[S], const uint32_t (&off0)[S]) {
#pragma unroll
    for (int s = 0; s < S; s++) {
        L.st[s] = st0[s];
        L.a[s] = lds_addr(raw + off0[s]);
        L.w[s] = lds_read_u16(L.a[s]);
        L.e[s] = tab[L.st[s] & (kProbM - 1)];
    }
}

// One rANS decode step with the reference arithmetic (rans_gemv.cu:32-37):
// st = freq*(st>>12) + bias from the entry e = tab[st & 4095]; renormalise
// with the next stream word when st < 2^16; return the symbol's code.  The
// entry for the following symbol is read as soon as the new state exists,
// before the code conversion and the word-pointer update, so those overlap
// the LDS latency instead of sitting on the state's dependency chain.
//
// The next word w is always read ahead.  REFILL=false: every lane re-reads
// it each step (no divergence, the cheapest step when LDS is not the
// bottleneck).  REFILL=true: only the lanes that just consumed their word
// fetch the next one (an EXEC-masked read, about 1 lane in 5 at 3 bits per
// symbol), which cuts LDS bank traffic where many waves share the CU.
template <bool REFILL, class E>
__device__ __forceinline__ int32_t rans_step(uint32_t& st, uint32_t& a, uint32_t& w, E& e,
                                             const E* tab) {
    const E cur = e;
    const uint32_t ns = entry_next_state(cur, st);
    const bool need = ns < kRansL;
    st = need ? ((ns << 16) | w) : ns;
    e = tab[st & (kProbM - 1)];
    if (REFILL) {
        if (need) {
            a += 2u;
            w = lds_read_u16(a);
        }
    } else {
        a += need ? 2u : 0u;
        w = lds_read_u16(a);
    }
    return entry_code(cur);
}

// Tile row and tile column of a side-table position c*R + r (R is a
// compile-time constant, so the division is a multiply and shift).
template <int R>
__device__ __forceinline__ int esc_row(int pos) { return (int)((uint32_t)pos % (uint32_t)R); }
template <int R>
__device__ __forceinline__ uint32_t esc_tcol(int pos) { return (uint32_t)pos / (uint32_t)R; }

// Adds an escape entry at tile row re to the lane's accumulators; v[b] is
// value*step*x[b] (0 for a lane without an entry).  A 0/1 weight per row and
// one FMA per (row, batch): 2R + RB instructions rather than R + 2RB for a
// select and an add.
template <int R, int B>
__device__ __forceinline__ void add_escape(float (&acc)[R][B], int re, const float (&v)[B]) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float m = re == r ? 1.f : 0.f;
#pragma unroll
        for (int b = 0; b < B; b++) acc[r][b] = fmaf(m, v[b], acc[r][b]);
    }
}

// Adds v to a float in LDS (ds_add_f32; no value returned).
__device__ __forceinline__ void lds_add(float* p, float v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// bf16 of f, round to nearest even (gfx950's v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// bf16 of lo and hi in the two halves of a word (one v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t to_bf16x2(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// ------------------------------------------------------------------ host
WaveLayout wave_layout(const rans_w64_matrix* m) {
    WaveLayout L;
    L.raw_words = (m->max_tile_words + 8 + 7) & ~7;
    L.wave_words = L.raw_words;
    return L;
}

// Dynamic LDS bytes of a launch (the static arrays come on top).
size_t lds_bytes(int waves, const WaveLayout& L) { return (size_t)waves * L.wave_words * 2; }

// Largest byte extent a kernel addresses through one buffer resource
// (an R-row slice of a decoded int32 output): it must fit the 32-bit range.
bool fits_buffer_ranges(const rans_w64_matrix* m) {
    return (int64_t)m->R * m->cols * 4 <= (int64_t)INT32_MAX;
}

bool valid_geometry(const rans_w64_matrix* m) {
    if (!m ||
        (m->flags & ~(RANS_F_WORDS_MASK | RANS_F_NO_ESCAPES | RANS_F_TABLE4 | RANS_F_TABLE8)) ||
        (m->flags & RANS_F_WORDS_MASK) == RANS_F_WORDS_MASK ||
        ((m->flags & RANS_F_TABLE4) && (m->flags & RANS_F_TABLE8)))
        return false;
    if (m->rows <= 0 || m->cols <= 0 || m->R <= 0 || m->C <= 0 || m->S <= 0) return false;
    if (m->rows % m->R || m->cols % m->C || m->C % (64 * m->S)) return false;
    if (m->max_tile_words <= 0 || m->max_tile_words > 65536) return false;
    if (m->max_state_words <= 0 || m->max_state_words > m->max_tile_words) return false;
    return fits_buffer_ranges(m);
}

bool valid_pointers(const rans_w64_matrix* m) {
    return m->words && m->tile_off && m->slen && m->tile_meta && m->table_lds && m->step &&
           m->esc_tileptr && m->esc_pos && m->esc_val;
}

// Opt in to more than 64 KB of LDS once per kernel (bytes dynamic, plus
// static_bytes or more of static __shared__ arrays).
std::mutex g_attr_mu;
const void* g_attr_done[512];
int g_attr_n = 0;

hipError_t ensure_lds(const void* fn, size_t bytes, int static_bytes) {
    if (bytes + static_bytes <= 65536) return hipSuccess;
    std::lock_guard<std::mutex> lk(g_attr_mu);
    for (int i = 0; i < g_attr_n; i++)
        if (g_attr_done[i] == fn) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kLdsMax - static_bytes);
    if (e == hipSuccess && g_attr_n < 512) g_attr_done[g_attr_n++] = fn;
    return e;
}

// CUs of the current device, cached per device; 0 when the query fails.
std::atomic<int> g_cus[64];

int device_cus() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 0;
    if (dev < 64) {
        const int v = g_cus[dev].load(std::memory_order_relaxed);
        if (v > 0) return v;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    if (dev < 64) g_cus[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// Tiles taller than 16 rows take one state per lane.  R = 35 splits rows of
// 8960 = 256 x 35 into 256 tile rows, so that 8960 x 1536 (Qwen2.5-1.5B's
// gate and up projections) runs as 2048 tiles of 35 x 192: two waves on
// every SIMD.  R = 20 is for large matrices, whose launches take more than
// one round of resident workgroups: 25600 rows make 1280 tile rows instead
// of 1600 with R = 16, so the last of the rounds of 768 workgroups is two
// thirds full instead of 8% (25600x5120 at batch 1: 54.8 -> 51.9 us), with
// fewer, longer states (2.923 -> 2.880 bits/weight).
bool supported_rs(int R, int S) {
    return ((R == 1 || R == 2 || R == 3 || R == 4 || R == 8 || R == 16) && (S == 1 || S == 2 || S == 4)) ||
           ((R == 20 || R == 35) && S == 1);
}

}  // namespace

#endif  // VRAMC_RANS_DEVICE_H
