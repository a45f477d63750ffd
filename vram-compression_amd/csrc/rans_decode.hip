// Decode of the w64 stream to a dense matrix (bf16 code*step, or int32
// codes) on MI355X (gfx950).  The stream format is documented in
// include/vramc_rans.h, the decode step in rans_device.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "../../include/vramc_rans.h"
#include "rans_device.h"

namespace {

// Waves of a decode workgroup (tiles are taken linearly, any count works).
constexpr int kMaxDecodeWaves = 16;
constexpr int64_t kPairWeights = 108 << 20;
constexpr int kNonTemporal = 2;  // cache policy of a raw buffer store
constexpr int kDecodeStaticLds = (int)sizeof(TabEntry<false>) * (int)kProbM;

struct DecodeArgs {
    const uint16_t* words;
    const uint32_t* tile_off;
    const uint8_t* slen;
    const uint32_t* tile_meta;
    const uint4* table_lds;
    const int32_t* esc_tileptr;
    const uint16_t* esc_pos;  // tile-local index c*R + r
    const int16_t* esc_val;
    const float* step;
    void* out;
    int rows, cols, C, ncb, ntiles;
    int W;        // waves per workgroup
    int has_esc;  // 0: the side table is empty
    WaveLayout L;
};

// v of the lane that quad_perm CTRL pairs with this one.
template <int CTRL>
__device__ __forceinline__ uint32_t quad_swap(uint32_t v) {
    return __builtin_amdgcn_update_dpp(0u, v, CTRL, 0xF, 0xF, true);
}

// Decode only.  MODE 0 writes int32 codes, MODE 1 writes bf16(code*step[c]).
// One wave per tile at a time, the staging and decode step of the GEMV.
// Output goes through one buffer resource over the tile row's R output rows:
// a store's row is its scalar offset, its column step an immediate.  Once
// its own stores have completed, each wave overwrites the escape positions of
// its tile (decoded as 0) with their side-table values, so no second launch.
//
// What bounds a large decode is its writes: storing into a window of 16 tile
// rows, which stays in the caches, 25600x5120 takes 58 us instead of 100, and
// writing the same bytes without decoding about 50.  So a bf16 output that
// fills the 256 MB memory-side cache but for a sixth or less (kPairWeights)
// goes out in
//   - PAIR: one 4-byte store for two rows.  Lanes l and l^1 hold neighbouring
//     columns, so they exchange halves and the even lane stores both columns
//     of the first row, the odd lane both of the second: half the store
//     instructions, for two more VALU instructions per pair;
//   - non-temporal stores, which keep the caches for the coded input.
// 25600x5120 84.2 -> 56.3 us, with 1% escapes 100.3 -> 86.4; 5120x25600 88.9
// -> 61.9; 34816x5120 100.7 -> 75.0.  (Pairs alone change nothing, and pairs of
// column steps or stores of 512 contiguous bytes over 4 of them ran slower.)
// Smaller outputs are stored plainly: escapes, written over their tile's
// values, then find them in the cache, as does a matrix product that reads the
// output next.  Plain and non-temporal, us: 28672x4096 (224 MB) 70.8 and 53.1,
// with 1% escapes 86.9 and 76.6; 20480x5120 (200 MB) 49.5 and 46.2, with
// escapes 58.4 and 69.0, with a product of 32 rows 82.3 and 95.9; 16384x4096
// (128 MB) 31.7 and 30.4, 35.5 and 45.3, 54.1 and 62.1.
//
// LOOP: workgroups stay, one or two a CU; each wave takes tiles first, first +
// stride, ... and copies the next tile's block as soon as it has decoded the
// last, so the table is copied once per workgroup and a wave waits for no
// other.  5120x5120 in 8x1024 tiles (3200 of them, formerly in workgroups of
// one wave, 4 waves on a CU) 37.7 -> 17.6 us.
template <int R, int S, int MODE, bool PAIR, bool LOOP>
__global__ void __launch_bounds__(64 * kMaxDecodeWaves) rans_w64_decode_kernel(DecodeArgs a) {
    __shared__ __align__(16) TabEntry<false> tab[kProbM];
    extern __shared__ __align__(16) uint16_t dyn[];
    constexpr int nst = 64 * S;
    constexpr int ESZ = MODE == 0 ? 4 : 2;
    constexpr int KU = S >= 4 ? 2 : 4;
    const int W = a.W;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar tile math
    const int lane = threadIdx.x & 63;
    uint16_t* raw = dyn + (size_t)wave * a.L.wave_words;
    asm volatile("" ::"s"(a.tile_off), "s"(a.tile_meta), "s"(a.slen), "s"(a.table_lds),
                 "s"(a.words), "s"(a.step), "s"(a.esc_tileptr), "s"(a.out), "s"(a.C),
                 "s"(a.cols), "s"(a.L.raw_words), "s"(a.W), "s"(a.ncb), "s"(a.ntiles));
    // LOOP: tiles spread over the workgroups first, so that a last, partial
    // round leaves every CU with about as many waves; otherwise a workgroup's
    // tiles are neighbours, whose blocks are too
    const int stride = gridDim.x * W;
    int t = LOOP ? wave * gridDim.x + blockIdx.x : blockIdx.x * W + wave;
    const bool any = t < a.ntiles;

    // what a tile needs from memory besides its block: extent, side-table
    // range, meta word, lengths; held for the tile in hand and the next one
    struct Head {
        TileOff to;
        int tp;
        uint32_t tmv, len[S];
    };
    auto load_head = [&](int tile) {
        Head h;
        const int tc = min(tile, a.ntiles - 1);
        h.to = load_tile_off(a.tile_off, tc);
        h.tp = a.esc_tileptr[tc + min(lane, 1)];
        // keep these loads first: the block's copy waits for the extent, and
        // left alone the compiler takes its end after all the others
        asm volatile("" ::: "memory");
        h.tmv = a.tile_meta[tc];
#pragma unroll
        for (int s = 0; s < S; s++) h.len[s] = a.slen[tc * nst + 64 * s + lane];
        return h;
    };
    const int nk = a.C / nst;
    const __amdgpu_buffer_rsrc_t srs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.step), 0, a.cols * 4, kBufWord3);
    float sr[KU][S];  // steps of the next block of column steps
    auto load_steps = [&](int c0) {
#pragma unroll
        for (int u = 0; u < KU; u++)
#pragma unroll
            for (int s = 0; s < S; s++)
                sr[u][s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    srs, (c0 + 64 * (S * u + s)) * 4, 0, 0));
    };
    Head cur = load_head(t), next = cur;
    if constexpr (LOOP) next = load_head(t + stride);
    if (MODE == 1) load_steps(t % a.ncb * a.C + lane);
    uint32_t o0, n16;
    tile_extent(cur.to, any, a.L.raw_words, o0, n16);
    stage_tile(raw, a.words, o0, n16, lane);
    stage_table(tab, a.table_lds, wave, W, lane);
    wait_vm();
    __syncthreads();

    const bool odd = lane & 1;
    const uint32_t sel = odd ? 0x03020706u : 0x05040100u;
    while (t < a.ntiles) {  // wave-uniform
        const int rb = t / a.ncb, cb = t - rb * a.ncb;
        const int colbase = cb * a.C + lane;
        const int e_lo = __builtin_amdgcn_readlane(cur.tp, 0), e_hi = __builtin_amdgcn_readlane(cur.tp, 1);
        uint8_t* obase = static_cast<uint8_t*>(a.out) + (size_t)rb * R * a.cols * ESZ;
        const __amdgpu_buffer_rsrc_t ors =
            __builtin_amdgcn_make_buffer_rsrc(obase, 0, R * a.cols * ESZ, kBufWord3);
        Lanes<S, TabEntry<false>> L;
        uint32_t off0[S], bit0[S], st0[S];
        stream_layout<S>(cur.len, __builtin_amdgcn_readfirstlane(cur.tmv), off0, bit0);
#pragma unroll
        for (int s = 0; s < S; s++) st0[s] = initial_state(raw, bit0[s], cur.len[s]);
        init_lanes(L, tab, raw, st0, off0);
        // One block of NU <= KU column steps.  The loop below runs whole blocks
        // only (no early exit): exits after 1, 2 or 3 steps' stores would meet
        // at the loop latch, and the compiler would then wait there for the
        // stores of the longest path.  A partial last block follows it.
        auto run_block = [&](int k0, auto nu_) {
            constexpr int NU = decltype(nu_)::value;
            float sv[KU][S];
            if (MODE == 1) {
#pragma unroll
                for (int u = 0; u < KU; u++)
#pragma unroll
                    for (int s = 0; s < S; s++) {
                        asm volatile("" : "+v"(sr[u][s]));
                        sv[u][s] = sr[u][s];
                    }
                // unconditional: past the last block these read columns of the
                // next tile, or 0 past the end of the matrix, and go unused.  A
                // conditional prefetch merges two wait states at the join, and
                // the compiler then waits for this block's stores as well
                // (vmcnt counts stores too), once per block
                load_steps(colbase + nst * (k0 + KU));
                asm volatile("" ::: "memory");
            }
            const int vb = (colbase + nst * k0) * ESZ;
            // paired stores: the lane pair's first column, in odd lanes one
            // row further down
            const int vp = vb - 2 * (lane & 1) + (odd ? a.cols * 2 : 0);
#pragma unroll
            for (int u = 0; u < NU; u++) {
                float held[S];
#pragma unroll
                for (int r = 0; r < R; r++) {
#pragma unroll
                    for (int s = 0; s < S; s++) {
                        // symbol order within a state is k-major, r-minor, as in the GEMV
                        const int32_t code = rans_step<(R >= 8)>(L.st[s], L.a[s], L.w[s], L.e[s], tab);
                        const int vo = 64 * (S * u + s) * ESZ;
                        if constexpr (MODE == 0) {
                            __builtin_amdgcn_raw_buffer_store_b32(code, ors, vb + vo, r * a.cols * 4, 0);
                        } else {
                            const float v = (float)code * sv[u][s];
                            if (!PAIR || (r == R - 1 && R % 2)) {
                                __builtin_amdgcn_raw_buffer_store_b16(to_bf16(v), ors, vb + vo,
                                                                      r * a.cols * 2, PAIR ? kNonTemporal : 0);
                            } else if (r % 2 == 0) {
                                held[s] = v;
                            } else {
                                const uint32_t p = to_bf16x2(held[s], v);
                                __builtin_amdgcn_raw_buffer_store_b32(
                                    __builtin_amdgcn_perm(quad_swap<0xB1>(p), p, sel), ors, vp + vo,
                                    (r - 1) * a.cols * 2, kNonTemporal);
                            }
                        }
                    }
                }
            }
        };
        const int nk_full = nk - nk % KU;
        for (int k0 = 0; k0 < nk_full; k0 += KU) run_block(k0, std::integral_constant<int, KU>());
        switch (nk - nk_full) {
            case 1: run_block(nk_full, std::integral_constant<int, 1>()); break;
            case 2: if constexpr (KU > 2) run_block(nk_full, std::integral_constant<int, 2>()); break;
            case 3: if constexpr (KU > 2) run_block(nk_full, std::integral_constant<int, 3>()); break;
            default: break;
        }

        // The next tile's block into the wave's region, whose last word has
        // been read (its LDS reads have returned), its first steps and the
        // head of the tile after it, in flight together with this tile's
        // stores.  They are waited for here:
        // a load pending at the loop's entry would make every block wait for
        // the stores before it.
        const int tn = t + stride;
        Head after = next;
        if (LOOP && tn < a.ntiles) {  // wave-uniform
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            tile_extent(next.to, true, a.L.raw_words, o0, n16);
            stage_tile(raw, a.words, o0, n16, lane);
            after = load_head(tn + stride);
            if (MODE == 1) load_steps(tn % a.ncb * a.C + lane);
        } else if (!a.has_esc) {
            return;
        }
        wait_vm();
        // Escapes of this tile: its own side-table entries, written over the 0
        // each escape position was decoded as.  The wave's own stores have
        // completed, so the value lands after that 0.  Positions are clamped into
        // the tile, so no side-table content can address outside the output.
        if (a.has_esc) {
            const int cbase = cb * a.C;
            for (int e = e_lo + lane; e < e_hi; e += 64) {
                const int pos = a.esc_pos[e];
                const int r = esc_row<R>(pos);
                const int col = cbase + (int)min(esc_tcol<R>(pos), (uint32_t)(a.C - 1));
                const int32_t v = a.esc_val[e];
                if (MODE == 0)
                    __builtin_amdgcn_raw_buffer_store_b32(v, ors, (r * a.cols + col) * 4, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b16(to_bf16((float)v * a.step[col]), ors,
                                                          (r * a.cols + col) * 2, 0, 0);
            }
        }
        if (!LOOP) return;
        cur = next;
        next = after;
        t = tn;
    }
}

// Waves of a decode workgroup and workgroups of a launch.
struct DecodeShape {
    int waves;
    int64_t grid;
};

// The bf16 decode: workgroups that stay and loop over the tiles, one a CU, or
// two where the LDS holds two whose waves take the tiles in fewer rounds (a
// second table, but more waves to hide each other's latencies: 20480x2560 in
// 20x512 tiles 29.9 us in one of 10 waves, twice over, 26.8 in two of 10;
// 4096x4096 in 2x1024 tiles of two states 13.9 and 12.2).  Stored past the
// caches (pair) only one: HBM takes the fewer writers' stores faster
// (28672x4096 53.1 us in one, 57.6 in two).  No more waves than give each the
// same number of tiles, but 4 to copy the table (64x256 4.6 us with one wave a
// workgroup, 4.0 with four).
DecodeShape decode_shape_loop(const rans_w64_matrix* m, int64_t ntiles, int cus, bool pair) {
    const WaveLayout L = wave_layout(m);
    DecodeShape best = {0, 0};
    int64_t best_rounds = 0;
    for (int per_cu = 1; per_cu <= (pair ? 1 : 2); per_cu++) {
        int most = 0;
        while (most < kMaxDecodeWaves &&
               per_cu * (lds_bytes(most + 1, L) + kDecodeStaticLds) <= (size_t)kLdsMax)
            most++;
        if (!most) break;
        const int64_t groups = (int64_t)cus * per_cu;
        const int64_t rounds = (ntiles + groups * most - 1) / (groups * most);
        if (best.waves && rounds >= best_rounds) break;
        const int waves = std::max((int)((ntiles + groups * rounds - 1) / (groups * rounds)),
                                   std::min(4, most));
        best = {waves, std::min(groups, (ntiles + waves - 1) / waves)};
        best_rounds = rounds;
    }
    return best;
}

// The decode to int32 codes, whose time is its writes: of the counts that put
// the fewest waves on the busiest CU when the workgroups spread evenly the
// largest, from 4 up (workgroups of fewer waves fill the LDS with tables).
DecodeShape decode_shape_once(const rans_w64_matrix* m, int64_t ntiles, int cus) {
    const WaveLayout L = wave_layout(m);
    int most = 0;
    while (most < 10 && lds_bytes(most + 1, L) + kDecodeStaticLds <= (size_t)kLdsMax) most++;
    DecodeShape best = {0, 0};
    int64_t best_load = 0;
    for (int w = std::max(std::min(4, most), 1); w <= most; w++) {
        const int64_t grid = (ntiles + w - 1) / w;
        const int64_t load = (grid + cus - 1) / cus * w;
        if (!best.waves || load <= best_load) best = {w, grid}, best_load = load;
    }
    return best;
}

template <int R, int S, int MODE, bool PAIR, bool LOOP>
int launch_decode_p(const DecodeArgs& a, int waves, size_t lds, int grid, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&rans_w64_decode_kernel<R, S, MODE, PAIR, LOOP>);
    hipError_t e = ensure_lds(fn, lds, kDecodeStaticLds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((rans_w64_decode_kernel<R, S, MODE, PAIR, LOOP>), dim3(grid), dim3(64 * waves),
                       lds, stream, a);
    return (int)hipGetLastError();
}

template <int R, int S, int MODE>
int launch_decode_t(const DecodeArgs& a, bool pair, int waves, size_t lds, int grid,
                    hipStream_t stream) {
    if constexpr (MODE == 1) {
        const bool loop = (int64_t)grid * waves < a.ntiles;
        if constexpr (R > 1) {
            if (pair)
                return loop ? launch_decode_p<R, S, MODE, true, true>(a, waves, lds, grid, stream)
                            : launch_decode_p<R, S, MODE, true, false>(a, waves, lds, grid, stream);
        }
        if (loop) return launch_decode_p<R, S, MODE, false, true>(a, waves, lds, grid, stream);
    }
    return launch_decode_p<R, S, MODE, false, false>(a, waves, lds, grid, stream);
}

template <int MODE>
int dispatch_decode(const DecodeArgs& a, int R, int S, bool pair, int waves, size_t lds, int grid,
                    hipStream_t st) {
#define VRAMC_DEC_CASE(RR, SS) \
    if (R == RR && S == SS) return launch_decode_t<RR, SS, MODE>(a, pair, waves, lds, grid, st);
#define VRAMC_DEC_R(RR) VRAMC_DEC_CASE(RR, 1) VRAMC_DEC_CASE(RR, 2) VRAMC_DEC_CASE(RR, 4)
    VRAMC_DEC_R(1) VRAMC_DEC_R(2) VRAMC_DEC_R(3) VRAMC_DEC_R(4) VRAMC_DEC_R(8) VRAMC_DEC_R(16)
    VRAMC_DEC_CASE(20, 1) VRAMC_DEC_CASE(35, 1)
#undef VRAMC_DEC_R
#undef VRAMC_DEC_CASE
    return RANS_EUNSUPPORTED;
}

template <int MODE>
int launch_decode_common(const rans_w64_matrix* m, void* out, hipStream_t stream) {
    if (!valid_geometry(m)) return RANS_EGEOMETRY;
    if (!valid_pointers(m) || !out) return RANS_EARG;
    if (!supported_rs(m->R, m->S)) return RANS_EUNSUPPORTED;
    const int64_t ntiles = (int64_t)(m->rows / m->R) * (m->cols / m->C);
    const int cus = device_cus();
    if (cus <= 0) return (int)hipErrorInvalidDevice;
    // paired rows in 4-byte stores (rows are a multiple of 128 bytes: cols is
    // one of 64)
    const bool pair = MODE == 1 && m->R > 1 && (uintptr_t)out % 4 == 0 &&
                      (int64_t)m->rows * m->cols >= kPairWeights;
    const DecodeShape shape = MODE == 1 ? decode_shape_loop(m, ntiles, cus, pair)
                                        : decode_shape_once(m, ntiles, cus);
    const int waves = shape.waves;
    if (!waves) return RANS_EGEOMETRY;
    DecodeArgs a;
    a.words = m->words;
    a.tile_off = m->tile_off;
    a.slen = m->slen;
    a.tile_meta = m->tile_meta;
    a.table_lds = reinterpret_cast<const uint4*>(m->table_lds);
    a.esc_tileptr = m->esc_tileptr;
    a.esc_pos = m->esc_pos;
    a.esc_val = m->esc_val;
    a.step = m->step;
    a.out = out;
    a.rows = m->rows;
    a.cols = m->cols;
    a.C = m->C;
    a.ncb = m->cols / m->C;
    a.ntiles = (int)ntiles;
    a.W = waves;
    a.has_esc = !(m->flags & RANS_F_NO_ESCAPES);
    a.L = wave_layout(m);
    return dispatch_decode<MODE>(a, m->R, m->S, pair, waves, lds_bytes(waves, a.L), (int)shape.grid,
                                 stream);
}

}  // namespace

extern "C" int rans_w64_decode(const rans_w64_matrix* m, void* out_bf16, hipStream_t stream) {
    return launch_decode_common<1>(m, out_bf16, stream);
}

extern "C" int rans_w64_decode_codes(const rans_w64_matrix* m, int32_t* out, hipStream_t stream) {
    return launch_decode_common<0>(m, out, stream);
}
