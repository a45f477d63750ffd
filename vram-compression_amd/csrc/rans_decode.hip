// Decode of the w64 stream to a dense matrix (bf16 code*step, or int32
// codes) on MI355X (gfx950).  The stream format is documented in
// include/vramc_rans.h, the decode step in rans_device.h.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/vramc_rans.h"
#include "rans_device.h"

namespace {

// Waves of a decode workgroup (tiles are taken linearly, any count works).
constexpr int kMaxDecodeWaves = 10;
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

// Decode only.  MODE 0 writes int32 codes, MODE 1 writes bf16(code*step[c]).
// One wave per tile, the staging and decode step of the GEMV.  Output goes
// through one buffer resource over the tile row's R output rows: a store's
// row is its scalar offset, its column step an immediate.  After its own
// stores have completed, each wave overwrites the escape positions of its
// tile (decoded as 0) with their side-table values, so no second launch.
template <int R, int S, int MODE>
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
    const int t = blockIdx.x * W + wave;
    const bool active = t < a.ntiles;
    const int tc = active ? t : a.ntiles - 1;
    const int rb = tc / a.ncb, cb = tc - rb * a.ncb;
    asm volatile("" ::"s"(a.tile_off), "s"(a.tile_meta), "s"(a.slen), "s"(a.table_lds),
                 "s"(a.words), "s"(a.step), "s"(a.esc_tileptr), "s"(a.out), "s"(a.C),
                 "s"(a.cols), "s"(a.L.raw_words), "s"(a.W), "s"(a.ncb), "s"(a.ntiles));

    const TileOff to = load_tile_off(a.tile_off, tc);
    const int tp = a.esc_tileptr[tc + min(lane, 1)];
    asm volatile("" ::: "memory");  // keep these two loads first
    const uint32_t tmv = a.tile_meta[tc];
    uint32_t len0[S];
#pragma unroll
    for (int s = 0; s < S; s++) len0[s] = a.slen[tc * nst + 64 * s + lane];
    const int nk = a.C / nst;
    const int colbase = cb * a.C + lane;
    const __amdgpu_buffer_rsrc_t srs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.step), 0, a.cols * 4, kBufWord3);
    float sr[KU][S];
    auto load_steps = [&](int k0) {
        const int c0 = colbase + 64 * S * k0;
#pragma unroll
        for (int u = 0; u < KU; u++)
#pragma unroll
            for (int s = 0; s < S; s++)
                sr[u][s] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(srs, (c0 + 64 * (S * u + s)) * 4, 0, 0));
    };
    if (MODE == 1) load_steps(0);
    uint32_t o0, n16;
    tile_extent(to, active, a.L.raw_words, o0, n16);
    stage_tile(raw, a.words, o0, n16, lane);
    stage_table(tab, a.table_lds, wave, W, lane);
    wait_vm();
    __syncthreads();
    if (!active) return;

    uint8_t* obase = static_cast<uint8_t*>(a.out) + (size_t)rb * R * a.cols * ESZ;
    const __amdgpu_buffer_rsrc_t ors =
        __builtin_amdgcn_make_buffer_rsrc(obase, 0, R * a.cols * ESZ, kBufWord3);
    Lanes<S, TabEntry<false>> L;
    uint32_t off0[S], bit0[S], st0[S];
    stream_layout<S>(len0, __builtin_amdgcn_readfirstlane(tmv), off0, bit0);
#pragma unroll
    for (int s = 0; s < S; s++) st0[s] = initial_state(raw, bit0[s], len0[s]);
    init_lanes(L, tab, raw, st0, off0);
    // One block of nu <= KU column steps.  The loop below runs whole blocks
    // only (nu = KU, no early exit): exits after 1, 2 or 3 steps' stores
    // would meet at the loop latch, and the compiler would then wait there
    // for the stores of the longest path.  A partial last block follows it.
    auto run_block = [&](int k0, int nu) {
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
            load_steps(k0 + KU);
            asm volatile("" ::: "memory");
        }
        const int vb = (colbase + 64 * S * k0) * ESZ;
#pragma unroll
        for (int u = 0; u < KU; u++) {
            if (u >= nu) break;
#pragma unroll
            for (int r = 0; r < R; r++) {
#pragma unroll
                for (int s = 0; s < S; s++) {
                    // symbol order within a state is k-major, r-minor, as in the GEMV
                    const int32_t code = rans_step<(R >= 8)>(L.st[s], L.a[s], L.w[s], L.e[s], tab);
                    const int vo = vb + 64 * (S * u + s) * ESZ;
                    if (MODE == 0)
                        __builtin_amdgcn_raw_buffer_store_b32(code, ors, vo, r * a.cols * 4, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b16(to_bf16((float)code * sv[u][s]), ors,
                                                              vo, r * a.cols * 2, 0);
                }
            }
        }
    };
    const int nk_full = nk - nk % KU;
    for (int k0 = 0; k0 < nk_full; k0 += KU) run_block(k0, KU);
    if (nk_full < nk) run_block(nk_full, nk - nk_full);

    // Escapes of this tile: its own side-table entries, written over the 0
    // each escape position was decoded as.  The wave's own stores complete
    // first, so the value lands after that 0.  Positions are clamped into
    // the tile, so no side-table content can address outside the output.
    if (!a.has_esc) return;
    wait_vm();
    const int e_lo = __builtin_amdgcn_readlane(tp, 0), e_hi = __builtin_amdgcn_readlane(tp, 1);
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

// Waves per decode workgroup: among the counts whose LDS fits, the one that
// puts the fewest waves on the busiest CU when the workgroups spread evenly
// over the CUs, the largest such (fewer table copies).
int decode_waves(const rans_w64_matrix* m) {
    const WaveLayout L = wave_layout(m);
    const int64_t ntiles = (int64_t)(m->rows / m->R) * (m->cols / m->C);
    const int cus = device_cus();
    int best = 0;
    int64_t best_load = 0;
    for (int w = 1; w <= kMaxDecodeWaves; w++) {
        if (lds_bytes(w, L) + kDecodeStaticLds > (size_t)kLdsMax) break;
        const int64_t grid = (ntiles + w - 1) / w;
        const int64_t load = cus > 0 ? (grid + cus - 1) / cus * w : -w;
        if (!best || load <= best_load) best = w, best_load = load;
    }
    return best;
}

template <int R, int S, int MODE>
int launch_decode_t(const DecodeArgs& a, int waves, size_t lds, int grid, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&rans_w64_decode_kernel<R, S, MODE>);
    hipError_t e = ensure_lds(fn, lds, kDecodeStaticLds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((rans_w64_decode_kernel<R, S, MODE>), dim3(grid), dim3(64 * waves), lds,
                       stream, a);
    return (int)hipGetLastError();
}

template <int MODE>
int dispatch_decode(const DecodeArgs& a, int R, int S, int waves, size_t lds, int grid,
                    hipStream_t st) {
#define VRAMC_DEC_CASE(RR, SS) \
    if (R == RR && S == SS) return launch_decode_t<RR, SS, MODE>(a, waves, lds, grid, st);
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
    const int waves = decode_waves(m);
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
    a.ntiles = (m->rows / m->R) * a.ncb;
    a.W = waves;
    a.has_esc = !(m->flags & RANS_F_NO_ESCAPES);
    a.L = wave_layout(m);
    const int grid = (a.ntiles + waves - 1) / waves;
    return dispatch_decode<MODE>(a, m->R, m->S, waves, lds_bytes(waves, a.L), grid, stream);
}

}  // namespace

extern "C" int rans_w64_decode(const rans_w64_matrix* m, void* out_bf16, hipStream_t stream) {
    return launch_decode_common<1>(m, out_bf16, stream);
}

extern "C" int rans_w64_decode_codes(const rans_w64_matrix* m, int32_t* out, hipStream_t stream) {
    return launch_decode_common<0>(m, out, stream);
}
