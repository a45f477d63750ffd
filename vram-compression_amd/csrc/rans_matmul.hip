// Decode fused with a matrix product on the matrix cores: out = x * W^T + bias
// for up to 64 rows of x in bf16, W = bf16(code * step) as the decode to a
// dense matrix rounds it, sums in f32, on MI355X (gfx950).  The stream format
// is documented in include/vramc_rans.h, the decode step in rans_device.h.
//
// The GEMV's multiplies are per row of x, and beyond 8 or 16 rows bind it;
// decoding to memory, a dense product and a pass for bias and type spend most
// of their time outside the decode.  Here each wave decodes its tile 64
// columns (R symbols) at a time into LDS and the matrix cores multiply behind
// the decode; the weights never reach memory.  5120x5120 at 32 rows: 37.9 ->
// 26.2 us a call, 34.0 -> 25.1 in a replayed graph.
//
// Bound by the decode's instructions while x is short (5120x5120 at 17 rows
// 24.5 us, 18 of them what decoding to memory takes) and from there on by the
// reads of x, which every wave makes from the caches for its own columns, at
// 7 to 9 TB/s: hence T tile rows to a wave where those reads cost more than
// the waves given up for them.
//
// Shape: a workgroup holds one table copy and rpw groups of T whole tile rows,
// a wave to each T tiles of a column, up to 16 waves; the waves of a tile row
// meet in LDS in a fixed order, so no partial sums go through memory and
// results are deterministic.
// rpw is the count that puts the fewest waves on the busiest CU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/vramc_rans.h"
#include "rans_device.h"

namespace {

constexpr int kMmMaxWaves = 16;
constexpr int kMmMaxRows = 64;
constexpr int kMmCus = 256;  // of an MI355X, for the questions asked without a device
constexpr int kMmStaticLds = (int)sizeof(TabEntry<false>) * (int)kProbM;
// Row stride of a wave's R x 64 weights in LDS: 16 bytes beyond the 128, so
// that 16 rows read as 16-byte fragments spread over the banks.
constexpr int kMmStride = 144;

struct MatmulArgs {
    const uint16_t* words;
    const uint32_t* tile_off;
    const uint8_t* slen;
    const uint32_t* tile_meta;
    const uint4* table_lds;
    const int32_t* esc_tileptr;
    const uint16_t* esc_pos;  // tile-local index c*R + r
    const int16_t* esc_val;
    const float* step;
    const void* x;
    const float* bias;  // or null
    void* out;
    int rows, cols, C, ncb, nrb;
    int rpw;  // groups of T tile rows per workgroup
    int nb;   // rows of x
    int out_dtype, has_esc;
    WaveLayout L;
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// NB blocks of 16 rows of x.  Fragments of v_mfma_f32_16x16x32_bf16: lane l
// holds row l%16 and columns 8*(l/16) .. +7 of either operand (16 bytes of a
// row of x, and of the weights in LDS), and of the product column l%16 (the
// row of x) and rows 4*(l/16) .. +3 (tile rows).  Tile rows past R re-read
// the last one and are not stored.
template <int R, int T, int NB>
__global__ void __launch_bounds__(64 * kMmMaxWaves) rans_w64_matmul_kernel(MatmulArgs a) {
    __shared__ __align__(16) TabEntry<false> tab[kProbM];
    extern __shared__ __align__(16) uint16_t dyn[];
    constexpr int TR = T * R;  // rows of a wave
    constexpr int MB = (TR + 15) / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int W = a.rpw * a.ncb;
    const int wave_stride = T * a.L.wave_words + TR * kMmStride / 2;  // 16-bit words
    uint16_t* raw = dyn + (size_t)wave * wave_stride;
    uint8_t* wt = reinterpret_cast<uint8_t*>(raw + T * a.L.wave_words);
    const int rsub = wave / a.ncb, cb = wave - rsub * a.ncb;
    // tiles past the last tile row repeat that row's, unstored
    int t[T];
#pragma unroll
    for (int i = 0; i < T; i++)
        t[i] = min(((int)blockIdx.x * a.rpw + rsub) * T + i, a.nrb - 1) * a.ncb + cb;

    TileOff to[T];
    int tp[T];
#pragma unroll
    for (int i = 0; i < T; i++) {
        to[i] = load_tile_off(a.tile_off, t[i]);
        tp[i] = a.esc_tileptr[t[i] + min(lane, 1)];
    }
    asm volatile("" ::: "memory");
    uint32_t tmv[T], len0[T];
#pragma unroll
    for (int i = 0; i < T; i++) {
        tmv[i] = a.tile_meta[t[i]];
        len0[i] = a.slen[(int64_t)t[i] * 64 + lane];
    }
    const int cbase = cb * a.C;
    const __amdgpu_buffer_rsrc_t srs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.step), 0, a.cols * 4, kBufWord3);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(a.x), 0, a.nb * a.cols * 2, kBufWord3);
    const int fc = 8 * (lane >> 4);  // this lane's first column of a fragment
    int xoff[NB];
#pragma unroll
    for (int n = 0; n < NB; n++)
        xoff[n] = (min(16 * n + (lane & 15), a.nb - 1) * a.cols + cbase + fc) * 2;
    float sr = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, (cbase + lane) * 4, 0, 0));
#pragma unroll
    for (int i = 0; i < T; i++) {
        uint32_t o0, n16;
        tile_extent(to[i], true, a.L.raw_words, o0, n16);
        stage_tile(raw + i * a.L.wave_words, a.words, o0, n16, lane);
    }
    stage_table(tab, a.table_lds, wave, W, lane);
    // x of 64 columns, loaded behind the products of the 64 before and so in
    // flight during a decode
    bf16x8 xf[NB][2];
    auto load_x64 = [&](int k) {
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                xf[n][h] = __builtin_bit_cast(
                    bf16x8, __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[n] + 64 * h, 128 * k, 0));
    };
    // Escapes run in column order, so those of 64 columns are the next few of
    // the side table; a lane holds one of the 64 next entries, with its
    // position past every tile once it is used.
    constexpr uint32_t kNoEsc = ~0u;
    int e_next[T], e_hi[T];
    uint32_t epos[T];
    uint16_t ebits[T];
    auto load_escapes = [&](int i) {
        epos[i] = kNoEsc;
        if (e_next[i] + lane < e_hi[i]) {
            epos[i] = a.esc_pos[e_next[i] + lane];
            const int col = cbase + (int)min(esc_tcol<R>((int)epos[i]), (uint32_t)(a.C - 1));
            ebits[i] = to_bf16((float)a.esc_val[e_next[i] + lane] * a.step[col]);
        }
        e_next[i] += 64;
    };
#pragma unroll
    for (int i = 0; i < T; i++) {
        e_next[i] = a.has_esc ? __builtin_amdgcn_readlane(tp[i], 0) : 0;
        e_hi[i] = a.has_esc ? __builtin_amdgcn_readlane(tp[i], 1) : 0;
        epos[i] = kNoEsc;
        ebits[i] = 0;
        if (e_next[i] < e_hi[i]) load_escapes(i);
    }
    wait_vm();
    __syncthreads();
    load_x64(0);

    f32x4 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int n = 0; n < NB; n++) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    Lanes<T, TabEntry<false>> L;
    {
        uint32_t off[T], st0[T];
#pragma unroll
        for (int i = 0; i < T; i++) {
            const uint32_t lb[1] = {len0[i]};
            uint32_t off1[1], bit1[1];
            stream_layout<1>(lb, __builtin_amdgcn_readfirstlane(tmv[i]), off1, bit1);
            off[i] = off1[0] + i * a.L.wave_words;
            st0[i] = initial_state(raw + i * a.L.wave_words, bit1[0], lb[0]);
        }
        init_lanes(L, tab, raw, st0, off);
    }
    uint16_t* const wcol = reinterpret_cast<uint16_t*>(wt) + lane;
    const int nk = a.C / 64;
    for (int k = 0; k < nk; k++) {
        asm volatile("" : "+v"(sr));
        const float sv = sr;
        const int kn = min(k + 1, nk - 1);  // the last loads are repeated, unused
        sr = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(srs, (cbase + lane) * 4, 256 * kn, 0));
        asm volatile("" ::: "memory");
        float held[T];
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int i = 0; i < T; i++) {
                const int32_t code = rans_step<(R >= 8)>(L.st[i], L.a[i], L.w[i], L.e[i], tab);
                const float v = (float)code * sv;
                uint16_t* const wrow = wcol + (i * R + r) * (kMmStride / 2);
                if (r % 2 == 0 && r + 1 < R) {
                    held[i] = v;
                } else if (r % 2) {
                    const uint32_t p = to_bf16x2(held[i], v);
                    wrow[-(kMmStride / 2)] = (uint16_t)p;
                    wrow[0] = (uint16_t)(p >> 16);
                } else {
                    wrow[0] = to_bf16(v);
                }
            }
        }
        asm volatile("" ::: "memory");
        if (a.has_esc) {
            const uint32_t end = (uint32_t)(k + 1) * (64 * R), begin = end - 64 * R;
#pragma unroll
            for (int i = 0; i < T; i++) {
                while (true) {  // wave-uniform
                    const bool mine = epos[i] < end;
                    if (mine && epos[i] >= begin) {
                        const int r = i * R + esc_row<R>((int)epos[i]);
                        const uint32_t c = esc_tcol<R>((int)epos[i]) & 63u;
                        *reinterpret_cast<uint16_t*>(wt + r * kMmStride + 2 * c) = ebits[i];
                    }
                    if (mine) epos[i] = kNoEsc;
                    if (e_next[i] >= e_hi[i] || __builtin_amdgcn_ballot_w64(epos[i] != kNoEsc)) break;
                    load_escapes(i);
                }
            }
            asm volatile("" ::: "memory");
        }
        // a wave's LDS operations complete in order: no barrier
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int m = 0; m < MB; m++) {
                const int row = min(16 * m + (lane & 15), TR - 1);
                const bf16x8 wf = __builtin_bit_cast(
                    bf16x8, *reinterpret_cast<const uint4*>(wt + row * kMmStride + 64 * h + 2 * fc));
#pragma unroll
                for (int n = 0; n < NB; n++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[n][h], acc[m][n], 0, 0, 0);
            }
        asm volatile("" ::: "memory");
        load_x64(kn);
    }

    // 16 rows of x at a time: each wave's TR x 16 sums over its weights in LDS
    // (64 of every 144 bytes), then one total per thread.
    const int tid = threadIdx.x, nthr = 64 * W;
    float* wred = reinterpret_cast<float*>(wt);
#pragma unroll
    for (int n = 0; n < NB; n++) {
        if (n) __syncthreads();  // totals of the block before are read
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int r = 16 * m + 4 * (lane >> 4) + i;
                if (r < TR) wred[r * 16 + (lane & 15)] = acc[m][n][i];
            }
        __syncthreads();
        for (int i = tid; i < a.rpw * TR * 16; i += nthr) {
            const int b = i / (a.rpw * TR), j = i - b * (a.rpw * TR);  // j: row within the workgroup
            const int rs = j / TR, r = j - rs * TR;
            const int64_t row = (int64_t)blockIdx.x * a.rpw * TR + j;
            if (row >= a.rows || 16 * n + b >= a.nb) continue;
            float v = 0.f;
            for (int w = 0; w < a.ncb; w++)
                v += reinterpret_cast<const float*>(dyn + (size_t)(rs * a.ncb + w) * wave_stride +
                                                    T * a.L.wave_words)[r * 16 + b];
            if (a.bias) v += a.bias[row];
            const int64_t o = (int64_t)(16 * n + b) * a.rows + row;
            if (a.out_dtype == RANS_X_F32)
                static_cast<float*>(a.out)[o] = v;
            else if (a.out_dtype == RANS_X_BF16)
                static_cast<__bf16*>(a.out)[o] = (__bf16)v;
            else
                static_cast<_Float16*>(a.out)[o] = (_Float16)v;
        }
    }
}

// Tile rows a wave can take at once: as many as fill the matrix cores' 16
// rows, and two of 16.  Every wave reads its columns of x for itself, so with
// T of them x is read T times less; in exchange T times fewer waves each
// decode T times the symbols, one tile's after the other's.
constexpr int mm_tiles(int R) { return R <= 4 ? 4 : R <= 16 ? 2 : 1; }

// What T decides of a launch's time, in ps: a wave decodes a symbol in 50 ns
// alone on its SIMD and in 14 for every wave the SIMD holds, and escapes cost
// three symbols a column step and tile; x comes from the caches at 9 TB/s; a
// column step of a 16x16 block of the product takes its SIMD 40 ns.  Of 45
// matrices at 17 to 64 rows the better T by this is within 0.3% of the faster
// one on average and within 12% at worst (a limit on the bytes of x was 3.6%
// and 61% off).  One and T tile rows, us from a replayed graph: 5120x5120 in
// 8-row tiles, 32 rows, 34.8 and 26.5; 6400x5120, 17 rows, 31.6 and 23.9;
// 25600x1024 in 16-row tiles, 24 rows, 27.4 and 22.5; 4096x4096 in 8-row
// tiles, 24 rows, 17.7 and 21.6; 10240x3200 in 16-row tiles, 24 rows, 22.3 and
// 29.0; 1536x8960 in 3-row tiles, 32 rows, 35.5 and 26.2, with escapes 36.2
// and 35.8; 2048x8192 in 4-row tiles with escapes, 17 rows, 23.5 and 37.9.
int64_t matmul_cost(const rans_w64_matrix* m, int nb, int T, int cus) {
    const int64_t nrb = m->rows / m->R, steps = m->C / 64, simds = 4 * cus;
    const int64_t waves = (nrb + T - 1) / T * (m->cols / m->C);
    const int64_t symbols = steps * (m->R + (m->flags & RANS_F_NO_ESCAPES ? 0 : 3));
    const int64_t blocks = waves * steps * ((T * m->R + 15) / 16) * ((nb + 15) / 16);
    return symbols * T * std::max<int64_t>(50000, 14000 * waves / simds) +
           nrb * nb * m->cols * 2 / T / 9 + 40000 * blocks / simds;
}

// Groups of T tile rows per workgroup: of the counts that put the fewest
// waves on the busiest CU when the workgroups spread evenly the largest
// (waves that share a table leave more LDS to others).  0 when not even one
// fits.
int matmul_rpw(const rans_w64_matrix* m, int T, int cus) {
    const int ncb = m->cols / m->C, groups = (m->rows / m->R + T - 1) / T;
    const size_t wave = (size_t)T * (wave_layout(m).wave_words * 2 + m->R * kMmStride);
    int best = 0;
    int64_t best_load = 0;
    for (int rpw = 1; rpw * ncb <= kMmMaxWaves; rpw++) {
        if (rpw * ncb * wave + kMmStaticLds > (size_t)kLdsMax) break;
        const int64_t grid = (groups + rpw - 1) / rpw;
        const int64_t load = (grid + cus - 1) / cus * rpw * ncb;
        if (!best || load <= best_load) best = rpw, best_load = load;
    }
    return best;
}

// T of a launch and its groups per workgroup (0 when none fits).
struct MatmulShape {
    int T, rpw;
};

MatmulShape matmul_shape(const rans_w64_matrix* m, int nb, int cus) {
    const int T = mm_tiles(m->R);
    if (T > 1 && matmul_cost(m, nb, T, cus) < matmul_cost(m, nb, 1, cus))
        if (const int rpw = matmul_rpw(m, T, cus)) return {T, rpw};
    return {1, matmul_rpw(m, 1, cus)};
}

// The rows up to which this path is taken: twice the rows a wave takes
// (some 4 bytes of x read per weight, what writing and reading the weight
// takes), in whole blocks of 16, or all 64 for matrices of up to 4M weights,
// whose time is in the launches.  Against decoding, the dense product and the
// last pass (us, from a replayed graph over three copies, without the host's
// part, which is 37 us for those three): 5120x5120 at 32 rows 26.5 to 34.2, at
// 64 47.2 to 38.2; 1536x1536 at 64 11.4 to 16.4; 12800x2048 in 16-row tiles at
// 64 27.7 to 33.6; 8960x1536 in 35-row tiles at 64 18.4 to 27.8; 1536x8960 in
// 3-row tiles at 32 26.2 to 34.3.  Of 45 matrices it is behind at its limit
// for five: by 5% for 1536x8960 with escapes at 32 (36.2 to 34.3), 6% for
// 2048x8192 in 4-row tiles with escapes (34.0 to 31.9), 5% for 9600x3200 at 64
// (38.8 to 36.8), 1% for the others.  Where x is short beside the weight the
// line is on the safe side: 4096x4096 at 48 rows would take 20.6 (29.3),
// 1536x17920 54.4 (74.4), 5120x5120 39.2 (40.4).  Shorter tiles than 3 rows
// stay on the dense product (2560x9728 in 2-row tiles at 32 rows 39.1 to 37.5).
int matmul_max_rows(const rans_w64_matrix* m, int cus) {
    if (!matmul_rpw(m, 1, cus)) return 0;
    if ((int64_t)m->rows * m->cols <= (4 << 20)) return kMmMaxRows;
    const int T = matmul_rpw(m, mm_tiles(m->R), cus) ? mm_tiles(m->R) : 1;
    return std::min(kMmMaxRows, (2 * T * m->R + 15) / 16 * 16);
}

bool matmul_compiled(const rans_w64_matrix* m) {
    return m->S == 1 && (m->R == 3 || m->R == 4 || m->R == 8 || m->R == 16 || m->R == 20 ||
                         m->R == 35);
}

template <int R, int T, int NB>
int launch_matmul_t(const MatmulArgs& a, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&rans_w64_matmul_kernel<R, T, NB>);
    const int waves = a.rpw * a.ncb, groups = (a.nrb + T - 1) / T;
    const size_t lds = (size_t)waves * T * (a.L.wave_words * 2 + R * kMmStride);
    const hipError_t e = ensure_lds(fn, lds, kMmStaticLds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((rans_w64_matmul_kernel<R, T, NB>), dim3((groups + a.rpw - 1) / a.rpw),
                       dim3(64 * waves), lds, stream, a);
    return (int)hipGetLastError();
}

template <int R, int T>
int launch_matmul_nb(const MatmulArgs& a, hipStream_t stream) {
    switch ((a.nb + 15) / 16) {
        case 1: return launch_matmul_t<R, T, 1>(a, stream);
        case 2: return launch_matmul_t<R, T, 2>(a, stream);
        case 3: return launch_matmul_t<R, T, 3>(a, stream);
        default: return launch_matmul_t<R, T, 4>(a, stream);
    }
}

template <int R>
int launch_matmul(const MatmulArgs& a, int T, hipStream_t stream) {
    if constexpr (mm_tiles(R) > 1)
        if (T > 1) return launch_matmul_nb<R, mm_tiles(R)>(a, stream);
    return launch_matmul_nb<R, 1>(a, stream);
}

}  // namespace

extern "C" int rans_matmul_rows(const rans_w64_matrix* m) {
    if (!valid_geometry(m)) return RANS_EGEOMETRY;
    if (!matmul_compiled(m) || (int64_t)kMmMaxRows * m->cols * 2 > INT32_MAX) return 0;
    return matmul_max_rows(m, kMmCus);
}

extern "C" int rans_matmul_tiles(const rans_w64_matrix* m, int batch) {
    if (!valid_geometry(m)) return RANS_EGEOMETRY;
    if (batch <= 0) return RANS_EARG;
    if (!matmul_compiled(m) || batch > kMmMaxRows || (int64_t)batch * m->cols * 2 > INT32_MAX) return 0;
    const MatmulShape shape = matmul_shape(m, batch, kMmCus);
    return shape.rpw ? shape.T : 0;
}

extern "C" int rans_w64_matmul(const rans_w64_matrix* m, const void* x, int batch, const float* bias,
                               void* out, int out_dtype, hipStream_t stream) {
    if (!valid_geometry(m)) return RANS_EGEOMETRY;
    if (!valid_pointers(m) || !x || !out || batch <= 0) return RANS_EARG;
    if (out_dtype != RANS_X_F32 && out_dtype != RANS_X_BF16 && out_dtype != RANS_X_F16)
        return RANS_EARG;
    if (!matmul_compiled(m) || batch > kMmMaxRows) return RANS_EUNSUPPORTED;
    // 16-byte loads of x, addressed with 32 bits
    if ((uintptr_t)x % 16 || (int64_t)batch * m->cols * 2 > INT32_MAX) return RANS_EGEOMETRY;
    const int cus = device_cus();
    if (cus <= 0) return (int)hipErrorInvalidDevice;
    MatmulArgs a;
    const MatmulShape shape = matmul_shape(m, batch, cus);
    const int T = shape.T;
    a.rpw = shape.rpw;
    if (!a.rpw) return RANS_EGEOMETRY;
    a.words = m->words;
    a.tile_off = m->tile_off;
    a.slen = m->slen;
    a.tile_meta = m->tile_meta;
    a.table_lds = reinterpret_cast<const uint4*>(m->table_lds);
    a.esc_tileptr = m->esc_tileptr;
    a.esc_pos = m->esc_pos;
    a.esc_val = m->esc_val;
    a.step = m->step;
    a.x = x;
    a.bias = bias;
    a.out = out;
    a.rows = m->rows;
    a.cols = m->cols;
    a.C = m->C;
    a.ncb = m->cols / m->C;
    a.nrb = m->rows / m->R;
    a.nb = batch;
    a.out_dtype = out_dtype;
    a.has_esc = !(m->flags & RANS_F_NO_ESCAPES);
    a.L = wave_layout(m);
    switch (m->R) {
        case 3: return launch_matmul<3>(a, T, stream);
        case 4: return launch_matmul<4>(a, T, stream);
        case 8: return launch_matmul<8>(a, T, stream);
        case 16: return launch_matmul<16>(a, T, stream);
        case 20: return launch_matmul<20>(a, T, stream);
        default: return launch_matmul<35>(a, T, stream);
    }
}
