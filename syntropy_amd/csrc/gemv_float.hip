// Gemv over F16 and BF16 weights on gfx950 (crates/kernels-cpu/src/gemv/portable.rs:30-45
// float_rows with the fold of gemv.rs:506-516): per output, 32 F32 accumulators; element i goes
// into accumulator i % 32 with one fused multiply-add, in increasing i; then the halving fold
// acc[j] += acc[j + h] for h = 16, 8, 4, 2, 1.  The activations stay F32 (no quantization).
//
// The accumulators on the matrix cores.  v_mfma_f32_4x4x1_16b_f32 is sixteen independent 4 x 4
// outer products with one product a sum, each D = fma(A, B, C): one fused multiply-add, rounded
// once, subnormals and zero signs kept (checked against fmaf on the device over random finite
// operands, subnormal results among them).  So the sixteen blocks are sixteen accumulators of
// 4 weight rows x 4 activation rows: lane l = 4 b + i holds, of weight row i of the tile, the
// dword of elements 32 m + 2 b and + 1 (accumulators 2 b and 2 b + 1: two instructions), and of
// activation row i the same two F32 values.
//
// What bounds it.  The weights' bytes, read once for up to 16 activation rows.  A wavefront takes
// R tiles of 4 weight rows x C tiles of 4 activation rows over the whole row length, KC elements a
// stage.  Weights (each wavefront its own rows) and activation rows (one set for the workgroup) are
// copied into LDS by global_load_lds in whole kilobytes of a row, NS - 1 stages ahead.
// Measured on 32064 x 4096 F16 (263 MB), against one 16-byte load a lane and F32 FMAs on four
// activation rows a pass: 54 us (4.9 TB/s) against 78 at one row, 75 against 288 at 9, 87 against
// 450 at 16, 174 against 833 at 32.  4096 x 4096: 9.6 against 41 us at one row.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace syn {

typedef float v4f_f __attribute__((ext_vector_type(4)));

template <int C, int R, int WV, int KC, int NS>
struct GfCfg {
    static constexpr int MC = KC / 32;             // steps of 32 elements a stage
    static constexpr int RPC = 1024 / (2 * KC);    // weight rows a copy instruction moves (1 KB)
    // A piece of LDS a copy instruction fills, and 32 bytes more: the four weight rows of a tile (one
    // dword a lane) and the four activation rows of a tile (two dwords) then start 32 bytes apart
    // modulo the 128 bytes that a group of lanes reads at once, which no two lanes share a bank in.
    static constexpr int WPIECE = 1024 + 32;
    static constexpr int WCOPIES = 4 * R / RPC;    // per wavefront a stage
    static constexpr int WBYTES = WCOPIES * WPIECE;
    static constexpr int XROW = 4 * KC + 32;
    static constexpr int XPIECES = 4 * C * KC * 4 / 1024;
    static constexpr int XCOPIES = (XPIECES + WV - 1) / WV;
    static constexpr int STAGE = WV * WBYTES + 4 * C * XROW;
    static constexpr int COPIES = WCOPIES + XCOPIES;
    static constexpr size_t LDS = (size_t)NS * STAGE;
    static_assert(RPC >= 1 && R % RPC == 0, "a copy takes row i of RPC tiles");
    static_assert(COPIES * (NS - 2) <= 63, "the wait count fits vmcnt");
    static_assert(LDS <= 160 * 1024, "LDS");
};

// VEC: rows of whole 16-byte pieces at 16-byte aligned addresses.  Else a stage copies the KC elements'
// space from the aligned piece that its first element lies in and takes KC - 32 of them, which leaves
// every row's offset in its piece the same in all stages.  An aligned piece that holds a byte of a row
// lies in the same page as that byte, so the reads around a row's ends stay on its pages.
template <int BF16, int VEC, int C, int R, int WV, int KC, int NS>
__global__ __launch_bounds__(64 * WV, 1) void k_gemv_float(const uint8_t* __restrict__ W, int n_out, int k,
                                                          const float* __restrict__ x, int rows,
                                                          float* __restrict__ y,
                                                          const uint32_t* __restrict__ active, int groups) {
    using G = GfCfg<C, R, WV, KC, NS>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    rows = active_rows(active, 0, rows);
    // activation groups of the same weight rows run on the same XCD (workgroups go to the 8 XCDs
    // in turn), one after the other, so that the later ones find the weights in its L2
    const int id = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int wb = groups == 1 ? id : 8 * (id / (8 * groups)) + (id & 7);
    const int t0 = groups == 1 ? 0 : 4 * C * ((id >> 3) % groups);
    if (t0 >= rows || (int64_t)wb * WV * 4 * R >= n_out) return;  // uniform
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = lane >> 2, i = lane & 3;
    const int row0 = (wb * WV + wave) * 4 * R;
    constexpr int KS = VEC ? KC : KC - 32;  // elements a stage
    const int ns = k / KS + (k % KS != 0);
    const uint32_t rb = 2u * (uint32_t)k;
    v4f_f acc[R][C][2];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[r][c][j] = v4f_f{0.0f, 0.0f, 0.0f, 0.0f};

    // weight copy u: row i' = u % 4 of tiles RPC (u / 4) .. + RPC - 1, 64 / RPC lanes each; rows past
    // the matrix re-read its last one, bytes past a row its last piece (neither is used)
    const uint8_t* wbase = W + (uint64_t)(row0 < n_out ? row0 : n_out - 1) * rb;
    const int last = n_out - 1 - (row0 < n_out ? row0 : n_out - 1);  // the last row, from wbase
    auto issue = [&](int s) {
        uint8_t* st = lds + (s % NS) * G::STAGE;
        // a stage past the row: of two, none flies but the next (the wait is for all); of more, the last
        // again, so that the counts stay
        if (NS == 2 && s >= ns) return;
        const int sc = s < ns ? s : ns - 1;
#pragma unroll
        for (int u = 0; u < G::WCOPIES; ++u) {
            const int tr = G::RPC * (u / 4) + lane / (64 / G::RPC);
            const int row = 4 * tr + (u & 3) < last ? 4 * tr + (u & 3) : last;
            const uint32_t to = lds_addr(st) + (uint32_t)(wave * G::WBYTES + u * G::WPIECE);
            if constexpr (VEC) {
                const uint32_t at = 2u * KC * (uint32_t)sc + 16u * (uint32_t)(lane % (64 / G::RPC));
                lds_dma16<true>((uint32_t)row * rb + (at < rb ? at : rb - 16), wbase, to);
            } else {
                // from the piece of the first of the copy's rows (two rows, of less than 2^25 bytes: 4
                // rows apart)
                const int r0 = 4 * G::RPC * (u / 4) + (u & 3) < last ? 4 * G::RPC * (u / 4) + (u & 3) : last;
                const uint8_t* from = wbase + (uint64_t)r0 * rb;
                const uint32_t mis = (uint32_t)((uintptr_t)from & 15);
                const uint64_t at = 2ull * KS * (uint64_t)sc;
                const uint32_t start = G::RPC == 1 ? mis : mis + (uint32_t)(row - r0) * rb;
                const uint64_t end = (((uint64_t)start + rb - 1) & ~15ull) - (start & ~15u) - at;  // the row's last piece
                const uint32_t off = 16u * (uint32_t)(lane % (64 / G::RPC));
                lds_dma16<true>((start & ~15u) + (off < end ? off : (uint32_t)end), from - mis + at, to);
            }
        }
        uint8_t* xst = st + WV * G::WBYTES;
#pragma unroll
        for (int u = 0; u < G::XCOPIES; ++u) {
            const int q0 = wave + WV * u, q = q0 < G::XPIECES ? q0 : G::XPIECES - 1;  // the last piece again
            constexpr int PR = KC / 256;  // pieces of an activation row
            const int t = t0 + q / PR < rows ? t0 + q / PR : rows - 1;
            const uint32_t dst = (uint32_t)((q / PR) * G::XROW + 1024 * (q % PR));
            const float* from = x + (int64_t)t * k;
            if constexpr (VEC) {
                const uint32_t at = 4u * KC * (uint32_t)sc + 1024u * (uint32_t)(q % PR) + 16u * (uint32_t)lane;
                lds_dma16<true>(at < 2 * rb ? at : 2 * rb - 16, from, lds_addr(xst) + dst);
            } else {
                const uint32_t mis = (uint32_t)((uintptr_t)from & 15);
                const uint64_t at = 4ull * KS * (uint64_t)sc, end = ((mis + 2 * (uint64_t)rb - 1) & ~15ull) - at;
                const uint32_t off = 1024u * (uint32_t)(q % PR) + 16u * (uint32_t)lane;
                lds_dma16<true>(off < end ? off : (uint32_t)end, reinterpret_cast<const uint8_t*>(from) - mis + at,
                                lds_addr(xst) + dst);
            }
        }
    };
    // (not VEC) where the lane's rows start in their pieces
    uint32_t woff[R], xoff[C];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = 4 * r + i < last ? 4 * r + i : last;
        woff[r] = VEC ? 0u : (uint32_t)((uintptr_t)(wbase + (uint64_t)row * rb) & 15);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int t = t0 + 4 * c + i < rows ? t0 + 4 * c + i : rows - 1;
        xoff[c] = VEC ? 0u : (uint32_t)((uintptr_t)(x + (int64_t)t * k) & 15);
    }
    auto cvt = [](uint32_t h) { return BF16 ? __builtin_bit_cast(float, h << 16) : f16_to_f32(h); };
    // `tail`: a stage that the row may end in; the others run without a branch, so that the LDS
    // reads of a step are issued under the products of the one before
    auto stage = [&](auto tail, int s) __attribute__((always_inline)) {
        const uint8_t* st = lds + (s % NS) * G::STAGE;
        const uint8_t* ws = st + wave * G::WBYTES + i * G::WPIECE + 4 * b;
        const uint8_t* xs = st + WV * G::WBYTES + i * G::XROW + 8 * b;
#pragma unroll
        for (int m = 0; m < KS / 32; ++m) {
            if (decltype(tail)::value && KS * s + 32 * m >= k) break;  // uniform
            float2 xb[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint8_t* p = xs + 4 * c * G::XROW + 128 * m + xoff[c];
                if constexpr (VEC)
                    xb[c] = *reinterpret_cast<const float2*>(p);
                else
                    xb[c] = make_float2(reinterpret_cast<const float*>(p)[0], reinterpret_cast<const float*>(p)[1]);
            }
            float a[R][2];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint8_t* p = ws + (r / G::RPC) * 4 * G::WPIECE + (r % G::RPC) * 2 * KC + 64 * m + woff[r];
                uint32_t w;
                if constexpr (VEC)
                    w = *reinterpret_cast<const uint32_t*>(p);
                else
                    w = reinterpret_cast<const uint16_t*>(p)[0] | (uint32_t)reinterpret_cast<const uint16_t*>(p)[1] << 16;
                a[r][0] = cvt(w & 0xFFFFu);
                a[r][1] = BF16 ? __builtin_bit_cast(float, w & 0xFFFF0000u) : cvt(w >> 16);
            }
            if constexpr (decltype(tail)::value) {  // elements past the row: 0 times -0.0, which no sum sees
                const uint32_t e = (uint32_t)KS * (uint32_t)s + 32u * m + 2u * b, n = (uint32_t)k;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    a[r][0] = e < n ? a[r][0] : 0.0f;
                    a[r][1] = e + 1 < n ? a[r][1] : 0.0f;
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    xb[c].x = e < n ? xb[c].x : -0.0f;
                    xb[c].y = e + 1 < n ? xb[c].y : -0.0f;
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    acc[r][c][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[r][0], xb[c].x, acc[r][c][0], 0, 0, 0);
                    acc[r][c][1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[r][1], xb[c].y, acc[r][c][1], 0, 0, 0);
                }
        }
    };
    if (ns > 0) {
        const int whole = k / KS;
#pragma unroll
        for (int s = 0; s < NS - 1; ++s) issue(s);
        for (int s = 0; s < ns; ++s) {
            // stage s has landed (the NS - 2 after it may fly), the previous one is read out, and the
            // next copies go into its place
            wait_vm<G::COPIES * (NS - 2)>();
            lds_barrier();
            issue(s + NS - 1);
            if (s < whole)
                stage(std::false_type{}, s);
            else
                stage(std::true_type{}, s);
        }
        wait_vm<0>();  // the last (repeated) copies have landed before the workgroup ends
    }
    // the halving fold: accumulators 2 b + j and 16 on (block b + 8), 8 on (b + 4), 4 on (b + 2),
    // 2 on (b + 1), then the lane's own two.  The first two steps take two and then four of the tile's
    // rows at once, each half or quarter of the lanes another row, so that a tile's 16 sums end in a
    // lane each: lanes 16 p + i hold activation row i of weight row 0, 2, 1, 3 for p = 0 to 3.
    const int q = (lane >> 3 & 2) | (lane >> 5);
    auto halves = [](float a, float b) __attribute__((always_inline)) {
        const auto v = __builtin_amdgcn_permlane32_swap(f2u(a), f2u(b), false, false);
        return u2f(v[0]) + u2f(v[1]);
    };
    auto quarters = [](float a, float b) __attribute__((always_inline)) {
        const auto v = __builtin_amdgcn_permlane16_swap(f2u(a), f2u(b), false, false);
        return u2f(v[0]) + u2f(v[1]);
    };
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float v[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v4f_f a = acc[r][c][j];
                float f = quarters(halves(a[0], a[1]), halves(a[2], a[3]));
                f = f + u2f(dpp_u32<0x128>(f2u(f)));  // row_ror:8
                v[j] = f + u2f(dpp_u32<0x124>(f2u(f)));  // row_ror:4
            }
            const int t = t0 + 4 * c + i, row = row0 + 4 * r + q;
            if ((lane & 12) == 0 && t < rows && row < n_out) y[(int64_t)t * n_out + row] = v[0] + v[1];
        }
}

constexpr int64_t GF_MAX_X = 1 << 20;

template <int BF16, int VEC, int C, int R, int WV, int KC, int NS>
static void launch_float(const uint8_t* W, int n_out, int k, const float* x, int rows, float* y, hipStream_t stream,
                         const uint32_t* active) {
    using G = GfCfg<C, R, WV, KC, NS>;
    const int groups = (rows + 4 * C - 1) / (4 * C);
    int64_t wgs = (n_out + 4 * R * WV - 1) / (4 * R * WV);
    if (groups > 1) wgs = (wgs + 7) / 8 * 8 * groups;
    // once per process, thread-safe (a function-local static); a refusal shows as the launch's error
    static const hipError_t attr = hipFuncSetAttribute((const void*)k_gemv_float<BF16, VEC, C, R, WV, KC, NS>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS);
    (void)attr;
    // a dimension of the grid holds less than 2^32 threads: whole rounds of the XCDs in x, the rest in y
    const dim3 grid((unsigned)(wgs < GF_MAX_X ? wgs : GF_MAX_X), (unsigned)((wgs + GF_MAX_X - 1) / GF_MAX_X));
    hipLaunchKernelGGL((k_gemv_float<BF16, VEC, C, R, WV, KC, NS>), grid, dim3(64 * WV), G::LDS, stream, W, n_out, k, x,
                       rows, y, active, groups);
}

// Workgroups of 64 weight rows (eight wavefronts of eight) from this many of them on, else of
// sixteen (four wavefronts of four), which spread fewer rows over more CUs: 14336 x 4096 at 2 rows
// 24.3 us in 224 workgroups against 33.6 in 896, 4096 x 4096 at 24 rows 36 us in 128 against 33.
constexpr int GF_WIDE_WGS = 129;

// Short rows have few stages to hide a workgroup's first copies and its fold behind: they take two stages
// a ring and half the wavefronts, so that a CU holds several workgroups and one starts while another
// ends.  Up to four activation rows, rows of medium length too are better off with two workgroups of two
// stages than with one of four.  Four stages of eight wavefronts | two of eight | two of four: one row of
// 50000 x 768 21 | 16 | 15 us, 50000 x 2048 35 | 35 | 38, 32064 x 4096 46 | 43 | 52, 14336 x 14336 86 | 90 | 83;
// 16 rows of 50000 x 768 38 | 35 | 30, 50000 x 4096 137 | 135 | 126.  (Rows of 32 to 128 values stay up to 15 %
// slower at one row, and up to 10 % at 17 to 20, than one 16-byte load a lane and F32 FMAs: 100000 x 64 at one row
// 8.7 against 7.9 us, at five 10.9 against 14.0.)
constexpr int GF_SHORT = 1024, GF_MID = 4096;

// Beyond 16 activation rows, groups of 16 (32 in one workgroup leave one wavefront a SIMD: 32064 x
// 4096 at 32 rows 192 us against 174).
template <int BF16, int VEC>
static void launch_float_rows(const uint8_t* W, int n_out, int k, const float* x, int rows, float* y,
                              hipStream_t stream, const uint32_t* active) {
    // (rows of 2^24 elements and more: a copy within one row, whose offsets then fit 32 bits)
    const bool wide = k <= (1 << 24) && (int64_t)((n_out + 63) / 64) * ((rows + 15) / 16) >= GF_WIDE_WGS;
    if (wide && k <= GF_SHORT) {
        if (rows <= 4)
            launch_float<BF16, VEC, 1, 2, 4, 256, 2>(W, n_out, k, x, rows, y, stream, active);
        else if (rows <= 8)
            launch_float<BF16, VEC, 2, 2, 4, 256, 2>(W, n_out, k, x, rows, y, stream, active);
        else if (rows <= 12 || (rows + 11) / 12 * 3 < (rows + 15) / 16 * 4)  // 17 to 24 rows: two groups of 12
            launch_float<BF16, VEC, 3, 2, 4, 256, 2>(W, n_out, k, x, rows, y, stream, active);
        else
            launch_float<BF16, VEC, 4, 2, 4, 256, 2>(W, n_out, k, x, rows, y, stream, active);
    } else if (rows <= 4 && wide && k <= GF_MID)
        launch_float<BF16, VEC, 1, 2, 8, 256, 2>(W, n_out, k, x, rows, y, stream, active);
    else if (rows <= 4 && wide)
        launch_float<BF16, VEC, 1, 2, 8, 256, 4>(W, n_out, k, x, rows, y, stream, active);
    else if (rows <= 4)
        launch_float<BF16, VEC, 1, 1, 4, 512, 4>(W, n_out, k, x, rows, y, stream, active);
    else if (rows <= 8 && wide)
        launch_float<BF16, VEC, 2, 2, 8, 256, 3>(W, n_out, k, x, rows, y, stream, active);
    else if (rows <= 8)
        launch_float<BF16, VEC, 2, 1, 4, 512, 4>(W, n_out, k, x, rows, y, stream, active);
    else if (rows <= 12 && wide)
        launch_float<BF16, VEC, 3, 2, 8, 256, 3>(W, n_out, k, x, rows, y, stream, active);
    else if (wide)
        launch_float<BF16, VEC, 4, 2, 8, 256, 3>(W, n_out, k, x, rows, y, stream, active);
    else
        launch_float<BF16, VEC, 4, 1, 4, 512, 3>(W, n_out, k, x, rows, y, stream, active);
}

template <int BF16>
static void launch_float_fmt(const uint8_t* W, int n_out, int k, const float* x, int rows, float* y,
                             hipStream_t stream, const uint32_t* active) {
    if (k % 8 == 0 && k <= (1 << 24) && ((uintptr_t)W & 15) == 0 && ((uintptr_t)x & 15) == 0)
        launch_float_rows<BF16, 1>(W, n_out, k, x, rows, y, stream, active);
    else
        launch_float_rows<BF16, 0>(W, n_out, k, x, rows, y, stream, active);
}

void launch_gemv_float(int ty, const uint8_t* W, int n_out, int k, const float* x, int rows, float* y,
                       hipStream_t stream, const uint32_t* active) {
    if (ty == T_BF16)
        launch_float_fmt<1>(W, n_out, k, x, rows, y, stream, active);
    else
        launch_float_fmt<0>(W, n_out, k, x, rows, y, stream, active);
}

}  // namespace syn
