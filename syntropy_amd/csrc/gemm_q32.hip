// Q8_0 and Q4_0 products at many activation rows on the gfx950 matrix cores: the Gemv value
// (crates/kernels-cpu/src/gemv.rs:539-547, portable.rs:114-190: per 32-value block the exact I32 sum
// s and the term (dw * dx) * s, the terms added in ascending block order from +0.0) for a dense
// matrix in GGUF or SPLIT order, and for the experts of a MoeGrouped layer (crates/kernels-cpu/src/
// moe.rs:470-551 with Q8_0 experts).
//
// What bounds it: the F32 operations that the reference's rounding fixes for every (output, block),
// on the vector ALU.  Written out they are four (a conversion, dw * dx, the product, the sum); here
// two, the rest on the matrix cores:
//   s:  v_mfma_i32_32x32x32_i8, one block of 32 rows x 32 tokens, with C = 0x4B400000, the bits of
//       M = 3 * 2^22.  |s| < 2^22, so the integer C + s is the bits of the F32 number M + s: no
//       conversion.
//   dw * dx and -M * dw * dx: v_mfma_f32_32x32x1_2b, two outer products a instruction, one product a
//       sum.  Both scales are F16 numbers, so dw * dx has at most 22 significant bits and M dw dx at
//       most 24: exact.
//   fma(dw * dx, M + s, -M * dw * dx) is then dw * dx * s rounded once, the reference's product, and
//       one addition folds it.  (s = 0 gives +0.0 for either zero, which a sum from +0.0 does not
//       see.)  An infinite scale (dw or dx past F16's range) makes that a NaN where the reference
//       may have an infinity, so a tile that ends with NaNs takes them again, as written, from its
//       blocks whose scales are not finite (g32_settle).
// Q4_0: the int8 operand holds 16 (n - 8) (a nibble in the high half of its byte, its top bit
// flipped), and the scale is dw / 16: the same bound on s, the same exactness.
//
// Per 32 x 32 tile and block that is about 96 cycles of matrix products and 80 of vector operations, and
// the two add up on this chip (two wavefronts a SIMD: a loop of both alone takes 184).  Measured, with
// the operands' reads: about 250; 4096 x 14336 Q8_0 SPLIT at 512 rows 128 us against 155 for the
// four-operation form (gemv_split.hip), GGUF Q4_0 6144 x 4096 at 200 rows 59 us against 841.
//
// A wavefront takes 32 rows x 32 TT tokens of one matrix, a workgroup RG x TG of them (gate and up: of
// both matrices; the wavefronts that hold up hand it through LDS to those that hold gate).
// Four blocks of every operand a stage are copied into LDS by global_load_lds one stage ahead.
//   GGUF rows are 34- or 18-byte blocks, so a row's four blocks start at any even address: the stage
//   copies the aligned 16-byte pieces around them, and a lane reads the five dwords around its 16
//   code bytes and shifts them together.  An aligned piece that holds a byte of the matrix lies in
//   the same page as that byte, so the reads around the matrix's ends stay on its pages.
//   SPLIT rows are lines of 128 (Q8_0) or 64 (Q4_0) bytes; as for the tokens' 128-byte lines, piece
//   q of line c sits at piece q ^ (c & 7) (or (c >> 1) & 3), so that eight lanes of neighbouring lines
//   read eight different 16-byte bank groups.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace syn {

typedef int v4i_q __attribute__((ext_vector_type(4)));
typedef int v16i_q __attribute__((ext_vector_type(16)));
typedef float v16f_q __attribute__((ext_vector_type(16)));
typedef float v32f_q __attribute__((ext_vector_type(32)));

constexpr int G32_S = 4;  // blocks a stage
constexpr int G32_BIAS = 0x4B400000;       // the bits of M
constexpr float G32_M = 12582912.0f;       // 3 * 2^22

enum : int { G32_DENSE = 0, G32_GATEUP = 1, G32_DOWN = 2 };

template <int FMT, int SPLIT, int MODE, int RG, int TG, int TT>
struct G32Cfg {
    static constexpr int R = MODE == G32_GATEUP ? 2 : 1;   // matrices
    static constexpr int NW = RG * TG * R;
    static constexpr int ROWS = 32 * RG;                   // rows of each matrix
    static constexpr int NR = ROWS * R;                    // row lines in LDS
    static constexpr int TOK = 32 * TT * TG;
    static constexpr int CB = FMT == T_Q8_0 ? 32 : 16;     // code bytes a block
    static constexpr int BB = CB + 2;
    static constexpr int STEP = SPLIT ? G32_S * CB : G32_S * BB;       // bytes of a row a stage
    static constexpr int WCH = SPLIT ? STEP / 16 : (STEP + 14 + 15) / 16;  // 16-byte pieces of a row a stage
    static constexpr int WL = 16 * WCH;
    static constexpr int W_OFF = 0;
    static constexpr int WJ = (NR * WCH + 63) / 64;        // copy instructions: row codes,
    static constexpr int SC_OFF = W_OFF + 1024 * WJ;
    static constexpr int SJ = SPLIT ? NR * 3 / 64 : 0;     // row scales (SPLIT), 4 bytes a lane, 3 a row
    static constexpr int A_OFF = SC_OFF + 256 * SJ;
    static constexpr int AJ = TOK * 8 / 64;                // token codes
    static constexpr int DX_OFF = A_OFF + 1024 * AJ;
    static constexpr int DJ = TOK * G32_S / 64;            // token scales [block][token], 4 bytes a lane
    static constexpr int STAGE = DX_OFF + 256 * DJ;
    // a wavefront's copies of each kind a stage (past the end a kind's last one again, so that every
    // wavefront's are the same)
    static constexpr int WPW = (WJ + NW - 1) / NW, SPW = (SJ + NW - 1) / NW;
    static constexpr int APW = (AJ + NW - 1) / NW, DPW = (DJ + NW - 1) / NW;
    static constexpr int COPIES = WPW + SPW + APW + DPW;
    // ring stages: what half a CU's LDS holds (two workgroups a CU), 2 to 4
    static constexpr int NSF = 80 * 1024 / STAGE;
    static constexpr int NS = NSF < 2 ? 2 : NSF > 4 ? 4 : NSF;
    static constexpr int LDS = NS * STAGE;
    static_assert(COPIES * (NS - 2) <= 63, "unit parity; the wait count fits vmcnt");
};

struct G32Args {
    const uint8_t* w0;
    const uint8_t* w1;        // MODE 1: up
    const int8_t* xq;         // Q8_0 rows: codes [row][k],
    const float* xd;          // scales [row][k / 32]
    float* y;
    int n_out, k, T;
    const uint32_t* active;   // dense: a step descriptor's rows_active, or null
    // experts
    uint64_t mat_bytes;
    const uint32_t* offsets;
    const uint32_t* slots;
    const uint32_t* err;
    int top_k;
};

// A 32 x 32 tile's outputs that ended as NaN, settled from the blocks whose weight or token scale is an
// infinity or a NaN: the reference's terms (dw * dx) * s of those blocks alone.  Beside an infinite or
// NaN term the finite ones (below 2^52 each) change nothing, and without one no output is a NaN.  The
// wavefront looks at the scales 16 blocks at a time and stops where every NaN is known to stay one, so a
// NaN row of activations costs a few blocks and any other scale at most one pass over the rows' scales,
// whatever the number of NaNs: 4096 x 14336 Q8_0 at 64 rows 117 us, with a NaN row of activations 120,
// with one infinite or NaN scale at a row's end 172 to 178 (the outputs one by one in their lanes:
// 17300, 1340).
// drow: the lane's row's first scale (dstep bytes a block), qrow: its code bytes (qstep); xq, xd: its
// token's codes and scales.
template <int FMT>
SYN_DEV void g32_settle(v16f_q& acc, int nb, const uint8_t* drow, int dstep, const uint8_t* qrow, int qstep,
                        const int8_t* xq, const float* xd) {
    const int h = (threadIdx.x >> 5) & 1;
    // bit 31 where v is a NaN, and bit 15 - i where v[i] is: no lane masks, of which a comparison each
    // would take the scalar registers of the loop above
    auto nan = [](float v) { return 0x7F800000u - (f2u(v) & 0x7FFFFFFFu); };
    auto nans = [&](const v16f_q& v) {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = __builtin_amdgcn_alignbit(m, nan(v[i]), 31);
        return m;
    };
    const uint32_t was = nans(acc);
    if (__builtin_amdgcn_ballot_w64(was != 0) == 0) return;  // uniform
    v16f_q sum = {};
    bool more = true;
#pragma unroll 1
    for (int b0 = 0; more && b0 < nb; b0 += 16) {  // uniform
        uint32_t odd = 0;  // bit j: block b0 + 8 h + j of the lane's row or token
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int b = b0 + 8 * h + j < nb ? b0 + 8 * h + j : nb - 1;
            const uint32_t dw = *reinterpret_cast<const uint16_t*>(drow + (int64_t)b * dstep);
            const uint32_t dx = f2u(xd[b]);
            odd |= (dw & 0x7C00u) == 0x7C00u || (dx & 0x7F800000u) == 0x7F800000u ? 1u << j : 0u;
        }
        uint32_t blocks = 0;  // any lane's
#pragma unroll 1
        for (int j = 0; j < 8; ++j) {
            const uint64_t m = __builtin_amdgcn_ballot_w64((odd >> j & 1) != 0);
            blocks |= ((uint32_t)m != 0 ? 1u << j : 0u) | ((uint32_t)(m >> 32) != 0 ? 256u << j : 0u);
        }
#pragma unroll 1
        for (; more && blocks; blocks &= blocks - 1) {
            const int b = b0 + __builtin_ctz(blocks);
            if (b >= nb) break;  // (the last block again)
            uint32_t w[4];
            __builtin_memcpy(w, qrow + (int64_t)b * qstep + (FMT == T_Q8_0 ? 16 * h : 0), 16);
            if constexpr (FMT == T_Q4_0) {  // 16 (n - 8), as the products take them
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = ((w[i] << (h ? 0 : 4)) & 0xF0F0F0F0u) ^ 0x80808080u;
            }
            const v4i_q a = {(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            const v4i_q x = *reinterpret_cast<const v4i_q*>(xq + 32 * (int64_t)b + 16 * h);
            const float dw = f16_to_f32(*reinterpret_cast<const uint16_t*>(drow + (int64_t)b * dstep)) *
                             (FMT == T_Q4_0 ? 0.0625f : 1.0f);
            const v16i_q f = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, x, v16i_q{}, 0, 0, 0);
            const v32f_q p = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, xd[b], v32f_q{}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[i] = sum[i] + p[i] * (float)f[i];
            more = __builtin_amdgcn_ballot_w64((was & ~nans(sum)) != 0) != 0;  // one is still open
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t m = (uint32_t)((int32_t)nan(acc[i]) >> 31);
        acc[i] = u2f((f2u(sum[i]) & m) | (f2u(acc[i]) & ~m));
    }
}

template <int FMT, int SPLIT, int MODE, int RG, int TG, int TT>
__global__ __launch_bounds__(64 * RG * TG * (MODE == G32_GATEUP ? 2 : 1), 2) void k_gemm_q32(G32Args g) {
    using C = G32Cfg<FMT, SPLIT, MODE, RG, TG, TT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = wave % RG, tg = wave / RG % TG, mat = wave / (RG * TG);  // mat: gate or up
    const int c = lane & 31, h = lane >> 5;
    const int row0 = (int)blockIdx.x * C::ROWS;
    const int nb = g.k / 32, nst = (nb + G32_S - 1) / G32_S;
    uint32_t e0 = 0;
    int T, tile = (int)blockIdx.z, tiles_step = (int)gridDim.z;
    const uint8_t* wm[C::R];
    if constexpr (MODE == G32_DENSE) {
        T = active_rows(g.active, 0, g.T);
        tile = (int)blockIdx.y;
        tiles_step = 1 << 30;
        wm[0] = g.w0;
    } else {
        const int e = (int)blockIdx.y;
        e0 = g.offsets[e];
        T = (int)(g.offsets[e + 1] - e0);
        if (g.err[0]) return;
        wm[0] = g.w0 + (uint64_t)e * g.mat_bytes;
        if constexpr (MODE == G32_GATEUP) wm[1] = g.w1 + (uint64_t)e * g.mat_bytes;
    }
    const uint32_t rb = (uint32_t)nb * (uint32_t)(SPLIT ? C::CB : C::BB);
    // GGUF: the 16-byte piece the matrix starts in, the start's offset in it, its last byte's piece
    const uint8_t* wbase[C::R];
    uint32_t mis[C::R], wlast[C::R];
#pragma unroll
    for (int r = 0; r < C::R; ++r) {
        mis[r] = SPLIT ? 0u : (uint32_t)((uintptr_t)wm[r] & 15);
        wbase[r] = wm[r] - mis[r];
        wlast[r] = (mis[r] + (uint32_t)g.n_out * rb - 1u) & ~15u;
    }
    const uint8_t* wscale = SPLIT ? g.w0 + (uint64_t)C::CB * (uint64_t)g.n_out * (uint64_t)nb : nullptr;
    const uint32_t ring = lds_addr(lds);
    v16i_q bias;
#pragma unroll
    for (int i = 0; i < 16; ++i) bias[i] = G32_BIAS;
    asm volatile("" : "+v"(bias));  // kept in 16 registers: a known constant is written again for every product

    for (; (int64_t)tile * C::TOK < T; tile += tiles_step) {  // uniform
        const int t0 = tile * C::TOK;
        const int valid = T - t0 < C::TOK ? T - t0 : C::TOK;
        auto token = [&](int t) -> uint32_t {  // the row of the codes that position t reads
            const int tc = t0 + (t < valid ? t : valid - 1);
            if constexpr (MODE == G32_DENSE) return (uint32_t)tc;
            if constexpr (MODE == G32_GATEUP) return g.slots[e0 + (uint32_t)tc] / (uint32_t)g.top_k;
            return e0 + (uint32_t)tc;
        };
        // this wavefront's copies of a kind: number wave + NW i of it
        auto nth = [&](int i, int n) { return wave + C::NW * i < n ? wave + C::NW * i : n - 1; };
        // (SPLIT: the last pieces of the codes and of the scales, for what lies past them)
        const uint32_t code_lim = (uint32_t)g.n_out * rb - 16u;
        const uint32_t scale_lim = (2u * (uint32_t)g.n_out * (uint32_t)nb - 1u) & ~3u;
        uint32_t woff[C::WPW], soff[C::SPW > 0 ? C::SPW : 1], aoff[C::APW], doff[C::DPW];
#pragma unroll
        for (int i = 0; i < C::WPW; ++i) {
            const int id0 = 64 * nth(i, C::WJ) + lane;
            const int id = id0 < C::NR * C::WCH ? id0 : C::NR * C::WCH - 1;
            const int lr = id / C::WCH, q = id - lr * C::WCH;
            const int r = row0 + lr % C::ROWS < g.n_out ? row0 + lr % C::ROWS : g.n_out - 1;
            if constexpr (SPLIT)
                woff[i] = (uint32_t)r * rb + 16u * (uint32_t)(q ^ (C::WCH == 8 ? lr & 7 : (lr >> 1) & 3));
            else  // (piece q begins 16 q after the piece that the stage's first byte lies in)
                woff[i] = (C::R == 2 && lr >= C::ROWS ? mis[C::R - 1] : mis[0]) + (uint32_t)r * rb + 16u * (uint32_t)q;
        }
        if constexpr (SPLIT) {
#pragma unroll
            for (int i = 0; i < C::SPW; ++i) {
                // the three dwords around a row's four F16 scales (of an odd number of blocks a row
                // every other row's begin between two dwords)
                const int id = 64 * nth(i, C::SJ) + lane, lr = id / 3;
                const int r = row0 + lr < g.n_out ? row0 + lr : g.n_out - 1;
                soff[i] = (((uint32_t)r * (uint32_t)nb * 2u) & ~3u) + 4u * (uint32_t)(id - 3 * lr);
            }
        }
#pragma unroll
        for (int i = 0; i < C::APW; ++i) {
            const int id = 64 * nth(i, C::AJ) + lane, t = id >> 3;
            aoff[i] = token(t) * (uint32_t)g.k + 16u * (uint32_t)((id & 7) ^ (t & 7));
        }
#pragma unroll
        for (int i = 0; i < C::DPW; ++i) doff[i] = token((64 * nth(i, C::DJ) + lane) % C::TOK) * (uint32_t)nb;
        auto issue = [&](int sn, int slot) __attribute__((always_inline)) {
            const int s = sn < nst ? sn : nst - 1;  // a stage past the row repeats the last, so that the counts stay
            const uint32_t st = ring + (uint32_t)(C::STAGE * slot);
#pragma unroll
            for (int i = 0; i < C::WPW; ++i) {
                const int u = nth(i, C::WJ);
                if constexpr (SPLIT) {
                    const uint32_t at = woff[i] + (uint32_t)C::STEP * (uint32_t)s;
                    lds_dma16(at < code_lim ? at : code_lim, g.w0, st + (uint32_t)(C::W_OFF + 1024 * u));
                } else {
                    // an instruction's 64 pieces belong to one matrix
                    static_assert(C::R == 1 || C::ROWS * C::WCH % 64 == 0, "gate and up on whole copies");
                    const bool up = C::R == 2 && 64 * u >= C::ROWS * C::WCH;
                    const uint32_t at = (woff[i] + (uint32_t)C::STEP * (uint32_t)s) & ~15u;
                    const uint32_t lim = up ? wlast[C::R - 1] : wlast[0];
                    lds_dma16(at < lim ? at : lim, up ? wbase[C::R - 1] : wbase[0],
                              st + (uint32_t)(C::W_OFF + 1024 * u));
                }
            }
            if constexpr (SPLIT) {
#pragma unroll
                for (int i = 0; i < C::SPW; ++i) {
                    const uint32_t at = soff[i] + 8u * (uint32_t)s;
                    lds_dma4(at < scale_lim ? at : scale_lim, wscale, st + (uint32_t)(C::SC_OFF + 256 * nth(i, C::SJ)));
                }
            }
            // (a last stage past a row's end reads on into the next row, or the scales that follow
            // the codes: not used)
#pragma unroll
            for (int i = 0; i < C::APW; ++i)
                lds_dma16(aoff[i], reinterpret_cast<const uint8_t*>(g.xq) + (size_t)(32 * G32_S) * (size_t)s,
                          st + (uint32_t)(C::A_OFF + 1024 * nth(i, C::AJ)));
#pragma unroll
            for (int i = 0; i < C::DPW; ++i) {
                const int u = nth(i, C::DJ);
                const int b = G32_S * s + (64 * u + lane) / C::TOK;
                lds_dma4(4u * (doff[i] + (uint32_t)(b < nb ? b : nb - 1)), g.xd,
                         st + (uint32_t)(C::DX_OFF + 256 * u));
            }
        };
        v16f_q acc[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[t] = v16f_q{};
        const bool busy = 32 * TT * tg < valid;  // uniform: this wavefront's token group holds tokens
        // lanes of the first half hold dw, of the second -M dw (Q4_0: of a 16th)
        const float unit = (h ? -G32_M : 1.0f) * (FMT == T_Q4_0 ? 0.0625f : 1.0f);
        const int lr = mat * C::ROWS + 32 * rg + c;  // this lane's row line
        const int rowc = row0 + 32 * rg + c < g.n_out ? row0 + 32 * rg + c : g.n_out - 1;
        const uint32_t rowoff = (C::R == 2 && mat ? mis[C::R - 1] : mis[0]) + (uint32_t)rowc * rb;
        // The operands of one 32 x 32 tile and block: read from the stage in LDS, then (the reads being
        // under way meanwhile) made what the products take.  Past the row's last block both scales are
        // 0, whose term is +0.0 whatever the codes.
        struct RowRaw {
            uint32_t w[5], m, d16;
        };
        struct Row {
            v4i_q a;
            float dw;
        };
        struct Tok {
            v4i_q b;
            uint32_t dx;
        };
        auto read_row = [&](const uint8_t* st, int s, int j) __attribute__((always_inline)) {
            RowRaw x;
            if constexpr (SPLIT) {
                const int q = FMT == T_Q8_0 ? (2 * j + h) ^ (lr & 7) : j ^ ((lr >> 1) & 3);
                const uint4 v = *reinterpret_cast<const uint4*>(st + C::W_OFF + lr * C::WL + 16 * q);
                x.w[0] = v.x, x.w[1] = v.y, x.w[2] = v.z, x.w[3] = v.w, x.w[4] = 0, x.m = 0;
                x.d16 = *reinterpret_cast<const uint16_t*>(st + C::SC_OFF + lr * 12 + (int)((uint32_t)rowc * (uint32_t)nb * 2u & 2u) + 2 * j);
            } else {
                const uint32_t sh = (rowoff + (uint32_t)C::STEP * (uint32_t)s) & 15u;
                const uint32_t o = (uint32_t)(lr * C::WL) + sh + (uint32_t)(C::BB * j);  // even
                x.d16 = *reinterpret_cast<const uint16_t*>(st + C::W_OFF + o);
                const uint32_t oc = o + 2u + (FMT == T_Q8_0 ? 16u * (uint32_t)h : 0u);
                const uint32_t* p = reinterpret_cast<const uint32_t*>(st + C::W_OFF + (oc & ~3u));
#pragma unroll
                for (int i = 0; i < 5; ++i) x.w[i] = p[i];
                x.m = oc & 2u;
            }
            return x;
        };
        auto make_row = [&](auto whole, const RowRaw& x, int s, int j) __attribute__((always_inline)) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w[i] = SPLIT ? x.w[i] : __builtin_amdgcn_alignbyte(x.w[i + 1], x.w[i], x.m);
                if constexpr (FMT == T_Q4_0)  // 16 (n - 8): the low nibbles for the first half, the high ones
                    w[i] = __builtin_amdgcn_bitop3_b32(w[i] << (h ? 0u : 4u), 0xF0F0F0F0u, 0x80808080u, 0x6A);  // (a & b) ^ c
            }
            return Row{v4i_q{(int)w[0], (int)w[1], (int)w[2], (int)w[3]},
                       f16_to_f32(decltype(whole)::value || G32_S * s + j < nb ? x.d16 : 0u) * unit};
        };
        auto read_tok = [&](const uint8_t* st, int j, int t) __attribute__((always_inline)) {
            const int lt = 32 * (TT * tg + t) + c;
            return Tok{*reinterpret_cast<const v4i_q*>(st + C::A_OFF + lt * 128 + 16 * ((2 * j + h) ^ (lt & 7))),
                       *reinterpret_cast<const uint32_t*>(st + C::DX_OFF + 4 * (j * C::TOK + lt))};
        };
        auto scale_of = [&](auto whole, const Tok& x, int s, int j) __attribute__((always_inline)) {
            return u2f(decltype(whole)::value || G32_S * s + j < nb ? x.dx : 0u);
        };
        // A tile's products (M + s and the two scale products) and its fold, a tile apart: the matrix
        // cores work on one tile while the vector ALU folds the one before.  The compiler's own order
        // puts each fold right after its products, behind their whole latency.
        v16i_q f[2];
        v32f_q pc[2];
        f[1] = v16i_q{};
        pc[1] = v32f_q{};  // nothing before the first: + 0
        auto fold = [&](v16f_q& a, int k, int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
            for (int i = lo; i < hi; ++i) a[i] = a[i] + __builtin_fmaf(pc[k][i], u2f((uint32_t)f[k][i]), pc[k][16 + i]);
        };
#pragma unroll
        for (int s = 0; s < C::NS - 1; ++s) issue(s, s);
        auto arrive = [&](int s, int slot) __attribute__((always_inline)) {
            wait_vm<C::COPIES * (C::NS - 2)>();  // this wavefront's copies of stage s have landed
            lds_barrier();                       // everyone's have, and stage s - 1 is read out
            issue(s + C::NS - 1, (slot + C::NS - 1) % C::NS);
        };
        // NT: the 32-token tiles of this wavefront that hold tokens
        auto loop = [&](auto tiles) __attribute__((always_inline)) {
            constexpr int NT = decltype(tiles)::value, UNITS = G32_S * NT;  // an even number
            // whole: every block of the stage is the row's (no scale to clear); slot: a constant
            // where one token tile leaves registers, so that the LDS offsets are the instructions' own
            auto stage = [&](auto whole, int s, int slot) __attribute__((always_inline)) {
                arrive(s, slot);
                const uint8_t* st = lds + C::STAGE * slot;
                RowRaw wr = read_row(st, s, 0);
                Row w;
                Tok x = read_tok(st, 0, 0);
#pragma unroll
                for (int u = 0; u < UNITS; ++u) {
                    const int j = u / NT, t = u % NT, k = u & 1;
                    v16f_q& prev = acc[(u + UNITS - 1) % NT];
                    if (t == 0) w = make_row(whole, wr, s, j);
                    float dx = scale_of(whole, x, s, j);
                    asm volatile("" : "+v"(w.a), "+v"(prev));
                    f[k] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w.a, x.b, bias, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (u + 1 < UNITS) {  // the next tile's operands
                        x = read_tok(st, (u + 1) / NT, (u + 1) % NT);
                        if (t + 1 == NT) wr = read_row(st, s, j + 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    fold(prev, k ^ 1, 0, 6);
                    asm volatile("" : "+v"(w.dw), "+v"(prev));
                    pc[k] = __builtin_amdgcn_mfma_f32_32x32x1f32(w.dw, dx, v32f_q{}, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    fold(prev, k ^ 1, 6, 16);
                    asm volatile("" : "+v"(prev));
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if constexpr (TT == 1) {
                const int nw = nb / G32_S;  // whole stages
                for (int s = 0; s < nw; s += C::NS) {
#pragma unroll
                    for (int i = 0; i < C::NS; ++i) {
                        if (s + i >= nw) break;  // uniform
                        stage(std::true_type{}, s + i, i);
                    }
                }
                if (nw < nst) stage(std::false_type{}, nw, nw % C::NS);
            } else {  // (two token tiles leave no registers for it)
                for (int s = 0; s < nst; ++s) stage(std::false_type{}, s, s % C::NS);
            }
            fold(acc[NT - 1], 1, 0, 16);
        };
        if (!busy)
            for (int s = 0; s < nst; ++s) arrive(s, s % C::NS);
        else if (TT == 1 || valid - 32 * TT * tg > 32)
            loop(std::integral_constant<int, TT>{});
        else
            loop(std::integral_constant<int, 1>{});
        wait_vm<0>();  // the last (repeated) copies have landed
        if (busy) {
            const uint8_t* w = C::R == 2 && mat ? wm[C::R - 1] : wm[0];
            const uint8_t* q = w + (uint64_t)rowc * rb + (SPLIT ? 0 : 2);
            const uint8_t* d = SPLIT ? wscale + 2 * (uint64_t)rowc * (uint64_t)nb : q - 2;
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const uint64_t x = token(32 * (TT * tg + t) + c);
                g32_settle<FMT>(acc[t], nb, d, SPLIT ? 2 : C::BB, q, SPLIT ? C::CB : C::BB, g.xq + x * (uint64_t)g.k,
                                g.xd + x * (uint64_t)nb);
            }
        }
        const bool vec = (g.n_out & 3) == 0 && ((uintptr_t)g.y & 15) == 0;  // uniform
        if (MODE != G32_DENSE || !vec) lds_barrier();  // the last stages are read out
        v16f_q up[TT];
        if constexpr (MODE == G32_GATEUP) {  // [wavefront][tile][i][lane]
            float* ux = reinterpret_cast<float*>(lds) + (size_t)(wave % (RG * TG)) * TT * 1024;
            static_assert(RG * TG * TT * 4096 <= C::LDS, "up's outputs fit the ring");
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (mat) ux[1024 * t + 64 * i + lane] = acc[t][i];
            lds_barrier();
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) up[t][i] = ux[1024 * t + 64 * i + lane];
            lds_barrier();  // read before another tile's copies
        }
        if (!busy || (C::R == 2 && mat)) continue;
        if constexpr (MODE == G32_DENSE) {
            // Rows of y that do not start at 16 bytes: the tile goes through the wavefront's part of LDS, so
            // that 32 lanes write a token's 32 outputs side by side and not four bytes of 32 tokens (4098 x 512
            // Q8_0 SPLIT at 1411 rows 27.5 against 37.1 us, of 4100 outputs 25.8).
            if (!vec) {
                static_assert(C::NW * 32 * 33 * 4 <= C::LDS, "the tiles fit the ring");
                int id = lane;
                asm volatile("" : "+v"(id));  // what follows from it is not computed before the loop, which has no registers left
                const int col = id & 31, half = id >> 5, n = row0 + 32 * rg + col;
                float* tx = reinterpret_cast<float*>(lds) + wave * 32 * 33;  // [token][row]
#pragma unroll
                for (int t = 0; t < TT; ++t) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) tx[33 * col + 4 * half + 8 * (i >> 2) + (i & 3)] = acc[t][i];
                    __builtin_amdgcn_wave_barrier();
                    const int first = 32 * (TT * tg + t);
                    const int tokens = valid - first < 32 ? valid - first : 32;
                    float* yr = g.y + (uint64_t)(t0 + first + half) * (uint64_t)g.n_out + (uint64_t)n;
#pragma unroll 4
                    for (int lt = half; lt < 32; lt += 2) {
                        if (lt < tokens && n < g.n_out) *yr = tx[33 * lt + col];
                        yr += 2 * (uint64_t)g.n_out;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
                continue;
            }
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int tt = 32 * (TT * tg + t) + c;
            if (tt >= valid) continue;
            const int tk = t0 + tt;
            const int n0 = row0 + 32 * rg + 4 * h;
            float o[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) o[i] = MODE == G32_GATEUP ? ref_silu(acc[t][i]) * up[t][i] : acc[t][i];
            const uint64_t yrow = MODE == G32_DENSE ? (uint64_t)tk
                                  : MODE == G32_GATEUP ? (uint64_t)(e0 + (uint32_t)tk)
                                                       : (uint64_t)g.slots[e0 + (uint32_t)tk];
            float* yr = g.y + yrow * (uint64_t)g.n_out;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + 8 * q;
                if (MODE == G32_DENSE || vec) {
                    if (n < g.n_out) *reinterpret_cast<float4*>(yr + n) = make_float4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (n + i < g.n_out) yr[n + i] = o[4 * q + i];
                }
            }
        }
    }
}

template <int FMT, int SPLIT, int MODE, int RG, int TG, int TT>
static void launch_g32(const G32Args& g, dim3 grid, hipStream_t stream) {
    using C = G32Cfg<FMT, SPLIT, MODE, RG, TG, TT>;
    // once per process, thread-safe (a function-local static); a refusal shows as the launch's error
    static const hipError_t attr = hipFuncSetAttribute((const void*)k_gemm_q32<FMT, SPLIT, MODE, RG, TG, TT>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    (void)attr;
    hipLaunchKernelGGL((k_gemm_q32<FMT, SPLIT, MODE, RG, TG, TT>), grid, dim3(64 * C::NW), (size_t)C::LDS, stream, g);
}

template <int FMT, int SPLIT, int RG, int TG, int TT>
static void launch_g32_dense(const G32Args& g, hipStream_t stream) {
    using C = G32Cfg<FMT, SPLIT, G32_DENSE, RG, TG, TT>;
    launch_g32<FMT, SPLIT, G32_DENSE, RG, TG, TT>(
        g, dim3((unsigned)((g.n_out + C::ROWS - 1) / C::ROWS), (unsigned)((g.T + C::TOK - 1) / C::TOK)), stream);
}

// Whether the kernel's 32-bit offsets and grid take the shape.
bool gemm_q32_fits(int ty, int n_out, int k, int T) {
    const uint64_t nb = (uint64_t)k / 32;
    return (ty == T_Q8_0 || ty == T_Q4_0) && nb > 0 && n_out > 0 && T > 0 && (T + 31) / 32 < 65536 &&
           (uint64_t)n_out * nb * (uint64_t)block_bytes(ty) < (1ull << 32) - 65536 &&
           (uint64_t)T * (uint64_t)k < (1ull << 32) - 65536;
}

// Wavefronts of one 32 x 32 tile until there are four a SIMD's worth, then of two (each weight operand
// made once for both: 14336 x 4096 Q8_0 at 512 rows 143 us).  Workgroups of 64 x 64 or 64 x 128, two
// a CU; up to 32 tokens, of 64 x 32.
constexpr int64_t G32_WIDE_TILES = 4096;

template <int FMT, int SPLIT>
static void launch_g32_fmt(const G32Args& g, hipStream_t stream) {
    const int64_t tiles = (int64_t)((g.n_out + 31) / 32) * ((g.T + 31) / 32);
    if (g.T <= 32)
        launch_g32_dense<FMT, SPLIT, 2, 1, 1>(g, stream);
    else if (tiles < G32_WIDE_TILES)
        launch_g32_dense<FMT, SPLIT, 2, 2, 1>(g, stream);
    else
        launch_g32_dense<FMT, SPLIT, 2, 2, 2>(g, stream);
}

void launch_gemm_q32(int ty, int split, const uint8_t* W, int n_out, int k, const int8_t* xq, const float* xd, int T,
                     float* y, hipStream_t stream, const uint32_t* active) {
    G32Args g{};
    g.w0 = W;
    g.xq = xq;
    g.xd = xd;
    g.y = y;
    g.n_out = n_out;
    g.k = k;
    g.T = T;
    g.active = active;
    if (ty == T_Q8_0)
        split ? launch_g32_fmt<T_Q8_0, 1>(g, stream) : launch_g32_fmt<T_Q8_0, 0>(g, stream);
    else
        split ? launch_g32_fmt<T_Q4_0, 1>(g, stream) : launch_g32_fmt<T_Q4_0, 0>(g, stream);
}

// Q8_0 experts in GGUF order.  mode 0: xq the tokens' rows (entry i reads row slots[i] / top_k),
// h[entry][n_out] = silu(gate) * up; mode 1: xq the entries' rows, y[slot][n_out].  An expert's entries
// go 64 a workgroup (32 where the experts average 16 or fewer, and a workgroup's LDS is better
// spent on a deeper ring: 64 experts of 1408 x 2048 at 128 rows 204 against 212 us a layer, at 300
// 277 against 219); the grid holds twice the average (an unused workgroup costs about a microsecond of a CU's LDS), and
// what is beyond it is walked in steps of the grid.  max_entries: the rows.
// The layer (64 experts, top 6, hidden 2048, inter 1408) against the vector-ALU kernel of moe_q8.hip,
// eight entries a pass: 300 rows 219 us against 2603, 32 rows 194 against 535, one row 75 against 155.
void launch_moe_q32(int mode, const uint8_t* w0, const uint8_t* w1, uint64_t mat_bytes, int n_experts, int n_out, int k,
                    const uint32_t* offsets, const uint32_t* slots, const uint32_t* err, int top_k, int max_entries,
                    int avg_entries, const int8_t* xq, const float* xd, float* y, hipStream_t stream) {
    G32Args g{};
    g.w0 = w0;
    g.w1 = w1;
    g.mat_bytes = mat_bytes;
    g.offsets = offsets;
    g.slots = slots;
    g.err = err;
    g.top_k = top_k;
    g.xq = xq;
    g.xd = xd;
    g.y = y;
    g.n_out = n_out;
    g.k = k;
    const bool few = avg_entries <= 16;
    const int tok = few ? 32 : 64, rows = mode == 0 || few ? 64 : 128;
    const int most = (max_entries + tok - 1) / tok, usual = (2 * avg_entries + tok - 1) / tok + 1;
    const dim3 grid((unsigned)((n_out + rows - 1) / rows), (unsigned)n_experts, (unsigned)(most < usual ? most : usual));
    if (mode == 0) {
        if (few)
            launch_g32<T_Q8_0, 0, G32_GATEUP, 2, 1, 1>(g, grid, stream);
        else
            launch_g32<T_Q8_0, 0, G32_GATEUP, 2, 1, 2>(g, grid, stream);
    } else {
        if (few)
            launch_g32<T_Q8_0, 0, G32_DOWN, 2, 1, 1>(g, grid, stream);
        else
            launch_g32<T_Q8_0, 0, G32_DOWN, 4, 1, 2>(g, grid, stream);
    }
}

}  // namespace syn
