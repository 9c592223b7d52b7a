// Prefill Q4_K GEMM on the gfx950 matrix cores: Y[t][n] for many activation rows t, each
// output the exact Gemv value (crates/kernels-cpu/src/gemv.rs:435-547: per super-block the
// term (d*dx)*S1 - (dmin*dx)*S2 with S1 = sum_j sc_j D_j and S2 = sum_j m_j s_j exact, folded
// in super-block order from +0.0).  The reference's Gemm is the same value (its Gemm kind is
// Gemv at a larger bucket, crates/kernels/src/reference/linear.rs:11-13).
//
// Exact sums on F16 matrix cores.  v_mfma_f32_16x16x32_f16 multiplies F16 operands exactly and
// accumulates in F32; when every operand is an integer and every partial sum stays below 2^24
// in magnitude, the F32 result is the exact integer whatever the order of the additions.  Per
// super-block the kernel feeds, for k = 0..255:
//   A[t][k] = x code (Q8_K, |x| <= 127, written as F16 by k_gemm_act);
//   B[k][n] = sc_j(k) * q_k - 512   (|B| <= 512, exact F16: the 6-bit scale folded into the
//                                     4-bit code, offset so that 256 * 127 * 512 < 2^24)
// so one accumulator holds D = S1 - 512 X exactly, X = sum_k x_k (a per-token integer the
// activation kernel stores), and fma(512, X, D) = fl(S1): one rounding of the exact S1, which
// is the reference's `S1 as f32`.  S2 comes from a second product per tile: A = (l_j, 64 h_j)
// with s_j = 64 h_j + l_j, B = (m_j, m_j), also exact.  The term and the fold are plain F32
// operations in the reference's order.
//
// B from the packed nibbles, two codes per instruction: the code dword (or it shifted right by
// 8) masked to the low nibbles of its 16-bit halves and ORed with 0x6400 in each half is the
// F16 pair (1024 + q0, 1024 + q1), and one v_pk_fma_f16 with (sc, -(1024 sc + 512)) gives
// sc*q - 512; masked to the high nibbles it is (1024 + 16 q0, 1024 + 16 q1), and the FMA takes
// (sc/16, -(64 sc + 512)).  Both are exact: every constant is an exact F16 (1024 sc + 512 =
// 512 (2 sc + 1)) and the FMA rounds once, to an exact integer.  The k order inside
// a super-block is free (the sum is exact), so each lane's eight k slots of an instruction are
// the codes of four consecutive bytes, low nibbles then high: k_gemm_act writes the activations
// in the same order.
//
// Tiling.  A wavefront computes 16 MT tokens x 16 NT rows as MT x NT tiles of 16 x 16, a workgroup four
// of them, one below the other.  The tokens' codes, sums, scales and X stream into LDS by
// global_load_lds_dwordx4 (no registers held while they fly); a row's weights serve one wavefront and
// go straight to its registers.  What bounds it: the vector ALU and the matrix cores, whose times add
// (per super-block and 64 tokens x 32 rows about 1150 cycles of matrix products, 560 of the fold's
// seven F32 operations an output, 700 of building B), then one wavefront's issue rate where a shape
// gives a SIMD only one.  14336 x 4096, X8, 2048 rows: 388 us (620 TFLOP/s) against 491 for workgroups of
// eight 64 x 32 wavefronts, one a CU, whose weights went through LDS; 4096 x 14336 at 64 rows 63 us
// against 220.
#include <type_traits>
#include "common.hpp"
#include "kernels.hpp"

namespace syn {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// ============================================================================================
// Activation layout (GemmAct)
// ============================================================================================
//
// For tpad = T rounded up to 64 and nb = k / 256 super-blocks:
//   codes [nb][tpad][256] F16: chunk c = 8p + s (8 codes) of token t holds the values
//         64p + 4s + {0, 2, 1, 3, 32, 34, 33, 35} and sits at chunk position c ^ (t & 15), so the
//         16 lanes of a read touch 16 distinct 16-byte bank groups;
//   tail  [nb][ s2: tpad x 16 F16 | dx: tpad x F32 | X: tpad x F32 ]: s2 = (l_0..l_7,
//         64 h_0..64 h_7) with s_j = 64 h_j + l_j, 0 <= l_j < 64; dx the Q8_K scale; X the sum
//         of the block's 256 codes.
// Rows t >= T are zero.
constexpr int GM_TAIL_ROW = 40;  // tail bytes per token per super-block

size_t gemm_act_bytes(int64_t tpad, int k) {
    const int64_t nb = k / 256;
    return align_up((uint64_t)(nb * tpad * 512), 256) + align_up((uint64_t)(nb * tpad * GM_TAIL_ROW), 256);
}

GemmAct gemm_act_at(uint8_t* base, int64_t tpad, int k) {
    const int64_t nb = k / 256;
    GemmAct a;
    a.codes = base;
    a.tail = base + align_up((uint64_t)(nb * tpad * 512), 256);
    a.tpad = (int)tpad;
    return a;
}

// One wavefront per (super-block b, token t): the Q8_K block of crates/kernels-cpu/src/gemv/
// act.rs:351-373 (q8k_block_lane), written in the GEMM order.  Lane l holds values 4l..4l+3
// (v4, loaded by the caller): sub-block j = l / 8, k part p = l / 16, nibble half h = (l / 8) & 1,
// dword s = l & 7.  A padding position (live false) writes zeros.
SYN_DEV void gemm_act_block(float4 v4, bool live, int b, int t, GemmAct a, int lane) {
    uint32_t q = 0;
    int sum32 = 0, xsum = 0;
    float d = 0.0f;
    if (live) {  // uniform over the wavefront
        const Q8KLane r = q8k_block_lane(v4, lane);
        q = r.packed;
        sum32 = r.sum32;
        d = r.d;
        xsum = sum32;
        xsum += __shfl_xor(xsum, 8);
        xsum += __shfl_xor(xsum, 16);
        xsum += __shfl_xor(xsum, 32);
    }
    const int p = lane >> 4, h = (lane >> 3) & 1, s = lane & 7;
    auto code = [&](int i) { return (_Float16)(float)(int8_t)(q >> (8 * i)); };
    h2 lo = {code(0), code(2)}, hi = {code(1), code(3)};
    const int pos = (8 * p + s) ^ (t & 15);
    uint8_t* dst = a.codes + ((int64_t)b * a.tpad + t) * 512 + pos * 16 + 8 * h;
    uint2 v;
    v.x = __builtin_bit_cast(uint32_t, lo);
    v.y = __builtin_bit_cast(uint32_t, hi);
    *reinterpret_cast<uint2*>(dst) = v;
    uint8_t* tail = a.tail + (int64_t)b * a.tpad * GM_TAIL_ROW;
    if ((lane & 7) == 0) {
        const int j = lane >> 3;
        const int hj = sum32 >> 6;  // floor: s = 64 h + l with 0 <= l < 64
        const int lj = sum32 - 64 * hj;
        _Float16* s2 = reinterpret_cast<_Float16*>(tail + (int64_t)t * 32);
        s2[j] = (_Float16)(float)lj;
        s2[8 + j] = (_Float16)(float)(64 * hj);
    }
    if (lane == 0) {
        reinterpret_cast<float*>(tail + (int64_t)a.tpad * 32)[t] = d;
        reinterpret_cast<float*>(tail + (int64_t)a.tpad * 36)[t] = (float)xsum;
    }
}

// A wavefront takes BPW consecutive super-blocks of one row, their loads issued together before
// any is quantized: at many blocks (ACT_WIDE_ITEMS or more) four a wavefront, which keeps more
// bytes in flight per wavefront (14336-wide rows at 2048 tokens: 45 against 50 us; the MoE layer's
// h: 43 against 56 us); below that one, which keeps more wavefronts (4096-wide: 15 against
// 17 us).  Item = (block group g, position t), t fastest.
constexpr int64_t ACT_WIDE_ITEMS = 65536;

template <int BPW, class RowOf>
SYN_DEV void gemm_act_blocks(int nb, int64_t item, GemmAct a, int lane, RowOf row_of) {
    const int ng = (nb + BPW - 1) / BPW;
    if (item >= (int64_t)ng * a.tpad) return;
    const int g = (int)(item / a.tpad), t = (int)(item - (int64_t)g * a.tpad);
    const float* row = row_of(t);  // null: a padding position
    float4 v[BPW];
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        const int b = g * BPW + j;
        v[j] = row && b < nb ? reinterpret_cast<const float4*>(row + (int64_t)b * 256)[lane] : float4{0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        const int b = g * BPW + j;
        if (b < nb) gemm_act_block(v[j], row != nullptr, b, t, a, lane);  // uniform
    }
}

// Blocks a wavefront for nb super-blocks at tpad positions, and the wavefronts that takes.
SYN_HD inline int gemm_act_bpw(int nb, int64_t tpad) { return (int64_t)nb * tpad >= ACT_WIDE_ITEMS ? 4 : 1; }
SYN_HD inline int64_t gemm_act_items(int nb, int64_t tpad) {
    const int bpw = gemm_act_bpw(nb, tpad);
    return (int64_t)((nb + bpw - 1) / bpw) * tpad;
}

template <int BPW>
__global__ __launch_bounds__(256) void k_gemm_act(const float* __restrict__ x, int T, int k, GemmAct a,
                                                  const uint32_t* __restrict__ active) {
    T = active_rows(active, 0, T);  // inactive rows are written as padding
    const int lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    gemm_act_blocks<BPW>(k / 256, item, a, lane, [&](int t) { return t < T ? x + (int64_t)t * k : nullptr; });
}

void launch_gemm_act(const float* x, int T, int k, GemmAct a, hipStream_t stream, const uint32_t* active) {
    const int64_t items = gemm_act_items(k / 256, a.tpad);
    if (items == 0) return;
    const dim3 grid((unsigned)((items + 3) / 4));
    if (gemm_act_bpw(k / 256, a.tpad) == 4)
        hipLaunchKernelGGL(k_gemm_act<4>, grid, dim3(256), 0, stream, x, T, k, a, active);
    else
        hipLaunchKernelGGL(k_gemm_act<1>, grid, dim3(256), 0, stream, x, T, k, a, active);
}

// ============================================================================================
// The GEMM
// ============================================================================================

constexpr int GM_WAVES = 4;                         // wavefronts per workgroup

// NT: 16-row tiles of a wavefront.
constexpr int gemm_rows(int nt) { return GM_WAVES * 16 * nt; }  // rows per workgroup

// MT: 16-token tiles, of a workgroup as of each of its wavefronts.  A stage is half a super-block of
// the tokens' codes: k steps 4 h .. 4 h + 3 of the eight.
template <int MT>
struct GmCfg {
    static constexpr int TT = 16 * MT;              // tokens
    static constexpr int AB = TT * 256;             // token code bytes per stage
    static constexpr int TB = TT * GM_TAIL_ROW;     // s2 | dx | X bytes per super-block
    // HALVES: two stages and one super-block's tail; else two super-blocks with theirs
    template <bool HALVES>
    static constexpr int TAIL = (HALVES ? 2 : 4) * AB;
    template <bool HALVES>
    static constexpr int LDS = TAIL<HALVES> + (HALVES ? 1 : 2) * TB;
    static constexpr int APW = AB / 1024 / GM_WAVES;  // a wavefront's loads (64 x 16 bytes) of a stage
    static constexpr int TPW = (TB / 16 + 64 * GM_WAVES - 1) / (64 * GM_WAVES);
    static_assert(AB % (1024 * GM_WAVES) == 0, "stage copies split evenly");
};

struct GemmArgs {
    const uint8_t* W;
    int layout;  // LAYOUT_SOURCE, LAYOUT_X8 (rows of whole 8-block runs) or LAYOUT_TILE64 (the experts)
    const uint8_t* codes;
    const uint8_t* tail;
    float* y;
    int N, T, nb, tpad;
    uint32_t rb;  // weight row bytes
    // blockIdx.x, blockIdx.y are the row and token tiles or, in a 1-D grid,
    int xcd_tokens;  // not 0: an XCD takes this many token tiles;
    int row_tiles;   // not 0: whole eights of row tiles come first, token tile by token tile, then the other rows
    const uint32_t* active;  // a step descriptor's rows_active, or null
};

// A super-block of the lane's rows (16 nt + lane % 16 of the wavefront's 32): the row header and, of
// lane group p, bytes 32 p .. + 31 of the codes.  A row's weights serve one wavefront, so they go
// straight to its registers, half a super-block ahead.
template <int NT>
struct GemmW {
    v4u hdr[NT], q[NT][2];
};

SYN_DEV uint32_t gemm_chunk_step(int layout) { return layout == LAYOUT_X8 ? 128u : 16u; }
SYN_DEV uint32_t gemm_row_offset(int layout, uint32_t r, uint32_t rb) {
    return layout == LAYOUT_TILE64 ? (uint32_t)tile64_row_offset(r, rb) : r * rb;
}

// wb: the super-block of the matrix's row 0; off: the lane's rows from there; qoff: its chunks 1 + 2 p.
template <int NT>
SYN_DEV GemmW<NT> gemm_weights(const uint8_t* wb, const uint32_t (&off)[NT], const uint32_t (&qoff)[NT],
                               uint32_t chunk_step) {
    GemmW<NT> w;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        w.hdr[nt] = *reinterpret_cast<const v4u*>(wb + off[nt]);
        w.q[nt][0] = *reinterpret_cast<const v4u*>(wb + qoff[nt]);
        w.q[nt][1] = *reinterpret_cast<const v4u*>(wb + chunk_step + qoff[nt]);
    }
    return w;
}

// The source chunk of token copy u (half 0; half 1 has bit 2 flipped) for a token whose row is skewed
// by `skew`: line 4 u + lane / 16 holds logical chunk (p, s) at position (4 p + s) ^ (line & 15), so
// that the 16 lines of a read touch 16 different 16-byte bank groups.
SYN_DEV uint32_t gemm_achunk(int u, int lane, uint32_t skew) {
    const int slot = (lane & 15) ^ ((4 * u + (lane >> 4)) & 15);
    return (uint32_t)(8 * (slot >> 2) + (slot & 3)) ^ (skew & 15u);
}

// The lane's 32-bit offsets of its copies, relative to the part's base of the super-block: token codes
// (of copy 0: 16 tokens on for each further one; half 1 has bit 6 flipped) and tail.
template <int MT>
struct GemmSlots {
    uint32_t aoff;
    int left;  // positions that exist from t0 on (a multiple of 64); a tile past them re-reads the last
    uint32_t toff[GmCfg<MT>::TPW];
};

template <int MT>
SYN_DEV GemmSlots<MT> gemm_slots(int tpad, int wave, int lane, int t0) {
    using C = GmCfg<MT>;
    GemmSlots<MT> s;
    const int left = s.left = tpad - t0;
    const int t = 4 * wave + (lane >> 4);  // of copy 0
    s.aoff = (uint32_t)t * 512u + 16u * gemm_achunk(wave, lane, (uint32_t)t);
#pragma unroll
    for (int i = 0; i < C::TPW; ++i) {
        // tokens' s2 (two pieces a token), then scales and code sums (a piece for four tokens)
        const int ti = 64 * (wave + GM_WAVES * i) + lane;
        const int part = ti < C::TT * 2 ? 0 : ti < C::TT * 2 + C::TT / 4 ? 1 : 2;
        const int at = part == 0 ? ti : ti - C::TT * 2 - (part - 1) * (C::TT / 4);
        const int end = part == 0 ? left * 2 : left / 4;
        s.toff[i] = (uint32_t)tpad * (part == 0 ? 0u : 28u + 4u * (uint32_t)part) + (uint32_t)t0 * (part == 0 ? 32u : 4u) +
                    16u * (uint32_t)(at < end ? at : end - 1);
    }
    return s;
}

// Issues the wavefront's copies of half H of the tokens' super-block at `ab` to `stage`; half 1 brings
// the tail.
template <int MT, int H>
SYN_DEV void gemm_issue(const GemmSlots<MT>& s, const uint8_t* ab, const uint8_t* tb, int wave, int lane,
                        uint8_t* stage, uint8_t* tail) {
    using C = GmCfg<MT>;
#pragma unroll
    for (int i = 0; i < C::APW; ++i) {
        static_assert(GM_WAVES == 4, "16 tokens a round of copies");
        lds_dma16<true>(s.aoff ^ (64u * H), ab + 512u * (uint32_t)(16 * i < s.left ? 16 * i : s.left - 16),
                  lds_addr(stage) + 1024u * (uint32_t)(wave + GM_WAVES * i));
    }
    if constexpr (H == 1) {
#pragma unroll
        for (int i = 0; i < C::TPW; ++i) {
            const int u = wave + GM_WAVES * i;
            if (64 * u + lane < C::TB / 16) lds_dma16<true>(s.toff[i], tb, lds_addr(tail) + 1024u * (uint32_t)u);
        }
    }
}

// The F16 pair (1024 + 16 q0, 1024 + 16 q1) etc. from the nibbles under `mask`.
// (v & mask) | 0x64006400 is one v_bitop3_b32 (truth table 0xEA = (a & b) | c); written as two
// operations the compiler issues an AND and an OR.
SYN_DEV h2 magic_pair(uint32_t v, uint32_t mask) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_bitop3_b32(v, mask, 0x64006400u, 0xEA));
}

SYN_DEV h2 bcast(_Float16 v) { return h2{v, v}; }

// What a super-block's products and fold need from its row headers: the pairs (sc, -(1024 sc + 512)) of
// sub-block 2p and (sc/16, -(64 sc + 512)) of 2p + 1, d, dmin and the minimums.
template <int NT>
struct GemmHdr {
    h2 ka[NT], kb[NT];
    float dd[NT], dm[NT];
    uint32_t mn[NT][2];  // m_0..3, m_4..7
};

template <int NT>
SYN_DEV void gemm_header(const GemmW<NT>& w, int p, GemmHdr<NT>& h) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const v4u hdr = w.hdr[nt];
        h.dd[nt] = f16_to_f32(hdr.x);
        h.dm[nt] = f16_to_f32(hdr.x >> 16);
        // get_scale_min_k4 (gemv.rs:528-537) on packed bytes
        const uint32_t w0 = hdr.y, w1 = hdr.z, w2 = hdr.w;
        const uint32_t sc_lo = w0 & 0x3F3F3F3Fu;                                 // sc_0..3
        const uint32_t sc_hi = (w2 & 0x0F0F0F0Fu) | ((w0 >> 2) & 0x30303030u);   // sc_4..7
        h.mn[nt][0] = w1 & 0x3F3F3F3Fu;                                          // m_0..3
        h.mn[nt][1] = ((w2 >> 4) & 0x0F0F0F0Fu) | ((w1 >> 2) & 0x30303030u);     // m_4..7
        // this lane group's sub-blocks: 2p (low nibbles) and 2p + 1 (high nibbles)
        const uint32_t scw = p < 2 ? sc_lo : sc_hi;
        const int sa = (int)((scw >> (16 * (p & 1))) & 0xFFu), sb = (int)((scw >> (16 * (p & 1) + 8)) & 0xFFu);
        const float fa = (float)sa, fb = (float)sb;
        h.ka[nt] = h2{(_Float16)fa, (_Float16)(-(1024.0f * fa + 512.0f))};
        h.kb[nt] = h2{(_Float16)(fb * 0.0625f), (_Float16)(-(64.0f * fb + 512.0f))};
    }
}

// The S2 operand: m_0..m_7 in lane groups 0 and 1 (against l_j and 64 h_j), zero in 2 and 3.
SYN_DEV v8h gemm_mins(const uint32_t (&mn)[2], int p) {
    const _Float16 on = p < 2 ? (_Float16)1.0f : (_Float16)0.0f;
    const h2 k1 = bcast(on), k0 = bcast((_Float16)(-1024.0f) * on);
    h2 m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)  // bytes 2 i, 2 i + 1 into the low bits of two halves
        m[i] = __builtin_elementwise_fma(
            __builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, mn[i >> 1], i & 1 ? 0x0c030c02u : 0x0c010c00u) | 0x64006400u), k1, k0);
    return v8h{m[0].x, m[0].y, m[1].x, m[1].y, m[2].x, m[2].y, m[3].x, m[3].y};
}

// The matrix-core part of one stage of the wavefront's tokens x 32 rows: dacc = S1 - 512 X exactly
// once both halves have run (half 0 starts it).  Only the first NMT 16-token tiles are computed (a
// tile of fewer entries leaves the rest empty).
template <int MT, int NMT, int H, int NT>
SYN_DEV void gemm_mfma(const uint8_t* st, const GemmW<NT>& w, int lane, v4f (&dacc)[MT][NT], const GemmHdr<NT>& h) {
    const int c = lane & 15, p = lane >> 4;
    const uint8_t* at = st + c * 256;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        v8h bq[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            uint32_t v = w.q[nt][H][s];  // sub-block 2p (low nibbles) and 2p + 1 (high)
            // keeps a step's operands from being made before it (and spilling)
            asm volatile("" : "+v"(v) : : "memory");
            // (b0, b2) low nibbles, (b1, b3) low, (b0, b2) high, (b1, b3) high
            const h2 y3 = __builtin_elementwise_fma(magic_pair(v, 0x000F000Fu), bcast(h.ka[nt].x), bcast(h.ka[nt].y));
            const h2 y2 = __builtin_elementwise_fma(magic_pair(v >> 8, 0x000F000Fu), bcast(h.ka[nt].x), bcast(h.ka[nt].y));
            const h2 y1 = __builtin_elementwise_fma(magic_pair(v, 0x00F000F0u), bcast(h.kb[nt].x), bcast(h.kb[nt].y));
            const h2 y4 = __builtin_elementwise_fma(magic_pair(v >> 8, 0x00F000F0u), bcast(h.kb[nt].x), bcast(h.kb[nt].y));
            bq[nt] = v8h{y3.x, y3.y, y2.x, y2.y, y1.x, y1.y, y4.x, y4.y};
        }
#pragma unroll
        for (int mt = 0; mt < NMT; ++mt) {
            const v8h a = *reinterpret_cast<const v8h*>(at + 16 * mt * 256 + (((4 * p + s) ^ c) << 4));
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                dacc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    a, bq[nt], H == 0 && s == 0 ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : dacc[mt][nt], 0, 0, 0);
            if (mt % 4 == 3) {  // four tiles' operands at a time
                asm volatile("" : : : "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// S2 from the tail's code sums, then the super-block's terms folded into the accumulators in
// the reference's rounding order.
template <int MT, int NMT, int NT>
SYN_DEV void gemm_fold(const uint8_t* tl, int lane, const v4f (&dacc)[MT][NT], const GemmHdr<NT>& h,
                       v4f (&acc)[MT][NT]) {
    constexpr int TT = 16 * MT;
    const int c = lane & 15, p = lane >> 4;
    const v8h zero8 = {};
    v8h bm[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) bm[nt] = gemm_mins(h.mn[nt], p);
#pragma unroll
    for (int mt = 0; mt < NMT; ++mt) {
        const v8h as = p < 2 ? *reinterpret_cast<const v8h*>(tl + (16 * mt + c) * 32 + 16 * p) : zero8;
        const v4f dx = *reinterpret_cast<const v4f*>(tl + TT * 32 + (16 * mt + 4 * p) * 4);
        const v4f xs = *reinterpret_cast<const v4f*>(tl + TT * 36 + (16 * mt + 4 * p) * 4);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const v4f s2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(as, bm[nt], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float s1 = __builtin_fmaf(512.0f, xs[i], dacc[mt][nt][i]);  // fl(S1), exact operands
                const float a1 = (h.dd[nt] * dx[i]) * s1;
                const float a2 = (h.dm[nt] * dx[i]) * s2[i];
                acc[mt][nt][i] = acc[mt][nt][i] + (a1 - a2);
            }
        }
        asm volatile("" : "+v"(acc[mt][0]), "+v"(acc[mt][NT - 1]) : : "memory");  // as above: a tile's operands at a time
    }
}

// The stage loop of both GEMM kernels.  `issue(half, b, stage, tail)` issues the wavefront's copies of a
// half of super-block b, `weights(b)` loads its rows.  HALVES: one barrier a half; once every
// wavefront's copies of a half have landed and every wavefront has left the half before, the next
// half's copies go to that one's place (the tail, which comes with half 1, after the fold before).
// Otherwise the same with whole super-blocks: twice the LDS, half the barriers, and a super-block's
// time for the copies to land, which is what counts where a SIMD holds few wavefronts.  On return
// the LDS may still be read.
template <bool HALVES, int MT, int NMT, int NT, class Issue, class Weights>
SYN_DEV void gemm_loop(int nb, uint8_t* smem, int lane, Issue&& issue, Weights&& weights, v4f (&acc)[MT][NT]) {
    using C = GmCfg<MT>;
    std::integral_constant<int, 0> h0;
    std::integral_constant<int, 1> h1;
    uint8_t* tails = smem + C::template TAIL<HALVES>;
    issue(h0, 0, smem, tails);
    if (!HALVES) issue(h1, 0, smem + C::AB, tails);
    GemmW<NT> next = weights(0);
    for (int b = 0; b < nb; ++b) {
        v4f d[MT][NT];
        GemmHdr<NT> h;
        const int buf = HALVES ? 0 : b & 1;
        uint8_t *st = smem + buf * 2 * C::AB, *tl = tails + buf * C::TB;
        wait_vm<0>();
        lds_barrier();
        const GemmW<NT> w = next;
        if constexpr (HALVES) {
            issue(h1, b, st + C::AB, tl);
        } else if (b + 1 < nb) {
            uint8_t *sn = smem + (buf ^ 1) * 2 * C::AB, *tn = tails + (buf ^ 1) * C::TB;
            issue(h0, b + 1, sn, tn);
            issue(h1, b + 1, sn + C::AB, tn);
            next = weights(b + 1);
        }
        gemm_header(w, lane >> 4, h);
        gemm_mfma<MT, NMT, 0>(st, w, lane, d, h);
        if constexpr (HALVES) {
            wait_vm<0>();
            lds_barrier();
            if (b + 1 < nb) {
                issue(h0, b + 1, st, tl);
                next = weights(b + 1);
            }
        }
        gemm_mfma<MT, NMT, 1>(st + C::AB, w, lane, d, h);
        gemm_fold<MT, NMT>(tl, lane, d, h, acc);
    }
}

// The loop on the 16-token tiles that hold `valid` tokens.
template <bool HALVES, int MT, int NMT, int NT, class Issue, class Weights>
SYN_DEV void gemm_tiles(int valid, int nb, uint8_t* smem, int lane, Issue&& issue, Weights&& weights,
                        v4f (&acc)[MT][NT]) {
    if constexpr (NMT < MT) {
        if (valid > 16 * NMT) {
            gemm_tiles<HALVES, MT, NMT + (MT > 4 ? 2 : 1), NT>(valid, nb, smem, lane, issue, weights, acc);
            return;
        }
    }
    gemm_loop<HALVES, MT, NMT, NT>(nb, smem, lane, issue, weights, acc);
}

// GU: W stacks N / 2 gate rows and as many up rows; a wavefront's two row tiles are 16 gate rows and
// the same up rows, and y[t][N / 2] = silu(gate) * up (the product k_silu_mul makes of a written y).
template <bool HALVES, int MT, int NT, bool GU>
__global__ __launch_bounds__(64 * GM_WAVES, 2) void k_gemm_q4k(GemmArgs g) {
    static_assert(!GU || NT == 2, "a gate tile and an up tile");
    using C = GmCfg<MT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: copy bases in SGPRs
    const int c = lane & 15, p = lane >> 4;
    int nx = (int)blockIdx.x, ty = (int)blockIdx.y;
    if (g.xcd_tokens) {
        const int id = nx >> 3;
        ty = (nx & 7) * g.xcd_tokens + id % g.xcd_tokens, nx = id / g.xcd_tokens;
    } else if (g.row_tiles) {
        const int eights = g.row_tiles & ~7, first = eights * ((g.T + C::TT - 1) / C::TT);
        const bool rest = nx >= first;
        const int id = rest ? nx - first : nx, wide = rest ? g.row_tiles - eights : eights;
        ty = id / wide, nx = (rest ? eights : 0) + id % wide;
    }
    const int cols = GU ? g.N / 2 : g.N;
    const int n0 = GU ? nx * (gemm_rows(NT) / 2) + 16 * wave : nx * gemm_rows(NT) + 16 * NT * wave, t0 = ty * C::TT;
    const int T = active_rows(g.active, 0, g.T);
    if (t0 >= T) return;  // uniform: a token tile past the step's active rows
    const GemmSlots<MT> sl = gemm_slots<MT>(g.tpad, wave, lane, t0);
    uint32_t off[NT], qoff[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + (GU ? 0 : 16 * nt) + c;
        off[nt] = gemm_row_offset(g.layout, (uint32_t)((n < cols ? n : cols - 1) + (GU ? nt * cols : 0)), g.rb);
        qoff[nt] = off[nt] + gemm_chunk_step(g.layout) * (uint32_t)(1 + 2 * p);
    }
    v4f acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    auto issue = [&](auto half, int b, uint8_t* stage, uint8_t* tail) {
        gemm_issue<MT, decltype(half)::value>(sl, g.codes + ((size_t)b * g.tpad + t0) * 512,
                                              g.tail + (size_t)b * g.tpad * GM_TAIL_ROW, wave, lane, stage, tail);
    };
    // super-block b of row 0: in X8 block b sits in run b / 8 at position b % 8
    auto weights = [&](int b) {
        return gemm_weights(g.layout == LAYOUT_X8 ? g.W + 1152 * (size_t)(b >> 3) + 16 * (size_t)(b & 7)
                                                  : g.W + 144 * (size_t)b,
                            off, qoff, gemm_chunk_step(g.layout));
    };
    gemm_tiles<HALVES, MT, (MT > 4 ? 2 : 1), NT>(T - t0, g.nb, smem, lane, issue, weights, acc);

#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < (GU ? 1 : NT); ++nt) {
            const int n = n0 + 16 * nt + c;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = t0 + 16 * mt + 4 * p + i;
                if (t < T && n < cols)
                    g.y[(int64_t)t * cols + n] = GU ? ref_silu(acc[mt][0][i]) * acc[mt][NT - 1][i] : acc[mt][nt][i];
            }
        }
}

bool gemm_q4k_supported(int n_out, int k) {
    return k >= 256 && k % 256 == 0 && n_out > 0 &&
           (uint64_t)n_out * (uint64_t)(k / 256) * 144u < (1ull << 32);
}

// The wavefront tile.  A large one makes each weight operand once for more tokens and reads each token
// once for more rows, a small one gives the SIMDs wavefronts: one alone issues a vector operation
// every five cycles, two every two and a half.  Microseconds measured for 32 tokens x 16 rows | 64 x
// 16 | 64 x 32 (whole super-blocks, halves) | 128 x 32:
//                                                        X8                          GGUF
//   4096 x 4096 at 64 rows (512 wavefronts of 32 x 16)   21 | 27 | 45, 44 | 48       22 | 28 | 43, 42 | 47
//   4096 x 4096 at 200 (1792)                            34 | 35 | 50, 49 | 75       29 | 32 | 46, 45 | 73
//   4096 x 4096 at 333 (1536 of 64 x 16)                 53 | 47 | 54, 52 | 78       40 | 41 | 48, 47 | 75
//   8192 x 2048 at 333 (3072)                                                        34 | 32 | 36, 36 | 42
//   14336 x 4096 at 200 (3584)                          104 | 85 | 70, 80 | 82       71 | 62 | 59, 62 | 74
//   8192 x 2048 at 448 (3584)                                                        41 | 39 | 37, 36 | 43
//   14336 x 4096 at 333 (336 workgroups of 128 x 128)   154 | 127 | 112, 110 | 97    96 | 89 | 93, 81 | 80
//   11264 x 2048 at 512 (352)                                                        57 | 52 | 51, 47 | 54
//   11264 x 2048 at 600 (440)                                                        68 | 59 | 60, 59 | 55
//   14336 x 4096 at 600 (560)                          255 | 192 | 160, 161 | 155   160 | 136 | 127, 120 | 140
//   14336 x 4096 at 1024 (896)                          424 | 314 | 246, 255 | 215   258 | 218 | 204, 181 | 187
//   4096 x 4096 at 2048 (512)                                                       153 | 133 | 119, 117 | 108
//   14336 x 4096 at 2048 (1792)                         878 | 639 | 487, 497 | 388   514 | 425 | 386, 346 | 332
// X8 reaches the 128-token form first: a 16-byte chunk of a block shares its 128-byte line with seven
// other blocks' chunks, so a workgroup draws eight times its weight bytes through its L1, and twice
// the tokens halve that.  The 128-token form holds 512 workgroups on the chip, the 64-token one 768; in
// GGUF order it is the better one where its last round is nearly full or one of several.  64 x 32 with whole
// super-blocks holds two workgroups a CU, halves three: the former while two hold them all.
// Against eight wavefronts of 64 x 32 a CU, whose weights went through LDS, GGUF order is up to 7 % slower where
// that form's 256 workgroups just filled the chip (4096 x 14336 at 850 rows 202 against 189 us, 8192 x 2048
// at 448 36.5 against 35.2; eight wavefronts with the weights in registers are no faster).
constexpr int64_t GM_SMALL_WAVES = 2048, GM_MID_WAVES = 3072, GM_WIDE_X8 = 320, GM_WIDE = 420;
constexpr int64_t GM_WIDE_ROUND = 512, GM_WIDE_NEXT = 896;

template <bool HALVES, int MT, int NT, bool GU = false>
static void launch_gemm_tiles(GemmArgs g, hipStream_t stream) {
    using C = GmCfg<MT>;
    // once per process, thread-safe (a function-local static); a refusal shows as the launch's error
    static const hipError_t attr =
        hipFuncSetAttribute((const void*)k_gemm_q4k<HALVES, MT, NT, GU>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            C::template LDS<HALVES>);
    (void)attr;
    const int cols = GU ? g.N / 2 : g.N, wide = GU ? gemm_rows(NT) / 2 : gemm_rows(NT);
    const unsigned nx = (unsigned)((cols + wide - 1) / wide), ny = (unsigned)((g.T + C::TT - 1) / C::TT);
    // Workgroups go to the 8 XCDs in turn.  Row tile by row tile, an XCD's L2 sees an eighth of the
    // weights and all tokens; where the tokens are the larger operand (512 bytes a super-block
    // against 144) and give every XCD as many tiles, an eighth of the tokens and all weights (GGUF 2048
    // x 8192 at 2048 rows 145 against 155 us; X8, whose lines are read eight times, 4096 x 14336 451
    // against 400).
    g.xcd_tokens = g.layout != LAYOUT_X8 && ny % 8 == 0 && nx < (1u << 23) / ny &&
                           (int64_t)g.T * 512 > (int64_t)g.N * 144 ? (int)(ny / 8) : 0;
    // Where the row tiles are no multiple of 8, a row's tile goes to another XCD at every token tile, and
    // each L2 sees all weights.  In X8, whose lines are read eight times, that took up to four times as
    // long (6000 x 4096, 47 tiles: 144 us at 600 rows, 285 at 2048; 14000 x 4096, 110 tiles: 323 at 1024),
    // so the odd tiles go last (74, 181, 216); up to 16 tiles they are too large a part (14 tiles of 8192: 148
    // against 154 us).  GGUF order does not need it (within 2 %).
    g.row_tiles = g.layout == LAYOUT_X8 && nx % 8 != 0 && nx > 16 && nx < (1u << 23) / ny ? (int)nx : 0;
    const bool flat = g.xcd_tokens || g.row_tiles;
    const dim3 grid(flat ? nx * ny : nx, flat ? 1u : ny);
    hipLaunchKernelGGL((k_gemm_q4k<HALVES, MT, NT, GU>), grid, dim3(64 * GM_WAVES), C::template LDS<HALVES>, stream, g);
}

static GemmArgs gemm_args(int layout, const uint8_t* W, int n_out, int k, GemmAct a, int T, float* y,
                          const uint32_t* active) {
    GemmArgs g{};
    g.active = active;
    g.W = W;
    g.layout = layout;
    g.codes = a.codes;
    g.tail = a.tail;
    g.y = y;
    g.N = n_out;
    g.T = T;
    g.nb = k / 256;
    g.tpad = a.tpad;
    g.rb = (uint32_t)(k / 256) * 144u;
    return g;
}

static bool gemm_mid(int64_t n, int64_t t) { return (n + 15) / 16 * ((t + 63) / 64) <= GM_MID_WAVES; }

template <bool GU>
static void launch_gemm_wide(const GemmArgs& g, hipStream_t stream) {
    const int64_t n = g.N, t = g.T;
    const int64_t wide = (n + 127) / 128 * ((t + 127) / 128);  // workgroups of 128 tokens
    if (g.layout == LAYOUT_X8 ? wide >= GM_WIDE_X8
                              : wide >= GM_WIDE_NEXT || (wide >= GM_WIDE && wide <= GM_WIDE_ROUND))
        launch_gemm_tiles<true, 8, 2, GU>(g, stream);
    else if ((n + 127) / 128 * ((t + 63) / 64) <= 512)
        launch_gemm_tiles<false, 4, 2, GU>(g, stream);
    else
        launch_gemm_tiles<true, 4, 2, GU>(g, stream);
}

void launch_gemm_q4k(int layout, const uint8_t* W, int n_out, int k, GemmAct a, int T, float* y,
                     hipStream_t stream, const uint32_t* active) {
    const GemmArgs g = gemm_args(layout, W, n_out, k, a, T, y, active);
    const int64_t n = n_out, t = T;
    if ((n + 15) / 16 * ((t + 31) / 32) <= GM_SMALL_WAVES)
        launch_gemm_tiles<false, 2, 1>(g, stream);
    else if (gemm_mid(n, t))
        launch_gemm_tiles<true, 4, 1>(g, stream);
    else
        launch_gemm_wide<false>(g, stream);
}

// Where the product takes tiles of two 16-row tiles a wavefront: GateUpAct's gate and up then meet in
// one (no [T][2 n] product written and read back: 5632 x 2048 at 333 rows 43.1 -> 38.8 us); below, the
// smaller tiles and k_silu_mul.
bool gemm_q4k_gate_up_fits(int n, int T) {
    const int64_t n2 = 2 * (int64_t)n;
    return (n2 + 15) / 16 * ((T + 31) / 32) > GM_SMALL_WAVES && !gemm_mid(n2, T);
}

void launch_gemm_q4k_gate_up(int layout, const uint8_t* W, int n, int k, GemmAct a, int T, float* y,
                             hipStream_t stream, const uint32_t* active) {
    launch_gemm_wide<true>(gemm_args(layout, W, 2 * n, k, a, T, y, active), stream);
}

// ============================================================================================
// The MoE layer at many tokens: the grouped expert FFN on the same matrix cores
// ============================================================================================
//
// Each expert's entries (the packed lists of k_moe_pack: offsets, slots) are padded to whole
// 64-entry tiles: tile i belongs to expert tile_e[i], and its padded position p = 64 i + t holds
// entry offsets[e] + p - pad_off[e] when that is below offsets[e + 1] (padding positions'
// outputs are dropped).  An entry's row is quantized exactly as the expert quantizes it
// (moe.rs:479-492), which depends on the row alone, so:
//   gate/up: the tokens' rows are quantized to Q8_K once, in the GEMM layout, and each stage
//     gathers position p's row from its entry's token (slots[i] / top_k); a workgroup takes
//     (tile, 64 weight rows); its 128-row weight tile is those 64 rows of the tile's gate
//     matrix followed by the same 64 rows of its up matrix, so wavefronts 0-1 hold g and
//     wavefronts 2-3 hold u of the same outputs, and h = silu(g) * u per entry
//     (moe.rs:529-551);
//   down: the entries' h rows quantized at their padded positions; (tile, 128 rows) of the
//     expert's down matrix; each output goes to its entry's slot (moe.rs:500-515).
// Every product is the Gemv value (the same exact sums and term fold as the dense GEMM).

// One workgroup: an inclusive scan of the experts' tile counts (E <= 256).
__global__ __launch_bounds__(256) void k_moe_tiles(const uint32_t* __restrict__ offsets, int n_experts,
                                                   const uint32_t* __restrict__ err, MoeTiles mt) {
    __shared__ uint32_t cnt[256];
    const int e = threadIdx.x;
    const bool bad = err[0] != 0;  // uniform: the layer writes nothing
    const uint32_t n = (!bad && e < n_experts) ? offsets[e + 1] - offsets[e] : 0u;
    const uint32_t tiles = (n + 63u) / 64u;
    cnt[e] = tiles;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t v = e >= off ? cnt[e - off] : 0u;
        __syncthreads();
        cnt[e] += v;
        __syncthreads();
    }
    const uint32_t end = cnt[e], begin = end - tiles;
    if (e < n_experts) mt.pad_off[e] = 64u * begin;
    if (e == n_experts - 1) {
        mt.pad_off[n_experts] = 64u * end;
        mt.n_tiles[0] = end;
    }
    for (uint32_t i = begin; i < end; ++i) mt.tile_e[i] = (uint32_t)e;
}

void launch_moe_tiles(const uint32_t* offsets, int n_experts, const uint32_t* err, MoeTiles mt,
                      hipStream_t stream) {
    hipLaunchKernelGGL(k_moe_tiles, dim3(1), dim3(256), 0, stream, offsets, n_experts, err, mt);
}

// The entries' h rows at their padded positions (row i of h for entry i).  Positions in tiles
// past the used ones are not written (no workgroup reads them).
template <int BPW>
__global__ __launch_bounds__(256) void k_moe_gemm_act(const float* __restrict__ h, int k,
                                                      const uint32_t* __restrict__ offsets, MoeTiles mt,
                                                      const uint32_t* __restrict__ err, GemmAct a) {
    if (err[0]) return;
    const int lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t ng = (k / 256 + BPW - 1) / BPW;
    if (item >= ng * a.tpad) return;
    const uint32_t tile = (uint32_t)(item - (item / a.tpad) * a.tpad) / 64u;
    if (tile >= mt.n_tiles[0]) return;  // a tile past the used ones: nothing reads it
    gemm_act_blocks<BPW>(k / 256, item, a, lane, [&](int pos) {
        const uint32_t e = mt.tile_e[tile];
        const uint32_t i = offsets[e] + ((uint32_t)pos - mt.pad_off[e]);
        return i < offsets[e + 1] ? h + (int64_t)i * k : nullptr;
    });
}

void launch_moe_gemm_act(const float* h, int k, const uint32_t* offsets, MoeTiles mt, const uint32_t* err,
                         GemmAct a, hipStream_t stream) {
    const int64_t items = gemm_act_items(k / 256, a.tpad);
    if (items == 0) return;
    const dim3 grid((unsigned)((items + 3) / 4));
    if (gemm_act_bpw(k / 256, a.tpad) == 4)
        hipLaunchKernelGGL(k_moe_gemm_act<4>, grid, dim3(256), 0, stream, h, k, offsets, mt, err, a);
    else
        hipLaunchKernelGGL(k_moe_gemm_act<1>, grid, dim3(256), 0, stream, h, k, offsets, mt, err, a);
}

struct MoeGemmArgs {
    const uint8_t* W0;  // gate (MODE 0) or down (MODE 1), stacked by expert
    const uint8_t* W1;  // up (MODE 0)
    uint64_t ebytes;    // bytes of one expert's matrix
    GemmAct act;
    int nb;             // super-blocks along k
    uint32_t rb;        // weight row bytes
    int row_tiles;      // workgroups per entry tile
    const uint32_t* offsets;
    MoeTiles mt;
    const uint32_t* err;
    const uint32_t* slots;
    float* out;         // h [entries][cols] (MODE 0) or out [slots][cols] (MODE 1)
    int cols;           // inter (MODE 0) or hidden (MODE 1)
    int layout;         // LAYOUT_SOURCE or LAYOUT_TILE64 (the row tiles are whole 64-row runs)
    int top_k;          // MODE 0: act holds the tokens' rows, position p of a tile reads its
                        // entry's token slots[i] / top_k
};

constexpr int GM_MT = 4;  // 16-entry tiles of an entry tile
constexpr int GM_NT = 2, GM_ROWS = gemm_rows(GM_NT);

// MODE 0 (gate/up, 64 weight rows of each per workgroup) or 1 (down, 128 rows).
template <int MODE>
__global__ __launch_bounds__(64 * GM_WAVES, 3) void k_moe_gemm(MoeGemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    if (g.err[0]) return;
    const int tile = (int)blockIdx.x / g.row_tiles, rt = (int)blockIdx.x - tile * g.row_tiles;
    if ((uint32_t)tile >= g.mt.n_tiles[0]) return;  // uniform per workgroup
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t e = g.mt.tile_e[tile];
    const int t0 = 64 * tile;
    const uint32_t i0 = g.offsets[e] + ((uint32_t)t0 - g.mt.pad_off[e]);
    const uint32_t left = g.offsets[e + 1] - i0;
    const int nvalid = left < 64u ? (int)left : 64;
    constexpr int ROWS = MODE == 0 ? GM_ROWS / 2 : GM_ROWS;  // rows of each matrix
    using C = GmCfg<GM_MT>;
    const int c = lane & 15, p = lane >> 4;
    // MODE 0: wavefronts 0-1 take the gate matrix's rows, 2-3 the same rows of up
    const bool upper = MODE == 0 && wave >= GM_WAVES / 2;
    const uint8_t* wm = (upper ? g.W1 : g.W0) + (uint64_t)e * g.ebytes + (uint64_t)rt * ROWS * g.rb;
    uint32_t off[GM_NT], qoff[GM_NT];
#pragma unroll
    for (int nt = 0; nt < GM_NT; ++nt) {
        off[nt] = gemm_row_offset(g.layout, (uint32_t)(16 * GM_NT * (wave - (upper ? GM_WAVES / 2 : 0)) + 16 * nt + c), g.rb);
        qoff[nt] = off[nt] + 16u * (uint32_t)(1 + 2 * p);
    }
    // super-block b of the tile's rows: 144 b on in GGUF order, 64 rows' blocks on in TILE64
    const size_t bstep = g.layout == LAYOUT_TILE64 ? (size_t)TILE64_ROWS * 144 : 144;
    auto weights = [&](int b) { return gemm_weights(wm + bstep * (size_t)b, off, qoff, 16u); };
    // MODE 0 gathers each position's token row from the tokens' quantized rows: a token's chunks are
    // skewed by its own number, the stage's lines by the position's.  Tail: wavefronts 0-1 the s2
    // halves, 2 the scales, 3 the code sums, one position a lane (padding positions read token 0;
    // their outputs are dropped)
    GemmSlots<GM_MT> sl = gemm_slots<GM_MT>(g.act.tpad, wave, lane, t0);
    static_assert(C::TT == 64 && C::TPW == 1, "one tail part a wavefront");
    const uint32_t tp = (uint32_t)g.act.tpad;
    auto token_of = [&](int pa) -> uint32_t {
        return pa < nvalid ? g.slots[i0 + (uint32_t)pa] / (uint32_t)g.top_k : 0u;
    };
    uint32_t aoff[C::APW];
    if constexpr (MODE == 0) {
#pragma unroll
        for (int i = 0; i < C::APW; ++i) {
            const int u = wave + GM_WAVES * i;
            const uint32_t tok = token_of(4 * u + (lane >> 4));
            aoff[i] = tok * 512u + 16u * gemm_achunk(u, lane, tok);
        }
        sl.toff[0] = wave < 2 ? token_of((64 * wave + lane) >> 1) * 32u + 16u * (uint32_t)(lane & 1)
                              : tp * (wave == 2 ? 32u : 36u) + token_of(lane) * 4u;
    }
    auto issue = [&](auto half, int b, uint8_t* stage, uint8_t* tail) {
        constexpr int H = decltype(half)::value;
        // super-block bases in 64 bits (2 * hidden * tp bytes of codes may pass 2^32); the offsets
        // within one super-block's rows stay below 2^25
        const uint8_t* ab = g.act.codes + ((size_t)b * tp + (MODE == 0 ? 0 : t0)) * 512u;
        const uint8_t* tb = g.act.tail + (size_t)b * tp * (uint32_t)GM_TAIL_ROW;
        if constexpr (MODE == 1) {
            gemm_issue<GM_MT, H>(sl, ab, tb, wave, lane, stage, tail);
        } else {
            const uint32_t tl = lds_addr(tail);
#pragma unroll
            for (int i = 0; i < C::APW; ++i)
                lds_dma16<true>(aoff[i] ^ (64u * H), ab, lds_addr(stage) + 1024u * (uint32_t)(wave + GM_WAVES * i));
            if constexpr (H == 1) {
                if (wave < 2)
                    lds_dma16<true>(sl.toff[0], tb, tl + 1024u * (uint32_t)wave);
                else
                    lds_dma4<true>(sl.toff[0], tb, tl + (wave == 2 ? 2048u : 2304u));
            }
        }
    };
    v4f acc[GM_MT][GM_NT];
#pragma unroll
    for (int mt = 0; mt < GM_MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < GM_NT; ++nt) acc[mt][nt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    // the 16-token tiles holding entries (the padding of an expert's last tile is not computed;
    // its outputs are dropped)
    gemm_tiles<true, GM_MT, 1, GM_NT>(nvalid, g.nb, smem, lane, issue, weights, acc);
    if constexpr (MODE == 0) {
        // u (the upper wavefronts) through LDS to the wavefronts holding g of the same outputs
        float* ux = reinterpret_cast<float*>(smem);  // [64 tokens][64 rows]
        lds_barrier();                               // the last stage is read out
        if (wave >= GM_WAVES / 2) {
#pragma unroll
            for (int mt = 0; mt < GM_MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < GM_NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        ux[(16 * mt + 4 * p + i) * ROWS + 16 * GM_NT * (wave - GM_WAVES / 2) + 16 * nt + c] = acc[mt][nt][i];
        }
        lds_barrier();
        if (wave < GM_WAVES / 2) {
#pragma unroll
            for (int mt = 0; mt < GM_MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < GM_NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int t = 16 * mt + 4 * p + i, r = 16 * GM_NT * wave + 16 * nt + c;
                        if (t < nvalid) {
                            const float u = ux[t * ROWS + r];
                            g.out[(int64_t)(i0 + t) * g.cols + rt * ROWS + r] = ref_silu(acc[mt][nt][i]) * u;
                        }
                    }
        }
    } else {
#pragma unroll
        for (int mt = 0; mt < GM_MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < GM_NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int t = 16 * mt + 4 * p + i, r = 16 * GM_NT * wave + 16 * nt + c;
                    if (t < nvalid) g.out[(int64_t)g.slots[i0 + t] * g.cols + rt * ROWS + r] = acc[mt][nt][i];
                }
    }
}

void launch_moe_gemm(int mode, const uint8_t* w0, const uint8_t* w1, int n_experts, int rows, int k,
                     GemmAct act, int max_tiles, const uint32_t* offsets, MoeTiles mt, const uint32_t* err,
                     const uint32_t* slots, float* out, hipStream_t stream, int top_k, int layout) {
    static_assert(GM_ROWS == 2 * TILE64_ROWS, "row tiles of whole TILE64 runs");
    MoeGemmArgs g;
    g.top_k = top_k;
    g.layout = layout == LAYOUT_TILE64 ? (int)LAYOUT_TILE64 : (int)LAYOUT_SOURCE;
    g.W0 = w0;
    g.W1 = w1;
    g.nb = k / 256;
    g.rb = (uint32_t)g.nb * 144u;
    g.ebytes = (uint64_t)rows * g.rb;
    g.act = act;
    g.row_tiles = mode == 0 ? rows / (GM_ROWS / 2) : rows / GM_ROWS;
    g.offsets = offsets;
    g.mt = mt;
    g.err = err;
    g.slots = slots;
    g.out = out;
    g.cols = rows;
    const dim3 grid((unsigned)(max_tiles * g.row_tiles));
    if (mode == 0) {
        static const hipError_t ok0 = hipFuncSetAttribute((const void*)k_moe_gemm<0>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, GmCfg<GM_MT>::LDS<true>);
        (void)ok0;  // a refusal shows as the launch's error
        hipLaunchKernelGGL(k_moe_gemm<0>, grid, dim3(64 * GM_WAVES), GmCfg<GM_MT>::LDS<true>, stream, g);
    } else {
        static const hipError_t ok1 = hipFuncSetAttribute((const void*)k_moe_gemm<1>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, GmCfg<GM_MT>::LDS<true>);
        (void)ok1;
        hipLaunchKernelGGL(k_moe_gemm<1>, grid, dim3(64 * GM_WAVES), GmCfg<GM_MT>::LDS<true>, stream, g);
    }
}

// Row tiles: gate/up 64 rows, down 128.
bool moe_gemm_supported(int hidden, int inter) { return hidden % GM_ROWS == 0 && inter % (GM_ROWS / 2) == 0; }

}  // namespace syn
