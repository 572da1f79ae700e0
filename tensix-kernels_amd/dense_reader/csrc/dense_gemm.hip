// dense_gemm.hip: the matmul of many rows (prefill), a tiled MFMA kernel over the packed weights.
//
// A workgroup of four wavefronts sums 32 MT rows by 256 columns (128 with a GLU), 64 columns a wavefront (the weights'
// rows of the MFMA, so that a lane ends with runs of columns), or (KS) 64 rows by 64 columns with each wavefront a
// quarter of K. What bounds it, and why this split:
// - the MFMA is 32x32x16: on MI355X it takes 13.7 ns a wavefront's SIMD (32 cycles), 2.4 PFLOP/s on a few CUs and about
//   1.7 on all of them with random values (power); 16x16x32 takes 13 ns for half the work, whatever the wavefronts;
// - a weight decoded from block-float costs 2.5 VALU instructions (bfloat8_b) of about 5 cycles, so a wavefront decodes
//   each once for all of its rows, in registers, one 64-k step ahead, the pairs of values spread between the MFMAs;
// - x is shared through LDS, four stages of 64 k: 64 columns a wavefront keep its LDS reads at half the MFMA's time (at
//   32 columns they take all of it). Its loads go straight to LDS (no registers, no writes by the wavefronts) three
//   steps ahead, the weights' codes to registers three steps ahead;
// - one workgroup a CU: 256 accumulators a lane at 256 rows, so that the stream of one wavefront must keep the SIMD
//   busy by itself, which the step's barrier at its middle (the next stage's operands are then read ahead across the
//   step's end) and the decode between the MFMAs are for. One step of 256 rows takes 1.28 us (bf16) or 1.39 us
//   (block-float) of its 0.87 us of MFMA at full clocks.
// bfloat8_b 1000 rows K = 4096 N = 14336 454 us in passes of 32 rows -> 111 us (1.06 PFLOP/s); bfloat4_b gate and up
// 333 rows 425 -> 85 us.

#include "dense_gemm.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace drk {

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// s of lane I of this row of 16
template <int I>
__device__ __forceinline__ float row_bcast(float s) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(s), 0x150 + I, 0xF, 0xF, true));
}
template <int B>
__device__ __forceinline__ float sbyte(uint32_t w) {
    return (float)(int)(signed char)(w >> (8 * B));
}

__device__ __forceinline__ f32x16 mfma32(uint4 w, uint4 x, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}

// The wavefront's LDS reads done and all but its newest VM vector memory loads landed, then (BAR) the workgroup's
// barrier. The x loads write LDS when they return, which the compiler's own waits follow by the LDS variable (each
// stage is one of its own) but not across wavefronts: this wait and barrier are what orders them.
template <int VM, bool BAR>
__device__ __forceinline__ void step_barrier() {
    static_assert(VM < 64, "step_barrier: vmcnt counts to 63");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));  // vmcnt(VM) lgkmcnt(0)
    if constexpr (BAR) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int I>
using ic = std::integral_constant<int, I>;
// f(ic<0>), .. f(ic<N - 1>)
template <int N, typename F, int I = 0>
__device__ __forceinline__ void unroll(F&& f) {
    if constexpr (I < N) {
        f(ic<I>{});
        unroll<N, F, I + 1>(static_cast<F&&>(f));
    }
}

// The workgroup's column tile and first row: workgroups go to the XCDs in turn, each XCD takes a run of tiles, the row
// tiles of one column tile after each other, so that the weights come into its L2 once.
__device__ __forceinline__ void gemm_tile(const GemmArgs& a, int bm, int& nt, int& m0) {
    const int total = a.tm * a.tn, xcd = blockIdx.x & 7;
    const int w = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
    nt = w / a.tm;
    m0 = (w - nt * a.tm) * bm;
}

// A lane's operands of one 64-k step: the weights' codes, one 16-byte load or more a 32-column tile
template <int FMT>
struct StepCodes {
    uint4 c[2][FMT == DR_BFP8 ? 2 : FMT == DR_BFP4 ? 1 : 4];
};

// MT row tiles of 32, two column tiles of 32 a wavefront (with GLU the gate's and the up's). KS: the wavefronts split
// K instead of lying side by side. acc: lane l's sums, row 32 t + l % 32, columns 8 g + 4 (l / 32) + 0 .. 3 of tile n in
// words 4 g + 0 .. 3.
// F32 (a float32 y, which shows the sums' rounding): the accumulators are carried over into further sums before they grow
// long. One accumulator for all of K rounds at each of its K / 16 MFMAs, which at K = 4096 and 14336 was 2.5 and 4.5 times
// the error of the passes of 32 rows (bfloat8_b 2.0e-7 against 8.0e-8, 4.7e-7 against 1.04e-7). At 64 rows they hold 256 k
// at a time, added up in three levels of eight; at 128 (block-float, up to K = F32_MT4_K), where the registers leave room for
// one more sum of each (bfloat8_b: but for two, kept in scratch), 256 k up to K = 2048 and 512 past it, added up in turn,
// much as the passes' wavefronts do. No larger an error than the passes' at any K (7.4e-8, at 128 rows 8.0e-8, and 8.7e-8; measured at K = 96 to
// 28672, each format). 1000 rows K = 4096 N = 14336 444 us in passes, 126 with one accumulator, 235 in tiles of 64 rows,
// 168 of 128.
template <int MT, int FMT, bool GLU, bool KS, bool F32>
__device__ __forceinline__ void gemm_k_loop(const GemmArgs& a, int nt, int m0, f32x16 (&acc)[2][MT], uint4* x0, uint4* x1,
                                            uint4* x2, uint4* x3) {
    constexpr int OT = GLU ? 1 : 2;                            // output tiles a wavefront
    constexpr int XW = KS ? 1 : GEMM_W;                        // wavefronts that stage one x together
    constexpr int NX = 32 * MT * 8 / (64 * XW);                // 16-byte x chunks a lane stages a step
    constexpr int NC = FMT == DR_BFP8 ? 2 : FMT == DR_BFP4 ? 1 : 4;
    constexpr int NG = 4 * MT;                                 // groups of two MFMAs a step
    constexpr int PF = F32 && MT > 2 ? 1 : 3;                  // x operands read ahead (fewer where registers are short)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, p = (lane >> 4) & 1, h = lane >> 5;
    const int t0 = KS ? nt * OT : (nt * GEMM_W + wave) * OT;   // the wavefront's first output tile

    // the two column tiles' bases; a lane reads panel p's columns
    const uint8_t* cb[2];
    const uint8_t* eb[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int to = min(GLU ? t0 : t0 + n, a.tiles - 1);
        const bool up = GLU && n == 1 && a.seg.glu == 2;
        const int tw = GLU && a.seg.glu == 1 ? 2 * to + n : to;
        cb[n] = (up ? a.seg.codes_up : a.seg.codes) + (size_t)(2 * tw) * a.seg.pstride;
        eb[n] = (up ? a.seg.exps_up : a.seg.exps) + (size_t)(2 * tw) * a.k_pad;
    }
    const uint32_t co = (uint32_t)p * a.seg.pstride + (uint32_t)(16 * h + c) * 16u;
    const uint32_t eo = (uint32_t)(p * a.k_pad + 4 * (16 * h + c));

    // K in groups of 256 (four steps): every wavefront all of them, or (KS) its share
    const int groups = a.k_pad >> 8;
    const int g0 = KS ? groups * wave / GEMM_W : 0, g1 = KS ? groups * (wave + 1) / GEMM_W : groups;
    if (KS && g0 == g1) return;
    const int s1 = 4 * g1 - 1;  // (the last step)

    // x: row r's chunk u' = 2 u + h (8 k: those MFMA u takes in lane half h) sits at slot 8 r + (u' ^ ((r >> 1) & 7)). A
    // lane's slots are 64 (wave + XW i) + lane, its chunk the same for all of them.
    const int wx = KS ? 0 : wave;
    const int ch = (lane & 7) ^ ((4 * wx + (lane >> 4)) & 7);
    auto chunk_k = [](int ch) {
        const int u = ch >> 1, hh = ch & 1;
        return FMT == DR_BFP8 ? 16 * (2 * (u >> 1) + hh) + 8 * (u & 1) : FMT == DR_BFP4 ? 32 * hh + 8 * u : 8 * ch;
    };
    const int xk[2] = {chunk_k(ch), chunk_k(KS ? ch ^ 4 : ch)};  // (KS: odd loads' rows are 8 further)
    // buffer loads from the tile's first row to its last (rows past x read as zeros)
    const uint32_t ldx2 = 2u * (uint32_t)a.ldx;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + (size_t)m0 * a.ldx), (short)0, (int)(ldx2 * (uint32_t)min(a.m - m0, 32 * MT)), 0x00020000);
    const uint32_t xo = (uint32_t)(8 * wx + (lane >> 3)) * ldx2;
    const int xbase = KS ? wave * 32 * MT * 8 : 0;  // (KS: the wavefront's own part of each stage)
    auto load_x = [&](int s, uint4* b) {
        const uint32_t ko = 128u * (uint32_t)min(s, s1);
#pragma unroll
        for (int i = 0; i < NX; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(b + xbase + 64 * (wx + XW * i)), 16,
                                                     xo + 2u * (uint32_t)xk[i & 1] + (ko + 8 * XW * i * ldx2), 0, 0, 0);
    };
    // a ragged K's last steps: the columns past K of the lane's own chunks (landed) become zeros
    const bool ragged = a.k != a.k_pad;
    auto zero_x = [&](int s, uint4* b) {
        if (ragged && 64 * (s + 1) > a.k) {
#pragma unroll
            for (int i = 0; i < NX; ++i)
                if (64 * s + xk[i & 1] >= a.k) b[xbase + 64 * (wx + XW * i) + lane] = make_uint4(0u, 0u, 0u, 0u);
        }
    };
    const int xrow = lane & 31;
    auto read_x = [&](const uint4* b, int u, int t) {
        return b[xbase + (32 * t + xrow) * 8 + ((2 * u + h) ^ ((xrow >> 1) & 7))];
    };

    auto load_c = [&](int s, StepCodes<FMT>& k) {
        s = min(s, s1);
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int v = 0; v < NC; ++v) {
                const uint32_t o = FMT == DR_BFP8 ? (uint32_t)s * 1024u + 512u * v
                                   : FMT == DR_BFP4 ? (uint32_t)s * 512u
                                                    : (uint32_t)s * 2048u + 512u * v;
                k.c[n][v] = *reinterpret_cast<const uint4*>(cb[n] + (co + o));
            }
    };
    uint32_t e[2][2], en[2][2];  // exponents of the group that the decode is in, and of the next
    auto load_e = [&](int g, uint32_t (&d)[2][2]) {
        if constexpr (FMT != DR_BF16) {
            g = min(g, g1 - 1);
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int v = 0; v < 2; ++v)
                    d[n][v] = *reinterpret_cast<const uint32_t*>(eb[n] + (eo + (uint32_t)g * 256u + 128u * v));
        }
    };

    // decode of step j of its group, in 32 pairs of values, those of the MFMAs needed first before the others
    struct Scales {
        float s[2][2];
        uint32_t lo, hi;
    } sc;
    auto scales = [&](auto jj) {
        constexpr int j = decltype(jj)::value;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            if constexpr (FMT == DR_BFP8) {
#pragma unroll
                for (int v = 0; v < 2; ++v) sc.s[n][v] = __builtin_ldexpf(1.f, (int)((e[n][v] >> (8 * j)) & 0xFFu) - 133);
            } else if constexpr (FMT == DR_BFP4) {
                const uint32_t w = e[n][j & 1] >> (16 * (j >> 1));
                sc.s[n][0] = __builtin_ldexpf(1.f, (int)(w & 0xFFu) - 133);
                sc.s[n][1] = __builtin_ldexpf(1.f, (int)((w >> 8) & 0xFFu) - 133);
            }
        }
    };
    auto decode = [&](auto pi, const StepCodes<FMT>& k, uint4 (&B)[2][4]) {
        constexpr int P = decltype(pi)::value, unit = P >> 2, q = P & 3, u = unit >> 1, n = unit & 1;
        float v0, v1;
        if constexpr (FMT == DR_BFP8) {
            const uint4& w4 = k.c[n][u >> 1];
            constexpr int d = 2 * (u & 1) + (q >> 1);
            const uint32_t w = d == 0 ? w4.x : d == 1 ? w4.y : d == 2 ? w4.z : w4.w;
            const float s = sc.s[n][u >> 1];
            v0 = sbyte<2 * (q & 1)>(w) * row_bcast<8 * (u & 1) + 2 * q>(s);
            v1 = sbyte<2 * (q & 1) + 1>(w) * row_bcast<8 * (u & 1) + 2 * q + 1>(s);
        } else {
            const uint4& w4 = k.c[n][0];
            const uint32_t w = u == 0 ? w4.x : u == 1 ? w4.y : u == 2 ? w4.z : w4.w;
            // nibble u' = m + 8 at the top of a byte, its top bit flipped: 16 m as a signed byte (the scale has the 1 / 16)
            if constexpr (q == 0) {
                sc.lo = ((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
                sc.hi = (w & 0xF0F0F0F0u) ^ 0x80808080u;
            }
            const uint32_t b = q < 2 ? sc.lo : sc.hi;
            v0 = sbyte<2 * (q & 1)>(b) * row_bcast<4 * u + q>(sc.s[n][0]);
            v1 = sbyte<2 * (q & 1) + 1>(b) * row_bcast<4 * u + q>(sc.s[n][1]);
        }
        const uint32_t w = pack_bf16(v0, v1);
        if constexpr (q == 0) B[n][u].x = w;
        if constexpr (q == 1) B[n][u].y = w;
        if constexpr (q == 2) B[n][u].z = w;
        if constexpr (q == 3) B[n][u].w = w;
    };

    constexpr int L = !F32 ? 0 : MT == 2 ? 3 : 1;  // sums beside the accumulators
    f32x16 lev[L ? L : 1][2][L ? MT : 1];            // (L 3: of 256, 2048 and 16384 k)
    if constexpr (F32) {
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int t = 0; t < MT; ++t) lev[l][n][t] = acc[n][t];  // (zeros)
    }
    StepCodes<FMT> k0, k1, k2, k3;  // step s's codes in k[s % 4], asked for three steps ahead
    uint4 B0[2][4], B1[2][4];       // the decoded operands of even and odd steps (bf16 weights: the codes themselves)
    uint4 A[PF + 1];
    // step s (its x in xc, its operands in Bc or kc): the next step's operands decoded between its MFMAs; at its middle
    // the next step's x is there for every wavefront, and the codes and x of step s + 3 are asked for
    auto step = [&](int s, auto jj, const uint4* xc, uint4* xn, uint4* xf, uint4 (&Bc)[2][4], uint4 (&Bn)[2][4],
                    StepCodes<FMT>& kc, StepCodes<FMT>& kn, StepCodes<FMT>& kf) {
        constexpr int j = decltype(jj)::value;
        if constexpr (FMT != DR_BF16) {
            if constexpr (j == 3) {
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int v = 0; v < 2; ++v) e[n][v] = en[n][v];
            }
            scales(ic<(j + 1) & 3>{});
        }
        unroll<NG>([&](auto gg) {
            constexpr int G = decltype(gg)::value, u = G / MT, t = G % MT;
            if constexpr (G == NG / 2) {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt((NX & 15) | (7 << 4) | (15 << 8) | ((NX >> 4) << 14));  // vmcnt(NX): x of s + 1
                if (s < s1) zero_x(s + 1, xn);
                step_barrier<NX, !KS>();
                load_c(s + 3, kf);
                if constexpr (j == 0) load_e((s >> 2) + 1, en);
                __builtin_amdgcn_sched_barrier(0);
                load_x(s + 3, xf);
                __builtin_amdgcn_sched_barrier(0);
            }
            // (the operand PF groups ahead: past this step's end the next step's first)
            constexpr int Gf = G + PF;
            if constexpr (Gf < NG)
                A[Gf % (PF + 1)] = read_x(xc, Gf / MT, Gf % MT);
            else
                A[Gf % (PF + 1)] = read_x(xn, (Gf - NG) / MT, (Gf - NG) % MT);
            const uint4 x = A[G % (PF + 1)];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                if constexpr (FMT == DR_BF16)
                    acc[n][t] = mfma32(kc.c[n][u], x, acc[n][t]);
                else
                    acc[n][t] = mfma32(Bc[n][u], x, acc[n][t]);
            }
            if constexpr (FMT != DR_BF16) {
                constexpr int P0 = G * 32 / NG, P1 = (G + 1) * 32 / NG;
                unroll<P1 - P0>([&](auto d) { decode(ic<P0 + decltype(d)::value>{}, kn, Bn); });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    static_assert(NG % (PF + 1) == 0, "the x operands' ring turns whole steps");

    const int s0 = 4 * g0;
    load_c(s0, k0);
    load_c(s0 + 1, k1);
    load_c(s0 + 2, k2);
    load_e(g0, e);
    __builtin_amdgcn_sched_barrier(0);
    load_x(s0, x0);
    load_x(s0 + 1, x1);
    load_x(s0 + 2, x2);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FMT != DR_BF16) {
        scales(ic<0>{});
        unroll<32>([&](auto d) { decode(d, k0, B0); });
    }
    __builtin_amdgcn_s_waitcnt(((2 * NX) & 15) | (7 << 4) | (15 << 8) | (((2 * NX) >> 4) << 14));
    zero_x(s0, x0);
    step_barrier<2 * NX, !KS>();
#pragma unroll
    for (int i = 0; i < PF; ++i) A[i] = read_x(x0, i / MT, i % MT);
    for (int g = g0; g < g1; ++g) {
        step(4 * g + 0, ic<0>{}, x0, x1, x3, B0, B1, k0, k1, k3);
        step(4 * g + 1, ic<1>{}, x1, x2, x0, B1, B0, k1, k2, k0);
        step(4 * g + 2, ic<2>{}, x2, x3, x1, B0, B1, k2, k3, k1);
        step(4 * g + 3, ic<3>{}, x3, x0, x2, B1, B0, k3, k0, k2);
        if constexpr (F32) {
            auto carry = [](f32x16 (&to)[2][MT], f32x16 (&from)[2][MT]) {
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        to[n][t] += from[n][t];
#pragma unroll
                        for (int i = 0; i < 16; ++i) from[n][t][i] = 0.f;
                    }
            };
            if constexpr (L == 1) {
                if (a.k_pad <= 2048 || ((g - g0) & 1)) carry(lev[0], acc);
            } else {
                carry(lev[0], acc);
                if (((g - g0) & 7) == 7) carry(lev[1], lev[0]);
                if (((g - g0) & 63) == 63) carry(lev[2], lev[1]);
            }
        }
    }
    if constexpr (F32) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if constexpr (L == 1) acc[n][t] = lev[0][n][t] + acc[n][t];
                else acc[n][t] = lev[2][n][t] + lev[1][n][t] + lev[0][n][t];
            }
    }
}

// the column scales of output columns oc .. oc + 3 (of the weight, or of the gate and the up)
struct ColScales {
    float g[4], u[4];
};
template <bool GLU>
__device__ __forceinline__ ColScales col_scales(const SegDev& sd, int oc) {
    ColScales s;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = min(oc + j, sd.n_out - 1);
        const int cg = GLU && sd.glu == 1 ? c + 32 * (c >> 5) : c;
        s.g[j] = load_scale(sd.scale, sd.scale_f32, cg);
        s.u[j] = !GLU ? 1.f
                 : sd.glu == 1 ? load_scale(sd.scale, sd.scale_f32, cg + 32)
                               : load_scale(sd.scale_up, sd.scale_f32, c);
    }
    return s;
}

// 4 output columns oc .. oc + 3 (within the weight's) of row m, summed in g (and u): the scales, the GLU and the
// residual, to y
template <bool GLU, bool F32>
__device__ __forceinline__ void gemm_store(const GemmArgs& a, int m, int oc, f32x4 g, f32x4 u, const ColScales& s) {
    const int left = a.seg.n_out - oc;
    const size_t ycol = (size_t)a.seg.col0 + oc;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (GLU) {
            v[j] = act_glu(g[j] * s.g[j], a.act) * (u[j] * s.u[j]);
        } else if (a.res != nullptr) {
            const float rv = j < left ? bf16_to_f32(a.res[(size_t)m * a.ldr + ycol + j]) : 0.f;
            v[j] = a.res_mode == 2 ? (rv + g[j]) * s.g[j] : g[j] * s.g[j] + rv;
        } else {
            v[j] = g[j] * s.g[j];
        }
    }
    const size_t idx = (size_t)m * a.ldy + ycol;
    if constexpr (F32) {
        float* y = reinterpret_cast<float*>(a.y) + idx;
        if (a.vec4 && left >= 4) {
            *reinterpret_cast<f32x4*>(y) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j < left) y[j] = v[j];
        }
    } else {
        uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + idx;
        uint32_t b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = f32_to_bf16(v[j]);
        if (a.vec4 && left >= 4) {
            *reinterpret_cast<uint2*>(y) = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j < left) y[j] = (uint16_t)b[j];
        }
    }
}

__device__ __forceinline__ f32x4 add4(f32x4 a, f32x4 b) {
    return f32x4{a[0] + b[0], a[1] + b[1], a[2] + b[2], a[3] + b[3]};
}

// two fp32 values as bf16 bits, to nearest even
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
__device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

// gemm_store where nothing is left to ask a row: bf16 y, no residual, all four columns in one aligned store
template <bool GLU>
__device__ __forceinline__ void gemm_store_plain(const GemmArgs& a, uint16_t* y, f32x4 g, f32x4 u, const ColScales& s) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        v[j] = GLU ? act_glu(g[j] * s.g[j], a.act) * (u[j] * s.u[j]) : g[j] * s.g[j];
    uint2 o = make_uint2(cvt2(v[0], v[1]), cvt2(v[2], v[3]));
    const float t = v[0] + v[1] + v[2] + v[3];
    if (t != t)  // (a NaN is 0x7FC0 here as in every kernel)
        o = make_uint2(f32_to_bf16(v[0]) | (f32_to_bf16(v[1]) << 16), f32_to_bf16(v[2]) | (f32_to_bf16(v[3]) << 16));
    *reinterpret_cast<uint2*>(y) = o;
}

template <int MT, int FMT, bool GLU, bool KS, bool F32>
__global__ __launch_bounds__(64 * GEMM_W, 1) void dr_gemm(const GemmArgs a) {
    constexpr int BM = 32 * MT, OT = GLU ? 1 : 2;
    constexpr int XN = BM * 8 * (KS ? GEMM_W : 1);  // 16-byte chunks a stage of x
    __shared__ uint4 x0[XN], x1[XN], x2[XN], x3[XN];
    int nt, m0;
    gemm_tile(a, BM, nt, m0);
    f32x16 acc[2][MT];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[n][t][i] = 0.f;
    gemm_k_loop<MT, FMT, GLU, KS, F32>(a, nt, m0, acc, x0, x1, x2, x3);
    // The sums through LDS, an x stage for each wavefront, so that a store covers whole runs of a row: row r's 16-byte
    // chunk k (columns 4 k .. + 3 of the two tiles) at 16 r + (k ^ (r % 16)). (The K loop ends with loads to the stages
    // in flight, which must have landed, every wavefront's, before sums are written there.)
    step_barrier<0, true>();
    constexpr int TP = KS ? MT : MT / 2;  // row tiles a pass
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    auto region = [&](int w) { return reinterpret_cast<f32x4*>(w == 0 ? x0 : w == 1 ? x1 : w == 2 ? x2 : x3); };
    f32x4* part = region(wave);
    // (a lane's column chunk is the same in every turn of the store loop)
    const int k = lane % (8 * OT), oc = 32 * OT * (KS ? nt : nt * GEMM_W + wave) + 4 * k;
    const ColScales cs = col_scales<GLU>(a.seg, oc);
    constexpr int RS = 64 / (8 * OT) * (KS ? GEMM_W : 1);  // rows a turn
    const int r0 = (KS ? (int)threadIdx.x : lane) / (8 * OT);
    const bool plain = a.vec4 && !F32 && a.res == nullptr && a.seg.n_out - oc >= 4;
#pragma unroll
    for (int tb = 0; tb < MT; tb += TP) {
        if (tb) __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < TP; ++t)
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& v = acc[n][tb + t];
                    part[(32 * t + r) * 16 + ((8 * n + 2 * g + h) ^ (r & 15))] =
                        f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
                }
        if constexpr (KS) __syncthreads();
        else __builtin_amdgcn_wave_barrier();  // (the wavefront's own region: its LDS instructions run in order)
        if (oc >= a.seg.n_out) continue;
        const int rows = min(a.m - m0 - 32 * tb, 32 * TP);
        auto sums = [&](int row, f32x4& g, f32x4& u) {
            const int ig = row * 16 + (k ^ (row & 15)), iu = row * 16 + ((k + 8) ^ (row & 15));
            g = part[ig];
            u = GLU ? part[iu] : g;
            if constexpr (KS) {  // the wavefronts' shares of K, in order
                g = region(0)[ig];
                if (GLU) u = region(0)[iu];
#pragma unroll
                for (int w = 1; w < GEMM_W; ++w) {
                    g = add4(g, region(w)[ig]);
                    if (GLU) u = add4(u, region(w)[iu]);
                }
            }
        };
        if (plain) {
            uint16_t* y = reinterpret_cast<uint16_t*>(a.y) + (size_t)(m0 + 32 * tb + r0) * a.ldy + a.seg.col0 + oc;
#pragma unroll 4
            for (int row = r0; row < rows; row += RS, y += (size_t)RS * a.ldy) {
                f32x4 g, u;
                sums(row, g, u);
                gemm_store_plain<GLU>(a, y, g, u, cs);
            }
        } else {
            for (int row = r0; row < rows; row += RS) {
                f32x4 g, u;
                sums(row, g, u);
                gemm_store<GLU, F32>(a, m0 + 32 * tb + row, oc, g, u, cs);
            }
        }
    }
}

template <int MT, bool KS, bool F32>
void launch_gemm_t(const GemmArgs& g, hipStream_t st) {
    const dim3 grid(g.tm * g.tn), b(64 * GEMM_W);
    const bool glu = g.seg.glu != 0;
    constexpr bool BF16 = !F32 || MT == 2;  // (gemm_plan's tiles)
    switch (g.seg.fmt) {
        case DR_BFP8:
            if (glu) hipLaunchKernelGGL((dr_gemm<MT, DR_BFP8, true, KS, F32>), grid, b, 0, st, g);
            else hipLaunchKernelGGL((dr_gemm<MT, DR_BFP8, false, KS, F32>), grid, b, 0, st, g);
            break;
        case DR_BFP4:
            if (glu) hipLaunchKernelGGL((dr_gemm<MT, DR_BFP4, true, KS, F32>), grid, b, 0, st, g);
            else hipLaunchKernelGGL((dr_gemm<MT, DR_BFP4, false, KS, F32>), grid, b, 0, st, g);
            break;
        default:
            if constexpr (BF16) {
                if (glu) hipLaunchKernelGGL((dr_gemm<MT, DR_BF16, true, KS, F32>), grid, b, 0, st, g);
                else hipLaunchKernelGGL((dr_gemm<MT, DR_BF16, false, KS, F32>), grid, b, 0, st, g);
            }
            break;
    }
}

}  // namespace

hipError_t launch_gemm(const GemmArgs& g, int mt, bool ks, hipStream_t st) {
    if (g.y_f32 && mt == 4) launch_gemm_t<4, false, true>(g, st);
    else if (g.y_f32) ks ? launch_gemm_t<2, true, true>(g, st) : launch_gemm_t<2, false, true>(g, st);
    else if (ks) launch_gemm_t<2, true, false>(g, st);
    else if (mt == 8) launch_gemm_t<8, false, false>(g, st);
    else if (mt == 6) launch_gemm_t<6, false, false>(g, st);
    else if (mt == 4) launch_gemm_t<4, false, false>(g, st);
    else launch_gemm_t<2, false, false>(g, st);
    return hipGetLastError();
}

}  // namespace drk
