// qgemm_wide.hip — the GEMMs for many activation rows (prompt prefill, wide
// verifies): Q4_K and Q6_K on one kernel, Q8_0 on its own.
//
// The prefill pushes a chunk of the prompt through the trunk as one batch of
// rows (engine.rs:1922-1953, step_greedy -> run_general, qwen35.rs:1125-1302),
// so every ggml_mul_mat there has tens to hundreds of activation rows.  The
// numbers are exactly those of the skinny kernel (qgemm.hip): for activation
// row m, weight row n and 256-element unit u (Q4_K)
//     isum = sum_j sc_j * dot_j      imin = sum_j mn_j * (codes of sub-block j)
//     term = rint(dws * da * isum) - rint(dms * da * imin)        (binary64)
// and the terms of all units are summed exactly, so the outputs are
// bit-identical to the skinny path's whatever the split.
//
// Mapping.  A workgroup of 4 waves owns one 64-row weight tile and up to 128
// activation rows (Q8_0: 64), over all of K or one slice of it.  Wave w takes
// weight rows 16w..16w+15 against all of them, in 16 x 16 output blocks.  The
// activation codes of one unit are staged in LDS for the four waves,
// double-buffered, while the next unit's codes and weights are in flight.  In
// the MFMA's lane layout (A row and B column = lane % 16, C rows 4 (lane / 16)
// + i of column lane % 16) a lane of the K-quants' kernel holds one weight row,
// so its scales are decoded once per unit; one of Q8_0's (the weights as A)
// holds one activation row and four weight rows.
#include <math.h>

#include "cpv_internal.h"

namespace {

constexpr int WT = 256;                 // threads per workgroup (4 waves)
constexpr int MAX_NMT = 8;              // 16-row activation blocks per workgroup, K-quants
constexpr int MAX_NMT_Q80 = 4;          //   and Q8_0 (its scales' LDS at 4 lets three share a CU)
// workgroups per CU: three waves per SIMD hold 168 registers (K-quants: up to
// two blocks)
constexpr int wide_per_cu(bool q80, int nmt) { return !q80 && nmt > 2 ? 2 : 3; }

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short v2u __attribute__((ext_vector_type(2)));

struct WideArgs {
    const uint8_t* w;      // repacked tiles: [tile][unit][pieces: Q4_K 9, Q6_K 13, Q8_0 17][64 rows][16 B]
    const int32_t* ew;     // [n_pad] row exponents
    const int8_t* qa;      // [rows][U*256] activation codes
    const float* da;       // [rows][U] activation scales
    double* gsum;          // [rows][n_pad], zero on entry
    int64_t n_pad;
    int U, M, win;
    int tiles, mblocks, ksplit, upk;   // grid = tiles * mblocks * ksplit; upk units per K slice
    const int32_t* bs16;   // [rows][U*16] sums of 16 codes (Q8_K)
    float* y;              // outputs [rows][n], or null: the sums stay in gsum
    int64_t n;             // weight rows
    bool vec;              // y takes 16-byte stores (n a multiple of 4, y aligned)
    int nfull;             // (tile, row block) pairs that run over all of K
};

__device__ __forceinline__ int64_t pack2(uint32_t lo, uint32_t hi)
{
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ v4i mfma16(int64_t a, int64_t b, v4i c)
{
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
}

// 16 bytes per lane from g into LDS at dst + 16 lane (dst wave-uniform), past
// the registers.  Written out because the builtin makes the compiler wait for
// the transfer before the next LDS read of any address (it cannot tell the two
// buffers apart): the unit then stalled for its successor's loads (17408 x 5120
// at 256 rows: 95 us a call, 90 this way).  The caller waits
// (wide_dma_wait) before the barrier that publishes dst.  (The s_nop: a wait
// state between the write of m0 and its use.)
__device__ __forceinline__ void wide_dma16(const void* g, void* dst)
{
    const uint32_t l = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)dst;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 : : "v"(g), "s"(__builtin_amdgcn_readfirstlane(l)) : "m0", "memory");
}
__device__ __forceinline__ void wide_dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

struct WidePart { int pair, u0, u1; bool whole; };

// workgroup -> (tile, row block) pair and its units.  Pairs 0 .. nfull - 1 run
// whole; each later one in a.ksplit slices of a.upk units.  Consecutive
// workgroups go to different XCDs, so the order is laid out per XCD: the row
// blocks of one tile (which read the same weights) run side by side on one
// XCD's L2.
__device__ __forceinline__ WidePart wide_part(const WideArgs& a, int b)
{
    WidePart p;
    if (b < a.nfull) {
        p.pair = (a.nfull & 7) == 0 ? (b & 7) * (a.nfull >> 3) + (b >> 3) : b;
        p.u0 = 0;
        p.u1 = a.U;
        p.whole = true;
        return p;
    }
    const int rest = (int)gridDim.x - a.nfull, c = b - a.nfull;
    const int l = (rest & 7) == 0 ? (c & 7) * (rest >> 3) + (c >> 3) : c;
    // (slices of the row blocks of a tile side by side)
    const int np = rest / a.ksplit, ks = l / np;
    p.pair = a.nfull + (l - ks * np);
    p.u0 = ks * a.upk;
    p.u1 = min(a.U, p.u0 + a.upk);
    p.whole = a.ksplit == 1;
    return p;
}

// Ea(m) of the block's 16 NMT rows: the exponent of the row's largest |scale|
// (several lanes a row, so that a row's loads are in flight together)
template <int NMT>
__device__ __forceinline__ void wide_row_exponents(const WideArgs& a, int rbase, int nda, double* s_sm, int* s_ea)
{
    constexpr int R = 16 * NMT, TPR = NMT > 4 ? 2 : NMT > 2 ? 4 : NMT > 1 ? 8 : 16;
    const int r = threadIdx.x / TPR, sub = threadIdx.x % TPR;
    const float* d = a.da + (int64_t)min(rbase + (r < R ? r : R - 1), a.M - 1) * nda;
    float mx = 0.0f;
#pragma unroll 8
    for (int u = sub; u < nda; u += TPR) mx = fmaxf(mx, fabsf(d[u]));
    mx = cpv_group_reduce<TPR>(mx, cpv_op_max());
    if (sub == 0 && r < R) {
        const int e = cpv_exp_of_max(mx);
        s_ea[r] = e;
        s_sm[r] = e == CPV_E_EMPTY ? 0.0 : ldexp(1.0, a.win - e);
    }
}

// the block's sums: outputs directly when y is asked for and the workgroup
// covers all of K; else stored in the accumulator (whole) or added to it
template <int NMT>
__device__ __forceinline__ void wide_store(const WideArgs& a, const WidePart& wp, int tile, int rbase, int nrow, int g,
                                           int er, const int* s_ea, const double (&S)[NMT][4])
{
    const int64_t n = (int64_t)tile * 64 + nrow;
#pragma unroll
    for (int mt = 0; mt < NMT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = mt * 16 + 4 * g + i, m = rbase + r;
            if (m >= a.M) continue;
            if (a.y && wp.whole) {
                if (n < a.n) a.y[(int64_t)m * a.n + n] = cpv_gout_value(S[mt][i], er, s_ea[r], a.win);
            } else {
                double* p = a.gsum + (int64_t)m * a.n_pad + n;
                if (wp.whole) *p = S[mt][i];
                else unsafeAtomicAdd(p, S[mt][i]);
            }
        }
}

// the outputs of the sliced pairs (from a.nfull on): y from the accumulator,
// which is left zero.  One workgroup per pair and 16-row block.
__global__ __launch_bounds__(WT) void wide_finalize_kernel(WideArgs a, int nda, int rows)
{
    const int pair = a.nfull + blockIdx.x, tile = pair / a.mblocks, mb = pair - tile * a.mblocks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n = (int64_t)tile * 64 + lane;
    const int e = a.ew[n];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int m = mb * rows + blockIdx.y * 16 + wave + 4 * q;
        const int mc = min(m, a.M - 1);
        float mx = 0.0f;
        for (int u = lane; u < nda; u += 64) mx = fmaxf(mx, fabsf(a.da[(int64_t)mc * nda + u]));
        mx = cpv_wave_reduce(mx, cpv_op_max());
        if (m >= a.M) continue;
        double* p = a.gsum + (int64_t)m * a.n_pad + n;
        const double S = *p;
        *p = 0.0;
        if (n < a.n) a.y[(int64_t)m * a.n + n] = cpv_gout_value(S, e, cpv_exp_of_max(mx), a.win);
    }
}

// ---------------------------------------------------------------- Q4_K and Q6_K
// What bounds these kernels is VALU issue: per 16 x 16 outputs and unit the
// contract's binary64 terms cost 40 instructions (Q4_K; 20 for Q6_K) at about
// 2.1 ns each, and an int8 MFMA takes two of those issue slots and 7 ns of its
// pipe whether it is 32 or 64 deep.  So everything else is made rare:
//  * the sub-block scales enter through the B operands.  Q4_K: a code times
//    the low (high) 3 bits of its scale is at most 15 * 7 = 105, so isum =
//    8 * (codes * high . a) + (codes * low . a), two chains of four 16x16x64
//    MFMAs, where 32-deep MFMAs per sub-block need 8 and a multiply-add per
//    output and sub-block.  Q6_K: code * scale (13 bits signed) as two signed
//    bytes, isum = 256 * high + low.  The bytes are built once per unit and
//    wave (75 instructions, Q6_K about 210) and meet up to 8 row blocks.
//  * Q4_K's imin = sum over the unit's 16-code groups of mn_j * (group sum) is
//    one 16x16x16 f16 MFMA on the quantizer's group sums: mn <= 63 and |sum|
//    <= 2032 are f16 values, every partial sum an integer below 2^21.
//  * a lane loads whole 16-byte weight pieces: MFMA k of a unit takes its k
//    slots from the pieces g and g + 4 of lane group g = lane / 16 (the
//    reduction runs in any order; the activations are read in the same one).
//  * activation codes go from memory to LDS without passing registers.
//  * one block's binary64 terms run beside the next block's MFMAs.
//  * outputs leave the kernel directly where it covers all of K.
// 17408 x 5120 at 256 rows, whole call: Q4_K 141 -> 94 us, Q6_K 210 -> 85;
// at 64 rows 62 -> 45 and 77 -> 49.
template <int TYPE, int NMT>
struct KqLds {
    static constexpr int R = 16 * NMT;
    static constexpr bool MIN = TYPE == CPV_Q4_K;
    uint8_t codes[2][R][256];            // 16-byte piece p of row r at slot p ^ (r % 16)
    double dad[2][R];                    // da * 2^(win - Ea) per staged row
    double sm[R];                        // 2^(win - Ea(m)), 0 for an all-zero row
    _Float16 bs[MIN ? 2 : 1][MIN ? R : 1][16];   // the group sums (exact in f16)
};

template <int TYPE, int NMT>
__global__ __launch_bounds__(WT) __attribute__((amdgpu_waves_per_eu(wide_per_cu(false, NMT)))) void qgemm_wide_kq_kernel(WideArgs a)
{
    constexpr bool Q4 = TYPE == CPV_Q4_K;
    constexpr int R = 16 * NMT, PCS = Q4 ? 9 : 13;
    __shared__ __align__(16) KqLds<TYPE, NMT> s;
    __shared__ int s_ea[R];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int U = a.U, M = a.M;
    const int64_t Kp = (int64_t)U * 256;
    const WidePart wp = wide_part(a, blockIdx.x);
    const int tile = wp.pair / a.mblocks, rbase = (wp.pair - tile * a.mblocks) * R, u0 = wp.u0, u1 = wp.u1;

    wide_row_exponents<NMT>(a, rbase, U, s.sm, s_ea);

    // staging of one unit: the codes go from memory into LDS directly, 4 rows
    // per wave and load (LDS slot = lane, so the swizzle is in the source
    // address); the row scales and (Q4_K) the rows' 16 group sums, 8 per
    // thread, pass through registers.  Surplus threads repeat another's row
    // (the same values to the same place: no branch)
    int soff[NMT];
#pragma unroll
    for (int q = 0; q < NMT; q++) {
        const int r = (q * 4 + wave) * 4 + (lane >> 4);
        soff[q] = (min(rbase + r, M - 1) - rbase) * (int)Kp + ((lane & 15) ^ (r & 15)) * 16;
    }
    const int8_t* qbase = a.qa + (int64_t)rbase * Kp;
    const int drow = tid % R, brow = (tid >> 1) % R;
    const float* sda = a.da + (int64_t)min(rbase + drow, M - 1) * U;
    const int32_t* sbs = a.bs16 + (int64_t)min(rbase + brow, M - 1) * U * 16 + 8 * (tid & 1);
    struct Stage { v4i b[Q4 ? 2 : 1]; float d; };
    auto stage_load = [&](int u, int buf, Stage& t) {
#pragma unroll
        for (int q = 0; q < NMT; q++)
            wide_dma16(qbase + soff[q] + u * 256, &s.codes[buf][(q * 4 + wave) * 4][0]);
        if constexpr (Q4) {
            t.b[0] = *(const v4i*)(sbs + u * 16);
            t.b[1] = *(const v4i*)(sbs + u * 16 + 4);
        }
        t.d = sda[u];
    };
    auto stage_store = [&](int buf, const Stage& t) {
        if constexpr (Q4) {
            // (a sum's low 16 bits: a unit whose largest value is below 127 /
            // FLT_MAX has out-of-range codes, stored as 0 or 127 but summed as
            // 32-bit integers, which agree in those bits)
            v8h h;
#pragma unroll
            for (int i = 0; i < 8; i++) h[i] = (_Float16)(float)(short)t.b[i >> 2][i & 3];
            *(v8h*)&s.bs[buf][brow][8 * (tid & 1)] = h;
        }
        s.dad[buf][drow] = (double)t.d * s.sm[drow];
    };

    // this lane's weight row, its pieces g and g + 4 of the codes (and for
    // Q6_K the pieces of the high bits beside them) and the scale piece
    const int nl = lane & 15, g = lane >> 4;
    const int nrow = wave * 16 + nl;
    const uint8_t* wrow = a.w + (int64_t)tile * U * PCS * 1024 + nrow * 16;
    const uint16_t* wd = (const uint16_t*)(a.w + (int64_t)(a.n_pad / 64) * U * 13 * 1024) + (int64_t)tile * U * 64 + nrow;
    struct Wt { v4i q[2]; v4i h[Q4 ? 1 : 2]; v4i s; uint32_t d; };
    auto wload = [&](int u, Wt& t) {
        const uint8_t* p = wrow + (int64_t)u * PCS * 1024;
        t.q[0] = *(const v4i*)(p + g * 1024);
        t.q[1] = *(const v4i*)(p + (4 + g) * 1024);
        if constexpr (!Q4) {
            t.h[0] = *(const v4i*)(p + (8 + (g & 1)) * 1024);
            t.h[1] = *(const v4i*)(p + (10 + (g & 1)) * 1024);
            t.d = wd[(int64_t)u * 64];
        }
        t.s = *(const v4i*)(p + (PCS - 1) * 1024);
    };
    const int er = a.ew[(int64_t)tile * 64 + nrow];
    // the activations of MFMA k: piece 8 (k >> 1) + (Q4_K: 2, Q6_K: 4) (k & 1)
    // above the lane group's, at its swizzled slot
    int aoff[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        aoff[k] = nl * 256 + (((Q4 ? 4 * (g >> 1) + (g & 1) : g) + 8 * (k >> 1) + (Q4 ? 2 : 4) * (k & 1)) ^ nl) * 16;

    double S[NMT][4];
#pragma unroll
    for (int mt = 0; mt < NMT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) S[mt][i] = 0.0;

    Wt wc, wn;
    Stage st;
    wload(u0, wc);
    stage_load(u0, 0, st);
    __syncthreads();                     // s.sm
    stage_store(0, st);
    wide_dma_wait();
    __syncthreads();

    for (int u = u0; u < u1; u++) {
        const int buf = (u - u0) & 1;
        const int un = u + 1 < u1 ? u + 1 : u;   // (the last one reloads itself: no branch)
        wload(un, wn);
        stage_load(un, buf ^ 1, st);

        // B operands of the unit's four 64-deep steps: high and low limbs
        v4i bh[4], bl[4];
        v4h bm;
        double dws, dms = 0.0;
        if constexpr (Q4) {
            const uint32_t h0 = (uint32_t)wc.s[0], hy = (uint32_t)wc.s[1], hz = (uint32_t)wc.s[2], hw = (uint32_t)wc.s[3];
            dws = ldexp((double)cpv_h2f((uint16_t)(h0 & 0xffffu)), -er);
            dms = ldexp((double)cpv_h2f((uint16_t)(h0 >> 16)), -er);
            // scales and mins of sub-blocks 0-3 and 4-7; this lane's are 2 (g >> 1), + 1 of each four
            const uint32_t sc[2] = {hy & 0x3f3f3f3fu, (hw & 0x0f0f0f0fu) | ((hy >> 2) & 0x30303030u)};
            const uint32_t mlo = hz & 0x3f3f3f3fu, mhi = ((hw >> 4) & 0x0f0f0f0fu) | ((hz >> 2) & 0x30303030u);
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const uint32_t sl = sc[hf] & 0x07070707u, sh = (sc[hf] >> 3) & 0x07070707u;
#pragma unroll
                for (int nb = 0; nb < 2; nb++) {
                    // the sub-block's byte in both 16-bit halves
                    const uint32_t sel = (g >> 1) ? (nb ? 0x0c030c03u : 0x0c020c02u) : (nb ? 0x0c010c01u : 0x0c000c00u);
                    const v2u ml = __builtin_bit_cast(v2u, __builtin_amdgcn_perm(sl, sl, sel));
                    const v2u mh = __builtin_bit_cast(v2u, __builtin_amdgcn_perm(sh, sh, sel));
#pragma unroll
                    for (int x = 0; x < 4; x++) {
                        const uint32_t w = (uint32_t)wc.q[hf][x];
                        const v2u c = __builtin_bit_cast(v2u, (nb ? w >> 4 : w) & 0x0f0f0f0fu);
                        bl[2 * hf + nb][x] = __builtin_bit_cast(int, c * ml);   // (bytes <= 105: no carry)
                        bh[2 * hf + nb][x] = __builtin_bit_cast(int, c * mh);
                    }
                }
            }
            // mn of k slots 4 g .. 4 g + 3: the 16-code groups of sub-blocks 2 g and 2 g + 1
            // (0x6400 | b is 1024 + b in f16)
            const uint32_t mw = ((g >> 1) ? mhi : mlo) >> (16 * (g & 1));
            const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, mw, 0x04000400u);
            const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, mw, 0x04010401u);
            const v2h k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
            const v2h m0 = __builtin_bit_cast(v2h, p0) - k1024, m1 = __builtin_bit_cast(v2h, p1) - k1024;
            bm = v4h{m0[0], m0[1], m1[0], m1[1]};
        } else {
            dws = ldexp((double)cpv_h2f((uint16_t)wc.d), -er);
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
#pragma unroll
                for (int nb = 0; nb < 2; nb++) {
                    // the 16-code group's scale; product + 128 per code, so that its
                    // high byte is the high limb and its low byte the low limb + 128
                    const int sc = (int)(int8_t)((uint32_t)wc.s[2 * hf + nb] >> (8 * g));
                    const uint32_t su = (uint32_t)(sc & 0xffff), cu = (uint32_t)((128 - 32 * sc) & 0xffff);
                    const v2u s2 = __builtin_bit_cast(v2u, su * 0x10001u), c2 = __builtin_bit_cast(v2u, cu | (cu << 16));
                    const int qsh = 2 * (g >> 1) + 4 * nb;
#pragma unroll
                    for (int x = 0; x < 4; x++) {
                        const uint32_t w = (uint32_t)wc.q[hf][x];
                        const uint32_t q = ((nb ? w >> 4 : w) & 0x0f0f0f0fu) |
                                           ((((uint32_t)wc.h[hf][x] >> qsh) & 0x03030303u) << 4);
                        const v2u e = __builtin_bit_cast(v2u, q & 0x00ff00ffu), o = __builtin_bit_cast(v2u, (q >> 8) & 0x00ff00ffu);
                        const uint32_t pe = __builtin_bit_cast(uint32_t, e * s2 + c2), po = __builtin_bit_cast(uint32_t, o * s2 + c2);
                        bl[2 * hf + nb][x] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
                        bh[2 * hf + nb][x] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
                    }
                }
        }
        // block mt's binary64 terms run beside block mt + 1's MFMAs, whose A
        // operands were read one block earlier
        const uint8_t* cb = &s.codes[buf][0][0];
        v4i av[4];
        v4h ab;
        struct Acc { v4i hi, lo; v4f mn; };
        auto mma = [&](int mt, Acc& c, bool more) {
            c.hi = c.lo = v4i{0, 0, 0, 0};
            if constexpr (Q4) {
                c.mn = __builtin_amdgcn_mfma_f32_16x16x16f16(ab, bm, v4f{0, 0, 0, 0}, 0, 0, 0);
                if (more) ab = *(const v4h*)&s.bs[buf][(mt + 1) * 16 + nl][4 * g];
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                c.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[k], bh[k], c.hi, 0, 0, 0);
                c.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[k], bl[k], c.lo, 0, 0, 0);
                if (more) av[k] = *(const v4i*)(cb + aoff[k] + (mt + 1) * 4096);
            }
        };
        struct Da { double v[4]; };
        auto da_of = [&](int mt) {
            Da d;
#pragma unroll
            for (int i = 0; i < 4; i++) d.v[i] = s.dad[buf][mt * 16 + 4 * g + i];
            return d;
        };
        Acc c[2];
#pragma unroll
        for (int k = 0; k < 4; k++) av[k] = *(const v4i*)(cb + aoff[k]);
        if constexpr (Q4) ab = *(const v4h*)&s.bs[buf][nl][4 * g];
        mma(0, c[0], NMT > 1);
        Da dc = da_of(0), dn = dc;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < NMT; mt++) {
            if (mt + 1 < NMT) {
                mma(mt + 1, c[(mt + 1) & 1], mt + 2 < NMT);
                dn = da_of(mt + 1);
            }
            const Acc& x = c[mt & 1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double da = dc.v[i];
                if constexpr (Q4) S[mt][i] += rint(dws * da * (double)(x.hi[i] * 8 + x.lo[i])) - rint(dms * da * (double)x.mn[i]);
                else S[mt][i] += rint(dws * da * (double)(x.hi[i] * 256 + x.lo[i]));
            }
            if (mt + 1 < NMT) {
                if constexpr (Q4) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);       // the next block's group sums and row scales
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, Q4 ? 5 : 3, 0);   // VALU
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x002, Q4 ? 5 : 3, 0);
                }
            }
            dc = dn;
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_store(buf ^ 1, st);
        wide_dma_wait();
        __syncthreads();
        wc = wn;
    }
    wide_store<NMT>(a, wp, tile, rbase, nrow, g, er, s_ea, S);
}

// ---------------------------------------------------------------- Q8_0
// The same for Q8_0 weights and activations (ggml's Q8_0 vec_dot_type).  Per
// (activation row m, weight row n, 32-element block j) the dot is one
// 16x16x32 MFMA's entry, and the block's term is rounded on its own:
//     term = rint(dw_j * da_j * 2^-g * dot)          (binary64)
// eight terms per 256-element unit, so VALU issue bounds this kernel: four
// instructions a term.  The product is exact (11 + 11 + 20 bits), so one fma
// with +-1.5 * 2^52 rounds it to its integer as rint does (|term| < 2^51);
// the terms of blocks 2 p and 2 p + 1 carry opposite offsets, and their sum is
// the two integers' (exact, and infinities and NaN pass as they did).  A lane
// holds one activation row and 4 weight rows (the weights are the MFMA's A
// operand): a block's activation scale is then one 8-byte LDS read per 4
// terms, where 4 rows' scales were 4 reads and LDS the bound.  The two MFMAs
// of the next block pair and row block run beside a pair's terms.
// 7168 x 5120 at 201 rows, whole call: 121 -> 63 us; 17408 x 5120 at 256 rows: 226 -> 148.
// A unit's 17 pieces: 16 of codes (block j in pieces 2j, 2j + 1), then the 8
// block scales (f16).
template <int NMT>
__global__ __launch_bounds__(WT) __attribute__((amdgpu_waves_per_eu(3))) void qgemm_wide_q80_kernel(WideArgs a)
{
    constexpr int R = 16 * NMT, STEPS = 4 * NMT;
    struct Lds {
        uint8_t codes[2][R][256];        // 16-byte piece p of row r at slot p ^ (r % 16)
        double dad[2][8][R];             // da_j * 2^(win - Ea) per block and staged row
        double dw[2][8][64];             // dw_j * 2^-Ew per block and weight row
        double sm[R];                    // 2^(win - Ea(m)), 0 for an all-zero row
    };
    __shared__ __align__(16) Lds s;
    __shared__ int s_ea[R];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int U = a.U, M = a.M, NDA = 8 * a.U;
    const int64_t Kp = (int64_t)U * 256;
    const WidePart wp = wide_part(a, blockIdx.x);
    const int tile = wp.pair / a.mblocks, rbase = (wp.pair - tile * a.mblocks) * R, u0 = wp.u0, u1 = wp.u1;

    wide_row_exponents<NMT>(a, rbase, NDA, s.sm, s_ea);

    // staging of one unit: the codes from memory into LDS directly (as the
    // K-quants'); the scales of two blocks per thread, of the activations (8 R
    // / 2 threads, the others repeat them) and of the weights
    const int8_t* qbase = a.qa + (int64_t)rbase * Kp;
    int soff[NMT];
#pragma unroll
    for (int q = 0; q < NMT; q++) {
        const int r = (q * 4 + wave) * 4 + (lane >> 4);
        soff[q] = (min(rbase + r, M - 1) - rbase) * (int)Kp + ((lane & 15) ^ (r & 15)) * 16;
    }
    const int arow = (tid >> 2) % R, ablk = 2 * (tid & 3), wsrow = tid & 63, wsblk = 2 * (tid >> 6);
    const float* sda = a.da + (int64_t)min(rbase + arow, M - 1) * NDA + ablk;
    const uint8_t* wtile = a.w + (int64_t)tile * U * 17 * 1024;
    const int ews = a.ew[(int64_t)tile * 64 + wsrow];
    struct Stage { float2 d; uint32_t w; };
    auto stage_load = [&](int u, int buf, Stage& t) {
#pragma unroll
        for (int q = 0; q < NMT; q++)
            wide_dma16(qbase + soff[q] + u * 256, &s.codes[buf][(q * 4 + wave) * 4][0]);
        t.d = *(const float2*)(sda + 8 * u);
        t.w = *(const uint32_t*)(wtile + ((int64_t)u * 17 + 16) * 1024 + wsrow * 16 + wsblk * 2);
    };
    auto stage_store = [&](int buf, const Stage& t) {
        s.dad[buf][ablk][arow] = (double)t.d.x * s.sm[arow];
        s.dad[buf][ablk + 1][arow] = (double)t.d.y * s.sm[arow];
        s.dw[buf][wsblk][wsrow] = ldexp((double)cpv_h2f((uint16_t)(t.w & 0xffffu)), -ews);
        s.dw[buf][wsblk + 1][wsrow] = ldexp((double)cpv_h2f((uint16_t)(t.w >> 16)), -ews);
    };

    // this lane's weight row and k slot: 8 codes of block j (bytes 8 (g & 1)
    // .. of piece 2j + (g >> 1))
    const int nl = lane & 15, g = lane >> 4;
    const uint8_t* wrow = wtile + (wave * 16 + nl) * 16 + (g >> 1) * 1024 + 8 * (g & 1);
    struct Wt { v2i q[8]; };
    auto wload = [&](int u, Wt& t) {
#pragma unroll
        for (int j = 0; j < 8; j++) t.q[j] = *(const v2i*)(wrow + ((int64_t)u * 17 + 2 * j) * 1024);
    };
    // the lane's outputs: weight rows n0 .. n0 + 3
    const int64_t n0 = (int64_t)tile * 64 + wave * 16 + 4 * g;
    const double MAGIC = 0x1.8p52;

    double S[NMT][4];
#pragma unroll
    for (int mt = 0; mt < NMT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) S[mt][i] = 0.0;

    Wt wc, wn;
    Stage st;
    wload(u0, wc);
    stage_load(u0, 0, st);
    __syncthreads();                     // s.sm
    stage_store(0, st);
    wide_dma_wait();
    __syncthreads();

    for (int u = u0; u < u1; u++) {
        const int buf = (u - u0) & 1;
        const int un = u + 1 < u1 ? u + 1 : u;   // (the last one reloads itself: no branch)
        wload(un, wn);
        stage_load(un, buf ^ 1, st);
        const uint8_t* cb = &s.codes[buf][0][0] + nl * 256 + 8 * (g & 1);
        // step t: block pair p = t / NMT, row block t % NMT
        int64_t av[2];
        double da[2], dan[2], dw[2][4];
        auto fetch = [&](int t) {
            const int p = t / NMT, mt = t % NMT;
#pragma unroll
            for (int h = 0; h < 2; h++)
                av[h] = *(const int64_t*)(cb + mt * 4096 + ((2 * (2 * p + h) + (g >> 1)) ^ nl) * 16);
        };
        auto fetch_d = [&](int t) {
            const int p = t / NMT, mt = t % NMT;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                dan[h] = s.dad[buf][2 * p + h][mt * 16 + nl];
            }
        };
        auto fetch_w = [&](int p) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 4; i++) dw[h][i] = s.dw[buf][2 * p + h][wave * 16 + 4 * g + i];
        };
        struct Acc { v4i d[2]; };
        auto mma = [&](int t, Acc& c) {
            const int p = t / NMT;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int j = 2 * p + h;
                c.d[h] = mfma16(pack2((uint32_t)wc.q[j][0], (uint32_t)wc.q[j][1]), av[h], v4i{0, 0, 0, 0});
            }
        };
        Acc c[2];
        fetch(0);
        fetch_d(0);
        fetch_w(0);
        mma(0, c[0]);
        fetch(1 < STEPS ? 1 : 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < STEPS; t++) {
            const int mt = t % NMT;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                da[h] = dan[h];
            }
            if (t + 1 < STEPS) {
                mma(t + 1, c[(t + 1) & 1]);
                if (t + 2 < STEPS) fetch(t + 2);
                fetch_d(t + 1);
            }
            const Acc& x = c[t & 1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double ta = __builtin_fma(dw[0][i] * da[0], (double)x.d[0][i], MAGIC);
                const double tb = __builtin_fma(dw[1][i] * da[1], (double)x.d[1][i], -MAGIC);
                S[mt][i] += ta + tb;
            }
            if (mt == NMT - 1 && t + 1 < STEPS) fetch_w((t + 1) / NMT);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_store(buf ^ 1, st);
        wide_dma_wait();
        __syncthreads();
        wc = wn;
    }

    // the outputs directly, or the sums to the accumulator: from a transposed
    // copy in LDS, so that 16 lanes' adds are 16 weight rows of one activation
    // row (adds scattered over rows took twice the whole launch)
    if (a.y && wp.whole) {
        int er[4];
#pragma unroll
        for (int i = 0; i < 4; i++) er[i] = a.ew[n0 + i];
#pragma unroll
        for (int mt = 0; mt < NMT; mt++) {
            const int m = rbase + mt * 16 + nl;
            if (m >= M) continue;
            float* y = a.y + (int64_t)m * a.n + n0;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = cpv_gout_value(S[mt][i], er[i], s_ea[mt * 16 + nl], a.win);
            if (a.vec) {   // (n a multiple of 4, y 16-byte aligned: the four rows exist together)
                if (n0 < a.n) *(float4*)y = float4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (n0 + i < a.n) y[i] = v[i];
            }
        }
        return;
    }
    static_assert(sizeof(s.codes) >= 64 * R * sizeof(double), "the sums fit the staged codes' space");
    double* sS = (double*)&s.codes[0][0][0] + wave * 16 * R;   // (the loop's last barrier is past: the codes are read)
#pragma unroll
    for (int mt = 0; mt < NMT; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) sS[(mt * 16 + nl) * 16 + 4 * g + i] = S[mt][i];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4 * NMT; q++) {
        const int r = 4 * q + g, m = rbase + r;
        if (m >= M) continue;
        const double v = sS[r * 16 + nl];
        double* p = a.gsum + (int64_t)m * a.n_pad + (int64_t)tile * 64 + wave * 16 + nl;
        if (wp.whole) *p = v;
        else unsafeAtomicAdd(p, v);
    }
}

}  // namespace

bool cpv_qgemm_wide_ok(const cpv_weight* w, int64_t m)
{
    // (Q6_K and Q8_0 from 9 rows: one 16-row block streams the weights once
    // where Q6_K's skinny kernel takes them in 8-row passes and Q8_0's runs
    // one wave per SIMD; Q4_K from 17, past its own 16-row kernel: at 24
    // rows 34 against 46 us, at 16 the 16-row kernel's 27 against 28 us)
    return (w->type == CPV_Q4_K && m > 16) || ((w->type == CPV_Q6_K || w->type == CPV_Q8_0) && m > 8);
}

namespace {

// Rows per workgroup and the deal of the (tile, row block) pairs over the
// chip's slots (workgroups in flight).  Whole rounds of pairs run over all of
// K; the pairs that are left run in ks K slices of at least 4 units each.
// Chosen by an estimate in us, fitted to 5120, 7168, 12288, 17408 and 34816 x
// 5120 and 5120 x 17408 at 64 to 256 rows (at 9 to 48, those and five smaller
// weights, whole calls: Q8_0 0.60 to 0.92 of the fixed 64-row blocks' and their
// finalize launch's time, the K-quants' none above theirs): a unit of nmt row blocks takes 0.5 +
// 0.315 nmt with two workgroups on a CU (Q8_0: 0.95 nmt with three) and 0.62
// of that with one, a workgroup's start (row exponents, first loads) 3, and a
// million atomic adds of a slice's sums 3.5 (they bypass the XCD's L2).  E.g.
// Q4_K 17408 x 5120 at 128 rows: 8 blocks in 272 pairs 70 us a call, 4 in 544
// pairs 55; 5120 x 17408 at 256 rows: 8 blocks in 160 pairs x 3 slices 112, 4
// in 320 whole pairs 146; Q8_0 7168 x 5120 at 201 rows: 3 blocks in 560 pairs
// 75, 2 in 784 pairs 63.
// Returns false where no deal's workgroups fit a grid.
struct WidePlan { int nmt, mblocks, nfull, ksplit, upk; };

bool wide_plan(bool q80, int64_t tiles, int M, int U, int cus, WidePlan* p)
{
    // (the staging offsets within a row block are 32-bit: very long rows in smaller blocks)
    int maxb = q80 ? MAX_NMT_Q80 : MAX_NMT;
    while (16LL * maxb * U * 256 > INT32_MAX) maxb--;
    const int nb16 = (M + 15) / 16;
    double best = 1e30;
    for (int mb = (nb16 + maxb - 1) / maxb; mb <= nb16; mb++) {
        const int nmt = (nb16 + mb - 1) / mb;
        if ((nb16 + nmt - 1) / nmt != mb) continue;   // (the same blocks in fewer workgroups)
        const int slots = cus * wide_per_cu(q80, nmt);
        const int64_t pairs = tiles * mb, full = pairs / slots * slots, rest = pairs - full;
        if (full + 16LL * slots > (int64_t)(UINT32_MAX / WT)) break;
        const double t = q80 ? 0.95 * nmt : (0.5 + 0.315 * nmt) * wide_per_cu(q80, nmt) / 2, t1 = 0.62 * t, s0 = 3.0;
        const double tf = (double)(full / slots) * (U * t + s0);
        for (int ks = 1; ks == 1 || (rest && ks <= U / 4 && ks <= 16); ks++) {
            const int upk = (U + ks - 1) / ks, k2 = (U + upk - 1) / upk;
            if (k2 != ks) continue;
            const int64_t w = rest * ks, last = w % slots;
            double tr = (double)(w / slots) * (upk * t + s0);
            if (last) tr += upk * (last > cus ? t : t1) + s0;   // (past cus the fullest CU decides)
            if (ks > 1) tr += (double)w * nmt * 1024 * 3.5e-6 + 1.5;
            if (tf + tr < best) {
                best = tf + tr;
                *p = {nmt, mb, (int)(ks > 1 ? full : pairs), ks, upk};
            }
        }
        if (nmt <= 2) break;
    }
    return best < 1e30;
}

void q80_launch(const WideArgs& a, int nmt, unsigned grid, hipStream_t stream)
{
    switch (nmt) {
    case 1: qgemm_wide_q80_kernel<1><<<grid, WT, 0, stream>>>(a); break;
    case 2: qgemm_wide_q80_kernel<2><<<grid, WT, 0, stream>>>(a); break;
    case 3: qgemm_wide_q80_kernel<3><<<grid, WT, 0, stream>>>(a); break;
    default: qgemm_wide_q80_kernel<4><<<grid, WT, 0, stream>>>(a); break;
    }
}

template <int TYPE>
void kq_launch(const WideArgs& a, int nmt, unsigned grid, hipStream_t stream)
{
    switch (nmt) {
    case 1:   // (9 to 16 rows: Q6_K only)
        if constexpr (TYPE == CPV_Q6_K) qgemm_wide_kq_kernel<TYPE, 1><<<grid, WT, 0, stream>>>(a);
        break;
    case 2: qgemm_wide_kq_kernel<TYPE, 2><<<grid, WT, 0, stream>>>(a); break;
    case 3: qgemm_wide_kq_kernel<TYPE, 3><<<grid, WT, 0, stream>>>(a); break;
    case 4: qgemm_wide_kq_kernel<TYPE, 4><<<grid, WT, 0, stream>>>(a); break;
    case 5: qgemm_wide_kq_kernel<TYPE, 5><<<grid, WT, 0, stream>>>(a); break;
    case 6: qgemm_wide_kq_kernel<TYPE, 6><<<grid, WT, 0, stream>>>(a); break;
    case 7: qgemm_wide_kq_kernel<TYPE, 7><<<grid, WT, 0, stream>>>(a); break;
    default: qgemm_wide_kq_kernel<TYPE, 8><<<grid, WT, 0, stream>>>(a); break;
    }
}

}  // namespace

cpv_status cpv_qgemm_wide(cpv_ctx* ctx, const cpv_weight* w, const cpv_act* act, double* gsum, int win, float* y)
{
    const bool q80 = w->type == CPV_Q8_0, q6k = w->type == CPV_Q6_K;
    if ((w->type != CPV_Q4_K && !q80 && !q6k) || act->kq == q80 || act->U != (int)w->units ||
        !cpv_qgemm_wide_ok(w, act->m) || act->m > INT32_MAX / 2)
        return cpv_fail(ctx, CPV_EINVAL, "qgemm_wide: weight or activation format not supported");
    if (64LL * act->U * 256 > INT32_MAX)
        return cpv_fail(ctx, CPV_EUNSUPPORTED, "qgemm_wide: k=%lld too long", (long long)w->k);
    WideArgs a;
    a.w = (const uint8_t*)w->data;
    a.ew = w->ew;
    a.qa = act->qa;
    a.da = act->da;
    a.gsum = gsum;
    a.n_pad = w->n_pad;
    a.U = act->U;
    a.M = (int)act->m;
    a.win = win;
    a.tiles = (int)(w->n_pad / 64);
    a.bs16 = act->bs16;
    a.y = y;
    a.n = w->n;
    a.vec = (w->n & 3) == 0 && ((uintptr_t)y & 15) == 0;
    WidePlan p;
    if (!wide_plan(q80, a.tiles, a.M, a.U, ctx->cu_count, &p))
        return cpv_fail(ctx, CPV_EUNSUPPORTED, "qgemm_wide: %d tiles by %d rows", a.tiles, a.M);
    const int nmt = p.nmt;
    a.mblocks = p.mblocks;
    a.nfull = p.nfull;
    a.ksplit = p.ksplit;
    a.upk = p.upk;
    const int64_t blocks = (int64_t)a.tiles * a.mblocks;
    const int64_t rest = blocks - a.nfull, grid = a.nfull + rest * a.ksplit;
    const int ev = cpv_prof_mark(ctx);
    auto go = [=]() {
        if (q80) q80_launch(a, nmt, (unsigned)grid, ctx->stream);
        else if (q6k) kq_launch<CPV_Q6_K>(a, nmt, (unsigned)grid, ctx->stream);
        else kq_launch<CPV_Q4_K>(a, nmt, (unsigned)grid, ctx->stream);
        if (y && rest)
            wide_finalize_kernel<<<dim3((unsigned)rest, (unsigned)nmt), WT, 0, ctx->stream>>>(
                a, a.U * (q80 ? 8 : 1), nmt * 16);
    };
    go();
    CPV_HIP(ctx, hipGetLastError());
    if (ev >= 0) {  // algorithmic bytes: the weight, f32 activations in, f32 outputs
        const double wrow_b = q80 ? (double)(w->k / 32) * 34.0 : (double)(w->k / 256) * (q6k ? 210.0 : 144.0);
        const double bytes = (double)w->n * wrow_b + 4.0 * a.M * (double)w->k + 4.0 * a.M * (double)w->n;
        const int cls = q80 ? CPV_PROF_Q8_0_WIDE : q6k ? CPV_PROF_Q6_K_WIDE : CPV_PROF_Q4_K_WIDE;
        cpv_prof_add(ctx, ev, cls, bytes);
        cpv_prof_keep(ctx, cls, bytes, go);
    }
    return CPV_OK;
}

extern "C" int cpv_qgemm_wide_plan(int type, int64_t n, int64_t k, int64_t m, int cus, int out[5])
{
    WidePlan p{};
    const int64_t U = (k + 255) / 256;
    if (m < 1 || m > INT32_MAX / 2 || 64 * U * 256 > INT32_MAX ||
        !wide_plan(type == CPV_Q8_0, (n + 63) / 64, (int)m, (int)U, cus, &p))
        return 0;
    out[0] = p.nmt;
    out[1] = p.mblocks;
    out[2] = p.nfull;
    out[3] = p.ksplit;
    out[4] = p.upk;
    return 1;
}
