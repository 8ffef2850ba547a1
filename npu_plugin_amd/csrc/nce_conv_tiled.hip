// CONV task, LDS-tiled implicit GEMM on v_mfma_i32_16x16x64_i8 for tasks with many output pixels and channels.
//
// A workgroup owns BM = 16*TM*WM output pixels x BN = 16*TN*WN channels. Both operands of a reduction step (128 bytes of the
// OYXI weight rows; the same part of every pixel's window) are staged in LDS once per workgroup and shared by its waves: the
// WN waves along the channels read the same activation rows, the WM waves along the pixels the same weight rows. Per 64-byte
// half of a step a wave reads TN + TM operand fragments for TN*TM matrix instructions.
//
// Staging: global_load_lds_dwordx4 moves 16 bytes per lane from global memory straight into LDS (no registers, no LDS
// store). One instruction fills a 1 KiB block of 8 rows x 128 bytes: eight neighbouring lanes fetch one row's 128 bytes, a
// whole cache line. (With blocks of 16 rows x 64 bytes the two halves of a line are fetched a step apart, and by then a tile
// of 512 rows has pushed the line out of the 32 KiB L1: the same loop then moved twice the bytes from L2 and a 256 x 256
// tile took 0.69 us per 64 bytes of the reduction.) Which 16-byte piece of its row a lane FETCHES is the layout: piece
// j ^ swz8(row / 2) at position j, which spreads the operand reads over all banks (below). NS steps form a ring.
//
// The loop is software-pipelined through registers: while the matrix instructions of one half of a step run, the operands of
// the next half are read from LDS, dealt out between them, and a pixel fragment is re-biased (u8 storage: x ^ 0x80) one
// group ahead of its use, so that no matrix instruction waits for an LDS or vector one. One barrier per step: it says that
// every wave's requests of the next step have landed and that every wave holds this step in registers, so its ring slot is
// free and is requested again at once. Taps outside the image fetch a line holding the input zero point. With an input
// zero point away from the storage offset the per-channel weight sums come out of the matrix unit against ones; the WM waves
// that read the same weight fragments share that out.
//
// What bounds it: for 256 x 256 tiles the matrix cores at the clock their power leaves them (a loop of nothing but the operand
// reads, re-biasing and matrix instructions on random bytes holds 3.4 POP/s on the whole chip, 4.4 on a sixteenth of it);
// for the smaller tiles, which the smaller tasks need to fill 256 CUs, the barrier and LDS round trip of a step. Measured
// against a loop without the register pipeline that fetched 16 x 64 byte blocks: 3x3 over 256 channels, 32 x 56 x 56, input
// zero point 0: 85-89 -> 71 us (1.66 POP/s); 128 x 7 x 7 x 512: 25.9 -> 21.6 us; 5x5 over 112 channels (a gather kernel
// before): 70 -> 31 us.
//
// Conditions (checked on the host): kernel up to 15 x 15. Semantics and the fused PPE are those of the weights-resident kernel
// (nce_conv_epi.h).
#include "nce_conv_epi.h"
#include "nce_conv_lds.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace nce {

namespace {

using namespace wres_detail;

struct TiledArgs {
    ConvArgs a;
    int32_t nsteps;   // 128-byte reduction steps, rounded up
    int32_t nc128;    // TILED_CHUNKS: 128-byte chunks along IC
    uint32_t ntm;     // pixel tiles
    uint32_t ntn;     // channel tiles
    FastDiv div_ntn;
    WarmArgs warm;
    int32_t wraps;    // TILED_UNITS: taps eight consecutive units can reach into (1 .. 8)
    int64_t row_adv;  // input offset from the last tap of a kernel row to the first of the next: in_sh - KX * in_sw
    FuseAdd fz;       // FZ kernels only
};

using namespace lds_detail;  // vmcnt_imm, load_to_lds_16

// Blocks of 8 rows x 128 bytes, two per operand fragment of 16 rows: piece p (0..7) of row r (0..15) sits at
// r * 128 + ((p ^ swz8(r >> 1)) << 4). A ds_read_b128 of an operand is served in clocks of sixteen lanes that hold rows 0-3 and
// 12-15 with one piece and rows 4-11 with its neighbour (nce_conv_lds.h); rows of equal parity share the eight bank groups
// of half the banks, so for those eight rows the positions p ^ {0, 1, 6, 7} and p ^ 1 ^ {3, 2, 5, 4} have to be eight
// different ones - they are.
__device__ __forceinline__ int swz8(int k) {
    return (0x76452310 >> (4 * k)) & 7;
}

// GEN: TILED_CHUNKS - input channels a multiple of 128: a step lies in one tap, its position is scalar. TILED_UNITS - any
// multiple of 16: a step is eight 16-byte units (tap, 16 channels) of their own and each lane walks the unit of the piece it
// fetches; past the reduction's end the weights read zeros. TILED_UNITS_ASUM - units, and weights whose zero point differs
// from their storage offset by dw: the per-pixel activation sums come out of the matrix unit (one more instruction per pixel
// fragment and half step, against ones; past the end and outside the image a fetch is the zero point, a' = -da, which the
// constant nsteps * 128 * da * dw takes back).
enum { TILED_CHUNKS = 0, TILED_UNITS = 1, TILED_UNITS_ASUM = 2 };

// OCC: waves per SIMD the register budget has to allow.
template <int WM, int WN, int TM, int TN, int NS, int OCC, bool FZ, int GEN>
__global__ __launch_bounds__(64 * WM * WN, OCC) void conv_tiled_kernel(TiledArgs w) {
    prefetch_kernel_arguments<sizeof(TiledArgs)>();
    constexpr bool UNITS = GEN != TILED_CHUNKS;
    constexpr bool ASUM = GEN == TILED_UNITS_ASUM;
    constexpr int NW = WM * WN;
    constexpr int BM = 16 * TM * WM;
    constexpr int BN = 16 * TN * WN;
    constexpr int CW = 16 * TN;              // channels per wave
    constexpr int NA = BN / 8 / NW;          // blocks of the weight tile one wave fetches per step
    constexpr int NB = BM / 8 / NW;          // blocks of the activation tile
    constexpr int STAGE = (BM + BN) * 128;   // bytes of one ring slot: weight rows, then activation rows
    static_assert(TN == 2 || TN == 4, "channel fragments per wave");
    static_assert((BN / 8) % NW == 0 && (BM / 8) % NW == 0 && NW % 2 == 0, "blocks divide among the waves");
    static_assert(!FZ || TN == 4, "fused add: a lane holds 16 channels");
    static_assert(NS >= 2 && (NS - 1) * (NA + NB) < 64, "ring depth against the 6-bit load counter");
    const ConvArgs& a = w.a;

    WarmLines warm;
    warm.request(w.warm, (blockIdx.x >> 3) * NW + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));

    extern __shared__ __attribute__((aligned(16))) uint8_t sT[];  // [slot][weights BN rows | activations BM rows] x 128 bytes
    __shared__ int64_t sOutOff[BM];   // output byte offset of the tile's pixels (channel 0 of the tensor)
    __shared__ int32_t sW2[BN], sBias[BN], sWsum[BN];
    __shared__ int32_t sCorr[BN];     // integer path: da * sum of weights; high-word path: scaled multiplier
    __shared__ double sM[BN], sBfull[BN];
    __shared__ int32_t sFlags;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN;  // position along channels
    const int wm = wave / WN;  // position along pixels
    const int c16 = lane & 15;

    const uint32_t ntotal = w.ntm * w.ntn;
    const uint32_t lid = xcd_tile(blockIdx.x, ntotal);
    if (lid >= ntotal) return;  // uniform for the whole workgroup
    const uint32_t mt = fdiv(lid, w.div_ntn), nt = lid - mt * w.ntn;
    const int32_t oc0 = a.z0 + (int32_t)nt * BN;
    const int32_t noc = min(BN, a.z0 + a.bc - oc0);
    const int32_t m0 = (int32_t)mt * BM;

    // ---- what this thread fetches: row lane / 8 of the blocks wave, wave + NW, ... ; position lane % 8 -----------
    const int brow = (wave & 1) * 8 + (lane >> 3);  // row within its fragment of 16 (NW is even: the same for all its blocks)
    const int pj = (lane & 7) ^ swz8(brow >> 1);    // the piece that belongs at this lane's position
    uint32_t woff[NA];                              // byte offset from the first weight set of the tile
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int r = (wave + NW * i) * 8 + (lane >> 3);  // row of the weight tile: fragment r / 16, wave group r / CW
        const int cl = (r / CW) * CW + channel_of_frag_row<TN>((r % CW) >> 4, r & 15);
        const int ch = min(cl, noc - 1);  // rows past the box's last channel duplicate it (their results are not stored)
        woff[i] = (uint32_t)ch * (uint32_t)a.w_soc + (UNITS ? 0 : pj * 16);
    }
    const uint8_t* const wbase = a.w + (int64_t)oc0 * a.w_soc;
    const uint8_t* bsrc[NB];
    uint32_t taps[NB];  // bit ky: kernel row ky lies inside the image; bit 16 + kx: kernel column kx does
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int r = (wave + NW * i) * 8 + (lane >> 3);  // pixel of the tile
        const int32_t p = min(m0 + r, a.M - 1);           // pixels past the end duplicate the last one
        const int32_t rr = fdiv(p, a.div_bw);
        const int32_t bx = p - rr * a.bw;
        const int32_t n = fdiv(rr, a.div_bh);
        const int32_t by = rr - n * a.bh;
        const int32_t iy0 = (a.y0 + by) * a.SY - a.PT;
        const int32_t ix0 = (a.x0 + bx) * a.SX - a.PL;
        bsrc[i] = a.in + (int64_t)n * a.in_sn + (int64_t)iy0 * a.in_sh + (int64_t)ix0 * a.in_sw + (UNITS ? 0 : pj * 16);
        taps[i] = bit_range(max(0, -iy0), min(a.KY, a.H - iy0)) | bit_range(max(0, -ix0), min(a.KX, a.W - ix0)) << 16;
        if ((lane & 7) == 0) sOutOff[r] = (int64_t)n * a.out_sn + (int64_t)(a.y0 + by) * a.out_sh + (int64_t)(a.x0 + bx) * a.out_sw;
    }
    const uint8_t* const fillp = &g_fill.b[a.fill_raw][(pj & 3) * 16];
    if (tid < BN) sWsum[tid] = 0;
    if (tid == 0) sFlags = 0;

    // TILED_CHUNKS: scalar walk over (kernel row, kernel column, 128-byte channel chunk); additions only
    int32_t it_ky = 0, it_kx = 0, it_c = 0;
    int64_t it_off = 0, tap_off = 0;
    const uint8_t* it_w = wbase;
    // TILED_UNITS: this lane's walk over the 16-byte units pj, pj + 8, pj + 16 ... of the reduction
    const uint8_t* const wzero = &g_fill.b[a.w_xor & 0x80u][(pj & 3) * 16];  // (bytes that are zero once re-biased)
    int32_t u = pj, u_icg = pj, u_kx = 0, u_ky = 0;
    int64_t u_tap = 0;
    auto wrap_unit = [&]() {
        for (int i = 0; i < w.wraps; ++i) {  // (uniform)
            const bool over = u_icg >= a.ICG;
            const bool row = over && u_kx + 1 == a.KX;
            u_icg -= over ? a.ICG : 0;
            u_kx = row ? 0 : u_kx + (over ? 1 : 0);
            u_ky += row ? 1 : 0;
            u_tap += over ? a.in_sw : 0;
            u_tap += row ? w.row_adv : 0;
        }
    };
    if constexpr (UNITS) wrap_unit();
    // Request the next step's operands into ring slot `slot` (uniform) and move on.
    auto request = [&](int slot) {
        uint8_t* const st = sT + slot * STAGE + wave * 1024;
        if constexpr (UNITS) {
            const bool real = u < a.KG;
            const int64_t off = u_tap + 16 * u_icg;
#pragma unroll
            for (int i = 0; i < NA; ++i) load_to_lds_16(real ? wbase + woff[i] + 16 * u : wzero, st + NW * i * 1024);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const bool ok = real && ((taps[i] >> u_ky) & (taps[i] >> (16 + u_kx)) & 1u) != 0;
                load_to_lds_16(ok ? bsrc[i] + off : fillp, st + (BN / 8 + NW * i) * 1024);
            }
            u += 8;
            u_icg += 8;
            wrap_unit();
        } else {
#pragma unroll
            for (int i = 0; i < NA; ++i) load_to_lds_16(it_w, woff[i], st + NW * i * 1024);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const bool ok = ((taps[i] >> it_ky) & (taps[i] >> (16 + it_kx)) & 1u) != 0;
                load_to_lds_16(ok ? bsrc[i] + it_off : fillp, st + (BN / 8 + NW * i) * 1024);
            }
            it_w += 128;
            it_off += 128;
            if (++it_c == w.nc128) {
                it_c = 0;
                tap_off += a.in_sw;
                if (++it_kx == a.KX) {
                    it_kx = 0;
                    ++it_ky;
                    tap_off += w.row_adv;
                }
                it_off = tap_off;
            }
        }
    };

    const int S = w.nsteps;
#pragma unroll
    for (int j = 0; j < NS; ++j)
        if (j < S) request(j);
    // the table rows of the workgroup's channels travel while the first operands do
    int32_t tw2 = 0, tbias = 0;
    if (tid < noc) {
        const int32_t* trow = a.table + (int64_t)(oc0 + tid) * a.table_stride;
        tw2 = trow[2];
        tbias = trow[3];
    }

    // operand reads: lane (c16, q) reads row c16 of a fragment, piece q of half 0; half 1 is at the address with bit 6 flipped
    const int frag0 = c16 * 128 + (((lane >> 4) ^ swz8(c16 >> 1)) << 4);
    const int a_rd = (wn * TN) * 2048;
    const int b_rd = BN * 128 + (wm * TM) * 2048;

    v4i acc[TN][TM];
    constexpr int NWS = (TN + WM - 1) / WM;
    v4i wsa[NWS];  // sums of this wave's share of the weight fragments (input zero point away from the storage offset only)
    v4i asum[TM];  // ASUM: sums of the pixel fragments
#pragma unroll
    for (int f = 0; f < TN; ++f)
#pragma unroll
        for (int x = 0; x < TM; ++x) acc[f][x] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int x = 0; x < TM; ++x) asum[x] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NWS; ++i) wsa[i] = v4i{0, 0, 0, 0};
    const int axor = (int)a.a_xor, wxor = (int)a.w_xor;
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};

    // The reduction loop, compiled twice: with and without the weight sums.
    auto reduce = [&](auto with_sums) {
        constexpr bool WS = decltype(with_sums)::value;
        constexpr int R = TN + TM, G = TM > 1 ? TM - 1 : 1;  // operand reads of a half step, groups that carry them
        v4i fa[2][TN], fb[2][TM];
        auto read = [&](const uint8_t* st, int i, auto par) {  // par: half of the step, and register set
            constexpr int P = decltype(par)::value;
            const uint8_t* const at = st + (frag0 ^ (64 * P));
            if (i < TN) fa[P][i] = *reinterpret_cast<const v4i*>(at + a_rd + i * 2048);
            else fb[P][i - TN] = *reinterpret_cast<const v4i*>(at + b_rd + (i - TN) * 2048);
        };
        auto prepare_next = [&](auto par) {
            constexpr int P = decltype(par)::value;
            if (wxor != 0) {  // uniform
#pragma unroll
                for (int f = 0; f < TN; ++f) fa[P][f] ^= wxor;
            }
            fb[P][0] ^= axor;
        };
        // One half step from the registers of set P, while the operands of the next half are read from ring slot `next` into the
        // other set; req() issues requests.
        auto half = [&](const uint8_t* next, auto par, auto&& req) {
            constexpr int P = decltype(par)::value;
            const auto other = std::integral_constant<int, P ^ 1>{};
#pragma unroll
            for (int x = 0; x < TM; ++x) {
#pragma unroll
                for (int f = 0; f < TN; ++f) acc[f][x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[P][f], fb[P][x], acc[f][x], 0, 0, 0);
                if constexpr (WS) {
                    if (x == 0) {
#pragma unroll
                        for (int f = 0; f < TN; ++f)
                            if (f % WM == wm) wsa[f / WM] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[P][f], ones, wsa[f / WM], 0, 0, 0);
                    }
                }
                if constexpr (ASUM) asum[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, fb[P][x], asum[x], 0, 0, 0);
                if (x + 1 < TM) fb[P][x + 1] ^= axor;
#pragma unroll
                for (int i = 0; i < R; ++i)
                    if (i * G / R == x) read(next, i, other);
                if (x + 1 == TM) prepare_next(other);
#pragma unroll
                for (int g = 0; g < TN; ++g) {  // one matrix instruction, one vector instruction, and an LDS read behind the first two
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 1, 0);
                    if (g < 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (x == 0) {
                    req();
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        const auto P0 = std::integral_constant<int, 0>{};
        const auto P1 = std::integral_constant<int, 1>{};
        if (S >= NS) __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * (NA + NB)));
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        warm.release();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < R; ++i) read(sT, i, P0);
        prepare_next(P0);
        for (int s = 0; s < S; ++s) {
            const int slot = (int)((uint32_t)s % NS), next = (int)((uint32_t)(s + 1) % NS);
            half(sT + slot * STAGE, P0, [] {});
            // Step s + 1 has to be in LDS before it is read: the requests up to step s + NS - 1 are out, those younger than step
            // s + 1 may stay in flight. Every wave holds step s in registers before its slot is requested again.
            if (s + NS <= S) __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 2) * (NA + NB)));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            // (the bare barrier: __syncthreads() would first wait for all outstanding loads)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            // (the last step reads a slot that holds nothing of use)
            half(sT + next * STAGE, P1, [&] { if (s + NS < S) request(slot); });
        }
    };
    if (a.da != 0) reduce(std::true_type{});
    else reduce(std::false_type{});
    __syncthreads();

    // ---- per-channel constants (thread = channel), as in the weights-resident kernel -----------------------
    if (a.da != 0 && c16 == 0) {
        // every column of a sum fragment holds the same sums: lane (0, q) publishes rows 4q .. 4q + 3
#pragma unroll
        for (int i = 0; i < NWS; ++i) {
            const int f = WM * i + wm;
            if (f < TN) {
#pragma unroll
                for (int r = 0; r < 4; ++r) sWsum[wn * CW + channel_of_frag_row<TN>(f, 4 * (lane >> 4) + r)] = wsa[i][r];
            }
        }
    }
    const int64_t acc_bound = min((int64_t)a.ktot * 65025, (int64_t)2147483648LL);
    if (tid < BN) {
        const int32_t mult = table_mult(tw2), shift = table_shift(tw2);
        const bool bad = shift > kMaxF64Shift;
        const bool sat = ppe_may_saturate(acc_bound, tbias, mult, shift);
        bool hi_bad = false;
        if (tid < noc) {
            hi_bad = shift < 1 || shift > 32 || ((int64_t)mult << (32 - min(shift, 32))) > 0x7fffffffLL;
            const double cb = ((__builtin_fabs((double)tbias) + 4294967296.0) * (double)mult + 2147483648.0 + 384.0 * __builtin_ldexp(1.0, shift));
            hi_bad = hi_bad || __builtin_ldexp(cb, 32 - shift) >= 4611686018427387904.0;
        }
        const int wf = (bad ? 1 : 0) | (sat ? 2 : 0) | (hi_bad ? 4 : 0);
        if (wf) atomicOr(&sFlags, wf);
        sW2[tid] = tw2;
        sBias[tid] = tbias;
    }
    __syncthreads();
    const int flags = sFlags;
    const PpeF64 pu = ppe_f64_setup(a.ppe, (flags & 2) != 0);
    int pmode = ppe_mode_of(pu, (flags & 1) != 0);
    if (pmode == PPE_MODE_FOLDED && !(flags & 4)) pmode = PPE_MODE_HI;
    EpiPack ep = epi_pack_setup(pu);
    if (pmode == PPE_MODE_SLOPE && !(flags & 4)) {
        // slope = pm * 2^-ps with |slope| <= 1 in this mode; the high-word form needs slope * 2^32 in int32
        const int32_t pm = a.ppe.prelu_mult, ps = a.ppe.prelu_shift;
        if (ps <= 32 && (ps >= 1 || pm == 0)) {
            const int64_t q = (int64_t)pm * ((int64_t)1 << (32 - ps));
            if (q >= -0x7fffffffLL && q <= 0x7fffffffLL) {
                const int64_t zpf = pu.zp + (ep.flip ? 128 : 0);
                const int64_t half = ps >= 1 ? (int64_t)1 << (ps - 1) : 0;
                pmode = PPE_MODE_HI_SLOPE;
                ep.pmq = __builtin_amdgcn_readfirstlane((int32_t)q);
                ep.cpz = (half + zpf * ((int64_t)1 << ps) - zpf * pm) * ((int64_t)1 << (32 - ps));
            }
        }
    }
    if (tid < BN) {
        const int32_t mult = table_mult(tw2), shift = table_shift(tw2);
        // |da| <= 255, |sum w'| < 2^23; with a weight zero-point offset the constant term of the whole (padded) reduction joins
        const int32_t corr = a.da * sWsum[tid] + (ASUM ? w.nsteps * 128 * a.da * a.dw : 0);
        const double M = ppe_scale_M(mult, shift);
        double B = __builtin_fma((double)corr, M, ppe_scale_B(tbias, M, shift, a.ppe.round_mode));
        if (pmode != PPE_MODE_INT) B += ep.zp_fold;  // floor(x + zp) = floor(x) + zp
        sM[tid] = M;
        sBfull[tid] = B;
        sCorr[tid] = corr;
        if (pmode == PPE_MODE_HI || pmode == PPE_MODE_HI_SLOPE) {
            int32_t mq = 0;
            int64_t cq = 0;
            if (tid < noc) {
                const int64_t base = ((int64_t)tbias + corr) * mult + ((int64_t)1 << (shift - 1)) + ((int64_t)(pu.zp + (ep.flip ? 128 : 0)) << shift);
                mq = (int32_t)((uint32_t)mult << (32 - shift));
                cq = (int64_t)((uint64_t)base << (32 - shift));
            }
            sCorr[tid] = mq;
            reinterpret_cast<int64_t*>(sBfull)[tid] = cq;
        }
    }
    __syncthreads();

    // ---- PPE + store: this wave's CW channels of its 16 * TM pixels ---------------------------------------
    uint8_t* dst[TM];
    bool valid[TM];
    int32_t dws[TM];
#pragma unroll
    for (int x = 0; x < TM; ++x) {
        const int r = (wm * TM + x) * 16 + c16;
        valid[x] = m0 + r < a.M;
        dst[x] = a.out + sOutOff[r] + (int64_t)(oc0 + wn * CW) * a.out_sc;
        dws[x] = ASUM ? a.dw * asum[x][0] : 0;  // (every row of a sum fragment is the pixel's sum)
    }
    const int q = lane >> 4;
    const int nocw = noc - wn * CW;
    const EpiSmem ew = {sM + wn * CW, nullptr, sW2 + wn * CW, sBias + wn * CW, nullptr, nullptr};
    const double* const bw = sBfull + wn * CW;
    const int32_t* const cw = sCorr + wn * CW;
    // (at most EX pixel fragments at a time: over more of them the epilogue's state does not fit beside the accumulators)
    constexpr int EX = TM > 4 ? 2 : TM;
    static_assert(TM == EX || TM == 4 * EX, "epilogue rounds");
    const auto epilogue = [&](auto first) {
        constexpr int x0 = decltype(first)::value;
        v4i ax[TN][EX];
        uint8_t* dx[EX];
        bool vx[EX];
        int32_t wx[EX];
        uint4 other[FZ ? EX : 1];
#pragma unroll
        for (int x = 0; x < EX; ++x) {
#pragma unroll
            for (int f = 0; f < TN; ++f) ax[f][x] = acc[f][x0 + x];
            dx[x] = dst[x0 + x];
            vx[x] = valid[x0 + x];
            wx[x] = dws[x0 + x];
        }
        if constexpr (FZ) {
            if (nocw > 0) {  // uniform per wave; lanes past the last channel read a duplicate inside the tensor
                const int ch0 = min(16 * q, nocw - 16);
#pragma unroll
                for (int x = 0; x < EX; ++x) other[x] = *reinterpret_cast<const uint4*>(w.fz.other + ((dx[x] + ch0) - a.out));
            }
        }
        if (pmode == PPE_MODE_HI) wres_epilogue<TN, EX, PPE_MODE_HI, FZ>(a, ew, bw, cw, ax, wx, q, nocw, dx, vx, pu, ep, &w.fz, other);
        else if (pmode == PPE_MODE_HI_SLOPE) wres_epilogue<TN, EX, PPE_MODE_HI_SLOPE, FZ>(a, ew, bw, cw, ax, wx, q, nocw, dx, vx, pu, ep, &w.fz, other);
        else if (pmode == PPE_MODE_FOLDED) wres_epilogue<TN, EX, PPE_MODE_FOLDED, FZ>(a, ew, bw, cw, ax, wx, q, nocw, dx, vx, pu, ep, &w.fz, other);
        else if (pmode == PPE_MODE_SLOPE) wres_epilogue<TN, EX, PPE_MODE_SLOPE, FZ>(a, ew, bw, cw, ax, wx, q, nocw, dx, vx, pu, ep, &w.fz, other);
        else wres_epilogue<TN, EX, PPE_MODE_INT, FZ>(a, ew, bw, cw, ax, wx, q, nocw, dx, vx, pu, ep, &w.fz, other);
    };
    epilogue(std::integral_constant<int, 0>{});
    if constexpr (TM > EX) {
        epilogue(std::integral_constant<int, EX>{});
        epilogue(std::integral_constant<int, 2 * EX>{});
        epilogue(std::integral_constant<int, 3 * EX>{});
    }
}

template <int WM, int WN, int TM, int TN, int NS, int OCC>
hipError_t launch_shape(TiledArgs& w, bool fused, hipStream_t stream) {
    constexpr int BM = 16 * TM * WM;
    constexpr int BN = 16 * TN * WN;
    constexpr size_t lds = (size_t)NS * (BM + BN) * 128;
    const ConvArgs& a = w.a;
    w.ntm = (uint32_t)(((int64_t)a.M + BM - 1) / BM);
    w.ntn = (uint32_t)((a.bc + BN - 1) / BN);
    w.div_ntn = make_fastdiv(w.ntn);
    w.warm = make_warm(a.w + (int64_t)a.z0 * a.w_soc, (int64_t)a.bc * a.w_soc, std::min<int64_t>(xcd_grid(w.ntm * w.ntn) / kNumXcd, 32 * 4 * OCC / (WM * WN)) * (WM * WN));
    if ((uint64_t)w.ntm * w.ntn > 0x7ffffff0ull) return hipErrorNotSupported;
    const auto go = [&](auto kernel, LdsGrant& grant) {
        if (const hipError_t e = grant.ensure(reinterpret_cast<const void*>(kernel), lds, 48 * 1024); e != hipSuccess) return e;
        return emit(kernel, dim3(xcd_grid(w.ntm * w.ntn)), dim3(64 * WM * WN), lds, stream, w);
    };
    static LdsGrant grants[4];
    if (a.dw != 0) return fused ? hipErrorNotSupported : go(&conv_tiled_kernel<WM, WN, TM, TN, NS, OCC, false, TILED_UNITS_ASUM>, grants[0]);
    if (a.IC % 128 != 0) return fused ? hipErrorNotSupported : go(&conv_tiled_kernel<WM, WN, TM, TN, NS, OCC, false, TILED_UNITS>, grants[1]);
    if (!fused) return go(&conv_tiled_kernel<WM, WN, TM, TN, NS, OCC, false, TILED_CHUNKS>, grants[2]);
    if constexpr (TN == 4) return go(&conv_tiled_kernel<WM, WN, TM, TN, NS, OCC, true, TILED_CHUNKS>, grants[3]);
    return hipErrorNotSupported;
}

}  // namespace

// Shapes (pixels x channels): 1 = 256 x 256, 2 = 256 x 128, 3 = 128 x 128 (eight waves each), 4 = 128 x 64, 5 = 64 x 128,
// 6 = 64 x 64, 7 = 256 x 64 (four waves).
hipError_t launch_conv_tiled(const ConvArgs& a, hipStream_t stream, int shape, const FuseAdd* fuse) {
    if (a.KY > 15 || a.KX > 15) return hipErrorNotSupported;
    if (a.M > 0x7fffffff - 1024) return hipErrorNotSupported;
    if (fuse != nullptr && a.out_sc != 1) return hipErrorNotSupported;
    if (a.w_soc > 0x7fffffffLL / 256) return hipErrorNotSupported;  // (32-bit offsets within a tile's weights)
    // (weight zero-point offset: the activation sums times dw and the constant stay inside int32)
    if (a.dw != 0 && ((int64_t)a.ktot + 128) * 255 * 255 > 0x7fffffffLL) return hipErrorNotSupported;
    TiledArgs w;
    memset(&w, 0, sizeof(w));
    w.a = a;
    w.a.fill_raw = (a.fill ^ a.a_xor) & 0xFFu;
    if (fuse) w.fz = *fuse;
    w.nc128 = a.IC / 128;
    w.wraps = (a.ICG + 7) / a.ICG;
    w.nsteps = (a.KG + 7) / 8;
    w.row_adv = a.in_sh - (int64_t)a.KX * a.in_sw;
    const bool fz = fuse != nullptr;
    switch (shape) {
    case 1: return launch_shape<2, 4, 8, 4, 2, 2>(w, fz, stream);
    case 2: return launch_shape<4, 2, 4, 4, 2, 2>(w, fz, stream);
    case 3: return launch_shape<4, 2, 2, 4, 2, 4>(w, fz, stream);
    case 4: return launch_shape<4, 1, 2, 4, 2, 3>(w, fz, stream);
    case 5: return launch_shape<2, 2, 2, 4, 2, 3>(w, fz, stream);
    case 6: return launch_shape<4, 1, 1, 4, 2, 4>(w, fz, stream);
    case 7: return launch_shape<4, 1, 4, 4, 2, 2>(w, fz, stream);
    default: return hipErrorNotSupported;
    }
}

}  // namespace nce
