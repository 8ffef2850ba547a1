// CONV task, split-reduction implicit GEMM on v_mfma_i32_16x16x64_i8 for tasks with few output tiles.
//
// A convolution over one or a few images has too few tiles for 256 CUs, and the kernels that give a tile's whole reduction
// to one wave (weights-resident) or walk it step by step behind a barrier (LDS-tiled) then spend their time on one CU
// streaming a slice of weights: 3x3 over 256 channels on one 14 x 14 image took 9 us with 16 of 256 CUs at work. Here a
// workgroup owns ONE small tile - 16*BF pixels x 16*NF channels - and its W waves share out the REDUCTION: wave k takes the
// 64-byte slices k, k + W, k + 2W ... of it. The waves do not synchronise while they multiply: each streams both operands of
// its slices with global_load_lds_dwordx4 into an LDS ring of its own (D slices deep; short reductions are in flight all at
// once, so a wave sees about one round trip to memory) and waits for its own requests only. At the end the partial
// accumulators meet in LDS, and one wave per fragment adds them up, runs the PPE on four channels of one pixel per lane and
// stores a dword. What bounds it: launch, arguments, one or two memory round trips and the exchange - 3.5-5 us where the
// kernels above took 5-13; for long reductions the L2-to-LDS stream (about 30 bytes per clock and CU, (NF + BF) KiB per NF*BF
// matrix instructions).
//
// A slice is four 16-byte units (tap, 16 input channels), and every lane works out the unit it fetches (two multiply-high
// divisions), so any input channel count the validator accepts is served; units past the reduction's end read zero weights.
// SUMS: the zero-point terms. The per-channel weight sums and per-pixel activation sums come out of the matrix unit against
// ones and travel through the same exchange; the correction da * sum w' + dw * sum a' + K * da * dw is added to the
// accumulator modulo 2^32, which is the accumulator's own arithmetic, so no reduction is too long for it.
// Semantics are those of nce_conv.hip.
#include "nce_conv_epi.h"
#include "nce_conv_lds.h"

#include <algorithm>
#include <cstring>

namespace nce {
namespace {

using namespace wres_detail;
using namespace lds_detail;

struct SplitConvArgs {
    ConvArgs a;
    int32_t nslices;        // 64-byte slices of the reduction
    int32_t per_wave;       // slices of a wave, rounded up
    uint32_t ntm, ntn;      // pixel tiles, channel tiles
    int32_t channel_major;  // tile order: 1 = an XCD walks all pixels of a channel slice (weights outweigh activations)
    FastDiv div_icg, div_kx, div_ntm, div_ntn;
    int32_t in_sn32, in_sh32, in_sw32;
    FuseAdd fz;             // FZ kernels only
};

constexpr int kSplitWaves = 8;

template <int NF, int BF, int D, bool SUMS, bool FZ>
__global__ __launch_bounds__(64 * kSplitWaves) void conv_split_kernel(SplitConvArgs w) {
    prefetch_kernel_arguments<sizeof(SplitConvArgs)>();
    constexpr int F = NF + BF;             // blocks of 1 KiB per slice: weights, then pixels
    constexpr int OCT = 16 * NF, BP = 16 * BF;
    constexpr int SLOTS = NF * BF + (SUMS ? F : 0);  // fragments a wave hands to the exchange
    const ConvArgs& a = w.a;
    extern __shared__ __attribute__((aligned(16))) uint8_t sR[];  // [wave][D][F] x 1 KiB, then [wave][SLOTS] x 1 KiB

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nwaves = (int)blockDim.x >> 6;
    const int c16 = lane & 15, q = lane >> 4;

    const uint32_t total = w.ntm * w.ntn;
    const uint32_t lid = xcd_tile(blockIdx.x, total);
    if (lid >= total) return;  // uniform for the whole workgroup
    uint32_t mt, nt;
    if (w.channel_major) {
        nt = fdiv(lid, w.div_ntm);
        mt = lid - nt * w.ntm;
    } else {
        mt = fdiv(lid, w.div_ntn);
        nt = lid - mt * w.ntn;
    }
    const int32_t oc0 = a.z0 + (int32_t)nt * OCT;
    const int32_t noc = min(OCT, a.z0 + a.bc - oc0);
    const int32_t m0 = (int32_t)mt * BP;

    // ---- what this lane fetches: row lane / 4 of every block, the piece that belongs at position lane % 4 (nce_conv_lds.h)
    const int prow = lane >> 2;
    const int pj = (lane & 3) ^ swz(prow);
    const uint8_t* wsrc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f)  // rows past the box's last channel duplicate it (their results are not stored)
        wsrc[f] = a.w + (int64_t)(oc0 + min(channel_of_frag_row<NF>(f, prow), noc - 1)) * a.w_soc;
    const uint8_t* bsrc[BF];
    uint32_t rows[BF], cols[BF];
#pragma unroll
    for (int x = 0; x < BF; ++x) {
        const int32_t p = min(m0 + 16 * x + prow, a.M - 1);  // pixels past the end duplicate the last one
        const int32_t rr = fdiv(p, a.div_bw);
        const int32_t bx = p - rr * a.bw;
        const int32_t n = fdiv(rr, a.div_bh);
        const int32_t by = rr - n * a.bh;
        const int32_t iy0 = (a.y0 + by) * a.SY - a.PT;
        const int32_t ix0 = (a.x0 + bx) * a.SX - a.PL;
        bsrc[x] = a.in + (int64_t)n * w.in_sn32 + (int64_t)iy0 * w.in_sh32 + (int64_t)ix0 * w.in_sw32;
        rows[x] = bit_range(max(0, -iy0), min(a.KY, a.H - iy0));
        cols[x] = bit_range(max(0, -ix0), min(a.KX, a.W - ix0));
    }
    const uint8_t* const fillp = &g_fill.b[a.fill_raw][pj * 16];
    const uint8_t* const wzero = &g_fill.b[a.w_xor & 0x80u][pj * 16];  // (bytes that are zero once re-biased)

    uint8_t* const ring = sR + wave * (D * F * 1024);
    // Request slice st into ring slot `slot` (both uniform; slices past the end are all zeros and fill).
    auto request = [&](int st, int slot) {
        const int u = 4 * st + pj;
        const bool real = u < a.KG;
        const int tap = (int)fdiv((uint32_t)u, w.div_icg);
        const int icg = u - tap * a.ICG;
        const int ky = (int)fdiv((uint32_t)tap, w.div_kx);
        const int kx = tap - ky * a.KX;
        const int64_t off = (int64_t)ky * w.in_sh32 + (int64_t)kx * w.in_sw32 + 16 * icg;
        uint8_t* const dst = ring + slot * (F * 1024);
#pragma unroll
        for (int f = 0; f < NF; ++f) load_to_lds_16(real ? wsrc[f] + (int64_t)u * 16 : wzero, dst + f * 1024);
#pragma unroll
        for (int x = 0; x < BF; ++x) {
            const bool ok = real && ((rows[x] >> ky) & (cols[x] >> kx) & 1u) != 0;
            load_to_lds_16(ok ? bsrc[x] + off : fillp, dst + (NF + x) * 1024);
        }
    };
    const int n = w.per_wave;
#pragma unroll
    for (int j = 0; j < D; ++j)
        if (j < n) request(wave + j * nwaves, j);

    // ---- the output this thread finishes: fragment slots wave, wave + nwaves, ... of the tile; four channels of one pixel.
    // Table rows, addresses and the other operand of a fused add travel while the operands do. (vmcnt counts in order:
    // these loads are younger than the first D slices, and the waits below cover them where they have to.)
    auto epilogue_of = [&](int slot, const v4i& sum) {
        const int f = slot / BF, x = slot - f * BF;
        const int ch = 4 * NF * q + 4 * f;
        const int32_t p = m0 + 16 * x + c16;
        if (ch >= noc || p >= a.M) return;
        const int32_t rr = fdiv(p, a.div_bw);
        const int32_t bx = p - rr * a.bw;
        const int32_t nn = fdiv(rr, a.div_bh);
        const int32_t by = rr - nn * a.bh;
        uint8_t* const dst = a.out + (int64_t)nn * a.out_sn + (int64_t)(a.y0 + by) * a.out_sh + (int64_t)(a.x0 + bx) * a.out_sw + (int64_t)(oc0 + ch) * a.out_sc;
        uint32_t other = 0;
        if constexpr (FZ) other = *reinterpret_cast<const uint32_t*>(w.fz.other + (dst - a.out));
        const int32_t* const trow = a.table + (int64_t)(oc0 + ch) * a.table_stride;
        int2 tr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) tr[r] = *reinterpret_cast<const int2*>(trow + r * a.table_stride + 2);
        // High-word form (see nce_conv_wres.hip): everything scaled by 2^(32 - shift) so that the rounding shift is the
        // high word of one multiply-add. Its products stay below 2^63 by the conditions on mult and cq, hence nothing
        // leaves int32 either.
        const PpeDev& pp = a.ppe;
        const bool prelu = !(pp.prelu_mult == 1 && pp.prelu_shift == 0);
        const int32_t pm = pp.prelu_mult, ps = pp.prelu_shift;
        const int64_t slope = ps >= 1 && ps <= 32 ? (int64_t)pm * ((int64_t)1 << (32 - ps)) : 0x7fffffffffffLL;
        bool hi_ok = pp.round_mode == NCE_ROUND_HALF_UP && (!prelu || (slope >= -0x7fffffffLL && slope <= 0x7fffffffLL));
        int32_t mq[4];
        int64_t cq[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int32_t mult = table_mult(tr[r].x), shift = table_shift(tr[r].x);
            const int s = min(max(shift, 1), 32);
            const int64_t m64 = (int64_t)mult << (32 - s);
            const int64_t base = (int64_t)tr[r].y * mult + ((int64_t)1 << (s - 1)) + ((int64_t)pp.zp_out << s);  // (below 2^48)
            hi_ok = hi_ok && shift == s && m64 <= 0x7fffffffLL && base < ((int64_t)1 << (29 + s)) && base > -((int64_t)1 << (29 + s));
            mq[r] = (int32_t)m64;
            cq[r] = (int64_t)((uint64_t)base << (32 - s));
        }
        uint32_t packed = 0;
        if (__all(hi_ok)) {
            const int32_t ilo = pp.lo + pp.zp_out, ihi = pp.hi + pp.zp_out;
            const int32_t pmq = (int32_t)slope;
            const int64_t cpz = ps >= 1 && ps <= 32 ? (((int64_t)1 << (ps - 1)) + (int64_t)pp.zp_out * ((int64_t)1 << ps) - (int64_t)pp.zp_out * pm) * ((int64_t)1 << (32 - ps)) : 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int32_t y = (int32_t)(((int64_t)sum[r] * mq[r] + cq[r]) >> 32);
                if (prelu) y = max(y, (int32_t)(((int64_t)y * pmq + cpz) >> 32));  // (|slope| <= 1/2: it raises negative values only)
                packed |= ((uint32_t)clamp_med3(y, ilo, ihi) & 0xFFu) << (8 * r);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                packed |= ((uint32_t)ppe_apply(sum[r], tr[r].y, table_mult(tr[r].x), table_shift(tr[r].x), pp) & 0xFFu) << (8 * r);
        }
        if (a.out_sc == 1) {
            *reinterpret_cast<uint32_t*>(dst) = packed;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[r * a.out_sc] = (uint8_t)(packed >> (8 * r));
        }
        if constexpr (FZ) {  // the add on the bytes just stored (dense NHWC tensors: same offsets)
            const uint32_t ua = packed ^ w.fz.in_flip, ub = other ^ w.fz.in_flip;
            uint32_t r4 = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t pair = __builtin_amdgcn_perm(ub, ua, 0x0c040c00u + (uint32_t)i * 0x00010001u);
                const int32_t s = (int32_t)__builtin_amdgcn_udot2(__builtin_bit_cast(fz_u16x2, pair), __builtin_bit_cast(fz_u16x2, w.fz.mults),
                                                                   (uint32_t)w.fz.c0h, false);
                r4 |= (uint32_t)clamp_med3((int32_t)(((int64_t)s * w.fz.mq + w.fz.cq) >> 32), w.fz.ilo, w.fz.ihi) << (8 * i);
            }
            *reinterpret_cast<uint32_t*>(w.fz.out + (dst - a.out)) = r4 ^ w.fz.flip;
        }
    };

    // ---- the wave's share of the reduction ------------------------------------------------------------------------------
    const int frag_off = c16 * 64 + ((q ^ swz(c16)) << 4);
    v4i acc[NF][BF], wsum[SUMS ? NF : 1], asum[SUMS ? BF : 1];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int x = 0; x < BF; ++x) acc[f][x] = v4i{0, 0, 0, 0};
    if constexpr (SUMS) {
#pragma unroll
        for (int f = 0; f < NF; ++f) wsum[f] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int x = 0; x < BF; ++x) asum[x] = v4i{0, 0, 0, 0};
    }
    const int axor = (int)a.a_xor, wxor = (int)a.w_xor;
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    auto consume = [&](int slot) {
        const uint8_t* const src = ring + slot * (F * 1024) + frag_off;
        v4i fa[NF], fb[BF];
#pragma unroll
        for (int f = 0; f < NF; ++f) fa[f] = *reinterpret_cast<const v4i*>(src + f * 1024);
#pragma unroll
        for (int x = 0; x < BF; ++x) fb[x] = *reinterpret_cast<const v4i*>(src + (NF + x) * 1024);
#pragma unroll
        for (int f = 0; f < NF; ++f) fa[f] ^= wxor;
#pragma unroll
        for (int x = 0; x < BF; ++x) fb[x] ^= axor;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int x = 0; x < BF; ++x) acc[f][x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[f], fb[x], acc[f][x], 0, 0, 0);
        if constexpr (SUMS) {
#pragma unroll
            for (int f = 0; f < NF; ++f) wsum[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[f], ones, wsum[f], 0, 0, 0);
#pragma unroll
            for (int x = 0; x < BF; ++x) asum[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, fb[x], asum[x], 0, 0, 0);
        }
    };
    int slot = 0, i = 0;
    for (; i + D < n; ++i) {  // steady state: D - 1 younger slices stay in flight
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((D - 1) * F));
        asm volatile("" ::: "memory");
        consume(slot);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's operands are in registers
        request(wave + (i + D) * nwaves, slot);
        slot = slot == D - 1 ? 0 : slot + 1;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    asm volatile("" ::: "memory");
    for (; i < n; ++i) {
        consume(slot);
        slot = slot == D - 1 ? 0 : slot + 1;
    }

    // ---- exchange: every wave leaves its partial fragments, one wave per fragment adds them up -------------------------------
    // (lane layout throughout: accumulator fragment (f, x) has rows 4q .. 4q + 3 of pixel c16; a weight-sum fragment has the
    // same rows in every column, an activation-sum fragment the pixel's sum in every row)
    const int32_t kdd = SUMS ? w.per_wave * nwaves * 64 * a.da * a.dw : 0;  // (padding slices count: their activations are -da)
    __syncthreads();  // every wave has left its ring
    {
        uint8_t* const mine = sR + (wave * SLOTS) * 1024 + lane * 16;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int x = 0; x < BF; ++x) *reinterpret_cast<v4i*>(mine + (f * BF + x) * 1024) = acc[f][x];
        if constexpr (SUMS) {
#pragma unroll
            for (int f = 0; f < NF; ++f) *reinterpret_cast<v4i*>(mine + (NF * BF + f) * 1024) = wsum[f];
#pragma unroll
            for (int x = 0; x < BF; ++x) *reinterpret_cast<v4i*>(mine + (NF * BF + NF + x) * 1024) = asum[x];
        }
    }
    __syncthreads();
    for (int s = wave; s < NF * BF; s += nwaves) {
        v4i sum = {0, 0, 0, 0};
        const uint8_t* src = sR + s * 1024 + lane * 16;
#pragma unroll
        for (int k = 0; k < kSplitWaves; ++k)
            if (k < nwaves) sum += *reinterpret_cast<const v4i*>(src + k * SLOTS * 1024);
        if constexpr (SUMS) {
            const int f = s / BF, x = s - f * BF;
            v4i ws = {0, 0, 0, 0};
            int32_t as = 0;
#pragma unroll
            for (int k = 0; k < kSplitWaves; ++k)
                if (k < nwaves) {
                    ws += *reinterpret_cast<const v4i*>(sR + (k * SLOTS + NF * BF + f) * 1024 + lane * 16);
                    as += *reinterpret_cast<const int32_t*>(sR + (k * SLOTS + NF * BF + NF + x) * 1024 + lane * 16);
                }
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] += a.da * ws[r] + a.dw * as + kdd;
        }
        epilogue_of(s, sum);
    }
}

template <int NF, int BF, int D>
hipError_t launch_tile(SplitConvArgs& w, bool fused, hipStream_t stream) {
    constexpr int F = NF + BF;
    const ConvArgs& a = w.a;
    w.ntm = (uint32_t)(((int64_t)a.M + 16 * BF - 1) / (16 * BF));
    w.ntn = (uint32_t)((a.bc + 16 * NF - 1) / (16 * NF));
    if ((uint64_t)w.ntm * w.ntn > 0x7ffffff0ull) return hipErrorNotSupported;
    w.div_ntm = make_fastdiv(w.ntm);
    w.div_ntn = make_fastdiv(w.ntn);
    const bool sums = a.da != 0 || a.dw != 0;
    const int slots = NF * BF + (sums ? F : 0);
    // As many waves as the reduction has slices, up to eight (and up to what LDS holds at the exchange), and no more than keep
    // the waves' shares equal.
    const int most = std::min(kSplitWaves, 156 / slots);
    w.per_wave = (w.nslices + most - 1) / most;
    const int nwaves = (w.nslices + w.per_wave - 1) / w.per_wave;
    const size_t lds = (size_t)nwaves * 1024 * std::max(D * F, slots);
    const auto go = [&](auto kernel, LdsGrant& grant) {
        if (const hipError_t e = grant.ensure(reinterpret_cast<const void*>(kernel), lds, 48 * 1024); e != hipSuccess) return e;
        return emit(kernel, dim3(xcd_grid(w.ntm * w.ntn)), dim3(64 * nwaves), lds, stream, w);
    };
    static LdsGrant grants[4];
    if (fused) return sums ? go(&conv_split_kernel<NF, BF, D, true, true>, grants[0]) : go(&conv_split_kernel<NF, BF, D, false, true>, grants[1]);
    return sums ? go(&conv_split_kernel<NF, BF, D, true, false>, grants[2]) : go(&conv_split_kernel<NF, BF, D, false, false>, grants[3]);
}

}  // namespace

// shape 0: automatic. Else 1 .. 5: 16 px x 16 ch, 16 px x 32 ch, 32 x 32, 32 px x 64 ch, 64 x 64.
hipError_t launch_conv_split(const ConvArgs& a, hipStream_t stream, int shape, const FuseAdd* fuse) {
    if (a.KY > 31 || a.KX > 31 || a.M > 0x7fffffff - 1024) return hipErrorNotSupported;
    if (fuse != nullptr && a.out_sc != 1) return hipErrorNotSupported;
    for (const int64_t st : {a.in_sn, a.in_sh, a.in_sw})
        if (st < 0 || st > 0x7fffffffLL) return hipErrorNotSupported;
    SplitConvArgs w;
    memset(&w, 0, sizeof(w));
    w.a = a;
    w.a.fill_raw = (a.fill ^ a.a_xor) & 0xFFu;
    if (fuse) w.fz = *fuse;
    w.in_sn32 = (int32_t)a.in_sn;
    w.in_sh32 = (int32_t)a.in_sh;
    w.in_sw32 = (int32_t)a.in_sw;
    w.nslices = (a.KG + 3) / 4;
    w.div_icg = make_fastdiv((uint32_t)a.ICG);
    w.div_kx = make_fastdiv((uint32_t)a.KX);
    w.channel_major = (int64_t)a.bc * a.ktot >= (int64_t)a.M * a.SY * a.SX * a.IC;
    const bool fz = fuse != nullptr;
    switch (shape) {
    case 1: return launch_tile<1, 1, 8>(w, fz, stream);
    case 2: return launch_tile<2, 1, 5>(w, fz, stream);
    case 3: return launch_tile<2, 2, 4>(w, fz, stream);
    case 4: return launch_tile<4, 2, 3>(w, fz, stream);
    case 5: return launch_tile<4, 4, 2>(w, fz, stream);
    default: return hipErrorNotSupported;
    }
}

}  // namespace nce
