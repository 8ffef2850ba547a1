// CONV task, band kernel: implicit GEMM on v_mfma_i32_16x16x64_i8 for kernels larger than 1x1 over few input channels.
//
// A pixel of 16, 32 or 48 channels is one to three 16-byte units, and the kernels that fetch a tap's unit per lane from global
// memory (weights-resident, LDS-tiled) spend their time on addresses and on 16-byte pieces of cache lines. Here a workgroup
// owns runs of NW waves x 16*BF consecutive output pixels, one after the other, of one slice of 16*NF channels and keeps BOTH
// operands in LDS: the slice's weights, for as long as it lives, and a ring of the input rows that a run and the next one
// reach. Every input row is fetched once per workgroup, in whole cache lines; padding bytes are written into it; and the
// reduction has nothing but LDS reads at offsets from a table and matrix instructions.
//
// What bounds it: issue. Of the stem's time (7x7 over 16 channels, stride 2) the matrix pipe is busy 38 %, the vector pipe
// (epilogue, ring addresses) 51 % and the LDS 40 %, and a wave's chain of them does not overlap with itself. Hence twelve
// waves of 32 or 48 pixels rather than eight of 64 (111 -> 105 us at 128 images), and hence the skew: waves that leave one
// barrier together would do the same thing at the same time, so the second half of the waves is half a run behind: between two
// barriers the first half multiplies run t and then writes it out while the second half writes out run t - 1 and then
// multiplies run t. Rows of run t + 1 are requested before the products of run t and put into the ring after them, in rows
// that run t does not read.
//
// Measured against the kernels named above: stem, 128 images of 224 x 224: 121 -> 107 us; 3x3 over 32 channels to 160, 24 images
// of 96 x 106: 56.6 -> 28.3 us; 5x5 over 16 to 800, 2 x 100 x 100: 32.8 -> 16.7 us; 3x3 over 96 to 304 with a weight zero point,
// 44 x 32 x 32: 39.3 -> 24.9 us. Small tasks are slower (3.7-5 us before the first product), which the estimate in nce_conv.hip
// accounts for.
//
// Ring row: one plane per (16-channel group, column modulo the stride), so that the 16 pixels of a fragment are 16
// consecutive 16-byte units whatever the stride and the channel count (close to bank-conflict-free, nce_conv_lds.h). Rows are
// counted through the batch (every image with its padding rows), so runs cross images. Columns outside the image are filled
// once, rows outside it when they enter the ring.
//
// Semantics are those of nce_conv.hip.
#include "nce_conv_epi.h"
#include "nce_conv_lds.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace nce {
namespace {

using namespace wres_detail;
using namespace lds_detail;

constexpr int band_fetch(int nw) { return 64 / nw; }  // rows a wave fetches a unit of per lane
constexpr size_t kBandLds = 156 * 1024;

struct BandArgs {
    ConvArgs a;
    int32_t nsteps;            // reduction steps of four 16-byte units
    uint32_t ntiles, tpg;      // pixel runs; of a workgroup
    uint32_t groups, slices;   // workgroups per channel slice, channel slices
    FastDiv div_slices, div_vh, div_icg, div_kx, div_sx, div_ring;
    int32_t vh;                // rows of an image with its padding: (bh - 1) * SY + KY
    int32_t ring;              // rows of the ring
    int32_t ru;                // units of a row
    int32_t chunks;            // waves a row's units take: 1, 2, 4 or 8
    int32_t images;
    int32_t plane, row;        // bytes of a plane of a row, of a row
    int32_t band_at, offs_at;  // LDS offsets: ring, unit offsets
    int32_t run_rows, run_px;  // pixels of a run = run_rows * bw + run_px ...
    int32_t run_v;             // ... and run_rows * SY
    int32_t dense_out;         // output pixels at equal distances
    int32_t run_reach, run_fresh;  // rows a run reaches, rows that come new with it (bounds)
};

template <int NF, int BF, int NW, bool ASUM>
__global__ __launch_bounds__(64 * NW) void conv_band_kernel(BandArgs w) {
    prefetch_kernel_arguments<sizeof(BandArgs)>();
    constexpr int OCT = 16 * NF, BP = 16 * BF * NW, FETCH = band_fetch(NW);
    const ConvArgs& a = w.a;
    extern __shared__ __attribute__((aligned(16))) uint8_t sL[];  // weights: [step][NF] x 1 KiB; unit offsets; ring
    __shared__ int32_t sW2[OCT], sBias[OCT], sWsum[OCT], sCorr[OCT];
    __shared__ double sM[OCT], sBfull[OCT];
    __shared__ int32_t sFlags;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, q = lane >> 4;

    const uint32_t total = w.groups * w.slices;
    const uint32_t lid = xcd_tile(blockIdx.x, total);
    if (lid >= total) return;  // uniform for the whole workgroup
    const uint32_t group = fdiv(lid, w.div_slices), slice = lid - group * w.slices;
    const uint32_t t0 = group * w.tpg, t1 = min(t0 + w.tpg, w.ntiles);
    const int32_t oc0 = a.z0 + (int32_t)slice * OCT;
    const int32_t noc = min(OCT, a.z0 + a.bc - oc0);
    uint8_t* const band = sL + w.band_at;
    int32_t* const offs = reinterpret_cast<int32_t*>(sL + w.offs_at);

    // ---- what this thread fetches: one unit of the rows sub, sub + per_pass, ... (rows are uniform in a wave) ---------------
    const int32_t per_pass = NW / w.chunks, sub = wave / w.chunks;
    const int32_t rem = (wave - sub * w.chunks) * 64 + lane;
    const int32_t ux = (int32_t)fdiv((uint32_t)rem, w.div_icg), uc = rem - ux * a.ICG;
    const int32_t uxq = (int32_t)fdiv((uint32_t)ux, w.div_sx), uxr = ux - uxq * a.SX;
    const int32_t ix = ux + a.x0 * a.SX - a.PL;
    const bool writes = rem < w.ru && (uint32_t)ix < (uint32_t)a.W;
    const uint32_t column = writes ? (uint32_t)ix * (uint32_t)a.in_sw + 16u * uc : 0u;
    uint8_t* const put = band + (uc * a.SX + uxr) * w.plane + uxq * 16;
    const int32_t iy_base = a.y0 * a.SY - a.PT;
    const uint4 fill4 = make_uint4(a.fill, a.fill, a.fill, a.fill);

    auto row_of = [&](int32_t p) {  // row, in the batch, of a pixel's first tap
        const int32_t rr = fdiv(p, a.div_bw);
        const int32_t n = fdiv(rr, a.div_bh);
        return n * w.vh + (rr - n * a.bh) * a.SY;
    };
    const int32_t vbase = row_of((int32_t)(t0 * BP));  // its slot is 0
    auto end_of = [&](uint32_t t) { return row_of(min((int32_t)((t + 1) * BP), a.M) - 1) + a.KY; };
    // Row sub + j * per_pass of a fetch: its address and its ring offset are worked out by lane j, all rows at once, and handed to
    // the scalar unit - row by row in scalar code they were half of a run's time. Loads are unconditional (rows past the end or
    // outside the image read some row of it, which is not used) and consumed at one place: behind a branch the compiler
    // waits for every earlier load before the next one.
    uint4 unit[FETCH];
    uint32_t row_slot = 0;  // lane j: ring offset | 1 for a row outside the image
    auto fetch = [&](int32_t first) {  // rows first, first + 1, ...
        const int32_t v = first + sub + min(lane, FETCH - 1) * per_pass;
        const int32_t n = fdiv((uint32_t)v, w.div_vh), iy = v - n * w.vh + iy_base;
        const bool ok = n < w.images && (uint32_t)iy < (uint32_t)a.H;
        const uint64_t at = (uint64_t)(uint32_t)(ok ? n : 0) * (uint32_t)a.in_sn + (uint64_t)(uint32_t)(ok ? iy : 0) * (uint32_t)a.in_sh;
        const int32_t r = v - vbase;
        row_slot = (uint32_t)((r - (int32_t)fdiv((uint32_t)r, w.div_ring) * w.ring) * w.row) | (ok ? 0u : 1u);
#pragma unroll
        for (int j = 0; j < FETCH; ++j) {
            const uint64_t off = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)at, j) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(at >> 32), j) << 32;
            unit[j] = *reinterpret_cast<const uint4*>(a.in + off + column);
        }
    };
    auto place = [&](int32_t first, int32_t end) {
#pragma unroll
        for (int j = 0; j < FETCH; ++j) asm volatile("" : "+v"(unit[j].x), "+v"(unit[j].y), "+v"(unit[j].z), "+v"(unit[j].w));
        const int32_t rows = sub < per_pass ? end - first - sub : 0;
#pragma unroll
        for (int j = 0; j < FETCH; ++j) {
            const uint32_t slot = (uint32_t)__builtin_amdgcn_readlane((int)row_slot, j);
            uint4 u = fill4;
            if ((slot & 1u) == 0) {  // uniform
                u.x = unit[j].x ^ a.a_xor;
                u.y = unit[j].y ^ a.a_xor;
                u.z = unit[j].z ^ a.a_xor;
                u.w = unit[j].w ^ a.a_xor;
            }
            if (j * per_pass >= rows) break;  // uniform
            if (writes) *reinterpret_cast<uint4*>(put + (slot & ~1u)) = u;
        }
    };

    int32_t have = vbase + FETCH * per_pass;  // rows requested
    const int32_t first_end = end_of(t0);
    fetch(vbase);
    // ---- the slice's weights, in operand order (nce_conv_lds.h); offsets of the reduction's units in the band; table rows ------
    int32_t tw2 = 0, tbias = 0;
    if (tid < noc) {
        const int32_t* row = a.table + (int64_t)(oc0 + tid) * a.table_stride;
        tw2 = row[2];
        tbias = row[3];
    }
    {
        const int prow = lane >> 2, pj = (lane & 3) ^ swz(prow);
        for (int b = wave; b < w.nsteps * NF; b += NW) {
            const int s = b / NF, f = b - s * NF, u = 4 * s + pj;
            const int ch = channel_of_frag_row<NF>(f, prow);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (u < a.KG && ch < noc) {
                v = *reinterpret_cast<const uint4*>(a.w + (int64_t)(oc0 + ch) * a.w_soc + 16 * u);
                v.x ^= a.w_xor;
                v.y ^= a.w_xor;
                v.z ^= a.w_xor;
                v.w ^= a.w_xor;
            }
            *reinterpret_cast<uint4*>(sL + b * 1024 + lane * 16) = v;
        }
        for (int u = tid; u < 4 * w.nsteps; u += (64 * NW)) {
            const int tap = (int)fdiv((uint32_t)u, w.div_icg), icg = u - tap * a.ICG;
            const int ky = (int)fdiv((uint32_t)tap, w.div_kx), kx = tap - ky * a.KX;
            const int kq = (int)fdiv((uint32_t)kx, w.div_sx);
            // (units past the end read the first one, against zero weights)
            offs[u] = u < a.KG ? (icg * a.SX + kx - kq * a.SX) * w.plane + ky * w.row + kq * 16 : 0;
        }
    }
    for (int i = tid * 16; i < w.ring * w.row; i += (64 * NW) * 16) *reinterpret_cast<uint4*>(band + i) = fill4;
    if (tid == 0) sFlags = 0;
    __syncthreads();
    place(vbase, min(have, first_end));
    for (; have < first_end; have += FETCH * per_pass) {
        fetch(have);
        place(have, min(have + FETCH * per_pass, first_end));
    }
    have = first_end;

    const int frag_off = c16 * 64 + ((q ^ swz(c16)) << 4);
    // ---- per-channel constants (thread = channel), as in the weights-resident kernel -----------------------------------------
    if (a.da != 0) {
        const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
        if (wave < NF) {
            v4i ws = {0, 0, 0, 0};
            for (int s = 0; s < w.nsteps; ++s)
                ws = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i*>(sL + (s * NF + wave) * 1024 + frag_off), ones, ws, 0, 0, 0);
            if (c16 == 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) sWsum[channel_of_frag_row<NF>(wave, 4 * q + r)] = ws[r];
            }
        }
    }
    const int64_t acc_bound = min((int64_t)a.ktot * 65025, (int64_t)2147483648LL);
    if (tid < OCT) {
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
        const int32_t pm = a.ppe.prelu_mult, ps = a.ppe.prelu_shift;
        if (ps <= 32 && (ps >= 1 || pm == 0)) {
            const int64_t sl = (int64_t)pm * ((int64_t)1 << (32 - ps));
            if (sl >= -0x7fffffffLL && sl <= 0x7fffffffLL) {
                const int64_t zpf = pu.zp + (ep.flip ? 128 : 0);
                const int64_t half = ps >= 1 ? (int64_t)1 << (ps - 1) : 0;
                pmode = PPE_MODE_HI_SLOPE;
                ep.pmq = __builtin_amdgcn_readfirstlane((int32_t)sl);
                ep.cpz = (half + zpf * ((int64_t)1 << ps) - zpf * pm) * ((int64_t)1 << (32 - ps));
            }
        }
    }
    if (tid < OCT) {
        const int32_t mult = table_mult(tw2), shift = table_shift(tw2);
        const int32_t corr = (a.da != 0 ? a.da * sWsum[tid] : 0) + a.ktot * a.da * a.dw;
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
    const EpiSmem es = {sM, nullptr, sW2, sBias, nullptr, nullptr};

    // This lane's pixels: column, row in the image and row in the batch of the first tap; moved on from run to run.
    int32_t bx[BF], by[BF], bv[BF];
#pragma unroll
    for (int x = 0; x < BF; ++x) {
        const int32_t p = (int32_t)(t0 * BP) + (wave * BF + x) * 16 + c16;
        const int32_t rr = fdiv(p, a.div_bw);
        bx[x] = p - rr * a.bw;
        const int32_t n = fdiv(rr, a.div_bh);
        by[x] = rr - n * a.bh;
        bv[x] = n * w.vh + by[x] * a.SY;
    }
    const int32_t ring_bytes = w.ring * w.row;
    const bool ahead = wave < NW / 2;
    const auto barrier = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (uint32_t t = t0; t < t1; ++t) {
        if (ahead && t > t0) barrier();  // the rows of run t are in the ring, those of run t - 1 are no longer read
        const int32_t next_end = t + 1 < t1 ? end_of(t + 1) : have;
        if (t + 1 < t1) fetch(have);
        const int32_t p0 = (int32_t)(t * BP), v0 = row_of(p0);
        const int32_t s0 = v0 - vbase - (int32_t)fdiv((uint32_t)(v0 - vbase), w.div_ring) * w.ring;
        uint32_t pb[BF];  // offset of the pixel's first unit in the ring
#pragma unroll
        for (int x = 0; x < BF; ++x) {
            int32_t slot = s0 + min(bv[x] - v0, w.ring - 1);  // (pixels past the last one: any row)
            slot -= slot >= w.ring ? w.ring : 0;
            pb[x] = __umul24((uint32_t)slot, (uint32_t)w.row) + (uint32_t)bx[x] * 16u;
            // on to the next run
            bx[x] += w.run_px;
            const bool wrap = bx[x] >= a.bw;
            bx[x] -= wrap ? a.bw : 0;
            const int32_t dr = w.run_rows + (wrap ? 1 : 0);
            by[x] += dr;
            bv[x] += w.run_v + (wrap ? a.SY : 0);
            for (int32_t left = w.run_rows + 1; left > 0; left -= a.bh) {  // uniform; images passed
                const bool over = by[x] >= a.bh;
                by[x] -= over ? a.bh : 0;
                bv[x] += over ? a.KY - a.SY : 0;
            }
        }
        v4i acc[NF][BF], asum[ASUM ? BF : 1];
#pragma unroll
        for (int x = 0; x < BF; ++x) {
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f][x] = v4i{0, 0, 0, 0};
            if constexpr (ASUM) asum[x] = v4i{0, 0, 0, 0};
        }
        // Operands of the next step are read between this step's matrix instructions: by itself the compiler reads each
        // fragment right before its use, five LDS latencies per step.
        const uint8_t* fw = sL + frag_off;
        v4i fa[2][NF], fb[2][BF];
        int32_t off = offs[q];
        auto read_a = [&](auto p, int f) { fa[decltype(p)::value][f] = *reinterpret_cast<const v4i*>(fw + f * 1024); };
        auto read_b = [&](auto p, int x) { fb[decltype(p)::value][x] = *reinterpret_cast<const v4i*>(band + min(pb[x] + off, pb[x] + off - (uint32_t)ring_bytes)); };
        auto step = [&](auto p, int s) {
            constexpr int P = decltype(p)::value;
            const auto other = std::integral_constant<int, P ^ 1>{};
            constexpr int G = BF;  // groups of NF matrix instructions
            int32_t next_off = 0;
#pragma unroll
            for (int x = 0; x < G; ++x) {
                if constexpr (ASUM) {  // (units past the end do not count)
                    const int one = 4 * s + q < a.KG ? 0x01010101 : 0;
                    const v4i ones = {one, one, one, one};
                    asum[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, fb[P][x], asum[x], 0, 0, 0);
                }
#pragma unroll
                for (int f = 0; f < NF; ++f) acc[f][x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[P][f], fb[P][x], acc[f][x], 0, 0, 0);
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    if (f * G / NF == x) read_a(other, f);
                read_b(other, x);
                if (x == 0) next_off = offs[4 * min(s + 2, w.nsteps - 1) + q];
                __builtin_amdgcn_sched_barrier(0);
            }
            off = next_off;
            fw += NF * 1024;
        };
        const auto P0 = std::integral_constant<int, 0>{};
        const auto P1 = std::integral_constant<int, 1>{};
#pragma unroll
        for (int f = 0; f < NF; ++f) read_a(P0, f);
#pragma unroll
        for (int x = 0; x < BF; ++x) read_b(P0, x);
        fw += NF * 1024;
        off = offs[4 * min(1, w.nsteps - 1) + q];
        for (int s = 0;;) {  // (the last step reads operands that nothing uses)
            step(P0, s);
            if (++s == w.nsteps) break;
            step(P1, s);
            if (++s == w.nsteps) break;
        }
        if (t + 1 < t1) place(have, next_end);
        have = next_end;
        if (!ahead && t + 1 < t1) barrier();
        uint8_t* dst[BF];
        bool valid[BF];
#pragma unroll
        for (int x = 0; x < BF; ++x) {
            const int32_t p = p0 + (wave * BF + x) * 16 + c16;
            valid[x] = p < a.M;
            if (w.dense_out) {
                dst[x] = a.out + (int64_t)a.y0 * a.out_sh + (int64_t)a.x0 * a.out_sw + (int64_t)p * a.out_sw + (int64_t)oc0 * a.out_sc;
            } else {
                const int32_t rr = fdiv(p, a.div_bw);
                const int32_t n = fdiv(rr, a.div_bh);
                dst[x] = a.out + (int64_t)n * a.out_sn + (int64_t)(a.y0 + rr - n * a.bh) * a.out_sh + (int64_t)(a.x0 + p - rr * a.bw) * a.out_sw + (int64_t)oc0 * a.out_sc;
            }
        }
        int32_t dws[BF];
#pragma unroll
        for (int x = 0; x < BF; ++x) dws[x] = ASUM ? a.dw * asum[x][0] : 0;  // (every row of a sum fragment is the pixel's sum)
        if (pmode == PPE_MODE_HI) wres_epilogue<NF, BF, PPE_MODE_HI>(a, es, sBfull, sCorr, acc, dws, q, noc, dst, valid, pu, ep);
        else if (pmode == PPE_MODE_HI_SLOPE) wres_epilogue<NF, BF, PPE_MODE_HI_SLOPE>(a, es, sBfull, sCorr, acc, dws, q, noc, dst, valid, pu, ep);
        else if (pmode == PPE_MODE_FOLDED) wres_epilogue<NF, BF, PPE_MODE_FOLDED>(a, es, sBfull, sCorr, acc, dws, q, noc, dst, valid, pu, ep);
        else if (pmode == PPE_MODE_SLOPE) wres_epilogue<NF, BF, PPE_MODE_SLOPE>(a, es, sBfull, sCorr, acc, dws, q, noc, dst, valid, pu, ep);
        else wres_epilogue<NF, BF, PPE_MODE_INT>(a, es, sBfull, sCorr, acc, dws, q, noc, dst, valid, pu, ep);
    }
}

// Band geometry of a task for pixel runs of 16 * bf * nw; false: it does not fit.
bool band_plan(const ConvArgs& a, int nf, int bf, int nw, BandArgs* w) {
    const int64_t bp = 16 * bf * nw;
    const int64_t columns = (int64_t)(a.bw - 1) * a.SX + a.KX, ru = columns * a.ICG;
    if (ru > 512) return false;
    const int64_t images = a.M / ((int64_t)a.bw * a.bh), ntiles = (a.M + bp - 1) / bp;
    // rows that n consecutive pixels reach; rows that come new with a run
    const auto rows_of = [&](int64_t n) {
        const int64_t rows = std::min<int64_t>((n + a.bw - 2) / a.bw, images * a.bh - 1);
        const int64_t breaks = std::min<int64_t>((rows + a.bh - 1) / a.bh, images - 1);
        return rows * a.SY + breaks * std::max(0, a.KY - a.SY) + a.KY;
    };
    const int64_t slices = (a.bc + 16 * nf - 1) / (16 * nf), most = std::max<int64_t>(1, 256 / slices);
    const int64_t tpg = (ntiles + most - 1) / most;
    const int64_t ring = rows_of(tpg == 1 ? bp : 2 * bp);
    int64_t chunks = 1;
    while (chunks * 64 < ru) chunks *= 2;
    const int64_t per_pass = nw / chunks;
    const int64_t step = (bp + a.bw - 1) / a.bw;
    const int64_t fresh = step * a.SY + std::min((step + a.bh - 1) / a.bh, images - 1) * std::max(0, a.KY - a.SY);
    if (tpg > 1 && fresh > per_pass * band_fetch(nw)) return false;
    const int64_t px = (columns + a.SX - 1) / a.SX;  // units of a row in a plane
    const int64_t plane = (px + 15) / 16 * 16, row = (plane * (a.ICG * a.SX - 1) + px) * 16;
    const int64_t nsteps = (a.KG + 3) / 4, wbytes = nsteps * nf * 1024, obytes = (nsteps * 16 + 255) / 256 * 256;
    if (wbytes + obytes + ring * row > (int64_t)kBandLds) return false;
    w->nsteps = (int32_t)nsteps;
    w->ntiles = (uint32_t)ntiles;
    w->slices = (uint32_t)slices;
    w->tpg = (uint32_t)tpg;
    w->groups = (uint32_t)((ntiles + tpg - 1) / tpg);
    w->div_slices = make_fastdiv(w->slices);
    w->vh = (a.bh - 1) * a.SY + a.KY;
    w->div_vh = make_fastdiv((uint32_t)w->vh);
    w->div_icg = make_fastdiv((uint32_t)a.ICG);
    w->div_kx = make_fastdiv((uint32_t)a.KX);
    w->div_sx = make_fastdiv((uint32_t)a.SX);
    w->div_ring = make_fastdiv((uint32_t)ring);
    w->ring = (int32_t)ring;
    w->ru = (int32_t)ru;
    w->chunks = (int32_t)chunks;
    w->images = (int32_t)images;
    w->plane = (int32_t)(plane * 16);
    w->row = (int32_t)row;
    w->offs_at = (int32_t)wbytes;
    w->band_at = (int32_t)(wbytes + obytes);
    w->run_rows = (int32_t)(bp / a.bw);
    w->run_px = (int32_t)(bp % a.bw);
    w->run_v = w->run_rows * a.SY;
    w->run_reach = (int32_t)rows_of(bp);
    w->run_fresh = (int32_t)fresh;
    w->dense_out = a.out_sh == a.bw * a.out_sw && a.out_sn == a.bh * a.out_sh;
    return true;
}

template <int NF, int BF, int NW>
hipError_t launch_band(BandArgs& w, hipStream_t stream) {
    const ConvArgs& a = w.a;
    if (!band_plan(a, NF, BF, NW, &w)) return hipErrorNotSupported;
    const size_t lds = (size_t)w.band_at + (size_t)w.ring * w.row;
    const auto go = [&](auto kernel, LdsGrant& grant) {
        if (const hipError_t e = grant.ensure(reinterpret_cast<const void*>(kernel), lds, 48 * 1024); e != hipSuccess) return e;
        return emit(kernel, dim3(xcd_grid(w.groups * w.slices)), dim3(64 * NW), lds, stream, w);
    };
    static LdsGrant grants[2];
    return a.dw != 0 ? go(&conv_band_kernel<NF, BF, NW, true>, grants[0]) : go(&conv_band_kernel<NF, BF, NW, false>, grants[1]);
}

}  // namespace

BandShape band_shape_for(const ConvArgs& a, int shape) {
    static constexpr int kTiles[4][2] = {{1, 8}, {2, 8}, {2, 12}, {3, 12}};
    BandShape b = {};
    BandArgs w;
    const int nf = a.bc > 32 ? 4 : 2, nw = kTiles[shape - 1][1];
    if (!band_plan(a, nf, kTiles[shape - 1][0], nw, &w)) return b;
    const int per_pass = nw / w.chunks;
    b.ok = true;
    b.nf = nf;
    b.tpg = w.tpg;
    b.groups = (int64_t)w.groups * w.slices;
    b.first_passes = (w.run_reach + per_pass - 1) / per_pass;
    b.fresh_passes = w.tpg > 1 ? (w.run_fresh + per_pass - 1) / per_pass : 0;
    return b;
}

// shape 1 .. 4: eight waves of 16 or of 32 pixels, twelve of 32 or of 48.
hipError_t launch_conv_band(const ConvArgs& a, hipStream_t stream, int shape) {
    if (a.M > 0x7fffffff - 1024) return hipErrorNotSupported;
    // (row numbers through the batch stay inside int32)
    if ((int64_t)a.M / ((int64_t)a.bw * a.bh) * ((int64_t)(a.bh - 1) * a.SY + a.KY) > 0x7fffffff - 4096) return hipErrorNotSupported;
    BandArgs w;
    memset(&w, 0, sizeof(w));
    w.a = a;
    w.a.fill_raw = (a.fill ^ a.a_xor) & 0xFFu;
    for (const int64_t st : {a.in_sn, a.in_sh, a.in_sw})
        if (st < 0 || st > 0x7fffffffLL) return hipErrorNotSupported;
    if (a.in_sw > 0x7fffffff / a.W) return hipErrorNotSupported;  // (32-bit offsets within a row)
    if (a.bc > 32) {
        switch (shape) {
        case 1: return launch_band<4, 1, 8>(w, stream);
        case 2: return launch_band<4, 2, 8>(w, stream);
        case 3: return launch_band<4, 2, 12>(w, stream);
        case 4: return launch_band<4, 3, 12>(w, stream);
        default: return hipErrorNotSupported;
        }
    }
    switch (shape) {
    case 1: return launch_band<2, 1, 8>(w, stream);
    case 2: return launch_band<2, 2, 8>(w, stream);
    case 3: return launch_band<2, 2, 12>(w, stream);
    case 4: return launch_band<2, 3, 12>(w, stream);
    default: return hipErrorNotSupported;
    }
}

}  // namespace nce
