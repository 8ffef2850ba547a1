// DWCONV and AVEPOOL tasks on the matrix cores: v_mfma_i32_16x16x64_i8 with a diagonal weight operand.
//
// For one group of 16 channels a depthwise window is an implicit GEMM whose weight matrix is diagonal: reduction step s
// covers the taps 4s .. 4s + 3, lane (pixel c, quarter q) supplies the 16 channel bytes of tap 4s + q as they lie in memory, and
// row c of the weight operand is zero but for byte c, the tap's weight of channel c. One instruction does four taps of 256
// outputs in sixteen clocks where the vector form (nce_window.hip) spends a byte permute and half a dot product on each tap of
// each output: the 7x7 of 32 x 24 x 24 x 832 took 78 us, 49 taps x 1.4 instructions an output. An average pool has the weight 1.
//
// A workgroup owns a run of pixels of up to four channel groups (64 bytes of a pixel) of a column strip. The rows of input it
// reaches go to LDS once, out-of-image bytes filled in; a wave keeps its group's diagonal operands in registers for the
// whole run and reads LDS, one ds_read_b128 per matrix instruction. Layout as in nce_conv_band.hip: one plane per (group, row,
// column modulo the stride), so that 16 pixels are 16 consecutive units. Four accumulator fragments (64 pixels) are requantised
// at a time, four channels of a pixel per lane, and transposed with lane swaps into one 16-byte store per pixel.
// What bounds it: the fetch (rows overlap between runs: 1.3 to 3 times the input through L2) and LDS reads; several workgroups
// per CU cover each other. 7x7 over 32 x 24 x 24 x 832: 83 -> 35 us; 5x5 over 56 x 69 x 69 x 144: 92 -> 62 us.
//
// Zero points as in nce_conv.hip: a' = a ^ 0x80 for u8, sum (a - zp)(w - zpw) = sum a' (w' + dw) + da * sum (w' + dw), with the
// dw part as further instructions against a constant diagonal (128 does not fit a byte: twice 64).
#include "nce_conv_common.h"

#include <algorithm>
#include <cstring>

namespace nce {
namespace {

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kMaxRun = 512;
constexpr int kMaxSteps = 13;

struct WinMfmaArgs {
    TaskDev t;
    Box box;
    int32_t npix;              // pixels of a strip over all images (strip columns x rows x images)
    int32_t strips, tw;        // column strips and their width (the last one may be narrower)
    int32_t run;               // pixels of a workgroup, a multiple of 64
    uint32_t nruns, nslabs;    // runs of a strip; slabs of `groups` channel groups
    int32_t glog;              // log2 of the channel groups per workgroup
    FastDiv div_slabs, div_strips, div_tw, div_bh, div_vh, div_units, div_kx, div_sx;
    int32_t vh;                // rows of an image with its padding
    int32_t units, chunk, per_pass;  // 16-byte units of a row; of a fetch pass; rows of a pass
    int32_t plane, row, group; // LDS bytes: column plane, row, channel group
    int32_t a_xor;
    uint32_t fill;
    int32_t da, dw_step, dw_times;
    int32_t ntaps;
    bool depthwise;
};

// STEPS: reduction steps the kernel is unrolled for (taps past the window's last have zero weights).
template <int STEPS, bool DW2>
__global__ __launch_bounds__(kThreads) void window_mfma_kernel(WinMfmaArgs a) {
    prefetch_kernel_arguments<sizeof(WinMfmaArgs)>();
    const TaskDev& t = a.t;
    const Box& box = a.box;
    extern __shared__ __attribute__((aligned(16))) uint8_t sIn[];
    __shared__ int32_t sPos[kMaxRun];    // LDS offset of a pixel's first tap
    __shared__ int64_t sOut[kMaxRun];    // output offset of a pixel; -1: none

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, q = lane >> 4;

    const uint32_t total = a.nruns * a.nslabs * (uint32_t)a.strips;
    const uint32_t lid = xcd_tile(blockIdx.x, total);
    if (lid >= total) return;  // uniform for the whole workgroup
    const uint32_t r1 = fdiv(lid, a.div_slabs), slab = lid - r1 * a.nslabs;
    const uint32_t rn = fdiv(r1, a.div_strips), strip = r1 - rn * (uint32_t)a.strips;
    const int32_t p0 = (int32_t)rn * a.run, x0 = (int32_t)strip * a.tw;
    const int32_t ngroups = min(1 << a.glog, (box.bc >> 4) - (int32_t)(slab << a.glog));
    const int32_t oc0 = box.z0 + (int32_t)(slab << (a.glog + 4));

    // ---- this wave's group: weights of the lane's channel, table rows of its four channels (requested ahead of the rows) --------
    const int g = wave & ((1 << a.glog) - 1);
    const bool works = g < ngroups;
    const int32_t ch = oc0 + 16 * (works ? g : 0);
    const int ntaps = a.ntaps;
    uint8_t wb[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        wb[s] = 0;
        if (a.depthwise) wb[s] = t.weights[(int64_t)(ch + c16) * t.w_stride_oc + min(4 * s + q, ntaps - 1)];
    }
    int32_t tw2[4] = {0, 0, 0, 0}, tbias[4] = {0, 0, 0, 0};
    if (t.table != nullptr) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int2 row = *reinterpret_cast<const int2*>(t.table + (int64_t)(ch + 4 * q + r) * t.table_stride + 2);
            tw2[r] = row.x;
            tbias[r] = row.y;
        }
    }

    // ---- fetch: a thread owns one unit (column, group) of the rows sub, sub + per_pass, ... of each column chunk -----------------
    auto row_of = [&](int32_t p) {  // row, counted through the batch, of a pixel's first tap
        const int32_t rr = fdiv(p, a.div_tw);
        const int32_t n = fdiv(rr, a.div_bh);
        return n * a.vh + (rr - n * box.bh) * t.sy;
    };
    const int32_t v0 = row_of(p0);
    {
        const int32_t nrows = row_of(min(p0 + a.run, a.npix) - 1) - v0 + t.ky;
        const int32_t iy_base = box.y0 * t.sy - t.pt, ix_base = (box.x0 + x0) * t.sx - t.pl;
        constexpr int BATCH = 8;
        const int32_t sub = fdiv((uint32_t)tid, a.div_units), rem = tid - sub * a.chunk;
        for (int32_t c0 = 0; c0 < a.units; c0 += a.chunk) {
            const int32_t cu = c0 + rem, cg = cu & ((1 << a.glog) - 1), cx = cu >> a.glog, ix = ix_base + cx;
            const bool mine = sub < a.per_pass && cu < a.units;
            const bool col_ok = mine && (uint32_t)ix < (uint32_t)t.in.w && cg < ngroups;
            const int32_t xq = fdiv((uint32_t)cx, a.div_sx);
            uint8_t* const put = sIn + cg * a.group + (cx - xq * t.sx) * a.plane + xq * 16;
            const uint8_t* const src = t.in.data + (col_ok ? (int64_t)ix * t.in.sw + oc0 + 16 * cg : 0);
            int32_t n = fdiv((uint32_t)(v0 + sub), a.div_vh), y = v0 + sub - n * a.vh;
            for (int32_t r0 = sub; r0 < nrows; r0 += BATCH * a.per_pass) {
                uint4 v[BATCH];
                uint32_t in = 0;
#pragma unroll
                for (int j = 0; j < BATCH; ++j) {
                    const int32_t iy = y + iy_base;
                    const bool ok = col_ok && (uint32_t)iy < (uint32_t)t.in.h && n < t.in.n;
                    in |= ok ? 1u << j : 0u;
                    v[j] = *reinterpret_cast<const uint4*>(ok ? src + (int64_t)n * t.in.sn + (int64_t)iy * t.in.sh : t.in.data);
                    y += a.per_pass;
                    while (y >= a.vh) y -= a.vh, ++n;
                }
#pragma unroll
                for (int j = 0; j < BATCH; ++j) {
                    const bool ok = (in >> j) & 1u;
                    uint4 w;
                    w.x = ok ? v[j].x ^ (uint32_t)a.a_xor : a.fill;
                    w.y = ok ? v[j].y ^ (uint32_t)a.a_xor : a.fill;
                    w.z = ok ? v[j].z ^ (uint32_t)a.a_xor : a.fill;
                    w.w = ok ? v[j].w ^ (uint32_t)a.a_xor : a.fill;
                    if (mine && r0 + j * a.per_pass < nrows) *reinterpret_cast<uint4*>(put + (r0 + j * a.per_pass) * a.row) = w;
                }
            }
        }
        for (int i = tid; i < a.run; i += kThreads) {
            const int32_t p = min(p0 + i, a.npix - 1);
            const int32_t rr = fdiv(p, a.div_tw), x = p - rr * a.tw;
            const int32_t n = fdiv(rr, a.div_bh), y = rr - n * box.bh;
            sPos[i] = (n * a.vh + y * t.sy - v0) * a.row + x * 16;
            sOut[i] = p0 + i < a.npix && x0 + x < box.bw
                          ? (int64_t)n * t.out.sn + (int64_t)(box.y0 + y) * t.out.sh + (int64_t)(box.x0 + x0 + x) * t.out.sw + (int64_t)oc0 * t.out.sc
                          : -1;
        }
    }

    // ---- diagonal operands, constants of the lane's four channels ---------------------------------------------------------------
    v4i fa[STEPS];
    int32_t koff[STEPS];
    int32_t wsum = 0;
    const uint32_t wx = t.w_is_signed ? 0u : 0x80u;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int u = 4 * s + q;
        const int uc = u < ntaps ? u : 0;
        uint32_t w = 1;
        if (a.depthwise) w = wb[s] ^ wx;
        if (u >= ntaps) w = 0;
        wsum += u < ntaps ? (int32_t)(int8_t)w + (a.depthwise ? a.dw_step * a.dw_times : 0) : 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) fa[s][d] = (c16 >> 2) == d ? (int)((w & 0xFFu) << (8 * (c16 & 3))) : 0;
        const int ky = (int)fdiv((uint32_t)uc, a.div_kx), kx = uc - ky * t.kx;
        const int kq = (int)fdiv((uint32_t)kx, a.div_sx);
        koff[s] = ky * a.row + (kx - kq * t.sx) * a.plane + kq * 16 + g * a.group;
    }
    wsum += __shfl_xor(wsum, 16);
    wsum += __shfl_xor(wsum, 32);
    const PpeDev& pp = t.ppe;
    const bool prelu = !(pp.prelu_mult == 1 && pp.prelu_shift == 0);
    const int32_t pm = pp.prelu_mult, ps = pp.prelu_shift;
    const int64_t slope = ps >= 1 && ps <= 32 ? (int64_t)pm * ((int64_t)1 << (32 - ps)) : 0x7fffffffffffLL;
    // High-word form (see nce_conv_wres.hip): everything scaled by 2^(32 - shift), so that the rounding shift is the high
    // word of one multiply-add; its conditions keep the products below 2^63 and the results inside int32.
    bool hi_ok = pp.round_mode == NCE_ROUND_HALF_UP && (!prelu || (slope >= -0x7fffffffLL && slope <= 0x7fffffffLL));
    int32_t mult[4], shift[4], bias[4], corr[4], mq[4];
    int64_t cq[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        mult[r] = t.table != nullptr ? table_mult(tw2[r]) : pp.quant_mult;
        shift[r] = t.table != nullptr ? table_shift(tw2[r]) : pp.quant_shift;
        bias[r] = tbias[r];
        corr[r] = a.da * __shfl(wsum, 4 * q + r);
        const int s = min(max(shift[r], 1), 32);
        const int64_t m64 = (int64_t)mult[r] << (32 - s);
        const bool small = mult[r] >= 0 && mult[r] <= 0xFFFF;
        const int64_t base = ((int64_t)bias[r] + corr[r]) * (small ? mult[r] : 0) + ((int64_t)1 << (s - 1)) + ((int64_t)pp.zp_out << s);
        hi_ok = hi_ok && small && shift[r] == s && m64 <= 0x7fffffffLL && base < ((int64_t)1 << (29 + s)) && base > -((int64_t)1 << (29 + s));
        mq[r] = (int32_t)m64;
        cq[r] = (int64_t)((uint64_t)base << (32 - s));
    }
    const bool hi = __all(hi_ok);
    const int32_t ilo = pp.lo + pp.zp_out, ihi = pp.hi + pp.zp_out, pmq = (int32_t)slope;
    const int64_t cpz = ps >= 1 && ps <= 32 ? (((int64_t)1 << (ps - 1)) + (int64_t)pp.zp_out * ((int64_t)1 << ps) - (int64_t)pp.zp_out * pm) * ((int64_t)1 << (32 - ps)) : 0;
    __syncthreads();
    if (!works) return;  // (no barrier follows)

    v4i fd{0, 0, 0, 0}, fdl{0, 0, 0, 0};  // constant diagonal of the weight zero point: all steps but the last, the last
    int last = 0;
    if constexpr (DW2) {
        last = (ntaps - 1) / 4;
        const uint32_t b = (uint32_t)a.dw_step & 0xFFu;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            fd[d] = (c16 >> 2) == d ? (int)(b << (8 * (c16 & 3))) : 0;
            fdl[d] = 4 * last + q < ntaps ? fd[d] : 0;
        }
    }
    // Units of four fragments: 64 pixels, shared out among the waves of a group.
    for (int set = (wave >> a.glog) * 64; set < a.run && p0 + set < a.npix; set += 64 * (kWaves >> a.glog)) {
        int32_t pos[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) pos[x] = sPos[set + 16 * x + c16];
        v4i acc[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[x] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            v4i fb[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) fb[x] = *reinterpret_cast<const v4i*>(sIn + pos[x] + koff[s]);
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[s], fb[x], acc[x], 0, 0, 0);
            if constexpr (DW2) {
                if (s <= last) {  // uniform
                    const v4i f = s == last ? fdl : fd;
                    for (int i = 0; i < a.dw_times; ++i)
#pragma unroll
                        for (int x = 0; x < 4; ++x) acc[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f, fb[x], acc[x], 0, 0, 0);
                }
            }
        }
        uint32_t w[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            w[x] = 0;
            if (hi) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    int32_t y = (int32_t)(((int64_t)acc[x][r] * mq[r] + cq[r]) >> 32);
                    if (prelu) y = max(y, (int32_t)(((int64_t)y * pmq + cpz) >> 32));  // (|slope| <= 1/2: it raises negative values only)
                    w[x] |= ((uint32_t)clamp_med3(y, ilo, ihi) & 0xFFu) << (8 * r);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) w[x] |= ((uint32_t)ppe_apply(acc[x][r] + corr[r], bias[r], mult[r], shift[r], pp) & 0xFFu) << (8 * r);
            }
        }
        // w[x] of quarter q: channels 4q .. of pixel 16x + c. Transposed to: word k of lane: channels 4k .. of pixel `lane`.
        const auto s02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        const auto o01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
        const auto o23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
        const int64_t at = sOut[set + lane];
        if (at >= 0) store_channels16(t.out.data + at + (int64_t)16 * g * t.out.sc, t.out.sc, o01[0], o01[1], o23[0], o23[1]);
    }
}

template <int STEPS>
hipError_t launch_steps(const WinMfmaArgs& a, size_t lds, hipStream_t s) {
    const auto go = [&](auto kernel, LdsGrant& grant) {
        if (const hipError_t e = grant.ensure(reinterpret_cast<const void*>(kernel), lds, 48 * 1024); e != hipSuccess) return e;
        return emit(kernel, dim3(xcd_grid(a.nruns * a.nslabs * (uint32_t)a.strips)), dim3(kThreads), lds, s, a);
    };
    static LdsGrant grants[2];
    return a.dw_times != 0 ? go(&window_mfma_kernel<STEPS, true>, grants[0]) : go(&window_mfma_kernel<STEPS, false>, grants[1]);
}

}  // namespace

// hipErrorNotSupported: the window or its rows are beyond the kernel.
hipError_t launch_window_mfma(const TaskDev& t, const Box& box, bool depthwise, hipStream_t stream) {
    const int64_t ntaps = (int64_t)t.ky * t.kx, images = t.out.n;
    if (ntaps > 4 * kMaxSteps) return hipErrorNotSupported;
    const int64_t cgroups = box.bc >> 4;
    if (images * box.bh * box.bw == 0 || cgroups == 0) return hipSuccess;
    WinMfmaArgs a;
    memset(&a, 0, sizeof(a));
    a.t = t;
    a.box = box;
    a.depthwise = depthwise;
    a.ntaps = (int32_t)ntaps;
    a.glog = cgroups >= 4 ? 2 : cgroups >= 2 ? 1 : 0;
    a.nslabs = (uint32_t)((cgroups + (1 << a.glog) - 1) >> a.glog);
    a.vh = (box.bh - 1) * t.sy + t.ky;
    if (images * a.vh > 0x7fffffff - 4096) return hipErrorNotSupported;
    // Column strips and pixel runs: the pair with the least work of the fullest CU - units fetched, matrix steps, a share per
    // workgroup - among those that leave room for three workgroups per CU (one, where none does).
    const int steps = (int)((ntaps + 3) / 4);
    double best = 1e300;
    size_t lds = 0;
    for (const size_t room : {(size_t)48 * 1024, (size_t)96 * 1024}) {  // (the larger one only where nothing fits the smaller)
        if (best < 1e300) break;
        for (int32_t tw = box.bw;; tw = (tw + 1) / 2) {
            const int64_t strips = (box.bw + tw - 1) / tw, npix = images * box.bh * tw;
            const int64_t cols = (int64_t)(tw - 1) * t.sx + t.kx, px = (cols + t.sx - 1) / t.sx, plane = (px + 15) / 16 * 16, row = plane * (t.sx - 1) + px;
            for (int32_t run = kMaxRun; run >= 64 && npix <= 0x7fffffff - kMaxRun; run /= 2) {
                const int64_t rows = std::min<int64_t>((run + tw - 2) / tw, images * box.bh - 1);
                const int64_t breaks = std::min<int64_t>((rows + box.bh - 1) / box.bh, images - 1);
                const int64_t nrows = rows * t.sy + breaks * std::max(0, t.ky - t.sy) + t.ky;
                const int64_t group = (nrows * row + 15) / 16 * 256;
                const size_t bytes = (size_t)group << a.glog;
                if (bytes > room) continue;
                const int64_t nruns = (npix + run - 1) / run, groups = nruns * a.nslabs * strips;
                if (groups > 0x7ffffff0ll) continue;
                const double cost = (double)((groups + 255) / 256) * (0.4 * (double)((nrows * cols) << a.glog) + 0.3 * (double)((run * steps) << a.glog) + 600.0);
                if (cost < best) {
                    best = cost;
                    lds = bytes;
                    a.tw = tw;
                    a.strips = (int32_t)strips;
                    a.run = run;
                    a.nruns = (uint32_t)nruns;
                    a.npix = (int32_t)npix;
                    a.units = (int32_t)(cols << a.glog);
                    a.group = (int32_t)group;
                    a.plane = (int32_t)(plane * 16);
                    a.row = (int32_t)(row * 16);
                }
            }
            if (tw <= 8) break;
        }
    }
    if (best == 1e300) return hipErrorNotSupported;
    a.chunk = std::min(a.units, kThreads);
    a.per_pass = kThreads / a.chunk;
    a.div_slabs = make_fastdiv(a.nslabs);
    a.div_strips = make_fastdiv((uint32_t)a.strips);
    a.div_tw = make_fastdiv((uint32_t)a.tw);
    a.div_bh = make_fastdiv((uint32_t)box.bh);
    a.div_vh = make_fastdiv((uint32_t)a.vh);
    a.div_units = make_fastdiv((uint32_t)a.chunk);
    a.div_kx = make_fastdiv((uint32_t)t.kx);
    a.div_sx = make_fastdiv((uint32_t)t.sx);
    const int32_t off_a = t.in.is_signed ? 0 : 128;
    a.a_xor = t.in.is_signed ? 0 : (int32_t)0x80808080u;
    a.fill = (uint32_t)((t.in.zp - off_a) & 0xFF) * 0x01010101u;
    a.da = off_a - t.in.zp;
    const int32_t dw = depthwise ? (t.w_is_signed ? 0 : 128) - t.w_zp : 0;
    a.dw_times = dw == 0 ? 0 : dw == 128 ? 2 : 1;
    a.dw_step = dw == 128 ? 64 : dw;
    if (steps <= 3) return launch_steps<3>(a, lds, stream);
    if (steps <= 7) return launch_steps<7>(a, lds, stream);
    return launch_steps<13>(a, lds, stream);
}

}  // namespace nce
