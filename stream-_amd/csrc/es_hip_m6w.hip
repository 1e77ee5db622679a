// Batched Q6_K products with one wave per superblock: es_matvec_multi (src/es_quant.c:1818-1850) for Q6_K rows against
// activations read as the Q8_K rows they are (no pre-pass). The reference forms, per row, activation and superblock,
// tot = sum sc * q_u * x - 32 * sum_g sc_g * bsums_g with q_u the unsigned 6-bit code, then s += (y.d * d) * tot over the
// row's superblocks in order (src/es_quant.c:1602-1640).
//
// A workgroup of up to 8 waves takes 16 rows x 16 WN activations at a time; wave w the superblocks w, w + waves, ... of
// these rows. Only the last line above is sequential: every wave forms its superblock's integers for the whole tile and
// leaves them in LDS as floats, and after one barrier each (4 rows, activation) has a thread that runs the reference's chain
// over the superblocks at hand (rows of 1 to 3 superblocks have fewer threads than chains at 32 or 64 activations and run them
// in turns: 8192 x 768 at 64 activations 8.6 us against 9.6 with narrower tiles, which unpack every superblock twice). A
// product of few rows and many superblocks (a 2048 x 8192 down projection: 16 workgroups of 128 rows running 32 superblocks
// one after another, 94.9 us at 64 activations) so has its superblocks in flight on different waves; with at most as many
// superblocks as waves a wave keeps its activation operands in registers over all row groups of its workgroup, and no operand
// passes through LDS. Measured (tiled kernel before -> this one): 2048 x 8192 at 64 activations 94.9 us and 5 us of pre-pass
// -> 24 us, 8192 x 2048 29.5 -> 12.8 us. Bound by the address unit: 16 rows x 64 bytes a load instruction, every other
// superblock 2 bytes off a dword. On 2048 x 8192 at 64 it is busy for 88% of the launch, the vector units for 26% of it; at 16
// activations the kernel streams 2.3 TB/s of the head's weights, and a second item of weights in flight changed nothing.
//
// Integers: q_u * sc lies in -8064..8001 and is split into two signed bytes, q_u * sc = 256 hi + lo, so two int8 planes
// carry it exactly: sum q_u * sc * x = 256 D(hi) + D(lo). -32 corr goes through one f16 MFMA (-32 sc and the bsums are
// exact halves, every partial sum a multiple of 32 below 2^29: exact in f32). 9 MFMAs per 16 x 16 tile and superblock.
// K order of the operands: slice ks and lane group lg take scale group g = 4 ks + lg, i.e. with n = ks >> 1, qn = ks & 1,
// qo = lg >> 1, lh = lg & 1 the elements 128 n + 32 (2 qn + qo) + 16 lh + [0, 16): nibble qn of ql[64 n + 32 qo + 16 lh + i]
// and field 2 qn + qo of qh[32 n + 16 lh + i] (src/es_quant.c:158-176); the activation operand is the row's 16-byte chunk g.
#include "es_hip_common.h"

namespace esq {
namespace {

typedef int16_t s16x8 __attribute__((ext_vector_type(8)));
// the raw bytes a lane needs of its row's superblock: its pieces of ql and qh, all 16 scales, d
struct Raw6 { uint4 ql0, ql1, qh0, qh1, sc; uint32_t d; };
__device__ __forceinline__ void load_raw6(const uint8_t *blk, int lg, Raw6 &r) {
    const int qo = lg >> 1, lh = lg & 1;
    r.ql0 = ldg_u128_a2(blk + (32 * qo + 16 * lh));
    r.ql1 = ldg_u128_a2(blk + 64 + 32 * qo + 16 * lh);
    r.qh0 = ldg_u128_a2(blk + 128 + 16 * lh);
    r.qh1 = ldg_u128_a2(blk + 160 + 16 * lh);
    r.sc = ldg_u128_a2(blk + 192);
    r.d = ldg<uint16_t>(blk + 208);
}

struct A6 { v4i hi[4], lo[4]; v8h corr; };
__device__ __forceinline__ void build_a6(const Raw6 &r, int lg, A6 &A) {
    const uint32_t scw[4] = {r.sc.x, r.sc.y, r.sc.z, r.sc.w};
    const int qo2 = (lg >> 1) * 2;
    // the qh dwords shifted by this lane's field pair once: field 2 qn + qo of each byte then sits at bits 4 qn .. 4 qn + 1
    const uint32_t qs0[4] = {r.qh0.x >> qo2, r.qh0.y >> qo2, r.qh0.z >> qo2, r.qh0.w >> qo2};
    const uint32_t qs1[4] = {r.qh1.x >> qo2, r.qh1.y >> qo2, r.qh1.z >> qo2, r.qh1.w >> qo2};
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
        const int n = ks >> 1, qn = ks & 1;
        const uint32_t sc2 = q6_scale2(scw[ks], lg);
        const uint4 qlv = n ? r.ql1 : r.ql0;
        const uint32_t qlw[4] = {qlv.x, qlv.y, qlv.z, qlv.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t nib = qn ? (qlw[i] >> 4) & 0x0f0f0f0fu : qlw[i] & 0x0f0f0f0fu;
            const uint32_t qsw = n ? qs1[i] : qs0[i];
            uint32_t h, l;
            q6_planes(nib | ((qn ? qsw : qsw << 4) & 0x30303030u), sc2, h, l);
            A.hi[ks][i] = (int)h;
            A.lo[ks][i] = (int)l;
        }
    }
    A.corr = q6_corr(lg == 0 ? scw[0] : scw[2], lg == 0 ? scw[1] : scw[3], lg);
}

struct B6 { v4i x[4]; s16x8 m; float d; };
__device__ __forceinline__ void load_b6(const uint8_t *blk, int lg, B6 &b) {   // blk: the lane's activation's Q8_K block
#pragma unroll
    for (int ks = 0; ks < 4; ks++) b.x[ks] = __builtin_bit_cast(v4i, ldg<uint4>(blk + 4 + 16 * (4 * ks + lg)));
    b.m = __builtin_bit_cast(s16x8, ldg<uint4>(blk + 260 + 16 * (lg & 1)));
    b.d = ldg<float>(blk);
}

// Launches of a few jobs: the jobs as arguments, one block (the kernel's first and only parameter, at offset 0 of the argument
// segment). A job is read at the grid row's offset of the segment, in the round trip that brings the arguments themselves (found
// by its tile numbers it came a round trip later, 0.1 us a launch).
struct M6wArgs { MkJob j[GRID_ROWS]; };   // grid row i runs the gridDim.x tiles of j[i] from -j[i].tile0 on
__device__ __forceinline__ MkJob m6w_job() {
    static_assert(sizeof(MkJob) % 4 == 0 && offsetof(M6wArgs, j) == 0, "jobs are read as dwords");
    constexpr int N = sizeof(MkJob) / 4;
    typedef const __attribute__((address_space(4))) uint32_t *ArgPtr;
    const ArgPtr src = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr() + blockIdx.y * N;
    uint32_t v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = src[i];
    return uniform_job(__builtin_bit_cast(MkJob, v));
}

// KEEP: at most as many superblocks as waves (one round per row group, activation operands loaded once).
template <int WN, bool CONTRACT, bool KEEP>
__device__ __forceinline__ void m6w_body(const MkJob &J) {
    extern __shared__ __align__(16) float lds6[];   // two buffers of [wave][16 WN activations][16 rows] tot | d | y.d
    // all activation tiles of a row chunk on one XCD (workgroup g runs on XCD g % 8; a grid row is a multiple of 8)
    const int tile = blockIdx.x - J.tile0, kq = tile >> 3;
    const int chunk = (tile & 7) + 8 * (kq / J.ntok_tiles), tok0 = (kq % J.ntok_tiles) * 16 * WN;
    const int ngroup = (J.r1 - J.r0 + 15) / 16, g0 = chunk * J.rows_per_wg, g1 = min(ngroup, g0 + J.rows_per_wg);
    if (g0 >= g1) return;
    const int nbk = J.cols / 256, nw = blockDim.x >> 6, nround = KEEP ? 1 : (nbk + nw - 1) / nw;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    constexpr int TOT = WN * 256, PERW = TOT + 16 + 16 * WN;   // floats per wave: tot, the rows' d, the activations' d
    const int items = (g1 - g0) * nround;

    uint32_t aoff[WN];   // the lane's activation rows (past the last repeat it; not stored)
#pragma unroll
    for (int c = 0; c < WN; c++) aoff[c] = (uint32_t)min(tok0 + 16 * c + lr, J.na - 1) * (uint32_t)J.astride;
    // item it: row group g0 + it / nround, superblock (it % nround) * nw + wave. A wave past the row's end in the last round
    // keeps its former weights and takes the row's last activation block: no chain reads its terms.
    Raw6 raw;
    B6 B[WN];
    auto load_w = [&](int it) {
        const int g = g0 + (KEEP ? it : it / nround), b = (KEEP ? 0 : it % nround) * nw + wave;
        if (it < items && b < nbk) load_raw6(J.W + ((uint32_t)min(J.r0 + 16 * g + lr, J.r1 - 1) * (uint32_t)J.row_bytes + 210u * b), lg, raw);
    };
    auto load_x = [&](int rd) {
        const int b = min(rd * nw + wave, nbk - 1);
#pragma unroll
        for (int c = 0; c < WN; c++) load_b6(J.act + aoff[c] + 292u * b, lg, B[c]);
    };
    load_w(0);
    load_x(0);

    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int it = 0; it < items; it++) {
        const int g = g0 + (KEEP ? it : it / nround), rd = KEEP ? 0 : it % nround;
        float *buf = lds6 + (it & 1) * nw * PERW, *mine = buf + wave * PERW;
        A6 a6;
        build_a6(raw, lg, a6);
        if (lg == 0) mine[TOT + lr] = half_bits_to_float(raw.d);
        load_w(it + 1);
#pragma unroll
        for (int c = 0; c < WN; c++) {
            v8h m;
#pragma unroll
            for (int e = 0; e < 8; e++) m[e] = static_cast<_Float16>(B[c].m[e]);
            const v4f dc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a6.corr, m, v4f{0, 0, 0, 0}, 0, 0, 0);
            v4i hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a6.hi[0], B[c].x[0], v4i{0, 0, 0, 0}, 0, 0, 0);
            v4i lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a6.lo[0], B[c].x[0], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int ks = 1; ks < 4; ks++) {
                hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a6.hi[ks], B[c].x[ks], hi, 0, 0, 0);
                lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a6.lo[ks], B[c].x[ks], lo, 0, 0, 0);
            }
            float4 t;   // rows 4 lg .. + 3 of activation 16 c + lr
            t.x = static_cast<float>(((hi[0] << 8) + lo[0]) + (int)dc[0]);
            t.y = static_cast<float>(((hi[1] << 8) + lo[1]) + (int)dc[1]);
            t.z = static_cast<float>(((hi[2] << 8) + lo[2]) + (int)dc[2]);
            t.w = static_cast<float>(((hi[3] << 8) + lo[3]) + (int)dc[3]);
            *reinterpret_cast<float4 *>(mine + (16 * c + lr) * 16 + 4 * lg) = t;
            if (lg == 0) mine[TOT + 16 + 16 * c + lr] = B[c].d;
        }
        if constexpr (!KEEP) load_x((it + 1) % nround);
        lds_sync();   // the item's terms are complete; the other buffer's chains (before this barrier) are done with it
        auto chain = [&](int c, float (&s)[4]) {   // chain c: activation c / 4 of the tile, rows 4 (c % 4) .. + 3
            const int n = min(nw, nbk - rd * nw), cq = c >> 2, cr = 4 * (c & 3), q = tok0 + cq;
            const float *e = buf;
            for (int k = 0; k < n; k++, e += PERW) {
                const float4 t = *reinterpret_cast<const float4 *>(e + cq * 16 + cr), d = *reinterpret_cast<const float4 *>(e + TOT + cr);
                const float td = e[TOT + 16 + cq];
                if constexpr (CONTRACT) {
                    s[0] = __builtin_fmaf(td * d.x, t.x, s[0]);
                    s[1] = __builtin_fmaf(td * d.y, t.y, s[1]);
                    s[2] = __builtin_fmaf(td * d.z, t.z, s[2]);
                    s[3] = __builtin_fmaf(td * d.w, t.w, s[3]);
                } else {
                    s[0] = s[0] + td * d.x * t.x;
                    s[1] = s[1] + td * d.y * t.y;
                    s[2] = s[2] + td * d.z * t.z;
                    s[3] = s[3] + td * d.w * t.w;
                }
            }
            if (rd == nround - 1) {
                const int r = J.r0 + 16 * g + cr;
                if (q < J.na) {
                    float *yp = J.y + (size_t)q * J.ystride + r;
                    if (r + 3 < J.r1 && (reinterpret_cast<uintptr_t>(yp) & 15) == 0) {
                        stg<float4>(yp, make_float4(s[0], s[1], s[2], s[3]));
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (r + i < J.r1) stg<float>(yp + i, s[i]);
                    }
                }
                s[0] = s[1] = s[2] = s[3] = 0.0f;
            }
        };
        if constexpr (KEEP && WN > 1) {   // a row of fewer superblocks than the tile has 16 activations: fewer threads than chains
            for (int c = tid; c < WN * 64; c += blockDim.x) {
                float s0[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                chain(c, s0);
            }
        } else if (tid < WN * 64) {   // the sums live over the row's rounds, in the chain's one thread
            chain(tid, s);
        }
    }
}

template <int WN, bool CONTRACT, bool KEEP>
__global__ __launch_bounds__(512) void m6w_kernel(M6wArgs) {
    const MkJob J = m6w_job();
    m6w_body<WN, CONTRACT, KEEP>(J);
}
// Launches of more jobs, from their table on the device. A kernel of its own: with both sources in one every launch took 0.1 to
// 0.5 us more (2048 x 768 at 8 activations 3.71 -> 3.93 us, 2048 x 8192 at 64 22.1 -> 22.4, 64 x 2048 x 768 at 12 45.2 -> 45.7).
template <int WN, bool CONTRACT, bool KEEP>
__global__ __launch_bounds__(512) void m6w_kernel_table(const MkJob *__restrict__ jobs, int njobs) {
    const MkJob J = uniform_job(load_tile_job(jobs, njobs, blockIdx.x));
    m6w_body<WN, CONTRACT, KEEP>(J);
}

template <int WN>
hipError_t launch(int nw, bool keep, const MkJob *jobs, int njobs, const M6wArgs &A, dim3 grid, int order, hipStream_t s) {
    const bool contract = order == ES_HIP_ORDER_X86_CONTRACT;
    const auto kern = contract ? (keep ? m6w_kernel<WN, true, true> : m6w_kernel<WN, true, false>)
                               : (keep ? m6w_kernel<WN, false, true> : m6w_kernel<WN, false, false>);
    const auto table = contract ? (keep ? m6w_kernel_table<WN, true, true> : m6w_kernel_table<WN, true, false>)
                                : (keep ? m6w_kernel_table<WN, false, true> : m6w_kernel_table<WN, false, false>);
    const size_t lds = (size_t)2 * nw * (WN * 256 + 16 + 16 * WN) * sizeof(float);   // at most 70 KB
    if (lds > 60 * 1024) {
        hipError_t e = hipFuncSetAttribute(jobs ? reinterpret_cast<const void *>(table) : reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
    }
    if (jobs)
        hipLaunchKernelGGL(table, grid, dim3(64 * nw), lds, s, jobs, njobs);
    else
        hipLaunchKernelGGL(kern, grid, dim3(64 * nw), lds, s, A);
    return hipGetLastError();
}

}  // namespace

hipError_t m6w_launch(int wn, int nw, bool keep, const MkJob *jobs, int njobs, const MkJob *hjobs, int grid, int order,
                      hipStream_t s) {
    // over several rounds every chain needs a thread of its own
    if (nw < 1 || nw > M6W_WAVES || (!keep && nw < wn) || njobs < 1 || (!jobs && njobs > M6W_INLINE)) return hipErrorInvalidValue;
    M6wArgs A{};
    dim3 g(grid);
    if (!jobs) {
        int tiles[M6W_INLINE];   // (multiples of 8)
        for (int i = 0; i < njobs; i++) tiles[i] = (i + 1 < njobs ? hjobs[i + 1].tile0 : grid) - hjobs[i].tile0;
        const int width = grid_row_width(tiles, njobs, 8);
        int row = 0;
        for (int i = 0; i < njobs; i++)
            for (int t = 0; t < tiles[i]; t += width) {
                A.j[row] = hjobs[i];
                A.j[row++].tile0 = -t;
            }
        g = dim3(width, row);
    }
    switch (wn) {
    case 1: return launch<1>(nw, keep, jobs, njobs, A, g, order, s);
    case 2: return launch<2>(nw, keep, jobs, njobs, A, g, order, s);
    case 4: return launch<4>(nw, keep, jobs, njobs, A, g, order, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace esq
