// Activation preparation on the device: es_act_prepare (src/es_quant.c:499-512) for rows of fp32 values, fused with what
// produces them in the engine:
//   plain rows                       -> Q8_0 (quantize_q80, src/es_quant.c:489-497) and / or Q8_K (es_quantize_q8_K,
//                                       src/es_q2k.c:102-125) blocks;
//   rmsnorm (src/es_engine.c:189-194) -> the normalised row (optional) and its blocks;
//   SwiGLU of gate|up rows (dense_n / moe_n, src/es_engine.c:957-972, 913-914) -> h (optional) and its blocks.
// The reference builds these loops for baseline x86-64 (no FMA), so every product and sum rounds on its own; this file is
// built with -ffp-contract=off and spells no fused operation. Division and square root are IEEE (correctly rounded), in
// float and in double; expf follows glibc's method bit for bit (es_hip_expf.h).
#include "es_hip_common.h"
#include "es_hip_expf.h"
#include "es_hip_q8k.h"
#include "es_hip_seqsum.h"

namespace esq {
namespace {

constexpr int PER = 8;   // consecutive elements per thread

struct QuantOut {
    uint8_t *q80;   // this row's Q8_0 blocks, or null
    uint8_t *q8k;   // this row's Q8_K blocks, or null
};

// 16 bytes of fp32 values at their 4-byte alignment
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load_per(const float *p, float (&v)[PER]) {
    const f32x4_a4 a = *reinterpret_cast<const f32x4_a4 *>(p), b = *reinterpret_cast<const f32x4_a4 *>(p + 4);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = a[k];
        v[4 + k] = b[k];
    }
}
__device__ __forceinline__ void store_per(float *p, const float (&v)[PER]) {
    *reinterpret_cast<f32x4_a4 *>(p) = f32x4_a4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4_a4 *>(p + 4) = f32x4_a4{v[4], v[5], v[6], v[7]};
}

// Eight consecutive elements e .. e + 7 of a row per thread: the kernels here are bound by issuing vector instructions where
// every element forms its block's scale (three IEEE divisions each) and the workgroup synchronises per block: SwiGLU of
// 512 x 8192 took 19.0 us that way, 9.9 us in this form (38 MB at 3.9 TB/s), plain rows of 512 x 2048 6.0 and 4.3 us.
// e is a multiple of 8: four lanes hold a Q8_0 block, 32 lanes a
// Q8_K block, so a block's scale is formed once per eight elements, its maximum and sums are lane moves and nothing
// synchronises the workgroup. Lanes without elements (have false) are whole blocks; they take part in the lane moves.
__device__ __forceinline__ void quant_per(const float (&v)[PER], bool have, int e, const QuantOut &o) {
    const float a = amax_quad(v);
    if (o.q80 && have) {   // quantize_q80: d = amax / 127, id = 1 / d (0 when d is 0), q = (int)(v * id +- 0.5)
        const float d = a / 127.0f, id = d != 0.0f ? 1.0f / d : 0.0f;
        int q[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const float x = v[k] * id;
            q[k] = static_cast<int>(x < 0.0f ? x - 0.5f : x + 0.5f);
        }
        uint8_t *blk = o.q80 + (size_t)(e >> 5) * 36;
        *reinterpret_cast<uint32_t *>(blk + 4 + (e & 31)) = pack_i8(q[0], q[1], q[2], q[3]);
        *reinterpret_cast<uint32_t *>(blk + 8 + (e & 31)) = pack_i8(q[4], q[5], q[6], q[7]);
        if ((e & 31) == 0) *reinterpret_cast<float *>(blk) = d;
    }
    if (o.q8k) {
        float d;
        uint32_t lo, hi;
        int bsum;
        q8k_from8(v, a, d, lo, hi, bsum);
        if (have) {
            const int i = e & 255;
            uint8_t *blk = o.q8k + (size_t)(e >> 8) * 292;
            *reinterpret_cast<uint32_t *>(blk + 4 + i) = lo;
            *reinterpret_cast<uint32_t *>(blk + 8 + i) = hi;
            if ((i & 15) == 0) reinterpret_cast<int16_t *>(blk + 260)[i >> 4] = static_cast<int16_t>(bsum);
            if (i == 0) *reinterpret_cast<float *>(blk) = d;
        }
    }
}

// Rows of fp32 values: one thread per 8 elements, the rows' threads one after another (a row is a whole number of blocks,
// so no block's lanes straddle two rows' threads: 4 lanes per 32 elements, 32 per 256).
__global__ __launch_bounds__(256) void act_prep_plain(const float *__restrict__ x, uint64_t xs, int per_row, long items, uint8_t *q80,
                                                      uint64_t q80s, uint8_t *q8k, uint64_t q8ks) {
    const long it = (long)blockIdx.x * 256 + threadIdx.x;
    const bool have = it < items;
    const long r = have ? it / per_row : 0;
    const int e = have ? (int)(it - r * per_row) * PER : 0;
    float v[PER] = {};
    if (have) load_per(x + r * xs + e, v);
    quant_per(v, have, e, QuantOut{q80 ? q80 + r * q80s : nullptr, q8k ? q8k + r * q8ks : nullptr});
}

// SwiGLU of gate|up rows (gate at gu[r][0, ff), up at gu[r][ff, 2 ff)), the threads as in act_prep_plain.
__global__ __launch_bounds__(256) void act_prep_swiglu(const float *__restrict__ gu, uint64_t gs, int per_row, long items, int ff, float *h,
                                                       uint64_t hs, uint8_t *q80, uint64_t q80s, uint8_t *q8k, uint64_t q8ks) {
    __shared__ uint64_t tab[32];   // expf's table in LDS: its load goes out beside the row's
    {
        static constexpr uint64_t T[32] = ESQ_EXPF_TABLE;
        if (threadIdx.x < 32) tab[threadIdx.x] = T[threadIdx.x];
    }
    const long it = (long)blockIdx.x * 256 + threadIdx.x;
    const bool have = it < items;
    const long r = have ? it / per_row : 0;
    const int e = have ? (int)(it - r * per_row) * PER : 0;
    float v[PER] = {}, u[PER] = {};
    if (have) {
        load_per(gu + r * gs + e, v);
        load_per(gu + r * gs + ff + e, u);
    }
    lds_sync();
    if (have) {
#pragma unroll
        for (int k = 0; k < PER; k++) v[k] = v[k] / (1.0f + esq_expf_tab(-v[k], tab)) * u[k];
        if (h) store_per(h + r * hs + e, v);
    }
    quant_per(v, have, e, QuantOut{q80 ? q80 + r * q80s : nullptr, q8k ? q8k + r * q8ks : nullptr});
}

// ---- rmsnorm ----
// lanes shifted or broadcast as in an inclusive wave scan (row_shr 1, 2, 4, 8, row_bcast:15 into rows 1 and 3, row_bcast:31
// into rows 2 and 3); lanes that receive nothing get 0
template <int CTRL, int ROW_MASK> __device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, CTRL < 0x140);
}
template <int CTRL, int ROW_MASK> __device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)dpp_u32<CTRL, ROW_MASK>((uint32_t)b) |
                                          (uint64_t)dpp_u32<CTRL, ROW_MASK>((uint32_t)(b >> 32)) << 32);
}
template <int CTRL, int ROW_MASK> __device__ __forceinline__ void scan_add(double &v) { v = v + dpp_f64<CTRL, ROW_MASK>(v); }
// one step of the ordered scan of runs: the earlier lanes' composite joins this lane's unless an event lies in between
// (bit 2 of e: an event at this lane or since)
template <int CTRL, int ROW_MASK> __device__ __forceinline__ void scan_run(SeqRun &r) {
    const SeqRun x{dpp_f64<CTRL, ROW_MASK>(r.a0), dpp_f64<CTRL, ROW_MASK>(r.a1), dpp_u32<CTRL, ROW_MASK>(r.e)};
    const SeqRun j = seq_join(x, r);
    if (!(r.e & 4u)) r = SeqRun{j.a0, j.a1, j.e | (x.e & 4u)};
}

// what an event needs of the lanes before it and of its own terms
struct SumEvent {
    double a0, a1;       // the run of its wave's lanes since the previous event
    uint32_t e, binade;
    double q[PER];
};
constexpr int RMS_WAVES = 16;   // waves per workgroup at most: 8192 elements at once

// rmsnorm, then the blocks: one workgroup per row, 8 consecutive elements per thread, NCH passes of blockDim * 8 elements
// (the row stays in registers). The sum of squares is the reference's in-order one, evaluated in parallel (es_hip_seqsum.h):
// one thread adding a row's squares in order is a chain of dependent fp64 additions of about 10 ns each, which was the
// whole kernel (2048 columns: 21.6 us for one row, 27.8 us for 512); now the chain has 8 additions per doubling of the sum
// (back to back in a graph 5.1 and 6.9 us).
template <int NCH>
__global__ __launch_bounds__(RMS_WAVES * 64) void act_prep_rms(const float *__restrict__ x, uint64_t xs, const float *__restrict__ w,
                                                               float eps, int cols, float *xn, uint64_t xns, uint8_t *q80,
                                                               uint64_t q80s, uint8_t *q8k, uint64_t q8ks) {
    extern __shared__ __align__(16) SumEvent ev[];   // [wave][64]
    __shared__ double wtot[RMS_WAVES];
    __shared__ SumEvent tail[RMS_WAVES];             // each wave's run after its last event
    __shared__ int nev[RMS_WAVES];
    __shared__ double s_sum;
    __shared__ int s_ok;
    const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
    const float *xr = x + (size_t)r * xs;
    float v[NCH][PER], wt[NCH][PER];
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        const int e = (c * (int)blockDim.x + tid) * PER;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            v[c][k] = 0.0f;
            wt[c][k] = 1.0f;
        }
        if (e < cols) {
            load_per(xr + e, v[c]);
            if (w) load_per(w + e, wt[c]);   // (beside the row's: its latency would otherwise follow the sum's)
        }
    }
    double sum = 0.0;   // exact: the in-order sum of everything before this pass
    bool ok = true;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        double q[PER];
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const double d = static_cast<double>(v[c][k]);
            q[k] = d * d;   // exact: a float's square fits a double
            t = t + q[k];
        }
        double incl = t;   // the approximate prefix sums, only to find the binades
        scan_add<0x111, 0xF>(incl);
        scan_add<0x112, 0xF>(incl);
        scan_add<0x114, 0xF>(incl);
        scan_add<0x118, 0xF>(incl);
        scan_add<0x142, 0xA>(incl);
        scan_add<0x143, 0xC>(incl);
        if (lane == 63) wtot[wv] = incl;
        const double before = __shfl_up(incl, 1);
        lds_sync();
        double base = sum;
        double pre[4];   // (the first ones read together)
#pragma unroll
        for (int i = 0; i < 4; i++) pre[i] = wtot[min(i, nw - 1)];
#pragma unroll
        for (int i = 0; i < 4; i++) base = i < wv ? base + pre[i] : base;
        for (int i = 4; i < wv; i++) base = base + wtot[i];
        const double from = lane == 0 ? base : base + before, to = base + incl;
        const bool event = !seq_is_run(from, to);
        SeqRun run = event ? SeqRun{0.0, 0.0, 4u} : seq_run(q, seq_binade(from));
        scan_run<0x111, 0xF>(run);
        scan_run<0x112, 0xF>(run);
        scan_run<0x114, 0xF>(run);
        scan_run<0x118, 0xF>(run);
        scan_run<0x142, 0xA>(run);
        scan_run<0x143, 0xC>(run);
        const double p0 = __shfl_up(run.a0, 1), p1 = __shfl_up(run.a1, 1);
        const uint32_t pe = (uint32_t)__shfl_up((int)run.e, 1);
        const uint64_t events = __ballot(event);
        if (event) {
            SumEvent E;
            const bool some = lane > 0 && !(events >> (lane - 1) & 1u);   // the lane before is part of a run
            E.a0 = some ? p0 : 0.0;
            E.a1 = some ? p1 : 0.0;
            E.e = some ? pe : 0u;
            E.binade = some ? seq_binade(from) : 0x800u;
#pragma unroll
            for (int k = 0; k < PER; k++) E.q[k] = q[k];
            ev[wv * 64 + __popcll(events & ((1ull << lane) - 1))] = E;
        }
        if (lane == 63) {
            SumEvent &E = tail[wv];
            E.a0 = run.a0;
            E.a1 = run.a1;
            E.e = run.e;
            E.binade = event ? 0x800u : seq_binade(from);
            nev[wv] = __popcll(events);
        }
        lds_sync();
        if (wv == 0) {   // the exact sum through the runs and events in order, the same on every lane; 0x800: no run
            for (int i = 0; i < nw; i++) {
                const int n = nev[i];
                SumEvent next = ev[i * 64];   // (one record ahead: its reads overlap this one's additions)
                for (int k = 0; k < n; k++) {
                    const SumEvent E = next;
                    next = ev[i * 64 + min(k + 1, 63)];
                    if (E.binade != 0x800u) sum = seq_add_run(sum, SeqRun{E.a0, E.a1, E.e}, E.binade, ok);
#pragma unroll
                    for (int m = 0; m < PER; m++) sum = sum + E.q[m];
                }
                const SumEvent &E = tail[i];
                if (E.binade != 0x800u) sum = seq_add_run(sum, SeqRun{E.a0, E.a1, E.e}, E.binade, ok);
            }
            if (lane == 0) {
                s_sum = sum;
                s_ok = ok;
            }
        }
        lds_sync();
        sum = s_sum;
        ok = s_ok;
    }
    // A binade was misjudged (uniform over the workgroup): in order, one wave, from LDS, two batches of 16 in turn (2048 columns
    // 21 us; each thread for itself from memory 85 us). Out of line: in line, the other rows took 0.7% longer.
    if (__builtin_expect(!ok, 0)) {
        static_assert(sizeof(SumEvent) >= NCH * PER * sizeof(float), "the row fits where the events were");
        float *const row = reinterpret_cast<float *>(ev);
#pragma unroll
        for (int c = 0; c < NCH; c++) {
            const int e = (c * (int)blockDim.x + tid) * PER;
            if (e < cols) {
                *reinterpret_cast<float4 *>(row + e) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
                *reinterpret_cast<float4 *>(row + e + 4) = make_float4(v[c][4], v[c][5], v[c][6], v[c][7]);
            }
        }
        lds_sync();
        if (wv == 0) {
            const float4 *const r4 = reinterpret_cast<const float4 *>(row);
            float4 a[4], b[4];
            auto fetch = [&](int e, float4 (&f)[4]) {   // (past the row's end its last ones again)
#pragma unroll
                for (int k = 0; k < 4; k++) f[k] = r4[min(e, cols - 16) / 4 + k];
            };
            auto add = [&](const float4 (&f)[4]) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float q[4] = {f[k].x, f[k].y, f[k].z, f[k].w};
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const double d = static_cast<double>(q[m]);
                        sum = sum + d * d;
                    }
                }
            };
            sum = 0.0;
            fetch(0, a);
            for (int e = 0; e < cols; e += 32) {   // cols is a multiple of 32
                fetch(e + 16, b);
                add(a);
                fetch(e + 32, a);
                add(b);
            }
            if (lane == 0) s_sum = sum;
        }
        lds_sync();
        sum = s_sum;
    }
    const float s = static_cast<float>(1.0 / __builtin_sqrt(sum / static_cast<double>(cols) + static_cast<double>(eps)));
    const QuantOut o{q80 ? q80 + (size_t)r * q80s : nullptr, q8k ? q8k + (size_t)r * q8ks : nullptr};
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        const int e = (c * (int)blockDim.x + tid) * PER;
        const bool have = e < cols;
        if (have) {
#pragma unroll
            for (int k = 0; k < PER; k++) v[c][k] = v[c][k] * s * wt[c][k];
            if (xn) store_per(xn + (size_t)r * xns + e, v[c]);
        }
        quant_per(v[c], have, have ? e : 0, o);
    }
}

}  // namespace

hipError_t act_prep_launch(const float *x, uint64_t xs, int rows, int cols, uint8_t *q80, uint64_t q80s, uint8_t *q8k,
                           uint64_t q8ks, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const long items = (long)rows * (cols / PER);
    hipLaunchKernelGGL(act_prep_plain, dim3((uint32_t)((items + 255) / 256)), dim3(256), 0, s, x, xs, cols / PER, items, q80, q80s, q8k, q8ks);
    return hipGetLastError();
}

hipError_t act_prep_swiglu_launch(const float *gu, uint64_t gs, int rows, int ff, float *h, uint64_t hs, uint8_t *q80,
                                  uint64_t q80s, uint8_t *q8k, uint64_t q8ks, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const long items = (long)rows * (ff / PER);
    hipLaunchKernelGGL(act_prep_swiglu, dim3((uint32_t)((items + 255) / 256)), dim3(256), 0, s, gu, gs, ff / PER, items, ff, h, hs, q80, q80s,
                       q8k, q8ks);
    return hipGetLastError();
}

hipError_t act_prep_rms_launch(const float *x, uint64_t xs, const float *w, float eps, int rows, int cols, float *xn,
                               uint64_t xns, uint8_t *q80, uint64_t q80s, uint8_t *q8k, uint64_t q8ks, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    // one wave per 512 elements, up to 16 waves; longer rows take two passes
    const int waves = cols > RMS_WAVES * 64 * PER ? RMS_WAVES : (cols + 64 * PER - 1) / (64 * PER);
    static_assert(ACT_RMS_MAX_COLS <= 2 * RMS_WAVES * 64 * PER, "at most two passes");
    const auto kern = cols > RMS_WAVES * 64 * PER ? act_prep_rms<2> : act_prep_rms<1>;
    const size_t lds = (size_t)waves * 64 * sizeof(SumEvent);
    if (lds > 60 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(lds));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(rows), dim3(waves * 64), lds, s, x, xs, w, eps, cols, xn, xns, q80, q80s, q8k, q8ks);
    return hipGetLastError();
}

}  // namespace esq
