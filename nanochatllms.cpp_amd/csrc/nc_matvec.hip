// nc_matvec.hip -- decode/prefill matrix-vector products for gfx950.
//
// Replaces matmul_2d_impl + vec_dot_product_{q8,q8_q4,f16} (gten/ops.cpp:
// 208-242, 292-490, 579-614).  The reference's AVX dot products fix a
// summation order that these kernels keep exactly:
//   Q8/Q4: per 32-value block i, four int32 lane sums L_k(i) over the
//          elements j with (j mod 8) in {2k, 2k+1}; t_k(i) = float(L_k) *
//          (d_x * d_w); acc_k = ((0 + t_k(0)) + t_k(1)) + ... in block order;
//          result (acc_0 + acc_1) + (acc_2 + acc_3).
//   F16:   eight fp32 lanes (lane = index mod 8), acc_j = x*w + acc_j over
//          the 8-wide chunks in order, result f0 + f1 + ... + f7 left to right.
//
// Q8/Q4 kernel: a 256-thread workgroup owns R weight rows.  Every thread
// loads whole weight blocks (16 B of Q4 codes or 32 B of Q8 codes, lane-
// permuted at upload so each lane's 8 codes sit in one or two dwords),
// computes the four exact integer lane sums with v_dot4 and the four fp32
// terms, and parks the terms in LDS; then 4R threads each fold one
// (row, lane) chain in block order.  Loads and integer work are spread over
// every block of the workgroup's rows; only the cheap fp32 fold is serial.
// The activation row is staged once per workgroup in LDS with the lane
// permutation, its per-lane code sums (for the Q4 "-7" offset) and delta.
// Weights are held in registers across activation rows, so prefill reads
// every weight once per launch.
//
// F16 kernels: several rows on the matrix cores (k_mfma_f16); one row with
// thread = (row, lane j): each thread reads 16-byte runs of its own lane (the
// weight layout interleaves 64-column groups over 8-row groups, so a
// wavefront reads 1 KiB contiguous) and folds its chain in order; the eight
// lanes of a row meet through wavefront shuffles.
#include <hip/hip_ext.h>

#include <cstdio>
#include <type_traits>

#include "nc_kernels.h"
#include "nc_qdot.h"
#include "nc_seqsum.h"

namespace nc {

constexpr int kMvThreads = 256;
constexpr int kMvMaxItems = 4;  // weight blocks per thread held in registers

template <int WT, int R>
__global__ __launch_bounds__(kMvThreads) void k_matvec_q(const uint8_t* __restrict__ x, int x_pitch, int n_xrows,
                                                        const uint32_t* __restrict__ wq,
                                                        const uint16_t* __restrict__ wd, float* __restrict__ out,
                                                        int out_pitch, int N, int nb)
{
    constexpr int WD = WT == Q4 ? 4 : 8;  // code dwords per block
    extern __shared__ __align__(16) uint32_t lds[];
    uint32_t* xs = lds;
    const int tp = ((nb + 3) & ~3) + 4;
    float* T = reinterpret_cast<float*>(lds + nb * kStage);
    const int tid = threadIdx.x;
    const int row0 = blockIdx.x * R;
    const int nitems = R * nb;

    // the first activation row's block is requested first, then every weight
    // load of this thread (unconditionally, at a clamped index), so both
    // latencies overlap; x is consumed first
    XRaw x0{};
    if (tid < nb) x0 = load_x_block(x, nb, tid);
    uint4 w[kMvMaxItems][WD / 4];
    uint16_t dw16[kMvMaxItems];
    int tix[kMvMaxItems], bix[kMvMaxItems];
#pragma unroll
    for (int it = 0; it < kMvMaxItems; it++) {
        const int j = tid + it * kMvThreads;
        const int r = j / nb, i = j - r * nb;
        const bool ok = j < nitems && row0 + r < N;
        tix[it] = ok ? r * 4 * tp + i : -1;
        bix[it] = i;
        const size_t b = ok ? (size_t)(row0 + r) * nb + i : 0;
        const uint4* src = reinterpret_cast<const uint4*>(wq + b * WD);
#pragma unroll
        for (int v = 0; v < WD / 4; v++) w[it][v] = load_stream(src + v);
        dw16[it] = load_stream(wd + b);
    }
    for (int p = 0; p < n_xrows; p++) {
        const uint8_t* xr = x + (size_t)p * x_pitch;
        if (tid < nb) stage_x_block(p == 0 ? x0 : load_x_block(xr, nb, tid), xs + tid * kStage);
        __syncthreads();
#pragma unroll
        for (int it = 0; it < kMvMaxItems; it++) {
            if (tix[it] < 0) continue;
            float tv[4];
            q_block_terms<WT>(xs + bix[it] * kStage, w[it], dw16[it], tv);
            float* t = T + tix[it];
#pragma unroll
            for (int k = 0; k < 4; k++) t[k * tp] = tv[k];
        }
        __syncthreads();
        if (tid < kWave) {
            float acc = 0.0f;
            if (tid < 4 * R) acc = seq_sum<16>(T + tid * tp, nb);
            const int g = tid & ~3;
            const float a0 = __shfl(acc, g), a1 = __shfl(acc, g + 1), a2 = __shfl(acc, g + 2), a3 = __shfl(acc, g + 3);
            const float res = (a0 + a1) + (a2 + a3);
            const int row = row0 + (tid >> 2);
            if (tid < 4 * R && (tid & 3) == 0 && row < N) out[(size_t)p * out_pitch + row] = res;
        }
        __syncthreads();
    }
}

// One to seven activation rows times a Q4 / Q8 weight, stored as Q8 rows by
// the launch itself (k_matvec_q and write_rows in one): a workgroup owns the
// 32 columns of one output block.  512 or 960 threads hold its weight blocks in
// registers and park the lane terms in LDS; one more wavefront folds the
// chains and quantizes the block.
//
// What bounds it: latency.  One row (MULTI false): load, terms, one fold of
// nb dependent adds (two chains per lane, 128 in all), the quantize.  More
// rows (MULTI): the columns go in two halves of 16, each with a term buffer
// of its own, and in phase t = 2 p + half the terms of t are computed while
// that wavefront folds those of t - 1, one barrier per phase; the next
// row is staged in the phase before it is used.
// Measured with the fp32 pass it replaces (us): 1 row x 5632 x 2048 Q4 7.8 ->
// 4.3; 5 rows x 5760 x 2304 Q8 20.8 -> 12.4 (the terms' reads of the staged
// rows, 64 bytes of LDS per lane and block, set the pace there).
constexpr int kMaNarrow = 512, kMaWide = 960;  // term threads

template <int WT, int IH, bool MULTI, int kMaTerm>
__global__ __launch_bounds__(kMaTerm + kWave) void k_matvec_qa(const uint8_t* __restrict__ x, int x_pitch, int n_xrows,
                                                          const uint32_t* __restrict__ wq,
                                                          const uint16_t* __restrict__ wd, uint8_t* __restrict__ out,
                                                          int out_pitch, int N, int nb)
{
    constexpr int WD = WT == Q4 ? 4 : 8;
    extern __shared__ __align__(16) uint32_t lds[];
    const int tp = ((nb + 3) & ~3) + 4;
    const int xstride = nb * kStage;                                     // staged rows: MULTI two, else one
    float* T = reinterpret_cast<float*>(lds + (MULTI ? 2 : 1) * xstride);  // [half][64 chains][tp]
    const int tid = threadIdx.x;
    const int col0 = blockIdx.x * 32;

    if (tid < kMaTerm) {
        // the first row's block, then every weight block of this thread
        const bool stager = tid < nb;
        XRaw xr{};
        if (stager) xr = load_x_block(x, nb, tid);
        uint4 w[2][IH][WD / 4];
        uint16_t dw16[2][IH];
        int tix[IH], bix[IH];
#pragma unroll
        for (int it = 0; it < IH; it++) {
            const int j = tid + it * kMaTerm;
            const int r = j / nb, i = j - r * nb;
            tix[it] = j < 16 * nb ? r * 4 * tp + i : -1;
            bix[it] = i;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // columns past N (and items past the half) read a valid block
                const int c = min(col0 + 16 * h + min(r, 15), N - 1);
                const size_t b = (size_t)c * nb + i;
                const uint4* src = reinterpret_cast<const uint4*>(wq + b * WD);
#pragma unroll
                for (int v = 0; v < WD / 4; v++) w[h][it][v] = load_stream(src + v);
                dw16[h][it] = load_stream(wd + b);
            }
        }
        auto terms = [&](int h, const uint32_t* xs) {
#pragma unroll
            for (int it = 0; it < IH; it++) {
                // the codes are unpacked here, not once for all rows (which
                // would hold twice the registers)
#pragma unroll
                for (int v = 0; v < WD / 4; v++)
                    asm volatile("" : "+v"(w[h][it][v].x), "+v"(w[h][it][v].y), "+v"(w[h][it][v].z), "+v"(w[h][it][v].w));
                if (tix[it] < 0) continue;
                float tv[4];
                q_block_terms<WT>(xs + bix[it] * kStage, w[h][it], dw16[h][it], tv);
                float* t = T + h * 64 * tp + tix[it];
#pragma unroll
                for (int k = 0; k < 4; k++) t[k * tp] = tv[k];
            }
        };
        if (stager) stage_x_block(xr, lds + tid * kStage);
        lds_barrier();
        if constexpr (!MULTI) {
            terms(0, lds);
            terms(1, lds);
            lds_barrier();
        } else {
            for (int p = 0; p < n_xrows; p++) {
                const uint32_t* xs = lds + (p & 1) * xstride;
                const bool more = p + 1 < n_xrows;
                if (more && stager) xr = load_x_block(x + (size_t)(p + 1) * x_pitch, nb, tid);
                terms(0, xs);
                lds_barrier();  // phase 2 p
                terms(1, xs);
                if (more && stager) stage_x_block(xr, lds + ((p + 1) & 1) * xstride + tid * kStage);
                lds_barrier();  // phase 2 p + 1
            }
        }
        return;
    }

    // the fold wavefront: lane = chain (column lane >> 2 of a half, AVX lane
    // lane & 3)
    const int lane = tid & (kWave - 1);
    auto column = [&](float acc) {
        const int g = lane & ~3;
        const float a0 = __shfl(acc, g), a1 = __shfl(acc, g + 1), a2 = __shfl(acc, g + 2), a3 = __shfl(acc, g + 3);
        return (a0 + a1) + (a2 + a3);
    };
    auto store = [&](int p, float va, float vb) {
        // q8_quant_lane over the block's 32 columns (each on four lanes)
        const int ca = col0 + (lane >> 2), cb = ca + 16;
        float a = fmaxf(ca < N ? fabsf(va) : 0.0f, cb < N ? fabsf(vb) : 0.0f);
        a = half_wave_max(a);
        a = fmaxf(a, __shfl_xor(a, 32));
        const float delta = a / 127.0f;
        const float scale = delta != 0.0f ? 1.0f / delta : 0.0f;
        uint8_t* o = out + (size_t)p * out_pitch;
        if ((lane & 3) == 0) {
            if (ca < N) o[ca] = (uint8_t)(int8_t)roundf(va * scale);
            if (cb < N) o[cb] = (uint8_t)(int8_t)roundf(vb * scale);
        }
        if (lane == 0) reinterpret_cast<uint16_t*>(o + act_delta_offset(N))[col0 >> 5] = f2h(delta);
    };
    lds_barrier();  // the first row's staging
    if constexpr (!MULTI) {
        lds_barrier();  // the terms
        const float *ta = T + lane * tp, *tb = ta + 64 * tp;
        float sa = 0.0f, sb = 0.0f;
        int c = 0;
        for (; c + 16 <= nb; c += 16) {
            float4 a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                a[q] = reinterpret_cast<const float4*>(ta + c)[q];
                b[q] = reinterpret_cast<const float4*>(tb + c)[q];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                sa = sa + a[q].x;
                sb = sb + b[q].x;
                sa = sa + a[q].y;
                sb = sb + b[q].y;
                sa = sa + a[q].z;
                sb = sb + b[q].z;
                sa = sa + a[q].w;
                sb = sb + b[q].w;
            }
        }
        for (; c < nb; c++) {
            sa = sa + ta[c];
            sb = sb + tb[c];
        }
        const float va = column(sa), vb = column(sb);
        store(0, va, vb);
    } else {
        for (int p = 0; p < n_xrows; p++) {
            lds_barrier();  // phase 2 p: half 0's terms are there
            const float va = column(seq_sum<16>(T + lane * tp, nb));
            lds_barrier();  // phase 2 p + 1: half 1's
            const float vb = column(seq_sum<16>(T + (64 + lane) * tp, nb));
            store(p, va, vb);
        }
    }
}

static size_t matvec_qa_lds(int nb, bool multi)
{
    const int tp = ((nb + 3) & ~3) + 4;
    return ((size_t)(multi ? 2 : 1) * nb * kStage + (size_t)128 * tp) * 4;
}

// The k_matvec_qa launch of a product: its term threads and their weight blocks
// per half; items 0 where k_matvec_q and a pass that quantizes its fp32 rows
// (k_write_rows) take less time, or k_matvec_qa cannot hold the blocks.
struct QaShape {
    int term, items;
};

// The lines, measured back to back with cold weights on MI355X (us, staged /
// direct):
//  * k_matvec_q runs 1024 workgroups of four columns at once, so past 4096
//    columns its time steps up by half and k_matvec_qa wins at any row count:
//    7 rows x 4096 x 4096 Q4 17.4 / 17.3, x 5632 25.8 / 17.7; 7 x 5632 x 5632 Q8
//    33.3 / 28.0.
//  * up to there k_matvec_qa leaves CUs idle (a workgroup per 32 columns, its
//    rows in turn), for a time that grows with the rows, the blocks of the
//    fold's chain and the blocks per thread: the fewest columns it wins at are
//    linear in work = rows nb^2.  Q4: 4 rows x 2048 x 4096 11.3 / 11.2, 5 rows 12.7 /
//    13.1; 1 x 768 x 5632 6.6 / 6.6, 256 columns 5.9 / 6.4.  Q8 blocks take twice
//    the registers and LDS reads, so its lines lie higher, the more so past two
//    blocks per thread: 3 x 768 x 2048 7.6 / 7.5, 4 rows 8.6 / 8.7; 1 x 1024 x 2304
//    5.9 / 6.2, 2 x 2048 x 2304 7.9 / 7.8; and past three only tall weights win
//    (1 x 2048 x 3584 7.0 / 7.8), as Q4's past 180 blocks (1 x 2048 x 7680 8.0 / 8.3).
//  * 960 threads instead of 512 pay past five blocks per thread (1 x 2048 x
//    5632 Q4 7.6 with 512, 6.9 with 960; 1 x 2048 x 4096 5.5 / 6.0): below, the
//    extra wavefronts only wait for the fold.  Q8 past 180 blocks would spill
//    (2 x 2048 x 7680: 32 with five blocks per thread, 17.6 with four, staged 11.4).
static QaShape qa_shape(int n_rows, const nc_tensor* w)
{
    const int N = w->rows, nb = w->cols / 32;
    const bool q4 = w->dtype == NC_Q4;
    if ((!q4 && w->dtype != NC_Q8) || w->cols <= 0 || w->cols % 32 || N <= 0 || n_rows < 1 || n_rows >= kGemmMinRows)
        return {0, 0};
    if (nb > (q4 ? 256 : 180) || matvec_qa_lds(nb, n_rows > 1) > 160 * 1024) return {0, 0};
    if (N <= 4096) {
        const int work = n_rows * nb * nb;
        const bool wins = q4         ? nb <= 180 && 22 * N >= work - 20000
                          : nb <= 64 ? 8 * N >= work - 6000
                                     : nb <= 96 && 16 * (N - 1400) >= work;
        if (!wins) return {0, 0};
    }
    const int term = nb > 160 ? kMaWide : kMaNarrow;
    return {term, (16 * nb + term - 1) / term};
}

static int matvec_qa(const uint8_t* x, int x_pitch, int n_rows, const nc_tensor* w, uint8_t* out, int out_pitch,
                     hipStream_t st)
{
    const int N = w->rows, nb = w->cols / 32;
    const QaShape shape = qa_shape(n_rows, w);
    const dim3 grid((N + 31) / 32);
    auto go = [&](auto kern, bool multi, int term) {
        const size_t lds = matvec_qa_lds(nb, multi);
        hipLaunchKernelGGL(kern, grid, dim3(term + kWave), lds, st, x, x_pitch, n_rows, (const uint32_t*)w->data,
                           (const uint16_t*)w->deltas, out, out_pitch, N, nb);
        return launch_status("k_matvec_qa");
    };
    auto by_items = [&](auto wt, auto multi) {
        constexpr int WT = decltype(wt)::value;
        constexpr bool M = decltype(multi)::value;
        if (shape.term == kMaWide) {
            if (shape.items == 3) return go(k_matvec_qa<WT, 3, M, kMaWide>, M, kMaWide);
            if constexpr (WT == Q4) {
                if (shape.items == 4) return go(k_matvec_qa<WT, 4, M, kMaWide>, M, kMaWide);
                if constexpr (!M)  // several rows' shared memory ends at four
                    if (shape.items == 5) return go(k_matvec_qa<WT, 5, M, kMaWide>, M, kMaWide);
            }
        } else {
            switch (shape.items) {
            case 1: return go(k_matvec_qa<WT, 1, M, kMaNarrow>, M, kMaNarrow);
            case 2: return go(k_matvec_qa<WT, 2, M, kMaNarrow>, M, kMaNarrow);
            case 3: return go(k_matvec_qa<WT, 3, M, kMaNarrow>, M, kMaNarrow);
            case 4: return go(k_matvec_qa<WT, 4, M, kMaNarrow>, M, kMaNarrow);
            case 5: return go(k_matvec_qa<WT, 5, M, kMaNarrow>, M, kMaNarrow);
            }
        }
        return fail(NC_ERR_ARG, "matvec to Q8 rows: [%d x %d] weights, %d rows", N, w->cols, n_rows);
    };
    auto by_rows = [&](auto wt) {
        return n_rows > 1 ? by_items(wt, std::true_type{}) : by_items(wt, std::false_type{});
    };
    return w->dtype == NC_Q4 ? by_rows(std::integral_constant<int, Q4>{}) : by_rows(std::integral_constant<int, Q8>{});
}

// F16, prefill, on the matrix cores.  v_mfma_f32_16x16x1_4b_f32 multiplies
// four independent pairs of 16-vectors (one K step each) and adds them to
// four 16 x 16 fp32 accumulators: one fused multiply-add per entry, which on
// exact fp16 products is the reference's multiply then add.  So its four
// blocks hold four lane chains j of a 16 x 16 tile (rows of x times rows of
// w), two of them (j = 0..3, 4..7) all eight, and the K steps m of the
// 64-column groups run in the reference's order; the eight chains of an
// output end up in one thread, which sums them left to right.
//
// What bounds it: the matrix cores' fp32 rate, 128 multiply-adds per clock
// and CU (134 TFLOP/s measured with nothing else in the loop), twice the
// vector unit's without packed math; for few tiles, the chain of K steps one
// wavefront runs (32 cycles each and half).  x is staged widened to fp32 in
// the operand order [group][lane j][m / 4][row]; the weights come straight
// from their layout, one 16-byte load per lane giving eight K steps, and are
// widened beside the products.
// Measured (us, cold caches; before: register-tiled vector kernel):
//   1500 rows x 2048 x 2048     259 -> 134 (94 TFLOP/s)
//   128 rows x 11264 x 2048     126 -> 67, 5632 x 2048 72 -> 39
//   64 rows x 2560 x 2048       32 -> 17, 2048 x 5632 73 -> 39
//   2 rows x 5632 x 2048        21 -> 16 (before: one row at a time)
//
// RN row tiles and CN column tiles of 16 per wavefront (four wavefronts side
// by side in columns); GC groups staged at a time, PF (GC or GC / 2) groups
// of weights in flight; ODT F32 or F16 rows out (out_pitch in floats or
// bytes).
typedef float f16x_t __attribute__((ext_vector_type(16)));

template <int RN, int CN, int GC, int PF, int ODT>
__global__ __launch_bounds__(256) void k_mfma_f16(const uint8_t* __restrict__ x, int x_pitch, int n_rows,
                                                  const uint16_t* __restrict__ w, void* __restrict__ out, int out_pitch,
                                                  int N, int K)
{
    static_assert(GC % PF == 0, "a group's weight slot is fixed");
    constexpr int kRows = 16 * RN, TPT = kRows * GC * 4 / 256;
    static_assert(kRows * GC * 4 % 256 == 0, "staging tasks spread evenly");
    __shared__ __align__(16) float4 xs[2][GC][8][2][kRows];  // [buffer][group][lane j][m / 4][row]
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lc = lane & 15, lb = lane >> 4;
    const int r0 = blockIdx.y * kRows;
    const int c0 = (blockIdx.x * 4 + wv) * 16 * CN;
    const int G = K / 64, nck = (G + GC - 1) / GC;
    const size_t gstride = (size_t)((N + 7) & ~7) * 8;  // uint4s per group
    const uint4* wcol[CN];  // lane j = lb of this thread's columns; j + 4 follows 4 uint4s on
#pragma unroll
    for (int n = 0; n < CN; n++)
        wcol[n] = reinterpret_cast<const uint4*>(w) + (size_t)min(c0 + 16 * n + lc, N - 1) * 8 + lb;

    // staging: a task is two 8-value runs m = 2p, 2p + 1 of one (row, group),
    // widened into the operand order
    uint4 xq[TPT][2];
    int t_row[TPT], t_g[TPT], t_p[TPT];
#pragma unroll
    for (int i = 0; i < TPT; i++) {
        const int t = tid + i * 256;
        t_row[i] = t % kRows;
        t_g[i] = t / kRows % GC;
        t_p[i] = t / (kRows * GC);
    }
    auto x_load = [&](int ck) {
#pragma unroll
        for (int i = 0; i < TPT; i++) {
            const int g = min(ck * GC + t_g[i], G - 1);
            const uint4* xrow = reinterpret_cast<const uint4*>(x + (size_t)min(r0 + t_row[i], n_rows - 1) * x_pitch);
            xq[i][0] = xrow[g * 8 + 2 * t_p[i]];
            xq[i][1] = xrow[g * 8 + 2 * t_p[i] + 1];
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < TPT; i++) {
            const uint32_t a[4] = {xq[i][0].x, xq[i][0].y, xq[i][0].z, xq[i][0].w};
            const uint32_t b[4] = {xq[i][1].x, xq[i][1].y, xq[i][1].z, xq[i][1].w};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t va = j & 1 ? a[j >> 1] >> 16 : a[j >> 1] & 0xFFFFu;
                const uint32_t vb = j & 1 ? b[j >> 1] >> 16 : b[j >> 1] & 0xFFFFu;
                reinterpret_cast<float2*>(&xs[buf][t_g[i]][j][t_p[i] >> 1][t_row[i]])[t_p[i] & 1] =
                    make_float2(h2f((uint16_t)va), h2f((uint16_t)vb));
            }
        }
    };
    // the weights of the next PF groups, each group's slot refilled once its
    // products are issued
    uint4 wq[PF][CN][2];
    auto w_load = [&](int g, uint4 (&q)[CN][2]) {
        const size_t o = (size_t)min(g, G - 1) * gstride;
#pragma unroll
        for (int n = 0; n < CN; n++)
#pragma unroll
            for (int h = 0; h < 2; h++) q[n][h] = wcol[n][o + 4 * h];
    };
    f16x_t acc[RN][CN][2];
#pragma unroll
    for (int r = 0; r < RN; r++)
#pragma unroll
        for (int n = 0; n < CN; n++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[r][n][h][e] = 0.0f;
    // the weight operands of two K steps in fp32, converted while the
    // products of the two before them are issued (a conversion into a
    // register that a product in flight still reads would wait for it)
    auto convert = [&](const uint4 (&q)[CN][2], int mp, float (&b)[CN][2][2]) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int n = 0; n < CN; n++) {
                const uint4& u = q[n][h];
                const uint32_t d = mp == 0 ? u.x : mp == 1 ? u.y : mp == 2 ? u.z : u.w;
                b[n][h][0] = h2f((uint16_t)(d & 0xFFFFu));
                b[n][h][1] = h2f((uint16_t)(d >> 16));
            }
    };
    auto group = [&](int buf, int gl, const uint4 (&q)[CN][2]) {
        float4 xa[RN][2][2];  // [row tile][lane half][m / 4]
#pragma unroll
        for (int mh = 0; mh < 2; mh++)
#pragma unroll
            for (int r = 0; r < RN; r++)
#pragma unroll
                for (int h = 0; h < 2; h++) xa[r][h][mh] = xs[buf][gl][4 * h + lb][mh][16 * r + lc];
        float b[2][CN][2][2];
        convert(q, 0, b[0]);
#pragma unroll
        for (int mp = 0; mp < 4; mp++) {
            if (mp < 3) convert(q, mp + 1, b[(mp + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int r = 0; r < RN; r++) {
                        const float4 v = xa[r][h][mp >> 1];
                        const float a = mp & 1 ? (t ? v.w : v.z) : (t ? v.y : v.x);
#pragma unroll
                        for (int n = 0; n < CN; n++)
                            acc[r][n][h] = __builtin_amdgcn_mfma_f32_16x16x1f32(a, b[mp & 1][n][h][t], acc[r][n][h], 0, 0, 0);
                    }
        }
    };
    x_load(0);
#pragma unroll
    for (int p = 0; p < PF; p++) w_load(p, wq[p]);
    stage(0);
    x_load(min(1, nck - 1));
    __syncthreads();
    for (int ck = 0; ck < nck; ck++) {
        const int buf = ck & 1, g0 = ck * GC;
#pragma unroll
        for (int gl = 0; gl < GC; gl++) {
            if (g0 + gl < G) group(buf, gl, wq[gl % PF]);  // uniform
            w_load(g0 + gl + PF, wq[gl % PF]);
        }
        stage(buf ^ 1);  // past the end: the last chunk again, never read
        x_load(min(ck + 2, nck - 1));
        lds_barrier();
    }
#pragma unroll
    for (int r = 0; r < RN; r++)
#pragma unroll
        for (int n = 0; n < CN; n++) {
            const int col = c0 + 16 * n + lc;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = r0 + 16 * r + 4 * lb + i;
                float s = acc[r][n][0][i];
#pragma unroll
                for (int j = 1; j < 8; j++) s = s + acc[r][n][j >> 2][(j & 3) * 4 + i];
                if (row < n_rows && col < N) {
                    if constexpr (ODT == F32) reinterpret_cast<float*>(out)[(size_t)row * out_pitch + col] = s;
                    else reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(out) + (size_t)row * out_pitch)[col] = f2h(s);
                }
            }
        }
}

// F16, one activation row (decode): a 64-thread workgroup owns 8 rows, thread
// (row, lane j) folds lane j's chain over the 64-column groups in order
// and keeps two batches of kF16Batch weight
// runs in flight (the next batch is requested before the current one is
// folded), so the fold is not serialised behind one load per group.
constexpr int kF16Batch = 16;

template <bool H16>
__global__ __launch_bounds__(64) void k_matvec_f16_row(const uint8_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                      void* __restrict__ out, int N, int K)
{
    extern __shared__ __align__(16) float xsf[];  // [K/64][8 lanes][8]
    const int tid = threadIdx.x;
    const int j = tid & 7;
    const int row = blockIdx.x * 8 + (tid >> 3);
    const int G = K / 64;
    const int npad = (N + 7) & ~7;
    const int rowc = row < N ? row : N - 1;  // rows past N read a valid row and store nothing
    const uint4* wrow = reinterpret_cast<const uint4*>(w) + (size_t)rowc * 8 + j;  // group 0
    const size_t gstride = (size_t)npad * 8;                                         // uint4s per group
    // two weight batches in flight, used in turn: batch A holds groups
    // [g0, g0 + B), batch B the next B groups; each is refilled right after
    // it is folded (no register copies, which would wait for the loads)
    uint4 wa[kF16Batch], wb[kF16Batch];
    auto load = [&](uint4(&dst)[kF16Batch], int gbase) {
#pragma unroll
        for (int b = 0; b < kF16Batch; b++) {
            const int g = gbase + b;
            dst[b] = load_stream(wrow + (size_t)(g < G ? g : 0) * gstride);
        }
    };
    // the activation row first (8 halves per load, K <= 8192), then the
    // weights, so staging the row waits for the row only
    constexpr int kXMax = 8192 / 8 / 64;
    uint4 xv8[kXMax];
#pragma unroll
    for (int i = 0; i < kXMax; i++) {
        const int c = tid + i * 64;  // 8-value chunk
        xv8[i] = c * 8 < K ? reinterpret_cast<const uint4*>(x)[c] : make_uint4(0, 0, 0, 0);
    }
    load(wa, 0);
    load(wb, kF16Batch);
#pragma unroll
    for (int i = 0; i < kXMax; i++) {
        const int c = tid + i * 64;
        if (c * 8 < K) {
            const uint32_t q[4] = {xv8[i].x, xv8[i].y, xv8[i].z, xv8[i].w};
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int e = c * 8 + t;
                const int g = e >> 6, m = (e >> 3) & 7, jj = e & 7;
                xsf[(g * 8 + jj) * 8 + m] = h2f((uint16_t)(t & 1 ? q[t >> 1] >> 16 : q[t >> 1] & 0xFFFFu));
            }
        }
    }
    __syncthreads();
    float acc = 0.0f;
    auto fold = [&](const uint4(&wv4)[kF16Batch], int gbase) {
#pragma unroll
        for (int b = 0; b < kF16Batch; b++) {
            const int g = gbase + b;
            if (g < G) {
                const float4 xa = *reinterpret_cast<const float4*>(xsf + (g * 8 + j) * 8);
                const float4 xb = *reinterpret_cast<const float4*>(xsf + (g * 8 + j) * 8 + 4);
                const uint32_t wv[4] = {wv4[b].x, wv4[b].y, wv4[b].z, wv4[b].w};
                const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const uint16_t h = (uint16_t)(m & 1 ? wv[m >> 1] >> 16 : wv[m >> 1] & 0xFFFFu);
                    acc = __builtin_fmaf(xv[m], h2f(h), acc);  // exact product: same as mul then add
                }
            }
        }
    };
    for (int g0 = 0; g0 < G; g0 += 2 * kF16Batch) {
        fold(wa, g0);
        if (g0 + 2 * kF16Batch < G) load(wa, g0 + 2 * kF16Batch);
        fold(wb, g0 + kF16Batch);
        if (g0 + 3 * kF16Batch < G) load(wb, g0 + 3 * kF16Batch);
    }
    // lanes 0..7 of the row summed left to right
    const int base = tid & ~7;
    float s = __shfl(acc, base);
#pragma unroll
    for (int l = 1; l < 8; l++) s = s + __shfl(acc, base + l);
    if (j == 0 && row < N) {
        if constexpr (H16) static_cast<uint16_t*>(out)[row] = f2h(s);
        else static_cast<float*>(out)[row] = s;
    }
}

// Fold of one wavefront's 64 lane chains (8 rows x 8 lanes, thread (row,
// lane j) folds lane j's chain over the G 64-column groups in order, as
// k_matvec_f16_row does), fully unrolled so that each fold waits for its
// own loads only.  The weights come through the ring wv of D loads per
// thread (its first D loads issued by the caller; the load for group g + D
// is issued once group g is folded); the activation row is the fp16 copy xs
// in LDS in the [G][8 lanes][8] order, read P groups ahead of its fold (the
// fp16 x fp16 products go through v_fma_mix exactly as through fp32).
template <int G, int D, int P>
__device__ __forceinline__ float dmv_f16_fold(const uint16_t* xs, uint4 (&wv)[D], const uint4* wrow, size_t gstride,
                                              int j)
{
    static_assert(D <= G && P <= G && P <= 15, "ring depths");
    const uint4* xrow = reinterpret_cast<const uint4*>(xs) + j;  // group g at xrow[g * 8]
    uint4 xr[P];
#pragma unroll
    for (int i = 0; i < P; i++) xr[i] = xrow[i * 8];
    float acc = 0.0f;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const uint4 xc = xr[g % P];
        if (g + P < G) xr[g % P] = xrow[(g + P) * 8];
        const uint4 wc = wv[g % D];
        if (g + D < G) wv[g % D] = load_stream(wrow + (size_t)(g + D) * gstride);
        const uint32_t wq[4] = {wc.x, wc.y, wc.z, wc.w}, xq[4] = {xc.x, xc.y, xc.z, xc.w};
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const float a = h2f((uint16_t)(m & 1 ? xq[m >> 1] >> 16 : xq[m >> 1] & 0xFFFFu));
            const float b = h2f((uint16_t)(m & 1 ? wq[m >> 1] >> 16 : wq[m >> 1] & 0xFFFFu));
            acc = __builtin_fmaf(a, b, acc);  // exact product: same as mul then add
        }
        // keep the ring order: this group's adds are done and the reads for
        // g + P and g + D issued here (otherwise the adds sink below every
        // read, which then hold all their registers at once)
        asm volatile("" : "+v"(acc)::"memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

// Row of wavefront quad q's lane-row sub (8 rows per wavefront): plain, rows
// 8q .. 8q+7; GLU (w a fused gate|up [2f, K] weight, N = 2f), gate rows
// 4q .. 4q+3 and up rows f+4q .. f+4q+3.
template <bool GLU>
__device__ __forceinline__ int dmv_f16_row(int q, int sub, int N)
{
    return GLU ? (sub < 4 ? 4 * q + sub : N / 2 + 4 * q + sub - 4) : 8 * q + sub;
}

// Lanes 0..7 of each row summed left to right.  Plain: the fp32 dots to
// out.  GLU: the fp16 SwiGLU values m[4q + i] = Act(Act(silu(Act(g))) *
// Act(u)) as k_silu_mul does them (tinyllama/tinyllama.cpp:88-97 in the
// fp16 dtype).
// With H16 (not GLU) the fp16 values to m_out[row].
template <bool GLU, bool H16 = false>
__device__ __forceinline__ void dmv_f16_finish(float acc, int lane, int q, int row, int N, float* out,
                                               uint16_t* m_out)
{
    const int base = lane & ~7;
    float s = __shfl(acc, base);
#pragma unroll
    for (int l = 1; l < 8; l++) s = s + __shfl(acc, base + l);
    if (!GLU) {
        if ((lane & 7) == 0 && row < N) {
            if constexpr (H16) m_out[row] = f2h(s);
            else out[row] = s;
        }
        return;
    }
    const float gsum = __shfl(s, (lane & 3) * 8), usum = __shfl(s, ((lane & 3) + 4) * 8);
    if (lane < 4 && 4 * q + lane < N / 2) {
        const float g = f16_roundtrip(gsum);
        const float gs = f16_roundtrip(g / (1.0f + expf_ref(-g)));
        const float u = f16_roundtrip(usum);
        m_out[4 * q + lane] = f2h(gs * u);
    }
}

// F16, one activation row (decode), for the group counts G = K / 64 it is
// built for: one wavefront per 8 rows (dmv_f16_fold); the row is staged
// into LDS as fp16 in the fold's order while the weight ring is in flight.
template <int G, int D, int P, bool GLU, bool H16 = false>
__global__ __launch_bounds__(64) void k_dmv_f16(const uint8_t* __restrict__ x, const uint16_t* __restrict__ w,
                                               float* __restrict__ out, int N, uint16_t* __restrict__ m_out)
{
    constexpr int K = G * 64, XC = K / 8, XPT = (XC + 63) / 64;
    __shared__ __align__(16) uint16_t xs[K];  // [G][8 lanes][8] halves
    const int lane = threadIdx.x;
    const int j = lane & 7, q = blockIdx.x;
    const int row = dmv_f16_row<GLU>(q, lane >> 3, N);
    const int rowc = row < N ? row : N - 1;  // rows past N read a valid row and store nothing
    const size_t gstride = (size_t)((N + 7) & ~7) * 8;  // uint4s per group
    const uint4* wrow = reinterpret_cast<const uint4*>(w) + (size_t)rowc * 8 + j;
    // the activation row first, then the weight ring, so staging waits for the row only
    uint4 xv[XPT];
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int c = lane + i * 64;  // 8-value chunk: group c >> 3, m = c & 7
        xv[i] = (XC % 64 == 0 || c < XC) ? reinterpret_cast<const uint4*>(x)[c] : make_uint4(0, 0, 0, 0);
    }
    uint4 wv[D];
#pragma unroll
    for (int i = 0; i < D; i++) wv[i] = load_stream(wrow + (size_t)i * gstride);
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int c = lane + i * 64;
        if (XC % 64 == 0 || c < XC) {
            const uint32_t q4[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
#pragma unroll
            for (int t = 0; t < 8; t++)
                xs[((c >> 3) * 8 + t) * 8 + (c & 7)] = (uint16_t)(t & 1 ? q4[t >> 1] >> 16 : q4[t >> 1] & 0xFFFFu);
        }
    }
    __syncthreads();
    const float acc = dmv_f16_fold<G, D, P>(xs, wv, wrow, gstride, j);
    dmv_f16_finish<GLU, H16>(acc, lane, q, row, N, out, m_out);
}

// The norm of the row fused into the fp16 decode matvec that consumes it
// (Zephyr's layer_norm, gten/ops.cpp:669-698; the fp16 Llama, MiniCPM and
// OpenELM models' rms_norm, gten/ops.cpp:830-903).  Threads 0-255 build the
// row -- ADD: the residual sum h = a + Act(Act(braw) [* bscale], Act) stored
// to h_out by workgroup 0 -- and compute the norm, synchronizing among
// themselves through an LDS counter: layer_norm's mean as the exact
// workgroup sum of the fp16 values (nc_seqsum.h), the variance (or rms_norm's
// sum of squares) as the exact workgroup sum of non-negative terms, then
// y = ((x - mean) / (sqrt(var) + 1e-5)) * w + b, or y = x / (sqrt(ss / n) +
// 1e-6) * w, rounded to fp16 into the fold's LDS order.  The other 512
// threads (8 wavefronts, 64 rows) issue their whole weight ring at once and
// fold once the row is there: a wavefront issuing a large transfer waits at
// the issue until the memory system takes it, so the norm's wavefronts hold
// no weights.  They issue the ring only once the norm's row loads have
// returned (a CU serves its loads in order, and rows queued behind the
// ring's hundreds of KB arrive microseconds late).  Under graph replay
// (dpos) the a and h_out rows sit at the device-held position.
constexpr int kNrmNorm = kSsThreads;  // norm threads
constexpr int kNrmFold = 512;         // fold threads
enum { kNrmLayer = 0, kNrmRms = 1 };

template <int G, int D, int P, int KIND, bool ADD, bool GLU>
__global__ __launch_bounds__(kNrmNorm + kNrmFold) void k_dmv_f16_nrm(
    const uint8_t* __restrict__ a, int a_pitch, const float* __restrict__ braw, float bscale, uint8_t* __restrict__ h_out,
    int h_pitch, const uint16_t* __restrict__ nw, const uint16_t* __restrict__ nb, const uint16_t* __restrict__ w,
    float* __restrict__ out, uint16_t* __restrict__ m_out, int N, const int* __restrict__ dpos)
{
    constexpr int K = G * 64, C = K / kNrmNorm;  // values per norm thread
    static_assert(K % kNrmNorm == 0 && C <= kSsMaxPer, "row width");
    __shared__ __align__(16) float buf[K];
    __shared__ __align__(16) uint16_t xs[K];
    __shared__ SgShared sgh;
    __shared__ SsShared ssh;
    __shared__ int cnt, rows_in;
    const int tid = threadIdx.x;
    if (tid == 0) {
        cnt = 0;
        rows_in = 0;
    }
    lds_barrier();
    if (tid < kNrmNorm) {
        const size_t prow = dpos ? (size_t)load_pos(dpos) : 0;
        const uint16_t* arow = reinterpret_cast<const uint16_t*>(a + prow * a_pitch);
        float x[C], g[C], bb[C];
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int e = tid * C + k;
            x[k] = h2f(arow[e]);
            g[k] = h2f(nw[e]);
            bb[k] = KIND == kNrmLayer ? h2f(nb[e]) : 0.0f;
        }
        float bw[C];
        if (ADD) {
#pragma unroll
            for (int k = 0; k < C; k++) bw[k] = braw[tid * C + k];
        }
        // every row load of this wavefront has returned: the fold's
        // wavefronts may queue their weights
        wait_loads_done();
        if ((tid & (kWave - 1)) == 0) __hip_atomic_fetch_add(&rows_in, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (ADD) {
#pragma unroll
            for (int k = 0; k < C; k++) {
                const int e = tid * C + k;
                float bv = f16_roundtrip(bw[k]);  // the Linear output as an fp16 Act
                if (bscale != 1.0f) bv = f16_roundtrip(bv * bscale);
                const float sm = x[k] + bv;
                x[k] = f16_roundtrip(sm);
                if (blockIdx.x == 0) reinterpret_cast<uint16_t*>(h_out + prow * h_pitch)[e] = f2h(sm);
            }
        }
        SsWaveBarrier<kNrmNorm / kWave> bar{&cnt, 0};
        float mean = 0.0f;
        if (KIND == kNrmLayer) {
#pragma unroll
            for (int k = 0; k < C; k++) buf[tid * C + k] = x[k];
            bar();
            mean = block_seq_sum_grid<C, kNrmNorm>(buf, sgh, nullptr, bar) / (float)K;
#pragma unroll
            for (int k = 0; k < C; k++) buf[tid * C + k] = (x[k] - mean) * (x[k] - mean);
        } else {
#pragma unroll
            for (int k = 0; k < C; k++) buf[tid * C + k] = x[k] * x[k];
        }
        bar();
        const float ss = block_seq_sum_core<C>(buf, K, ssh, nullptr, bar);
        const float denom = KIND == kNrmLayer ? sqrtf(ss / (float)K) + 1e-05f : sqrtf(ss / (float)K) + 1e-6f;
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int e = tid * C + k;
            const float y = KIND == kNrmLayer ? ((x[k] - mean) / denom) * g[k] + bb[k] : x[k] / denom * g[k];
            xs[((e >> 6) * 8 + (e & 7)) * 8 + ((e >> 3) & 7)] = f2h(y);
        }
        lds_barrier();
        return;
    }
    const int ft = tid - kNrmNorm, lane = tid & (kWave - 1);
    const int j = lane & 7, q = (int)blockIdx.x * (kNrmFold / kWave) + ft / kWave;
    const int row = dmv_f16_row<GLU>(q, lane >> 3, N);
    const int rowc = row < N ? row : N - 1;  // rows past N read a valid row and store nothing
    const size_t gstride = (size_t)((N + 7) & ~7) * 8;
    const uint4* wrow = reinterpret_cast<const uint4*>(w) + (size_t)rowc * 8 + j;
    uint4 wv[D];
    while (__hip_atomic_load(&rows_in, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < kNrmNorm / kWave)
        __builtin_amdgcn_s_sleep(2);
#pragma unroll
    for (int i = 0; i < D; i++) wv[i] = load_stream(wrow + (size_t)i * gstride);
    lds_barrier();  // the normalized row is in xs
    const float acc = dmv_f16_fold<G, D, P>(xs, wv, wrow, gstride, j);
    dmv_f16_finish<GLU>(acc, lane, q, row, N, out, m_out);
}

// The group counts k_dmv_f16 is built for (d_model and d_ffn of the fp16
// models: 2048 / 5632 and 2304 / 5760), with the ring depths measured best.
template <bool GLU, bool H16 = false, class Launch>
bool dmv_f16_dispatch(int G, Launch&& go)
{
    switch (G) {
    case 32: go(k_dmv_f16<32, 32, 8, GLU, H16>); return true;
    case 36: go(k_dmv_f16<36, 36, 8, GLU, H16>); return true;
    case 88: go(k_dmv_f16<88, 32, 8, GLU, H16>); return true;
    case 90: go(k_dmv_f16<90, 32, 8, GLU, H16>); return true;
    default: return false;
    }
}

// fp16 products: rows of whole 64-value groups, up to 16384 values.
static bool f16_shape_ok(const nc_tensor* w) { return w->cols % 64 == 0 && w->cols > 0 && w->cols <= 16384; }

// The fp16 product of several rows.  Shapes by the number of 64-column tiles
// of 16 and 32 rows (us at the shapes around the lines, in that order):
// two row tiles share each weight operand once 640 such workgroups exist
// (704: 65 against 71; 352: 45 against 39); below, one row tile, with four
// groups of weights in flight up to 384 workgroups (256: 42 against 46) and
// two beyond (528: 37 against 39, 704: 40 against 43).
template <int ODT>
static int mfma_f16(const uint8_t* x, int x_pitch, int n_rows, const nc_tensor* w, void* out, int out_pitch,
                    hipStream_t st, hipEvent_t ev_start, hipEvent_t ev_stop)
{
    const int N = w->rows, K = w->cols;
    const int tc = (N + 63) / 64, t1 = tc * ((n_rows + 15) / 16), t2 = tc * ((n_rows + 31) / 32);
    auto go = [&](auto kern, int rows) {
        const dim3 grid(tc, (n_rows + rows - 1) / rows);
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, dim3(256), 0, st, ev_start, ev_stop, 0, x, x_pitch, n_rows,
                                  (const uint16_t*)w->data, out, out_pitch, N, K);
        else
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, x, x_pitch, n_rows, (const uint16_t*)w->data, out,
                               out_pitch, N, K);
    };
    if (t2 >= 640) go(k_mfma_f16<2, 1, 2, 2, ODT>, 32);
    else if (t1 > 384) go(k_mfma_f16<1, 1, 4, 2, ODT>, 16);
    else go(k_mfma_f16<1, 1, 4, 4, ODT>, 16);
    return launch_status("k_mfma_f16");
}

// One fp16 row (K up to 8192) times w: fp32 dots, or (H16) their fp16 values.
template <bool H16>
static int f16_row(const uint8_t* x, const nc_tensor* w, void* out, hipStream_t st, hipEvent_t ev_start,
                   hipEvent_t ev_stop)
{
    const int N = w->rows, K = w->cols;
    const dim3 grid((N + 7) / 8);
    float* of = H16 ? nullptr : static_cast<float*>(out);
    uint16_t* oh = H16 ? static_cast<uint16_t*>(out) : nullptr;
    auto go = [&](auto kern) {
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, dim3(64), 0, st, ev_start, ev_stop, 0, x, (const uint16_t*)w->data, of, N,
                                  oh);
        else
            hipLaunchKernelGGL(kern, grid, dim3(64), 0, st, x, (const uint16_t*)w->data, of, N, oh);
    };
    if (dmv_f16_dispatch<false, H16>(K / 64, go)) return launch_status("k_dmv_f16");
    const size_t lds = (size_t)K * 4;
    if (ev_start)
        hipExtLaunchKernelGGL(k_matvec_f16_row<H16>, grid, dim3(64), lds, st, ev_start, ev_stop, 0, x,
                              (const uint16_t*)w->data, out, N, K);
    else
        hipLaunchKernelGGL(k_matvec_f16_row<H16>, grid, dim3(64), lds, st, x, (const uint16_t*)w->data, out, N, K);
    return launch_status("k_matvec_f16_row");
}

// Whether two fp16 rows go one after the other through the one-row kernel: its
// launch of few columns is over long before k_mfma_f16's chain of K steps, which
// two rows hardly fill (us back to back, k_mfma_f16 / this: 2048 x 2048 14.8 / 6.8,
// 1280 x 1280 10.0 / 8.4, 2304 x 5760 37.5 / 14.7, 4096 x 1536 12.0 / 11.5; 5632 x 2048
// 15.3, two of 5.9 and a gap).
static bool f16_two_rows(int n_rows, const nc_tensor* w)
{
    return n_rows == 2 && w->rows <= 4096 && f16_shape_ok(w) && w->cols <= 8192;
}

// out[r, c] = dot(x[r], w[c]) for x rows [0, n_rows) (pointers already at
// the first row), fp32 out with `out_pitch` floats per row.
int matvec_raw(const uint8_t* x, int x_dtype, int x_pitch, int n_rows, const nc_tensor* w, float* out, int out_pitch,
               hipStream_t st, hipEvent_t ev_start, hipEvent_t ev_stop, const nc_tensor* wc)
{
    // with events, the dispatch itself records them (the kernel's own start and end)
#define NC_MV_LAUNCH(KERNEL, GRID, LDS, ...)                                                              \
    do {                                                                                                  \
        if (ev_start)                                                                                     \
            hipExtLaunchKernelGGL(KERNEL, GRID, dim3(kMvThreads), LDS, st, ev_start, ev_stop, 0, __VA_ARGS__); \
        else                                                                                              \
            hipLaunchKernelGGL(KERNEL, GRID, dim3(kMvThreads), LDS, st, __VA_ARGS__);                     \
    } while (0)
    const int N = w->rows, K = w->cols;
    if (w->dtype == NC_Q4 || w->dtype == NC_Q8) {
        if (x_dtype != NC_Q8) return fail(NC_ERR_ARG, "matmul: Q%d weights need Q8 activations", w->dtype == NC_Q4 ? 4 : 8);
        if (K % 32) return fail(NC_ERR_ARG, "matmul: K=%d is not a multiple of 32", K);
        if (n_rows >= kGemmMinRows)
            return gemm_q_raw(x, x_pitch, n_rows, w, out, out_pitch, st, ev_start, ev_stop, wc);
        const int nb = K / 32;
        constexpr int R = 4;
        if (R * nb > kMvThreads * kMvMaxItems) return fail(NC_ERR_ARG, "matmul: K=%d too large", K);
        const int tp = ((nb + 3) & ~3) + 4;
        const size_t lds = (size_t)nb * kStage * 4 + (size_t)R * 4 * tp * 4;
        const dim3 grid((N + R - 1) / R);
        if (w->dtype == NC_Q4)
            NC_MV_LAUNCH((k_matvec_q<Q4, R>), grid, lds, x, x_pitch, n_rows, (const uint32_t*)w->data,
                         (const uint16_t*)w->deltas, out, out_pitch, N, nb);
        else
            NC_MV_LAUNCH((k_matvec_q<Q8, R>), grid, lds, x, x_pitch, n_rows, (const uint32_t*)w->data,
                         (const uint16_t*)w->deltas, out, out_pitch, N, nb);
        return launch_status("k_matvec_q");
    }
    if (w->dtype == NC_F16) {
        if (x_dtype != NC_F16) return fail(NC_ERR_ARG, "matmul: F16 weights need F16 activations");
        if (K % 64) return fail(NC_ERR_ARG, "matmul: F16 path needs K %% 64 == 0, K=%d", K);
        if (!f16_shape_ok(w)) return fail(NC_ERR_ARG, "matmul: K=%d too large", K);
        if (n_rows == 1 && K <= 8192) return f16_row<false>(x, w, out, st, ev_start, ev_stop);
        if (!ev_start && f16_two_rows(n_rows, w)) {
            const int s = f16_row<false>(x, w, out, st, nullptr, nullptr);
            return s ? s : f16_row<false>(x + x_pitch, w, out + out_pitch, st, nullptr, nullptr);
        }
        return mfma_f16<F32>(x, x_pitch, n_rows, w, out, out_pitch, st, ev_start, ev_stop);
    }
    return fail(NC_ERR_ARG, "matmul: weight dtype %d", w->dtype);
#undef NC_MV_LAUNCH
}

bool matvec_f16_glu_supported(const nc_tensor* w)
{
    return w->dtype == NC_F16 && w->rows % 8 == 0 && w->cols % 64 == 0 &&
           dmv_f16_dispatch<true>(w->cols / 64, [](auto) {});
}

int matvec_f16_glu(const uint8_t* x, const nc_tensor* w, uint8_t* m_out, hipStream_t st, hipEvent_t ev_start,
                   hipEvent_t ev_stop)
{
    const int N = w->rows, K = w->cols;
    if (!matvec_f16_glu_supported(w))
        return fail(NC_ERR_ARG, "gate|up SwiGLU matvec: [%d x %d] dtype %d", N, K, w->dtype);
    const dim3 grid(N / 8);
    auto go = [&](auto kern) {
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, dim3(64), 0, st, ev_start, ev_stop, 0, x, (const uint16_t*)w->data,
                                  nullptr, N, (uint16_t*)m_out);
        else
            hipLaunchKernelGGL(kern, grid, dim3(64), 0, st, x, (const uint16_t*)w->data, nullptr, N,
                               (uint16_t*)m_out);
    };
    dmv_f16_dispatch<true>(K / 64, go);
    return launch_status("k_dmv_f16<GLU>");
}

bool dmv_f16_nrm_supported(const nc_tensor* w, int d, bool glu)
{
    return w->dtype == NC_F16 && w->cols == d && (d == 2048 || d == 2304) && (!glu || w->rows % 8 == 0);
}

int dmv_f16_nrm_launch(int kind, const uint8_t* a, int a_pitch, const float* braw, float bscale, uint8_t* h_out,
                       int h_pitch, const uint16_t* nw, const uint16_t* nb, const nc_tensor* w, float* out,
                       uint8_t* m_out, bool glu, hipStream_t st, const int* dpos, hipEvent_t ev_start,
                       hipEvent_t ev_stop)
{
    const int N = w->rows, K = w->cols;
    if (!dmv_f16_nrm_supported(w, K, glu) || (kind == kNrmLayer && !nb))
        return fail(NC_ERR_ARG, "norm + fp16 matvec: [%d x %d] dtype %d", N, K, w->dtype);
    const int quads = glu ? N / 8 : (N + 7) / 8;  // fold wavefronts: 8 rows each
    const dim3 grid((quads + kNrmFold / kWave - 1) / (kNrmFold / kWave));
    auto go = [&](auto kern) {
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, dim3(kNrmNorm + kNrmFold), 0, st, ev_start, ev_stop, 0, a, a_pitch, braw,
                                  bscale, h_out, h_pitch, nw, nb, (const uint16_t*)w->data, out, (uint16_t*)m_out, N,
                                  dpos);
        else
            hipLaunchKernelGGL(kern, grid, dim3(kNrmNorm + kNrmFold), 0, st, a, a_pitch, braw, bscale, h_out, h_pitch,
                               nw, nb, (const uint16_t*)w->data, out, (uint16_t*)m_out, N, dpos);
    };
    const bool add = braw != nullptr;
    // ADD x GLU for each norm kind and row width (32 or 36 groups of 64;
    // rows of 36 groups keep 24 in the register ring, the rest refilled
    // during the fold: a full ring would spill at 768 threads)
    auto pick = [&](auto kd) {
        constexpr int KD = decltype(kd)::value;
        if (K == 2048) {
            if (add && glu) go(k_dmv_f16_nrm<32, 32, 8, KD, true, true>);
            else if (add) go(k_dmv_f16_nrm<32, 32, 8, KD, true, false>);
            else if (glu) go(k_dmv_f16_nrm<32, 32, 8, KD, false, true>);
            else go(k_dmv_f16_nrm<32, 32, 8, KD, false, false>);
        } else {
            if (add && glu) go(k_dmv_f16_nrm<36, 24, 8, KD, true, true>);
            else if (add) go(k_dmv_f16_nrm<36, 24, 8, KD, true, false>);
            else if (glu) go(k_dmv_f16_nrm<36, 24, 8, KD, false, true>);
            else go(k_dmv_f16_nrm<36, 24, 8, KD, false, false>);
        }
    };
    if (kind == kNrmLayer) pick(std::integral_constant<int, kNrmLayer>{});
    else pick(std::integral_constant<int, kNrmRms>{});
    return launch_status("k_dmv_f16_nrm");
}

}  // namespace nc

// ================================================================ C-ABI ==

using namespace nc;

namespace {

// Library-owned fp32 staging for matmul_2d calls whose output is an
// activation dtype (grown on demand, never inside a captured graph).
float* g_stage = nullptr;
size_t g_stage_bytes = 0;

int stage_buffer(size_t bytes, float** out)
{
    if (bytes > g_stage_bytes) {
        if (g_stage) (void)hipFree(g_stage);
        g_stage = nullptr;
        g_stage_bytes = 0;
        hipError_t e = hipMalloc(&g_stage, bytes);
        if (e != hipSuccess) return fail(NC_ERR_NOMEM, "matmul staging (%zu bytes): %s", bytes, hipGetErrorString(e));
        g_stage_bytes = bytes;
    }
    *out = g_stage;
    return NC_OK;
}

}  // namespace

// nc_matmul_2d_noalloc's staging: a file-scope device array.  Every GPU the
// library runs on holds its own copy, at its own address, until the process
// ends.  In host code `scratch` only names a host-side stand-in; the device
// address comes from hipGetSymbolAddress, taken once per device with that
// device current (nc_init, or the entry point's first call on a device) and
// kept in g_scratch.  Kernels get that address as an argument.
static __device__ __align__(256) float scratch[NC_NOALLOC_STAGE_BYTES / sizeof(float)];

namespace {

constexpr size_t kNoAllocStageBytes = NC_NOALLOC_STAGE_BYTES;
constexpr int kMaxDevices = 64;
float* g_scratch[kMaxDevices] = {};

int scratch_for_current(float** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    int s = noalloc_scratch_setup(dev);
    if (s) return s;
    *out = g_scratch[dev];
    return NC_OK;
}

}  // namespace

namespace nc {

int noalloc_scratch_setup(int dev)
{
    if (dev < 0 || dev >= kMaxDevices) return fail(NC_ERR_ARG, "staging array: device %d", dev);
    if (g_scratch[dev]) return NC_OK;
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    g_scratch[dev] = static_cast<float*>(p);
    return NC_OK;
}

}  // namespace nc

namespace {

bool overlap(const void* a, size_t na, const void* b, size_t nb)
{
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return a && b && x < y + nb && y < x + na;
}

// Whether a launch that computes x rows times w can store activation rows of
// out_dtype itself: gemm_q_act's, k_matvec_qa's, the fp16 ones.
bool direct_rows(int x_dtype, int x_pitch, int rows, const nc_tensor* w, int out_dtype)
{
    if (out_dtype != x_dtype || w->cols <= 0) return false;
    if (x_dtype == NC_Q8) return gemm_q_act_supported(x_pitch, rows, w) || qa_shape(rows, w).items;
    return x_dtype == NC_F16 && w->dtype == NC_F16 && f16_shape_ok(w);
}

// Whether this call's launch stores out's rows itself: such a launch, and no
// output byte that the product still reads (a staged product has read
// everything before it writes).
bool stores_rows(const nc_tensor* x, const uint8_t* xr, const nc_tensor* w, const nc_tensor* out, const uint8_t* orow,
                 int rows)
{
    if (!direct_rows(x->dtype, x->pitch, rows, w, out->dtype)) return false;
    const size_t on = (size_t)rows * out->pitch;
    size_t cb, db;
    if (nc_weight_bytes(w->dtype, w->rows, w->cols, &cb, &db)) return false;
    return !overlap(orow, on, xr, (size_t)rows * x->pitch) && !overlap(orow, on, w->data, cb) &&
           !overlap(orow, on, w->deltas, db);
}

// nc_matmul_2d with the staging of an activation-dtype output given by
// stage(bytes, &ptr).
template <class Stage>
int matmul_2d(const char* name, const nc_tensor* x, const nc_tensor* w, nc_tensor* out, int start, int n_ctx,
              void* stream, Stage&& stage)
{
    NC_CHECK_ARG(x && w && out && x->data && w->data && out->data, "%s: null tensor", name);
    NC_CHECK_ARG(x->cols == w->cols, "%s: x has %d columns, w has %d", name, x->cols, w->cols);
    NC_CHECK_ARG(out->cols == w->rows, "%s: out has %d columns, w has %d rows", name, out->cols, w->rows);
    NC_CHECK_ARG(start >= 0 && start <= n_ctx && n_ctx <= x->rows && n_ctx <= out->rows, "%s: rows [%d, %d)", name,
                 start, n_ctx);
    const int rows = n_ctx - start;
    if (rows == 0) return NC_OK;
    hipStream_t st = stream_of(stream);
    const uint8_t* xr = (const uint8_t*)x->data + (size_t)start * x->pitch;
    uint8_t* orow = (uint8_t*)out->data + (size_t)start * out->pitch;
    if (out->dtype == NC_F32) {
        NC_CHECK_ARG(out->pitch % 4 == 0, "%s: fp32 pitch %d", name, out->pitch);
        return matvec_raw(xr, x->dtype, x->pitch, rows, w, (float*)orow, out->pitch / 4, st);
    }
    // staging comes first, also where the launch will not need it: what a call
    // allocates or refuses then depends on its sizes alone, and a call warmed up
    // before a capture has its staging whichever route a later one takes
    float* sp = nullptr;
    int s = stage((size_t)rows * w->rows * 4, rows, &sp);
    if (s) return s;
    if (stores_rows(x, xr, w, out, orow, rows)) {
        if (x->dtype == NC_Q8)
            return rows < kGemmMinRows ? matvec_qa(xr, x->pitch, rows, w, orow, out->pitch, st)
                                       : gemm_q_act(xr, x->pitch, rows, w, orow, out->pitch, st);
        if (rows == 1 && w->cols <= 8192) return f16_row<true>(xr, w, orow, st, nullptr, nullptr);
        if (f16_two_rows(rows, w)) {
            s = f16_row<true>(xr, w, orow, st, nullptr, nullptr);
            return s ? s : f16_row<true>(xr + x->pitch, w, orow + out->pitch, st, nullptr, nullptr);
        }
        return mfma_f16<F16>(xr, x->pitch, rows, w, orow, out->pitch, st, nullptr, nullptr);
    }
    if ((s = matvec_raw(xr, x->dtype, x->pitch, rows, w, sp, w->rows, st))) return s;
    return write_rows(sp, w->rows, orow, out->pitch, out->dtype, w->rows, rows, st);
}

}  // namespace

// The same as nc_matmul_2d, with an activation-dtype output staged in the
// device's fixed array instead of library-allocated memory: no allocation
// anywhere on this path.
extern "C" int nc_matmul_2d_noalloc(const nc_tensor* x, const nc_tensor* w, nc_tensor* out, int start, int n_ctx,
                                    void* stream)
{
    return matmul_2d("matmul_2d_noalloc", x, w, out, start, n_ctx, stream, [&](size_t need, int rows, float** p) {
        NC_CHECK_ARG(need <= kNoAllocStageBytes,
                     "matmul_2d_noalloc: %d rows x %d outputs need %zu staging bytes, more than the %zu-byte array",
                     rows, w->rows, need, kNoAllocStageBytes);
        return scratch_for_current(p);
    });
}

extern "C" int nc_matmul_2d(const nc_tensor* x, const nc_tensor* w, nc_tensor* out, int start, int n_ctx, void* stream)
{
    return matmul_2d("matmul_2d", x, w, out, start, n_ctx, stream,
                     [&](size_t need, int, float** p) { return stage_buffer(need, p); });
}

// The kernel that nc_matmul_2d takes for a product of whole, aligned tensors
// that do not overlap, and how its rows are stored.
extern "C" const char* nc_debug_matmul_route(int x_dtype, int w_dtype, int out_dtype, int rows, int N, int K)
{
    static thread_local char name[64];
    static const uint64_t aligned[2] = {0, 0};
    const nc_tensor w{(void*)aligned, (void*)aligned, w_dtype, N, K, 0};
    const int pitch = nc_act_pitch(x_dtype, K);
    const bool direct = out_dtype != NC_F32 && direct_rows(x_dtype, pitch, rows, &w, out_dtype);
    const char* tail = out_dtype == NC_F32 ? "" : direct ? ", rows" : " + k_write_rows";
    if (w_dtype != NC_F16 && rows < kGemmMinRows) {
        const QaShape q = qa_shape(rows, &w);
        if (direct) snprintf(name, sizeof name, "k_matvec_qa %dx%d%s", q.term, q.items, tail);
        else snprintf(name, sizeof name, "k_matvec_q%s", tail);
    } else {
        const bool one = (rows == 1 && K <= 8192) || f16_two_rows(rows, &w);
        snprintf(name, sizeof name, "%s%s",
                 w_dtype != NC_F16 ? gemm_route(pitch, rows, &w, direct) : one ? "one fp16 row" : "k_mfma_f16", tail);
    }
    return name;
}
