// nc_gemm.hip -- prefill matmul of Q8 activation rows with Q4 / Q8 weights
// on the matrix cores, with the reference's arithmetic.
//
// matmul_2d_impl (gten/ops.cpp:579-614) computes each output as the
// reference's block dot product (vec_dot_product_q8 / _q8_q4, ops.cpp:
// 292-490): per 32-value block b, four int32 lane sums L_k(b) over the
// elements {2k, 2k+1, 2k+8, 2k+9} and the same + 16, fp32 terms
// float(L_k) * (d_x * d_w), four fp32 chains acc_k folded in block order,
// and (acc_0 + acc_1) + (acc_2 + acc_3).
//
// The integer lane sums come from v_mfma_i32_16x16x32_i8 (K = 32 = one
// block), with the activation operand expanded by lane: matrix row 4r + k
// holds row r's lane-k codes in K group k and zeros in the other three
// groups, the weight operand holds column n's lane-g codes in K group g (the
// weights are stored lane-permuted, so a lane's eight codes are one dword
// (Q4) or two (Q8)).  Result entry (4r + k, n) is then exactly L_k(r, n),
// and the MFMA output layout puts the four lane sums of one (row, column)
// in one thread: thread (n, r) owns its chains and folds them in block
// order with plain fp32 multiplies and adds -- the reference's rounding
// steps, one per block and lane.  Q4 codes enter raw (0..14): the
// accumulator starts at -7 * (sum of the lane's activation codes), so the
// MFMA yields sum (code - 7) * x, as the reference's decoded values give.
//
// Three quarters of each activation operand are zeros: the matrix cores do
// four times the necessary integer work, which is cheap next to the
// vector-unit fold (13 fp32 operations per output and block).  k_gemm_qw
// (below) takes the same lane sums on the fp16 matrix cores and reads the
// weights' chunk-major copy when the caller has one; this kernel keeps the
// products it does not take (K not a multiple of 128).
#include <hip/hip_ext.h>

#include <type_traits>

#include "nc_kernels.h"
#include "nc_qdot.h"

namespace nc {

constexpr int kGmChunk = 4;                // activation blocks staged per step (double-buffered)

typedef int v4i __attribute__((ext_vector_type(4)));

// NG 16-wide column groups per wavefront, NW wavefronts per workgroup (all
// on the same rows, side by side in columns), MR groups of 4 rows (one MFMA
// row operand each) per workgroup; the first 4 MR x kGmChunk threads stage
// the activation blocks.  Kept for what k_gemm_qw does not take (gemm_shape): rows
// whose blocks do not come in fours, weights not at whole dwords, operands of
// 2 GiB and more.
template <int WT, int NG, int NW, int MR, int PF>
__global__ __launch_bounds__(64 * NW) void k_gemm_q(const uint8_t* __restrict__ x, int x_pitch, int n_rows,
                                                      const uint32_t* __restrict__ wq,
                                                      const uint16_t* __restrict__ wd, float* __restrict__ out,
                                                      int out_pitch, int N, int nb)
{
    constexpr int WV = WT == Q4 ? 1 : 2;  // code dwords of one lane of a weight block
    constexpr int WD = WT == Q4 ? 4 : 8;  // code dwords per weight block
    constexpr int kGmNg = NG;
    constexpr int kGmCols = 16 * NG * NW;  // columns per workgroup
    constexpr int kGmRows = 4 * MR;        // rows per workgroup
    // staged activation blocks (nc_qdot.h layout): [buffer][block][row]
    __shared__ __align__(16) uint32_t xs[2][kGmChunk][kGmRows][kStage];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lc = lane & 15, lg = lane >> 4;  // column within a 16-group; K group (AVX lane)
    const int r0 = blockIdx.y * kGmRows;
    const int c0 = blockIdx.x * kGmCols + wv * 16 * NG;
    const int nch = (nb + kGmChunk - 1) / kGmChunk;

    // staging: thread t < kGmRows x kGmChunk stages (row t % kGmRows, block
    // t / kGmRows) of each chunk; rows past the end repeat the last row
    // (their outputs are not stored)
    constexpr int kStagers = kGmRows * kGmChunk;
    static_assert(kStagers <= 64 * NW, "every staged (row, block) needs its own thread");
    const int srow = tid % kGmRows, sblk = (tid / kGmRows) & (kGmChunk - 1);
    const uint8_t* xrow = x + (size_t)min(r0 + srow, n_rows - 1) * x_pitch;
    auto stage_load = [&](int ch) { return load_x_block(xrow, nb, min(ch * kGmChunk + sblk, nb - 1)); };

    // this thread's weight columns (columns past the end repeat the last)
    size_t wrow[kGmNg];
#pragma unroll
    for (int n = 0; n < kGmNg; n++) wrow[n] = (size_t)min(c0 + 16 * n + lc, N - 1) * nb;
    auto w_load = [&](int ch, uint32_t (&w)[kGmChunk][kGmNg][WV], uint16_t (&d)[kGmChunk][kGmNg]) {
#pragma unroll
        for (int j = 0; j < kGmChunk; j++) {
            const int b = min(ch * kGmChunk + j, nb - 1);
#pragma unroll
            for (int n = 0; n < kGmNg; n++) {
                const uint32_t* blk = wq + (wrow[n] + b) * WD;
#pragma unroll
                for (int v = 0; v < WV; v++) w[j][n][v] = blk[WV * lg + v];
                d[j][n] = wd[wrow[n] + b];
            }
        }
    };

    float acc[MR][kGmNg][4];
#pragma unroll
    for (int m = 0; m < MR; m++)
#pragma unroll
        for (int n = 0; n < kGmNg; n++)
#pragma unroll
            for (int k = 0; k < 4; k++) acc[m][n][k] = 0.0f;

    // weights and activation blocks: a ring of PF chunks in registers;
    // chunk ch sits in slot ch % PF from its request (PF chunks ahead) until
    // it is used, so HBM latency hides behind PF chunks of work, and a slot
    // is refilled straight after use (no register copies, which would wait
    // for the loads).  Both are requested together because the vector
    // memory counter completes in order: the activation blocks staged at
    // the end of chunk ch (chunk ch + 1's) were requested PF - 1 chunks
    // earlier, so waiting for them waits only for loads that old.  Every
    // request is issued (chunks past the end re-read the last blocks), so
    // the waits are exact counts.
    uint32_t wr[PF][kGmChunk][kGmNg][WV];
    uint16_t dr[PF][kGmChunk][kGmNg];
    XRaw xq[PF];
#pragma unroll
    for (int p = 0; p < PF; p++) {
        w_load(p, wr[p], dr[p]);
        xq[p] = stage_load(min(p, nch - 1));
    }
    if (tid < kStagers) stage_x_block(xq[0], xs[0][sblk][srow]);
    lds_barrier();
    for (int cb = 0; cb < nch; cb += PF) {
#pragma unroll
        for (int p = 0; p < PF; p++) {
            const int ch = cb + p;
            if (ch >= nch) break;  // uniform
            const int buf = ch & 1;
            {
#pragma unroll
            for (int j = 0; j < kGmChunk; j++) {
                if (ch * kGmChunk + j >= nb) break;  // uniform
                // weight operands: column lc of group n, lane lg's eight codes
                long B[kGmNg];
                float dw[kGmNg];
#pragma unroll
                for (int n = 0; n < kGmNg; n++) {
                    if (WT == Q4) {
                        const uint32_t P = wr[p][j][n][0];
                        // high nibbles pair with codes {2k,2k+1,2k+8,2k+9},
                        // low nibbles with those + 16 (the staged xa_k, xb_k
                        // order)
                        B[n] = (long)(uint64_t)(((P >> 4) & 0x0F0F0F0Fu) | ((uint64_t)(P & 0x0F0F0F0Fu) << 32));
                    } else {
                        B[n] = (long)(uint64_t)(wr[p][j][n][0] | ((uint64_t)wr[p][j][n][1] << 32));
                    }
                    dw[n] = h2f(dr[p][j][n]);
                }
#pragma unroll
                for (int m = 0; m < MR; m++) {
                    // activation operand: matrix row lc = 4 r' + k of row
                    // group m holds row (4m + r')'s lane-k codes in K group
                    // k only
                    const uint32_t* sa = xs[buf][j][4 * m + (lc >> 2)];
                    const uint2 v = *reinterpret_cast<const uint2*>(sa + 2 * lg);
                    const bool own = lg == (lc & 3);
                    const long A = (long)(uint64_t)((own ? v.x : 0u) | ((uint64_t)(own ? v.y : 0u) << 32));
                    // this thread's outputs: row 4m + lg, lane sums k = 0..3
                    const uint32_t* sr = xs[buf][j][4 * m + lg];
                    const uint4 cs = *reinterpret_cast<const uint4*>(sr + 8);
                    const v4i cinit = WT == Q4 ? v4i{(int)cs.x, (int)cs.y, (int)cs.z, (int)cs.w} : v4i{0, 0, 0, 0};
                    const float dx = __uint_as_float(sr[12]);
#pragma unroll
                    for (int n = 0; n < kGmNg; n++) {
                        const v4i L = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B[n], cinit, 0, 0, 0);
                        const float dd = dx * dw[n];
#pragma unroll
                        for (int k = 0; k < 4; k++) acc[m][n][k] = acc[m][n][k] + (float)L[k] * dd;
                    }
                }
            }
            }
            // the slot's next chunk, then chunk ch + 1's activation blocks
            // into the other staging buffer
            w_load(ch + PF, wr[p], dr[p]);
            xq[p] = stage_load(min(ch + PF, nch - 1));
            if (ch + 1 < nch && tid < kStagers) stage_x_block(xq[(p + 1) % PF], xs[buf ^ 1][sblk][srow]);
            lds_barrier();
        }
    }
#pragma unroll
    for (int m = 0; m < MR; m++) {
        const int row = r0 + 4 * m + lg;
#pragma unroll
        for (int n = 0; n < kGmNg; n++) {
            const int col = c0 + 16 * n + lc;
            if (row < n_rows && col < N)
                out[(size_t)row * out_pitch + col] = (acc[m][n][0] + acc[m][n][1]) + (acc[m][n][2] + acc[m][n][3]);
        }
    }
}

// ---------------------------------------------------------------------------
// The same products with the lane sums taken on the fp16 matrix cores
// (v_mfma_f32_16x16x32_f16): codes enter as fp16 integers or exact sixteenths of
// them (see k_gemm_qw), so that each product and each partial sum the matrix
// core forms is an integer below 2^22, exactly representable in fp32, and the
// fp32 result is exactly float(L_k): the conversion the integer path needs per
// lane and block is gone, and the fold is 9 fp32 operations per (row, column,
// block) instead of 13.
//
// The activation operand is staged once per workgroup already expanded: for
// block j and row group m, lane l = (4r + k) + 16 g holds row 4m + r's lane-k
// codes as fp16 when g == k, and zeros otherwise (the zero entries are written
// once at kernel start and never touched again).  A lane reads its 16 bytes
// with one LDS load; rows of a group share them across the NW wavefronts.
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// Four bytes b0..b3 of `u` (each below 256) as fp16 1024 + b, two per dword:
// [b0, b1] and [b2, b3] (v_perm_b32 with the exponent byte 0x64 from a
// constant).
__device__ __forceinline__ void bytes_to_h1024(uint32_t u, uint32_t& lo, uint32_t& hi)
{
    lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
}

// The same, then plus `bias` (fp16, both halves): exact integers.
__device__ __forceinline__ void bytes_to_h(uint32_t u, uint32_t bias2, uint32_t& lo, uint32_t& hi)
{
    uint32_t a, b;
    bytes_to_h1024(u, a, b);
    const h2_t bb = __builtin_bit_cast(h2_t, bias2);
    lo = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, a) + bb);
    hi = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, b) + bb);
}
constexpr uint32_t kHm1152 = 0xE480E480u;  // fp16 -1152, twice: (1024 + c + 128) - 1152 = c

// Four signed int8 codes -> four fp16 values (two dwords).
__device__ __forceinline__ void s8x4_to_h(uint32_t v, uint32_t& lo, uint32_t& hi)
{
    bytes_to_h(v ^ 0x80808080u, kHm1152, lo, hi);
}

// Four signed int8 codes -> their fp16 values / 16 (two dwords): (1024 + c +
// 128) / 16 - 72, one rounding, exact.
__device__ __forceinline__ void s8x4_to_h16(uint32_t v, uint32_t& lo, uint32_t& hi)
{
    uint32_t a, b;
    bytes_to_h1024(v ^ 0x80808080u, a, b);
    const h2_t sc = {(_Float16)0.0625f, (_Float16)0.0625f}, off = {(_Float16)-72.0f, (_Float16)-72.0f};
    lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2_t, a), sc, off));
    hi = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2_t, b), sc, off));
}

// ---------------------------------------------------------------------------
// k_gemm_qw: a wavefront owns 4 MR rows x 16 NG columns, so each activation
// operand, accumulator start and row delta it reads from LDS serves NG weight
// operands, and each converted weight operand MR row groups; NW wavefronts
// side by side in columns share the staged rows; a chunk is CH blocks, one
// LDS barrier each.
//
// What bounds it with enough (row, column) tiles to fill the chip (NG = 2):
// the vector unit.  Per block a wavefront issues 9 fp32 operations per 64
// (row, column) pairs (the reference's rounding steps, none of which can go)
// beside 11 per weight operand.  With NG = 1 there the LDS reads are the
// limit instead: per block and row group 18 LDS cycles (two 16-byte reads and
// a dword per lane) on a unit that four SIMDs share, against 9 + 11 / MR
// vector operations of 4 cycles each on one.  With few tiles a SIMD has one
// wavefront or none, and the chain over the blocks is bound by latencies: NG
// = 1 then gives twice the wavefronts, CH = 8 halves the barriers and the
// LDS reads run RD steps ahead.
//
// The weights are read in their own layout, 16 bytes per lane: lane (column,
// g) of a 16 x 4 arrangement reads block b0 + g of its column, and a 4 x 4
// transpose over the four 16-lane rows (two lane swaps per pair of registers)
// hands every lane its AVX lane's codes of the four blocks; or (CL) from the
// chunk-major copy, where they lie in that order already.
//
// Codes enter raw, as fp16 1024 + byte (one v_perm_b32 per two), and the
// accumulators start at what that adds.  Q8: the byte is w + 128, so the
// products sum to sum (1152 + w) x and the start is -1152 sum x.  Q4: the
// low nibbles enter as 1024 + n against x, the high ones in place as 1024 +
// 16 n against x / 16 (exact in fp16), giving (64 + n) x; the start is -1031
// sum x over the low ones and -71 sum x over the high ones, which leaves sum
// (n - 7) x.  Every value on the way is an integer below 2^22.
//
// ODT: F32 stores the dot products (out_pitch floats per row); Q8 stores them
// as write_row_from_float does (out_pitch bytes per row), a block of 32
// columns being two column groups of one wavefront.
__device__ __forceinline__ void lane_rows_transpose4(uint32_t (&r)[4])
{
    // r[b] of lane row g <- r[g] of lane row b
    auto swap32 = [](uint32_t& a, uint32_t& b) {
        const auto t = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = t[0];
        b = t[1];
    };
    auto swap16 = [](uint32_t& a, uint32_t& b) {
        const auto t = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = t[0];
        b = t[1];
    };
    swap32(r[0], r[2]);
    swap32(r[1], r[3]);
    swap16(r[0], r[1]);
    swap16(r[2], r[3]);
}

template <int WT, int MR, int NG, int NW, int CH, int RD, bool CL, int WPE, int ODT>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE))) void k_gemm_qw(
        const uint8_t* __restrict__ x, int x_pitch, int n_rows, const uint32_t* __restrict__ wq,
        const uint16_t* __restrict__ wd, void* __restrict__ out, int out_pitch, int N, int nb)
{
    constexpr int WV = WT == Q4 ? 1 : 2;  // code dwords of one lane of a weight block
    constexpr int WD = WT == Q4 ? 4 : 8;  // code dwords per weight block
    constexpr int PF = 2;                 // chunks in flight
    constexpr int kRows = 4 * MR, kThreads = 64 * NW;
    static_assert(ODT != Q8 || NG % 2 == 0, "a Q8 output block is two column groups");
    __shared__ __align__(16) uint4 xa[2][CH][MR][64];                   // expanded operands (see above)
    __shared__ __align__(16) float xd[2][CH][4][MR];                    // deltas of rows 4m + g as [g][m]
    __shared__ __align__(16) float xc[2][CH][kRows][4];  // accumulator starts
    static_assert(MR >= 2, "the row deltas of two blocks are held in turn");
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int lc = lane & 15, lg = lane >> 4;
    const int r0 = blockIdx.y * kRows;
    const int c0 = (blockIdx.x * NW + wv) * 16 * NG;
    const int nch = nb / CH;

    for (int e = tid; e < 2 * CH * MR * 64; e += kThreads)
        if (((e & 15) & 3) != ((e >> 4) & 3)) (&xa[0][0][0][0])[e] = make_uint4(0, 0, 0, 0);

    // staging tasks: one AVX lane k of one (row, block) of the chunk
    constexpr int kTasks = 4 * kRows * CH;
    constexpr int TPT = (kTasks + kThreads - 1) / kThreads;
    static_assert(kThreads % 4 == 0, "a thread's tasks share their lane");
    const uint32_t psel = tid & 1 ? 0x07060302u : 0x05040100u;  // byte pairs of lanes k odd / even
    struct XLane {
        uint32_t d[4];
        uint16_t d16;
    };
    // 32-bit offsets from buffer resources: a chunk's position is the scalar
    // offset, so no address is formed per load
    const auto xres = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (unsigned)((size_t)n_rows * x_pitch), kBufferFlags);
    int t_row[TPT], t_blk[TPT], t_k[TPT], t_off[TPT], t_dof[TPT];
#pragma unroll
    for (int i = 0; i < TPT; i++) {
        const int t = min(tid + i * kThreads, kTasks - 1);
        t_k[i] = t & 3;
        t_row[i] = (t >> 2) % kRows;
        t_blk[i] = (t >> 2) / kRows;
        const int base = min(r0 + t_row[i], n_rows - 1) * x_pitch;
        t_off[i] = base + t_blk[i] * 32 + (t_k[i] >> 1) * 4;
        t_dof[i] = base + nb * 32 + t_blk[i] * 2;
    }
    auto x_load = [&](int ch, XLane (&q)[TPT]) {
        const int b0 = min(ch, nch - 1) * CH;
#pragma unroll
        for (int i = 0; i < TPT; i++) {
#pragma unroll
            for (int v = 0; v < 4; v++) q[i].d[v] = __builtin_amdgcn_raw_buffer_load_b32(xres, t_off[i] + 8 * v, b0 * 32, 0);
            q[i].d16 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(xres, t_dof[i], b0 * 2, 0);
        }
    };
    auto stage = [&](const XLane (&q)[TPT], int buf) {
#pragma unroll
        for (int i = 0; i < TPT; i++) {
            if (tid + i * kThreads >= kTasks) break;  // uniform per wave: kTasks is a multiple of 64
            const int k = t_k[i], r = t_row[i], j = t_blk[i];
            const uint32_t a = __builtin_amdgcn_perm(q[i].d[1], q[i].d[0], psel);  // pick_pair of lane k
            const uint32_t bq = __builtin_amdgcn_perm(q[i].d[3], q[i].d[2], psel);
            const int sa = __builtin_amdgcn_sdot4((int)a, 0x01010101, 0, false);
            const int sb = __builtin_amdgcn_sdot4((int)bq, 0x01010101, 0, false);
            uint4 hv;
            if constexpr (WT == Q4) {
                s8x4_to_h16(a, hv.x, hv.y);
                xc[buf][j][r][k] = (float)(-71 * sa - 1031 * sb);
            } else {
                s8x4_to_h(a, hv.x, hv.y);
                xc[buf][j][r][k] = (float)(-1152 * (sa + sb));
            }
            s8x4_to_h(bq, hv.z, hv.w);
            xa[buf][j][r >> 2][(r & 3) * 4 + k + 16 * k] = hv;
            if (k == 0) xd[buf][j][r & 3][r >> 2] = h2f(q[i].d16);
        }
    };

    // this thread's weight columns (columns past the end repeat the last)
    const size_t wbytes = (size_t)N * nb * WD * 4;
    const auto wres = __builtin_amdgcn_make_buffer_rsrc((void*)wq, 0, (unsigned)wbytes, kBufferFlags);
    const auto dres = __builtin_amdgcn_make_buffer_rsrc((void*)wd, 0, (unsigned)((size_t)N * nb * 2), kBufferFlags);
    int w_off[NG], d_off[NG];
#pragma unroll
    for (int n = 0; n < NG; n++) {
        const int col = min(c0 + 16 * n + lc, N - 1);
        w_off[n] = CL ? (col * 4 + lg) * 16 * WV : (col * nb + lg) * WD * 4;
        d_off[n] = CL ? col * 8 : col * nb * 2;
    }
    typedef uint32_t U4 __attribute__((ext_vector_type(4)));
    typedef uint32_t U2 __attribute__((ext_vector_type(2)));
    struct WChunk {
        // per four blocks: CL: block b's lane-lg codes; plain: block lg's codes, before the transpose
        uint32_t c[CH / 4][NG][WV][4];
        uint32_t d[CH / 4][NG][2];  // the four blocks' deltas
    };
    auto w_load = [&](int ch, WChunk& w) {
#pragma unroll
        for (int f = 0; f < CH / 4; f++) {
            const int cc = min(ch, nch - 1) * (CH / 4) + f;
            const int ws = CL ? cc * N * 64 * WV : cc * 4 * WD * 4, ds = CL ? cc * N * 8 : cc * 8;
#pragma unroll
            for (int n = 0; n < NG; n++) {
#pragma unroll
                for (int q = 0; q < WV; q++) {
                    const U4 t = __builtin_amdgcn_raw_buffer_load_b128(wres, w_off[n] + 16 * q, ws, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) w.c[f][n][q][e] = t[e];
                }
                const U2 d = __builtin_amdgcn_raw_buffer_load_b64(dres, d_off[n], ds, 0);
                w.d[f][n][0] = d[0];
                w.d[f][n][1] = d[1];
            }
        }
    };
    // one lane's code dwords of block b, after the transpose (plain) or as
    // the copy has them
    auto w_order = [&](uint32_t (&c)[WV][4]) {
        if constexpr (CL) {
            if constexpr (WV == 2) {
                // [block][2 dwords] in order -> [dword][block]
                uint32_t a[8];
#pragma unroll
                for (int e = 0; e < 8; e++) a[e] = c[e >> 2][e & 3];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    c[0][b] = a[2 * b];
                    c[1][b] = a[2 * b + 1];
                }
            }
        } else if constexpr (WV == 1) {
            lane_rows_transpose4(c[0]);
        } else {
            // dwords 2k, 2k + 1 of a block belong to lane k
            uint32_t lo[4] = {c[0][0], c[0][2], c[1][0], c[1][2]};
            uint32_t hi[4] = {c[0][1], c[0][3], c[1][1], c[1][3]};
            lane_rows_transpose4(lo);
            lane_rows_transpose4(hi);
#pragma unroll
            for (int b = 0; b < 4; b++) {
                c[0][b] = lo[b];
                c[1][b] = hi[b];
            }
        }
    };
    auto b_operand = [&](const WChunk& w, int n, int j, h8_t& Bh, float& dw) {
        uint4 B;
        const uint32_t(&c)[WV][4] = w.c[j / 4][n];
        if constexpr (WT == Q4) {
            // high nibbles in place: 1024 + 16 n
            const uint32_t P = c[0][j % 4];
            bytes_to_h1024(P & 0xF0F0F0F0u, B.x, B.y);
            bytes_to_h1024(P & 0x0F0F0F0Fu, B.z, B.w);
        } else {
            bytes_to_h1024(c[0][j % 4] ^ 0x80808080u, B.x, B.y);
            bytes_to_h1024(c[WV - 1][j % 4] ^ 0x80808080u, B.z, B.w);
        }
        Bh = __builtin_bit_cast(h8_t, B);
        dw = h2f((uint16_t)(w.d[j / 4][n][(j >> 1) & 1] >> (16 * (j & 1))));
    };

    float acc[MR][NG][4];
#pragma unroll
    for (int m = 0; m < MR; m++)
#pragma unroll
        for (int n = 0; n < NG; n++)
#pragma unroll
            for (int k = 0; k < 4; k++) acc[m][n][k] = 0.0f;

    // weights and activation blocks in a ring of PF chunks (requested PF
    // chunks ahead, every request issued so the waits are exact counts)
    WChunk wr[PF];
    XLane xq[PF][TPT];
#pragma unroll
    for (int p = 0; p < PF; p++) {
        w_load(p, wr[p]);
        x_load(p, xq[p]);
    }
    stage(xq[0], 0);
    lds_barrier();
    auto chunk = [&](int ch, auto pc) {
            constexpr int p = decltype(pc)::value, buf = p;
#pragma unroll
            for (int f = 0; f < CH / 4; f++)
#pragma unroll
                for (int n = 0; n < NG; n++) w_order(wr[p].c[f][n]);
            // steps s = (block j, row group m) in turn: step s's products are
            // issued, then step s - 1's are folded, with the LDS reads of the
            // next RD steps in flight; the fences keep that order (and the
            // registers a deeper interleaving would take)
            auto a_read = [&](int s, uint4& A, f4_t& ci) {
                A = xa[buf][s / MR][s % MR][lane];
                ci = *reinterpret_cast<const f4_t*>(&xc[buf][s / MR][4 * (s % MR) + lg][0]);
            };
            uint4 A[RD + 1];
            f4_t ci[RD + 1], L[2][NG];
            h8_t Bh[NG];
            float dw[2][NG], dx[2][MR];
#pragma unroll
            for (int s = 0; s < RD; s++) a_read(s, A[s], ci[s]);
#pragma unroll
            for (int m = 0; m < MR; m++) dx[0][m] = xd[buf][0][lg][m];
            auto fold = [&](int s) {
                const int j = s / MR, m = s % MR;
#pragma unroll
                for (int n = 0; n < NG; n++) {
                    const float dd = dx[j & 1][m] * dw[j & 1][n];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        acc[m][n][k] = acc[m][n][k] + L[s & 1][n][k] * dd;
                        asm volatile("" : "+v"(acc[m][n][k]));  // the add stays in this step
                    }
                }
            };
#pragma unroll
            for (int s = 0; s < CH * MR; s++) {
                const int j = s / MR, m = s % MR;
                if (m == 0) {
#pragma unroll
                    for (int n = 0; n < NG; n++) {
                        // convert here, not earlier
#pragma unroll
                        for (int q = 0; q < WV; q++) asm volatile("" : "+v"(wr[p].c[j / 4][n][q][j % 4]));
                        b_operand(wr[p], n, j, Bh[n], dw[j & 1][n]);
                    }
                }
                if (s + RD < CH * MR) a_read(s + RD, A[(s + RD) % (RD + 1)], ci[(s + RD) % (RD + 1)]);
                if (m == MR - 1 && j + 1 < CH) {
#pragma unroll
                    for (int mm = 0; mm < MR; mm++) dx[(j + 1) & 1][mm] = xd[buf][j + 1][lg][mm];
                }
#pragma unroll
                for (int n = 0; n < NG; n++)
                    L[s & 1][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, A[s % (RD + 1)]), Bh[n],
                                                                        ci[s % (RD + 1)], 0, 0, 0);
                if (s > 0) fold(s - 1);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            fold(CH * MR - 1);
            __builtin_amdgcn_sched_barrier(0);
            w_load(ch + PF, wr[p]);
            x_load(ch + PF, xq[p]);
            stage(xq[p ^ 1], buf ^ 1);  // past the end: the last chunk again, never read
            lds_barrier();
    };
    int ch = 0;
    for (; ch + 1 < nch; ch += 2) {
        chunk(ch, std::integral_constant<int, 0>{});
        chunk(ch + 1, std::integral_constant<int, 1>{});
    }
    if (ch < nch) chunk(ch, std::integral_constant<int, 0>{});
#pragma unroll
    for (int m = 0; m < MR; m++) {
        const int row = r0 + 4 * m + lg;
        const bool row_ok = row < n_rows;
        float v[NG];
#pragma unroll
        for (int n = 0; n < NG; n++) v[n] = (acc[m][n][0] + acc[m][n][1]) + (acc[m][n][2] + acc[m][n][3]);
        if constexpr (ODT == F32) {
            float* o = reinterpret_cast<float*>(out) + (size_t)row * out_pitch;
#pragma unroll
            for (int n = 0; n < NG; n++)
                if (row_ok && c0 + 16 * n + lc < N) o[c0 + 16 * n + lc] = v[n];
        } else {
            uint8_t* o = reinterpret_cast<uint8_t*>(out) + (size_t)row * out_pitch;
#pragma unroll
            for (int n = 0; n < NG; n += 2) {
                // q8_quant_lane over the block's 16 lanes x 2 columns
                const int ca = c0 + 16 * n + lc, cb2 = ca + 16;
                float a = fmaxf(ca < N ? fabsf(v[n]) : 0.0f, cb2 < N ? fabsf(v[n + 1]) : 0.0f);
                a = quad_max(a);
                a = fmaxf(a, dpp_f<0x141>(a));  // row_half_mirror
                a = fmaxf(a, dpp_f<0x140>(a));  // row_mirror
                const float delta = a / 127.0f;
                const float scale = delta != 0.0f ? 1.0f / delta : 0.0f;
                if (row_ok && ca < N) o[ca] = (uint8_t)(int8_t)roundf(v[n] * scale);
                if (row_ok && cb2 < N) o[cb2] = (uint8_t)(int8_t)roundf(v[n + 1] * scale);
                if (row_ok && lc == 0 && ca < N)
                    reinterpret_cast<uint16_t*>(o + act_delta_offset(N))[ca >> 5] = f2h(delta);
            }
        }
    }
}

// The chunk-major copy of a Q4 / Q8 weight [N, K] (K % 128 == 0) that the
// prefill matmul reads: codes [K/128][N][4 lanes][4 blocks][WV dwords] --
// for each group of four blocks, each row's lane-k code dwords of the four
// blocks side by side -- and deltas [K/128][N][4].
template <int WT>
__global__ void k_chunk_layout(const uint32_t* __restrict__ wq, const uint16_t* __restrict__ wd, int N, int nb,
                               uint32_t* __restrict__ cq, uint16_t* __restrict__ cd)
{
    constexpr int WV = WT == Q4 ? 1 : 2, WD = WV * 4;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one (row, block) each
    if (t >= (int64_t)N * nb) return;
    const int n = (int)(t / nb), b = (int)(t - (int64_t)n * nb);
    const size_t c4 = (size_t)(b >> 2) * N + n;
    const uint32_t* src = wq + t * WD;
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int v = 0; v < WV; v++) cq[((c4 * 4 + k) * 4 + (b & 3)) * WV + v] = src[WV * k + v];
    cd[c4 * 4 + (b & 3)] = wd[t];
}

bool chunk_layout_supported(const nc_tensor* w)
{
    return (w->dtype == NC_Q4 || w->dtype == NC_Q8) && w->cols > 0 && w->cols % 128 == 0 && w->rows > 0;
}

int chunk_layout_launch(const nc_tensor* w, void* codes, void* deltas, hipStream_t st)
{
    if (!chunk_layout_supported(w)) return fail(NC_ERR_ARG, "chunk layout: [%d x %d] dtype %d", w->rows, w->cols, w->dtype);
    const int nb = w->cols / 32;
    const int64_t n = (int64_t)w->rows * nb;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (w->dtype == NC_Q4)
        hipLaunchKernelGGL(k_chunk_layout<Q4>, grid, dim3(256), 0, st, (const uint32_t*)w->data,
                           (const uint16_t*)w->deltas, w->rows, nb, (uint32_t*)codes, (uint16_t*)deltas);
    else
        hipLaunchKernelGGL(k_chunk_layout<Q8>, grid, dim3(256), 0, st, (const uint32_t*)w->data,
                           (const uint16_t*)w->deltas, w->rows, nb, (uint32_t*)codes, (uint16_t*)deltas);
    return launch_status("k_chunk_layout");
}

// Workgroup shapes, measured on MI355X (us per launch, every launch after a
// 512 MB write that evicts L2 and the memory-side cache, as a prefill meets
// its weights; over the chunk-major copy / the weight's own layout; Q4, Q8 in
// brackets).
//   rows x N x K (groups)    8 x 32                     8 x 64
//   16 x 2048 x 2048 (64)    12.2 / 12.8 [13.1 / 13.9]  12.2 / 13.6 [14.0 / 15.0]
//   64 x 2560 x 2048 (320)   15.9 / 17.4 [17.6 / 20.1]  14.9 / 17.5 [17.9 / 21.1]
//   128 x 2048 x 5632 (512)  35.8 / 38.8 [40.2 / 46.7]  33.4 / 37.2 [38.9 / 45.1]
//   201 x 2048 x 2048 (832)  30.0 / 35.6 [36.9 / 43.8]  22.7 / 29.6 [32.0 / 37.8]
//   128 x 6144 x 2048 (1536) 47.8 / 57.5 [59.0 / 68.8]  32.3 / 42.8 [45.9 / 55.2]
//   512 x 6912 x 2304 (6912) 180 / 192 [203 / 220]      118 / 134 [163 / 171]
//                            16 x 64                    16 x 128
//   16 x 2048 x 2048         19.7 / 18.4 [21.2 / 22.6]  25.9 / 26.5 [28.3 / 30.7]
//   64 x 2560 x 2048         19.3 / 18.9 [21.4 / 22.8]  25.0 / 26.6 [27.9 / 29.8]
//   128 x 2048 x 5632        45.8 / 44.8 [50.2 / 52.6]  60.0 / 61.8 [66.0 / 71.6]
//   201 x 2048 x 2048        22.7 / 23.9 [24.9 / 26.0]  26.1 / 28.1 [28.7 / 30.8]
//   128 x 6144 x 2048        29.3 / 32.5 [32.6 / 37.2]  32.2 / 36.3 [36.6 / 39.8]
//   512 x 6912 x 2304        109 / 118 [119 / 127]      99 / 109 [112 / 123]
// 8 x 128 is not among them: of 1108 such calls it was the best by more than 3%
// in one.  The kernel before (one column group per wavefront, the compiler's
// order of LDS reads and folds): 201 x 2048 x 2048 27.0 / 31.5 [26.8 / 31.3], 512 x
// 6912 x 2304 136 / 194 [162 / 194].  At 512 x 11520 x 2304 the 16 x 128 launch keeps
// the vector unit busy (see the kernel); holding LDS operands two steps ahead
// or taking the d_x d_w products from the matrix cores changed nothing there.
//
// The rule follows the workgroups that 8 rows x 64 columns would have.  Up to
// kTiny of them Q8 takes half the columns each, for twice as many (Q4, with half
// the bytes to wait for, gains nothing: 8 x 1280 x 1280 9.4 / 9.6).  Up to three per
// CU 8 x 64, whose time then steps up (Q8 plain 160 x 2560 x 2048, 800 of them:
// 38.0, 16 x 64 26.1; 160 x 2304 x 2304, 720: 27.2 / 27.6); Q4 over the chunk-major
// copy, with the cheapest operands, up to five.  Then 16 x 64, which shares the
// converted weights over twice the rows, and from kBig 16 x 128, which shares
// the activation operands too.
constexpr int kTiny = 96, kBig = 1600;
constexpr int small_groups(int dtype, bool cl) { return dtype == NC_Q4 && cl ? 1280 : 768; }

static int64_t groups8x64(int N, int n_rows) { return (int64_t)((N + 63) / 64) * ((n_rows + 7) / 8); }

enum GemmShape { kGemmNone, kGemm8x32, kGemm8x64, kGemm8x128, kGemm16x64, kGemm16x128 };

// The k_gemm_qw shape of this product, kGemmNone when it is not taken: its
// chunks are four blocks, its loads need whole dwords, and its offsets are 32
// bits.  cl: w is the chunk-major copy.
static GemmShape gemm_shape(int x_pitch, int n_rows, const nc_tensor* w, bool cl)
{
    const int N = w->rows, nb = w->cols / 32;
    const size_t lim = (size_t)1 << 31;
    if (w->cols % 128 || ((uintptr_t)w->data & 3) || ((uintptr_t)w->deltas & 3)) return kGemmNone;
    if ((size_t)N * nb * (w->dtype == NC_Q4 ? 16 : 32) >= lim || (size_t)n_rows * x_pitch >= lim) return kGemmNone;
    const int64_t groups = groups8x64(N, n_rows);
    if (w->dtype == NC_Q8 && groups <= kTiny && nb % 8 == 0) return kGemm8x32;
    if (groups <= small_groups(w->dtype, cl)) return kGemm8x64;
    return groups <= kBig ? kGemm16x64 : kGemm16x128;
}

// The shape that stores Q8 rows itself, kGemmNone where the fp32 product and
// a pass that quantizes its rows take less time: a 32-column block needs both its
// column groups in one wavefront, so 16 x 128 where that is the product's own
// shape, else 8 x 128 for Q4 weights up to K = 2304, where it costs less than the
// pass (us back to back, 8 x 128 / 16 x 64 and the pass: 256 x 2048 x 1024 13.6 /
// 15.4, 160 x 4096 x 1536 22.6 / 23.6, 33 x 11264 x 2048 25.9 / 29.0; 201 x 2048 x 5632
// 56.2 / 53.3; Q8 weights 201 x 2048 x 2048 30.8 / 25.5).
static GemmShape gemm_act_shape(int x_pitch, int n_rows, const nc_tensor* w)
{
    const GemmShape shape = gemm_shape(x_pitch, n_rows, w, false);
    if (shape == kGemm16x64 && w->dtype == NC_Q4 && w->cols <= 2304) return kGemm8x128;
    return shape == kGemm16x128 ? shape : kGemmNone;
}

template <int ODT>
static int gemm_qw(const uint8_t* x, int x_pitch, int n_rows, const nc_tensor* w, bool cl, GemmShape shape, void* out,
                   int out_pitch, hipStream_t st, hipEvent_t ev_start, hipEvent_t ev_stop)
{
    const int N = w->rows, nb = w->cols / 32;
    const int rows = shape >= kGemm16x64 ? 16 : 8, cols = shape == kGemm8x32 ? 32 : shape == kGemm8x128 || shape == kGemm16x128 ? 128 : 64;
    auto go = [&](auto kern) {
        const dim3 grid((N + cols - 1) / cols, (n_rows + rows - 1) / rows), block(shape == kGemm8x32 ? 128 : 256);
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, block, 0, st, ev_start, ev_stop, 0, x, x_pitch, n_rows,
                                  (const uint32_t*)w->data, (const uint16_t*)w->deltas, out, out_pitch, N, nb);
        else
            hipLaunchKernelGGL(kern, grid, block, 0, st, x, x_pitch, n_rows, (const uint32_t*)w->data,
                               (const uint16_t*)w->deltas, out, out_pitch, N, nb);
    };
    auto by_layout = [&](auto wt, auto c) {
        constexpr int WT = decltype(wt)::value;
        constexpr bool CL = decltype(c)::value;
        if (shape == kGemm16x128) return go(k_gemm_qw<WT, 4, 2, 4, 4, 1, CL, 3, ODT>);
        if constexpr (ODT == Q8 && WT == Q4 && !CL) {
            if (shape == kGemm8x128) return go(k_gemm_qw<WT, 2, 2, 4, 4, 1, CL, 4, ODT>);
        }
        if constexpr (ODT == F32) {
            if (shape == kGemm16x64) return go(k_gemm_qw<WT, 4, 1, 4, 4, 1, CL, 2, ODT>);
            if constexpr (WT == Q8)
                if (shape == kGemm8x32) return go(k_gemm_qw<WT, 2, 1, 2, 8, 2, CL, 2, ODT>);
            // eight blocks per barrier while the workgroups are few (64 x 2560 x
            // 2048 Q4: 14.9, 16.1 with four), four where their smaller shared
            // memory lets more of them share a CU (256 x 2048 x 2048: 22.9, 23.7
            // with eight)
            if (nb % 8 == 0 && groups8x64(N, n_rows) <= 512) return go(k_gemm_qw<WT, 2, 1, 4, 8, 2, CL, 2, ODT>);
            return go(k_gemm_qw<WT, 2, 1, 4, 4, 1, CL, 2, ODT>);
        }
    };
    auto by_type = [&](auto wt) {
        if constexpr (ODT == F32) {
            if (cl) return by_layout(wt, std::true_type{});
        }
        by_layout(wt, std::false_type{});
    };
    if (w->dtype == NC_Q4) by_type(std::integral_constant<int, Q4>{});
    else by_type(std::integral_constant<int, Q8>{});
    return launch_status("k_gemm_qw");
}

const char* gemm_route(int x_pitch, int n_rows, const nc_tensor* w, bool act)
{
    switch (act ? gemm_act_shape(x_pitch, n_rows, w) : gemm_shape(x_pitch, n_rows, w, false)) {
    case kGemm8x32: return "k_gemm_qw 8x32";
    case kGemm8x64: return "k_gemm_qw 8x64";
    case kGemm8x128: return "k_gemm_qw 8x128";
    case kGemm16x64: return "k_gemm_qw 16x64";
    case kGemm16x128: return "k_gemm_qw 16x128";
    default: return "k_gemm_q";
    }
}

bool gemm_q_act_supported(int x_pitch, int n_rows, const nc_tensor* w)
{
    return (w->dtype == NC_Q4 || w->dtype == NC_Q8) && n_rows >= kGemmMinRows &&
           gemm_act_shape(x_pitch, n_rows, w) != kGemmNone;
}

int gemm_q_act(const uint8_t* x, int x_pitch, int n_rows, const nc_tensor* w, uint8_t* out, int out_pitch,
               hipStream_t st)
{
    if (!gemm_q_act_supported(x_pitch, n_rows, w))
        return fail(NC_ERR_ARG, "gemm to Q8 rows: [%d x %d] weights, %d rows", w->rows, w->cols, n_rows);
    return gemm_qw<Q8>(x, x_pitch, n_rows, w, false, gemm_act_shape(x_pitch, n_rows, w), out, out_pitch, st, nullptr,
                       nullptr);
}

int gemm_q_raw(const uint8_t* x, int x_pitch, int n_rows, const nc_tensor* w, float* out, int out_pitch,
               hipStream_t st, hipEvent_t ev_start, hipEvent_t ev_stop, const nc_tensor* wc)
{
    if (w->dtype != NC_Q4 && w->dtype != NC_Q8) return fail(NC_ERR_ARG, "gemm: Q4/Q8 weights only");
    if (w->cols % 32 || w->cols <= 0 || w->rows <= 0 || n_rows <= 0)
        return fail(NC_ERR_ARG, "gemm: [%d x %d] weights, %d rows", w->rows, w->cols, n_rows);
    const int N = w->rows, nb = w->cols / 32;
    if (wc && (wc->dtype != w->dtype || wc->rows != N || wc->cols != w->cols || !chunk_layout_supported(wc)))
        return fail(NC_ERR_ARG, "gemm: chunk copy [%d x %d] of a [%d x %d] weight", wc->rows, wc->cols, N, w->cols);
    // the chunk-major copy, when the caller has one
    const nc_tensor* wt = wc ? wc : w;
    if (const GemmShape shape = gemm_shape(x_pitch, n_rows, wt, wc != nullptr))
        return gemm_qw<F32>(x, x_pitch, n_rows, wt, wc != nullptr, shape, out, out_pitch, st, ev_start, ev_stop);
    // (NG, NW, MR, PF): 512 rows (1, 2, 8, 4), tall weights (2, 2, 8, 3);
    // 64 rows (1, 1, 4, 3), tall (1, 2, 8, 4)
    auto go = [&](auto kern, int mr, int ng, int nw) {
        const dim3 grid((N + 16 * ng * nw - 1) / (16 * ng * nw), (n_rows + 4 * mr - 1) / (4 * mr));
        if (ev_start)
            hipExtLaunchKernelGGL(kern, grid, dim3(64 * nw), 0, st, ev_start, ev_stop, 0, x, x_pitch, n_rows,
                                  (const uint32_t*)w->data, (const uint16_t*)w->deltas, out, out_pitch, N, nb);
        else
            hipLaunchKernelGGL(kern, grid, dim3(64 * nw), 0, st, x, x_pitch, n_rows, (const uint32_t*)w->data,
                               (const uint16_t*)w->deltas, out, out_pitch, N, nb);
    };
    const bool wide = n_rows >= 256, tall = N >= 8192;
    auto by_type = [&](auto t) {
        constexpr int WT = decltype(t)::value;
        if (wide && tall) go(k_gemm_q<WT, 2, 2, 8, 3>, 8, 2, 2);
        else if (wide || (tall && n_rows >= 32)) go(k_gemm_q<WT, 1, 2, 8, 4>, 8, 1, 2);
        else go(k_gemm_q<WT, 1, 1, 4, 3>, 4, 1, 1);
    };
    if (w->dtype == NC_Q4) by_type(std::integral_constant<int, Q4>{});
    else by_type(std::integral_constant<int, Q8>{});
    return launch_status("k_gemm_q");
}

}  // namespace nc
