// Wide int8 GEMM on the gfx950 matrix cores, for forwards of many token
// rows at once (prefill chunks, batched verify across sessions), and the
// elementwise producers of its quantized inputs.
//
// o[t][n] = 0.0f + (sum_s float(acc[t,n,s]) * xs[t][s]) * ws[n]
// with acc the exact int32 sum over the 32-element group s
// (lz_matmul_xq_nt -> matmul_q8_impl + epi_q8, src/ops_matmul.c:336-466,
// src/ops_epi.c:983-1017).  v_mfma_i32_16x16x32_i8 contracts exactly one
// 32-element group: started from a zero accumulator it returns the exact
// group sums of a 16 x 16 (row, token) tile, which the lanes then fold into
// fp32 in group order, one multiply and one add per group and output, as
// the reference's epilogue does (a one-group row, K == 32, takes the
// reference's r == 1 association instead: epi_one_group).  The result is bit-identical to the GEMV
// path for every token, whatever the number of tokens.
//
// Operand layout of the 16x16x32 int8 MFMA (64 lanes): lane l supplies
// A[l % 16][8 (l / 16) .. +8) and B[8 (l / 16) .. +8)[l % 16] as eight
// bytes each, and receives D[4 (l / 16) + v][l % 16] in result register v.
// A is the weight tile (rows), B the activation tile (tokens).
//
// Three kernels: k_mfma_q8t for K a multiple of 128 (every configuration of
// bench.py); for any other K (the toy models' 32, 64, 96, ..., an expert width
// of 704 or 1344) k_mfma_q8, blocks of 16 weight rows x 64 token columns (a wave
// per 16 columns), K through double-buffered LDS stages of MF_KC bytes (eight
// groups), and its narrow form k_mfma_q8n, 64 weight rows x 16 token columns.
#include "l98_devmath.h"
#include "l98_launch.h"

typedef int v4i_t __attribute__((ext_vector_type(4)));

#define MF_THREADS 256
#define MF_ROWS 16        // weight rows per block
#define MF_COLS 64        // token columns per block (16 per wave)
#define MF_KC 256         // K bytes (eight groups) per LDS stage
#define MF_LDS_ROW (MF_KC + 16)   // padded stage row: the lanes' 8-byte operand reads spread over the banks

// Columns of a launch: dense (column t is activation row t and output row
// t, t < M) or grouped (block z is group g: expert gexp[g], columns
// list[goff[g] .. goff[g] + gcnt[g]), activation row xmap[col] or col,
// output row col).
// Dense GEMMs over the same rows sharing a launch: job j covers block rows
// [blk0, next job's blk0) of the grid's x, with its own weights, input (X,
// Xs, K) and output; n == 0: the launch's own arguments.
#define MF_MAX_JOBS 6
struct MfJob {
    const int8_t *W;
    const float *ws;
    float *out;
    const int8_t *X;
    const float *Xs;
    int N, out_stride, blk0, K;
};
struct MfJobs {
    MfJob j[MF_MAX_JOBS];
    int n, pad[3];
};

struct MfCols {
    const int *gexp, *goff, *gcnt, *list, *xmap;
    const int *ng;           // groups actually present (device)
};

// One LDS stage of k_mfma_q8 in a thread's registers (set R: Aw0 .. At1): its
// 16-byte piece of a weight row and four of activation columns, and two of the
// block's 64 x 8 activation group scales (column tid / 4, groups 2 (tid % 4) and
// the next).  Plain locals (a struct would be kept in scratch memory across the
// scheduling barriers that hold the loads' issue in place).
static_assert(MF_KC == 256 && MF_THREADS == 256, "a stage: eight group scales per column, two per thread");
#define MF_STAGE_LOAD(R, st_)                                                                  \
    do {                                                                                       \
        const int off_ = imin((st_) * MF_KC + 16 * pc, K - 16);                                \
        R##w0 = *reinterpret_cast<const int4 *>(wl0 + off_);                                   \
        R##x0 = *reinterpret_cast<const int4 *>(xl0 + off_);                                   \
        R##x1 = *reinterpret_cast<const int4 *>(xl1 + off_);                                   \
        R##x2 = *reinterpret_cast<const int4 *>(xl2 + off_);                                   \
        R##x3 = *reinterpret_cast<const int4 *>(xl3 + off_);                                   \
        const int g_ = (st_) * (MF_KC / 32) + 2 * (tid & 3);                                   \
        R##t0 = xsl[imin(g_, nb - 1)];                                                         \
        R##t1 = xsl[imin(g_ + 1, nb - 1)];                                                     \
    } while (0)
#define MF_STAGE_PUT(R, b_)                                                                    \
    do {                                                                                       \
        *reinterpret_cast<int4 *>(&s_w[b_][rr][16 * pc]) = R##w0;                              \
        *reinterpret_cast<int4 *>(&s_x[b_][rr][16 * pc]) = R##x0;                              \
        *reinterpret_cast<int4 *>(&s_x[b_][rr + 16][16 * pc]) = R##x1;                         \
        *reinterpret_cast<int4 *>(&s_x[b_][rr + 32][16 * pc]) = R##x2;                         \
        *reinterpret_cast<int4 *>(&s_x[b_][rr + 48][16 * pc]) = R##x3;                         \
        *reinterpret_cast<float2 *>(&s_xs[b_][tid >> 2][2 * (tid & 3)]) = make_float2(R##t0, R##t1); \
    } while (0)

__device__ __forceinline__ void mf_fold(float (&f)[4], v4i_t d, float s, bool one) {
    f[0] += one ? (float)d[0] : (float)d[0] * s;
    f[1] += one ? (float)d[1] : (float)d[1] * s;
    f[2] += one ? (float)d[2] : (float)d[2] * s;
    f[3] += one ? (float)d[3] : (float)d[3] * s;
}
__device__ __forceinline__ void mf_stage(float (&f)[4], const int8_t (*sw)[MF_LDS_ROW], const int8_t (*sx)[MF_LDS_ROW],
                                         const float *sc, int ng, bool one, int wave, int lane, int kq) {
    const v4i_t zero = {0, 0, 0, 0};
#pragma unroll
    for (int gl = 0; gl < MF_KC / 32; gl++) {
        if (gl >= ng) break;                           // uniform
        const long b = *reinterpret_cast<const long *>(&sx[16 * wave + (lane & 15)][32 * gl + kq]);
        const long a = *reinterpret_cast<const long *>(&sw[(lane & 15)][32 * gl + kq]);
        mf_fold(f, __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, zero, 0, 0, 0), sc[gl], one);
    }
}

__global__ __launch_bounds__(MF_THREADS) void k_mfma_q8(const int8_t *__restrict__ W0, const float *__restrict__ ws0,
                                                         int N0, int K0, size_t w_group_stride,
                                                         const int8_t *__restrict__ X0, const float *__restrict__ Xs0,
                                                         int M, MfCols cols, float *__restrict__ out0,
                                                         int out_stride0, MfJobs jobs) {
    __shared__ __align__(16) int8_t s_w[2][MF_ROWS][MF_LDS_ROW];
    __shared__ __align__(16) int8_t s_x[2][MF_COLS][MF_LDS_ROW];
    __shared__ __align__(16) float s_xs[2][MF_COLS][MF_KC / 32];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int8_t *W = W0;
    const float *ws = ws0;
    float *out = out0;
    const int8_t *X = X0;
    const float *Xs = Xs0;
    int N = N0, K = K0, out_stride = out_stride0, bx = blockIdx.x;
    if (jobs.n) {
        // the job whose block rows hold this block (the index is uniform)
        int ji = 0;
#pragma unroll
        for (int k = 1; k < MF_MAX_JOBS; k++)
            if (k < jobs.n && bx >= jobs.j[k].blk0) ji = k;
        const MfJob jb = jobs.j[ji];
        W = jb.W;
        ws = jb.ws;
        out = jb.out;
        X = jb.X;
        Xs = jb.Xs;
        K = jb.K;
        N = jb.N;
        out_stride = jb.out_stride;
        bx -= jb.blk0;
    }
    const int n0 = bx * MF_ROWS;
    const int nb = K >> 5;
    int ncols = M, cbase = 0;
    const int8_t *Wg = W;
    const float *wsg = ws;
    if (cols.list) {
        const int g = blockIdx.z;
        if (g >= *cols.ng) return;
        ncols = cols.gcnt[g];
        cbase = cols.goff[g];
        const int e = cols.gexp[g];
        Wg = W + (size_t)e * w_group_stride;
        wsg = ws + (size_t)e * N;
    }
    // column tiles blockIdx.y, + gridDim.y, ... (a grouped launch has one
    // block row per group, which walks the group's tiles)
#pragma unroll 1
    for (int c0 = blockIdx.y * MF_COLS; c0 < ncols; c0 += gridDim.y * MF_COLS) {
        // this lane's B column and its output row
        const int cl = c0 + 16 * wave + (lane & 15);
        const int cc = cl < ncols ? cl : ncols - 1;
        const int orow = cols.list ? cols.list[cbase + cc] : cc;
        const int kq = 8 * (lane >> 4);
        // Stage loads: thread t takes the 16-byte piece pc of weight row rr and
        // activation columns rr + 16 j (j < 4) of the block: every row's MF_KC-byte
        // stage is read by 16 consecutive threads.  Rows past N and columns past
        // ncols repeat the last; pieces past K repeat the row's last piece (their
        // groups are not used).
        const int pc = tid & 15, rr = tid >> 4;
        auto xcol = [&](int j) {
            const int c = imin(c0 + rr + 16 * j, ncols - 1);
            int xr = c;
            if (cols.list) {
                const int o = cols.list[cbase + c];
                xr = cols.xmap ? cols.xmap[o] : o;
            }
            return X + (size_t)xr * K;
        };
        const int8_t *wl0 = Wg + (size_t)imin(n0 + rr, N - 1) * K;
        const int8_t *xl0 = xcol(0), *xl1 = xcol(1), *xl2 = xcol(2), *xl3 = xcol(3);
        // the activation scales this thread stages: column tid / 4
        const float *xsl;
        {
            const int c = imin(c0 + (tid >> 2), ncols - 1);
            int xr = c;
            if (cols.list) {
                const int o = cols.list[cbase + c];
                xr = cols.xmap ? cols.xmap[o] : o;
            }
            xsl = Xs + (size_t)xr * nb;
        }
        const int nst = (K + MF_KC - 1) / MF_KC;
        int4 Aw0, Ax0, Ax1, Ax2, Ax3;
        float At0, At1;
        float f[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        // one group (K == 32): f holds the exact group sum (|acc| < 2^24) for
        // epi_one_group's association
        const bool one = nb == 1;
        float s0 = 0.0f;
        MF_STAGE_LOAD(A, 0);
        MF_STAGE_PUT(A, 0);
        __syncthreads();
#pragma unroll 1
        for (int st = 0; st < nst; st++) {
            const int buf = st & 1;
            const float *sc = s_xs[buf][16 * wave + (lane & 15)];
            // the next stage's loads are in flight during this stage's MFMAs (the
            // last stage reloads itself into the idle buffer); the scheduling
            // barrier keeps their issue ahead of the MFMAs
            MF_STAGE_LOAD(A, st + 1 < nst ? st + 1 : st);
            __builtin_amdgcn_sched_barrier(0);
            mf_stage(f, s_w[buf], s_x[buf], sc, nb - st * (MF_KC / 32), one, wave, lane, kq);
            if (one) s0 = sc[0];
            MF_STAGE_PUT(A, buf ^ 1);
            __syncthreads();
        }
        // (after the last stage's barrier no wave reads this tile's LDS, so the
        // next tile may refill it)
        if (cl < ncols) {
            float *op = out + (size_t)orow * out_stride;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int n = n0 + 4 * (lane >> 4) + v;
                if (n < N) {
                    float sum = 0.0f;
                    if (one) sum = epi_one_group((int)f[v], s0, wsg[n]);
                    else sum += f[v] * wsg[n];
                    op[n] = sum;
                }
            }
        }
    }
}

#undef MF_STAGE_LOAD
#undef MF_STAGE_PUT

// The narrow form of k_mfma_q8: a block computes 64 weight rows x 16 token
// columns (wave w: rows 16 w .. 16 w + 15 of the same 16 columns), so each block
// streams four times the weights of k_mfma_q8's 16-row tile and stages only the
// 16 columns it uses, and the loads run two stages ahead (register sets A and B
// alternate) - for few columns per weight tile, where a stage's round trip, not
// the arithmetic, bounds the block (mf_narrow and the grouped launches say
// where).  Dense (cols.list null: column t is activation and output row t, t < M;
// jobs as in k_mfma_q8; a 1-D grid mapped onto the XCDs so that the column tiles
// of a weight tile share an L2) or grouped (block z is group g; a group's column
// tiles spread over the grid's y, whose extra blocks exit at once).  Same MFMAs
// and fold per (row, column) as k_mfma_q8, so the same bits.
#define MFN_ROWS 64
#define MFN_COLS 16
#define MFN_STAGE_LOAD(R, st_)                                                                 \
    do {                                                                                       \
        const int off_ = imin((st_) * MF_KC + 16 * pc, K - 16);                                \
        R##w0 = *reinterpret_cast<const int4 *>(wl0 + off_);                                   \
        R##w1 = *reinterpret_cast<const int4 *>(wl1 + off_);                                   \
        R##w2 = *reinterpret_cast<const int4 *>(wl2 + off_);                                   \
        R##w3 = *reinterpret_cast<const int4 *>(wl3 + off_);                                   \
        R##x0 = *reinterpret_cast<const int4 *>(xl0 + off_);                                   \
        if (tid < 64) {                                                                        \
            const int g_ = (st_) * (MF_KC / 32) + 2 * (tid & 3);                               \
            R##t0 = xsl[imin(g_, nb - 1)];                                                     \
            R##t1 = xsl[imin(g_ + 1, nb - 1)];                                                 \
        }                                                                                      \
    } while (0)
#define MFN_STAGE_PUT(R, b_)                                                                   \
    do {                                                                                       \
        *reinterpret_cast<int4 *>(&s_w[b_][rr][16 * pc]) = R##w0;                              \
        *reinterpret_cast<int4 *>(&s_w[b_][rr + 16][16 * pc]) = R##w1;                         \
        *reinterpret_cast<int4 *>(&s_w[b_][rr + 32][16 * pc]) = R##w2;                         \
        *reinterpret_cast<int4 *>(&s_w[b_][rr + 48][16 * pc]) = R##w3;                         \
        *reinterpret_cast<int4 *>(&s_x[b_][rr][16 * pc]) = R##x0;                              \
        if (tid < 64) *reinterpret_cast<float2 *>(&s_xs[b_][tid >> 2][2 * (tid & 3)]) = make_float2(R##t0, R##t1); \
    } while (0)
__global__ __launch_bounds__(MF_THREADS) void k_mfma_q8n(const int8_t *__restrict__ W0, const float *__restrict__ ws0,
                                                          int N0, int K0, size_t w_group_stride,
                                                          const int8_t *__restrict__ X0, const float *__restrict__ Xs0,
                                                          int M, MfCols cols, float *__restrict__ out0,
                                                          int out_stride0, MfJobs jobs) {
    __shared__ __align__(16) int8_t s_w[2][MFN_ROWS][MF_LDS_ROW];
    __shared__ __align__(16) int8_t s_x[2][MFN_COLS][MF_LDS_ROW];
    __shared__ __align__(16) float s_xs[2][MFN_COLS][MF_KC / 32];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int8_t *W = W0;
    const float *ws = ws0;
    float *out = out0;
    const int8_t *X = X0;
    const float *Xs = Xs0;
    int N = N0, K = K0, out_stride = out_stride0, bx = blockIdx.x;
    int cy = blockIdx.y, cys = gridDim.y;
    if (!cols.list) {
        // Dense: a 1-D grid of (row tiles rounded up to 8) x column tiles.
        // Blocks go to the 8 XCDs in turn by linear index, so block L runs on
        // XCD L % 8; give XCD x the row tiles x, x + 8, ... with all their
        // column tiles one after another, so the column tiles that share a
        // weight tile share that XCD's L2 (weights read from HBM once).
        const int ny = (M + MFN_COLS - 1) / MFN_COLS, xcd = bx & 7, sl = bx >> 3, q = sl / ny;
        bx = q * 8 + xcd;
        cy = sl - q * ny;
        cys = ny;
        const int nrt = jobs.n ? jobs.j[jobs.n - 1].blk0 + (jobs.j[jobs.n - 1].N + MFN_ROWS - 1) / MFN_ROWS
                               : (N0 + MFN_ROWS - 1) / MFN_ROWS;
        if (bx >= nrt) return;
    }
    if (jobs.n) {
        int ji = 0;
#pragma unroll
        for (int k = 1; k < MF_MAX_JOBS; k++)
            if (k < jobs.n && bx >= jobs.j[k].blk0) ji = k;
        const MfJob jb = jobs.j[ji];
        W = jb.W;
        ws = jb.ws;
        out = jb.out;
        X = jb.X;
        Xs = jb.Xs;
        K = jb.K;
        N = jb.N;
        out_stride = jb.out_stride;
        bx -= jb.blk0;
    }
    int ncols = M, cbase = 0;
    const int8_t *Wg = W;
    const float *wsg = ws;
    if (cols.list) {
        const int g = blockIdx.z;
        if (g >= *cols.ng) return;
        ncols = cols.gcnt[g];
        cbase = cols.goff[g];
        const int e = cols.gexp[g];
        Wg = W + (size_t)e * w_group_stride;
        wsg = ws + (size_t)e * N;
    }
    const int n0 = bx * MFN_ROWS, nb = K >> 5;
    const int pc = tid & 15, rr = tid >> 4;
    auto wrow = [&](int j) { const int r = n0 + rr + 16 * j; return Wg + (size_t)(r < N ? r : N - 1) * K; };
    const int8_t *wl0 = wrow(0), *wl1 = wrow(1), *wl2 = wrow(2), *wl3 = wrow(3);
    const int kq = 8 * (lane >> 4);
    const int nst = (K + MF_KC - 1) / MF_KC;
#pragma unroll 1
    for (int c0 = cy * MFN_COLS; c0 < ncols; c0 += cys * MFN_COLS) {
        auto xrow = [&](int c) {
            const int cc = imin(c0 + c, ncols - 1);
            if (!cols.list) return cc;
            const int o = cols.list[cbase + cc];
            return cols.xmap ? cols.xmap[o] : o;
        };
        const int8_t *xl0 = X + (size_t)xrow(rr) * K;                  // column rr's piece pc
        const float *xsl = Xs + (size_t)xrow(tid >> 2) * nb;            // threads < 64: column tid / 4
        const int cl = c0 + (lane & 15);
        int4 Aw0, Aw1, Aw2, Aw3, Ax0, Bw0, Bw1, Bw2, Bw3, Bx0;
        float At0 = 0.0f, At1 = 0.0f, Bt0 = 0.0f, Bt1 = 0.0f;
        float f[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        const bool one = nb == 1;
        float s0 = 0.0f;
        auto compute = [&](int buf, int st) {
            const float *sc = s_xs[buf][lane & 15];
            const v4i_t zero = {0, 0, 0, 0};
            const int ng = nb - st * (MF_KC / 32);
#pragma unroll
            for (int gl = 0; gl < MF_KC / 32; gl++) {
                if (gl >= ng) break;                               // uniform
                const long b = *reinterpret_cast<const long *>(&s_x[buf][lane & 15][32 * gl + kq]);
                const long a = *reinterpret_cast<const long *>(&s_w[buf][16 * wave + (lane & 15)][32 * gl + kq]);
                const v4i_t dd = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, zero, 0, 0, 0);
                mf_fold(f, dd, sc[gl], one);
            }
            if (one) s0 = sc[0];
        };
        // stage st in buffer st % 2; the loads of stages st + 1 and st + 2
        // in flight while it runs (stages past the last reload the last)
        MFN_STAGE_LOAD(A, 0);
        MFN_STAGE_PUT(A, 0);
        __syncthreads();
        MFN_STAGE_LOAD(A, imin(1, nst - 1));
#pragma unroll 1
        for (int st = 0; st < nst; st += 2) {
            MFN_STAGE_LOAD(B, imin(st + 2, nst - 1));
            __builtin_amdgcn_sched_barrier(0);
            compute(0, st);
            MFN_STAGE_PUT(A, 1);
            __syncthreads();
            if (st + 1 >= nst) break;                          // uniform
            MFN_STAGE_LOAD(A, imin(st + 3, nst - 1));
            __builtin_amdgcn_sched_barrier(0);
            compute(1, st + 1);
            MFN_STAGE_PUT(B, 0);
            __syncthreads();
        }
        if (cl < ncols) {
            float *op = out + (size_t)(cols.list ? cols.list[cbase + cl] : cl) * out_stride;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int n = n0 + 16 * wave + 4 * (lane >> 4) + v;
                if (n < N) {
                    float sum = 0.0f;
                    if (one) sum = epi_one_group((int)f[v], s0, wsg[n]);
                    else sum += f[v] * wsg[n];
                    op[n] = sum;
                }
            }
        }
    }
}
#undef MFN_STAGE_LOAD
#undef MFN_STAGE_PUT

// The tiled form, for many columns per weight row: a block of WR x WC waves
// computes 16 RT WR weight rows x 16 CT WC token columns, a wave 16 RT x 16 CT
// (RT x CT MFMA tiles per group, whose operands are read from LDS RT + CT
// times).  K goes through LDS in stages of 128 bytes (four groups) in four
// buffers, loaded by the LDS direct loads (no registers, no store
// instructions), three stages ahead.  A direct load's wave writes 64
// consecutive 16-byte pieces, so a stage's rows lie unpadded and their pieces
// are permuted instead: piece p of row r is at p ^ ((r >> 1) & 7), and the 16
// rows of an operand read fall on different banks.
//
// The fold takes the MFMA's result as a float without a conversion: the
// accumulator starts from the bits of 1.5 * 2^23, to which the integer sum
// |acc| <= 32 * 128 * 127 < 2^22 is added in the float's last places, and
// subtracting 1.5 * 2^23 leaves float(acc) exactly (a conversion takes twice
// a subtraction's cycles).
//
// Same group sums and the same multiply and add per group in order as
// k_mfma_q8, so the same bits.  K % 128 == 0.
#define MFT_KC 128
#define MFT_NB 4
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) void *mft_gptr;
typedef __attribute__((address_space(3))) void *mft_lptr;

// All but the last n of the wave's loads arrived, its LDS reads done, then
// the block's barrier: the next stage is whole and the buffer before it free.
template <int N>
__device__ __forceinline__ void mft_arrive() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

//
// PAIR (grouped only; RT = 2, WR = 2): the experts' w1 and w3 of the same 32
// rows as one block's 64, a wave's two tiles being its 16 rows of each, so
// that the lane holding w1's output holds w3's, and the block the whole
// 32-element group of a column: it leaves silu(w1) * w3 quantized per 32
// (mode 1 of k_wide_pro, the same arithmetic), and neither float matrix is
// written.
struct MfPair {
    const int8_t *W3;                   // w3's bank and scales
    const float *ws3;
    int8_t *q;                          // [pairs][N] and [pairs][N / 32]
    float *qs;
};
template <int RT, int CT, int WR, int WC, bool PAIR = false>
__global__ __launch_bounds__(64 * WR * WC) void k_mfma_q8t(const int8_t *W0, const float *ws0, int N0, int K0,
                                                           size_t w_group_stride, const int8_t *X0, const float *Xs0,
                                                           int M, MfCols cols, float *out0, int out_stride0,
                                                           MfJobs jobs, MfPair pair) {
    constexpr int TR = 16 * RT * WR, TC = 16 * CT * WC;   // the block's tile
    constexpr int ORT = PAIR ? TR / 2 : TR;               // output rows of a tile
    constexpr int AST = (PAIR ? 32 : 16) * MFT_KC;        // between a wave's tiles in LDS
    static_assert(!PAIR || (RT == 2 && WR == 2 && CT == 1), "a pair tile: 32 rows of each bank");
    constexpr int NTHR = 64 * WR * WC, PW = TR * 8 / NTHR, PX = TC * 8 / NTHR, SL = TC / (WR * WC);
    static_assert(TR * 8 % NTHR == 0 && TC * 8 % NTHR == 0 && SL <= 64, "whole direct loads");
    constexpr int LPS = PW + PX + 1;                      // direct loads of a wave per stage
    // a buffer: weight rows, activation columns, column scales.  One array: of
    // several the compiler would know which a direct load fills, and wait for
    // all loads in flight before reading any
    constexpr int XO = TR * MFT_KC, SO = XO + TC * MFT_KC, BUF = SO + TC * 16;
    __shared__ __align__(16) int8_t s_buf[MFT_NB][BUF];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int bx = blockIdx.x, cy = blockIdx.y, cys = gridDim.y;
    if (!cols.list) {
        // Dense: a 1-D grid over row tiles x column tiles.  Block L runs on XCD
        // L % 8; XCD x takes the x-th eighth of the tiles, columns innermost, so
        // the column tiles of a weight tile share an L2.
        const int nct = (M + TC - 1) / TC;
        const int nrt = jobs.n ? jobs.j[jobs.n - 1].blk0 + (jobs.j[jobs.n - 1].N + TR - 1) / TR : (N0 + TR - 1) / TR;
        const int per = gridDim.x >> 3, tile = (bx & 7) * per + (bx >> 3);
        if (tile >= nrt * nct) return;
        bx = tile / nct;
        cy = tile - bx * nct;
        cys = nct;
    }
    const int8_t *W = W0;
    const float *ws = ws0;
    float *out = out0;
    const int8_t *X = X0;
    const float *Xs = Xs0;
    int N = N0, K = K0, out_stride = out_stride0;
    if (jobs.n) {
        int ji = 0;
#pragma unroll
        for (int k = 1; k < MF_MAX_JOBS; k++)
            if (k < jobs.n && bx >= jobs.j[k].blk0) ji = k;
        const MfJob jb = jobs.j[ji];
        W = jb.W;
        ws = jb.ws;
        out = jb.out;
        X = jb.X;
        Xs = jb.Xs;
        K = jb.K;
        N = jb.N;
        out_stride = jb.out_stride;
        bx -= jb.blk0;
    }
    int ncols = M, cbase = 0;
    const int8_t *Wg = W, *Wg3 = PAIR ? pair.W3 : nullptr;
    const float *wsg = ws, *wsg3 = PAIR ? pair.ws3 : nullptr;
    if (cols.list) {
        const int g = blockIdx.z;
        if (g >= *cols.ng) return;
        ncols = cols.gcnt[g];
        cbase = cols.goff[g];
        const int e = cols.gexp[g];
        Wg = W + (size_t)e * w_group_stride;
        wsg = ws + (size_t)e * N;
        if constexpr (PAIR) {
            Wg3 += (size_t)e * w_group_stride;
            wsg3 += (size_t)e * N;
        }
    }
    float tabv = 0.0f;
    if constexpr (PAIR) tabv = c_exp_tab[tid & 31];
    const int n0 = bx * ORT, nb = K >> 5, nst = K / MFT_KC;
    // this thread's pieces of a stage: rows i NTHR / 8 + tid / 8, LDS place
    // tid % 8 (the row's bits 1..3 do not depend on i)
    const int prow = tid >> 3, gp = 16 * ((tid & 7) ^ ((prow >> 1) & 7));
    uint32_t wl[PW];
#pragma unroll
    for (int i = 0; i < PW; i++)
        wl[i] = (uint32_t)imin(n0 + (NTHR / 8 * i) % ORT + prow, N - 1) * (uint32_t)K + gp;
    // operand reads: lane l's 8 bytes 8 (l / 16) of group g of row l % 16
    const int r16 = lane & 15, q = lane >> 4;
    const int wr0 = (wave % WR) * 16 * (PAIR ? 1 : RT), wc0 = (wave / WR) * 16 * CT;
    int oa[4], ox[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const int o = r16 * MFT_KC + 16 * ((2 * g + (q >> 1)) ^ (r16 >> 1)) + 8 * (q & 1);
        oa[g] = wr0 * MFT_KC + o;
        ox[g] = XO + wc0 * MFT_KC + o;
    }
    const int os = SO + (wc0 + r16) * 16;
#pragma unroll 1
    for (int c0 = cy * TC; c0 < ncols; c0 += cys * TC) {
        auto xrow = [&](int c) {
            const int cc = imin(c0 + c, ncols - 1);
            if (!cols.list) return cc;
            const int o = cols.list[cbase + cc];
            return cols.xmap ? cols.xmap[o] : o;
        };
        // offsets from the uniform bases, so that a load takes no address
        // arithmetic (a weight matrix and the rows are below 4 GiB each)
        uint32_t xl[PX];
#pragma unroll
        for (int i = 0; i < PX; i++) xl[i] = (uint32_t)xrow(NTHR / 8 * i + prow) * (uint32_t)K + gp;
        // group scales: lanes below SL of each wave, a column's four each
        const uint32_t xsl = (uint32_t)xrow(wave * SL + imin(lane, SL - 1)) * (uint32_t)nb * 4;
        auto issue = [&](int st, int b) {
            const int8_t *wb = Wg + (size_t)st * MFT_KC, *wb3 = Wg3 + (size_t)st * MFT_KC;
            const int8_t *xb = X + (size_t)st * MFT_KC;
            const int8_t *sb = reinterpret_cast<const int8_t *>(Xs) + (size_t)st * 16;
#pragma unroll
            for (int i = 0; i < PW; i++)
                __builtin_amdgcn_global_load_lds((mft_gptr)((NTHR / 8 * i < ORT ? wb : wb3) + wl[i]),
                                                 (mft_lptr)(&s_buf[b][(NTHR * i + 64 * wave) * 16]), 16, 0, 0);
#pragma unroll
            for (int i = 0; i < PX; i++)
                __builtin_amdgcn_global_load_lds((mft_gptr)(xb + xl[i]),
                                                 (mft_lptr)(&s_buf[b][XO + (NTHR * i + 64 * wave) * 16]), 16, 0, 0);
            if (lane < SL)
                __builtin_amdgcn_global_load_lds((mft_gptr)(sb + xsl), (mft_lptr)(&s_buf[b][SO + wave * SL * 16]), 16,
                                                 0, 0);
        };
        float f[RT][CT][4];
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < CT; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) f[i][j][v] = 0.0f;
        v4i_t magic = {0x4B400000, 0x4B400000, 0x4B400000, 0x4B400000};     // 1.5 * 2^23
        asm volatile("" : "+v"(magic));                   // (kept in registers)
        auto compute = [&](int b) {
            const int8_t *p = s_buf[b];
            long ka[4][RT], kx[4][CT];
            v4f_t sc[CT];
#pragma unroll
            for (int g = 0; g < 4; g++) {
#pragma unroll
                for (int i = 0; i < RT; i++) ka[g][i] = *reinterpret_cast<const long *>(p + oa[g] + i * AST);
#pragma unroll
                for (int j = 0; j < CT; j++) kx[g][j] = *reinterpret_cast<const long *>(p + ox[g] + 16 * j * MFT_KC);
                if (g == 0)
#pragma unroll
                    for (int j = 0; j < CT; j++) sc[j] = *reinterpret_cast<const v4f_t *>(p + os + 256 * j);
            }
            v4i_t d[2][RT][CT];
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < CT; j++)
                    d[0][i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(ka[0][i], kx[0][j], magic, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // a group's fold runs beside the next group's MFMAs
#pragma unroll
            for (int g = 0; g < 4; g++) {
#pragma unroll
                for (int i = 0; i < RT; i++)
#pragma unroll
                    for (int j = 0; j < CT; j++) {
                        if (g < 3)
                            d[(g + 1) & 1][i][j] =
                                __builtin_amdgcn_mfma_i32_16x16x32_i8(ka[g + 1][i], kx[g + 1][j], magic, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            f[i][j][v] += (__int_as_float(d[g & 1][i][j][v]) - 12582912.0f) * sc[j][g];
                        if (g < 3) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA,
                        __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);                // a tile's fold
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        issue(0, 0);
        if (nst > 1) issue(1, 1);
        if (nst > 2) issue(2, 2);
        // (four stages per turn: the buffers are constants, LDS addresses
        // immediates)
#pragma unroll 1
        for (int st0 = 0; st0 < nst; st0 += MFT_NB) {
#pragma unroll
            for (int b = 0; b < MFT_NB; b++) {
                const int st = st0 + b;
                if (st >= nst) break;
                if (st + 2 < nst) mft_arrive<2 * LPS>();
                else if (st + 1 < nst) mft_arrive<LPS>();
                else mft_arrive<0>();
                if (st + 3 < nst) issue(st + 3, (b + 3) & (MFT_NB - 1));
                compute(b);
            }
        }
        // lane l: rows 4 (l / 16) .. + 3 of a tile, column l % 16
        if constexpr (PAIR) {
            // (in the stage buffers, which every wave has read)
            float *tab = reinterpret_cast<float *>(&s_buf[0][0]);
            uint32_t *s_am = reinterpret_cast<uint32_t *>(&s_buf[0][128]);        // [WR][TC]
            __syncthreads();
            if (tid < 32) tab[tid] = tabv;
            __syncthreads();
            const int n = n0 + wr0 + 4 * q, col = wc0 + r16, cl = c0 + col;
            float y[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int nc = imin(n + v, N - 1);
                const float h1 = 0.0f + f[0][0][v] * wsg[nc], h3 = 0.0f + f[1][0][v] * wsg3[nc];
                y[v] = d_silu(h1, tab) * h3;
            }
            const float4 y4 = make_float4(y[0], y[1], y[2], y[3]);
            uint32_t am = abs_bits4(y4);
            am = umax(am, (uint32_t)__shfl_xor((int)am, 16));
            am = umax(am, (uint32_t)__shfl_xor((int)am, 32));
            if (q == 0) s_am[(wave % WR) * TC + col] = am;
            __syncthreads();
            float sg;
            const uint32_t pk = quant4_amax(y4, f_from_u(umax(s_am[col], s_am[TC + col])), &sg);
            if (cl < ncols) {
                const size_t o = (size_t)cols.list[cbase + cl];
                *reinterpret_cast<uint32_t *>(pair.q + o * N + n) = pk;
                if (wave % WR == 0 && q == 0) pair.qs[o * (N >> 5) + (n0 >> 5)] = sg;
            }
        } else
#pragma unroll
        for (int j = 0; j < CT; j++) {
            const int cl = c0 + wc0 + 16 * j + r16;
            if (cl < ncols) {
                float *op = out + (size_t)(cols.list ? cols.list[cbase + cl] : cl) * out_stride;
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    const int n = n0 + wr0 + 16 * i + 4 * q;
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (n + v < N) op[n + v] = 0.0f + f[i][j][v] * wsg[n + v];
                }
            }
        }
        // another tile of this block: its loads wait for every wave's reads
        if (c0 + cys * TC < ncols) mft_arrive<0>();
    }
}

// ------------------------------------------------------ wide producers ---
//
// The quantized GEMM inputs of many rows, one 64-lane block per row, with
// the arithmetic of the GEMV prologues (l98_gemv.h) element for element:
//   mode 0: quantize src rows                       (PRO_QUANT)
//   mode 1: silu(src) * src2, then quantize          (PRO_SILU,
//           lz_ffn_gate_up, src/forward_kda.c:1067-1088)
//   mode 2: sum over the row's slots k < topk with sel_idx >= 0 of
//           sel_w * src[pair], in slot order from 0, then quantize
//           (PRO_COMBINE, src/forward_moe.c:128-200)
// Lane l holds float4 f = l + 64 j of the row, so a quantization group is
// an aligned lane octet.  n % 32 == 0, n <= 4096.
#define WP_MAXJ 16
struct WideProArgs {
    const float *src, *src2;
    const int *sel_idx;
    const float *sel_w;
    int8_t *xq;
    float *xqs, *fout;
    int mode, src_stride, topk, n;
};
__device__ __forceinline__ void wide_pro_body(int mode, const float *__restrict__ src, const float *__restrict__ src2,
                                              int src_stride, const int *__restrict__ sel_idx,
                                              const float *__restrict__ sel_w, int topk, int n,
                                              int8_t *__restrict__ xq, float *__restrict__ xqs,
                                              float *__restrict__ fout, int row, const float *tab) {
    const int lane = threadIdx.x;
    const int nf = n >> 2, nb = n >> 5;
    for (int j = 0; j < WP_MAXJ; j++) {
        if (64 * j >= nf) break;                   // wave-uniform
        const int f = lane + 64 * j;
        const int fc = f < nf ? f : nf - 1;
        float4 v;
        if (mode == 0) {
            v = reinterpret_cast<const float4 *>(src + (size_t)row * src_stride)[fc];
        } else if (mode == 1) {
            const float4 p = reinterpret_cast<const float4 *>(src + (size_t)row * src_stride)[fc];
            const float4 q = reinterpret_cast<const float4 *>(src2 + (size_t)row * src_stride)[fc];
            v = make_float4(d_silu(p.x, tab) * q.x, d_silu(p.y, tab) * q.y, d_silu(p.z, tab) * q.z,
                            d_silu(p.w, tab) * q.w);
        } else {
            float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int k = 0; k < topk; k++) {
                const int pair = row * topk + k;
                if (sel_idx[pair] < 0) continue;
                const float wk = sel_w[pair];
                const float4 hk = reinterpret_cast<const float4 *>(src + (size_t)pair * n)[fc];
                y = make_float4(y.x + wk * hk.x, y.y + wk * hk.y, y.z + wk * hk.z, y.w + wk * hk.w);
            }
            v = y;
        }
        if (fout && f < nf) reinterpret_cast<float4 *>(fout + (size_t)row * n)[f] = v;
        if (xq) {
            float sg;
            const uint32_t q = quant_octet(v, &sg);
            if (f < nf) {
                reinterpret_cast<uint32_t *>(xq + (size_t)row * n)[f] = q;
                if (!(f & 7)) xqs[(size_t)row * nb + (f >> 3)] = sg;
            }
        }
    }
}
__global__ __launch_bounds__(64) void k_wide_pro(int mode, const float *__restrict__ src,
                                                 const float *__restrict__ src2, int src_stride,
                                                 const int *__restrict__ sel_idx, const float *__restrict__ sel_w,
                                                 int topk, int n, int8_t *__restrict__ xq, float *__restrict__ xqs,
                                                 float *__restrict__ fout) {
    EXP_TAB_LOAD(tab);
    EXP_TAB_PUT(tab);
    __syncthreads();
    wide_pro_body(mode, src, src2, src_stride, sel_idx, sel_w, topk, n, xq, xqs, fout, blockIdx.x, tab);
}
// Two independent producers in one launch: blocks [0, rows_a) run a's rows,
// the rest b's.
__global__ __launch_bounds__(64) void k_wide_pro2(WideProArgs a, int rows_a, WideProArgs b) {
    EXP_TAB_LOAD(tab);
    EXP_TAB_PUT(tab);
    __syncthreads();
    const bool first = (int)blockIdx.x < rows_a;
    const WideProArgs &p = first ? a : b;
    wide_pro_body(p.mode, p.src, p.src2, p.src_stride, p.sel_idx, p.sel_w, p.topk, p.n, p.xq, p.xqs, p.fout,
                  first ? blockIdx.x : blockIdx.x - rows_a, tab);
}

// ---------------------------------------------------------- host glue ---

extern "C" int l98k_upload_exp_table_mfma(const float *tab) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(c_exp_tab), tab, 32 * sizeof(float));
}

// The tile of k_mfma_q8t's launches: 32 weight rows x 16 token columns for at
// most 16 columns, 64 x 32 where that still leaves MFT_BIG tiles or more (by its
// LDS three blocks to a CU, 768 on the chip), else 32 x 32.  Measured (us, rows
// x K at that many columns; 32 x 16 / 32 x 32 / 64 x 32 tiles; before, on tiles
// of 64 x 16 up to 128 columns and 16 x 64 above):
//     2048 x 1024 at   1:   5.0 /  5.2 /  7.2 (5.9)
//     4176 x 1024 at  12:   5.5 /  5.6 /  7.8 (6.8)
//    65536 x 1024 at   8:  14.4 / 15.2 / 16.8 (17.3)
//   131072 x 2048 at   4:  40.5 / 41.9 / 45.1 (47.1)
//   131072 x 2048 at  16:  43.0 / 45.5 / 46.6 (48.2)
//     2048 x 2048 at 128:   8.3 /  8.1 / 11.8 (9.8)
//     8336 x 2048 at 128:  16.9 / 16.8 / 16.5 (22.1)
//   131072 x 2048 at 128:   233 /  201 /  174 (254)
//     4176 x 1024 at 512:    -  / 17.3 / 17.7 (26.2)
//     8336 x 2048 at 512:    -  / 45.0 / 42.7 (74.7)
//     2048 x 2048 at 512:    -  / 13.9 / 13.7 (24.3)
// 64 x 64 tiles and blocks of eight waves were slower at every shape: too few
// blocks for the waits of one to be covered by another's work.
#define MFT_BIG 2048
enum { MFT_32x16, MFT_32x32, MFT_64x32 };
static int mft_tile_rows(int t) { return t == MFT_64x32 ? 64 : 32; }
static int mft_tile_cols(int t) { return t == MFT_32x16 ? 16 : 32; }
static void mft_launch(int t, dim3 grid, const int8_t *W, const float *ws, int N, int K, size_t w_group_stride,
                       const int8_t *X, const float *Xs, int M, const MfCols &c, float *out, int out_stride,
                       const MfJobs &jobs, hipStream_t st) {
    if (t == MFT_32x16)
        hipLaunchKernelGGL((k_mfma_q8t<1, 1, 2, 1>), grid, dim3(128), 0, st, W, ws, N, K, w_group_stride, X, Xs, M, c,
                           out, out_stride, jobs, MfPair{});
    else if (t == MFT_32x32)
        hipLaunchKernelGGL((k_mfma_q8t<1, 1, 2, 2>), grid, dim3(256), 0, st, W, ws, N, K, w_group_stride, X, Xs, M, c,
                           out, out_stride, jobs, MfPair{});
    else
        hipLaunchKernelGGL((k_mfma_q8t<2, 1, 2, 2>), grid, dim3(256), 0, st, W, ws, N, K, w_group_stride, X, Xs, M, c,
                           out, out_stride, jobs, MfPair{});
}
// k_mfma_q8t takes offsets of 32 bits into a weight matrix and into the rows.
static bool mft_ok(int N, int K, int rows) {
    return K % MFT_KC == 0 && (uint64_t)N * K < (1ull << 32) && (uint64_t)rows * K < (1ull << 32);
}

// Whether a dense launch of K not a multiple of 128 takes k_mfma_q8n: `blocks`
// 16-row weight tiles of all its jobs, `stages` the MF_KC-byte stages of those
// tiles.  Measured (us, rows x K at that many columns, k_mfma_q8n / k_mfma_q8):
//     2048 x 1056 at  4:  7.2 /  6.8      8192 x  352 at   4:  4.9 /  4.9
//    16384 x   96 at  4:  3.9 /  5.6     65536 x 1056 at   4: 18.8 / 42.1
//    65536 x 1056 at 32: 27.5 / 44.2     65536 x  352 at  64: 29.4 / 27.9
//    16384 x 1056 at 64: 15.6 / 15.3    131072 x 1056 at 128:  172 /  179
static bool mf_narrow(int M, size_t blocks, size_t stages) {
    if (M <= 32) return stages >= 1024;
    return M <= 128 && blocks >= 1024 && stages >= 4 * blocks;
}

// Several dense GEMMs over the same M rows in one launch: job j multiplies
// W[j] (N[j] x K[j], scales ws[j]) over the rows of X[j] / Xs[j] into out[j]
// (row stride out_stride[j]).  The blocks of job j follow those of job
// j - 1.  Returns 0, a HIP error, or -1 for shapes outside the kernels.
extern "C" int l98k_mfma_gemm_multi(int n_jobs, const int8_t *const *W, const float *const *ws, const int *N,
                                    float *const *out, const int *out_stride, const int *K,
                                    const int8_t *const *X, const float *const *Xs, int M, hipStream_t st) {
    if (n_jobs < 1 || n_jobs > MF_MAX_JOBS || M < 1) return -1;
    bool tiled = true;
    size_t rows = 0, tiles16 = 0, stages = 0;
    for (int j = 0; j < n_jobs; j++) {
        if (N[j] < 1 || out_stride[j] < N[j] || K[j] < 32 || (K[j] & 31)) return -1;
        tiled = tiled && mft_ok(N[j], K[j], M);
        rows += (size_t)N[j];
        tiles16 += (size_t)(N[j] + MF_ROWS - 1) / MF_ROWS;
        stages += (size_t)(N[j] + MF_ROWS - 1) / MF_ROWS * ((K[j] + MF_KC - 1) / MF_KC);
    }
    int t = M <= 16 ? MFT_32x16 : MFT_32x32;
    if (M > 16 && (rows / 64) * ((M + 31) / 32) >= MFT_BIG) t = MFT_64x32;
    const bool narrow = !tiled && mf_narrow(M, tiles16, stages);
    const int tr = tiled ? mft_tile_rows(t) : narrow ? MFN_ROWS : MF_ROWS;
    MfJobs jobs{};
    int blocks = 0;
    for (int j = 0; j < n_jobs; j++) {
        jobs.j[j] = MfJob{W[j], ws[j], out[j], X[j], Xs[j], N[j], out_stride[j], blocks, K[j]};
        blocks += (N[j] + tr - 1) / tr;
    }
    jobs.n = n_jobs > 1 ? n_jobs : 0;               // one GEMM: the launch's own arguments
    if (tiled) {
        const int tiles = blocks * ((M + mft_tile_cols(t) - 1) / mft_tile_cols(t));
        mft_launch(t, dim3((tiles + 7) & ~7), W[0], ws[0], N[0], K[0], 0, X[0], Xs[0], M, MfCols{}, out[0],
                   out_stride[0], jobs, st);
    } else if (narrow) {
        hipLaunchKernelGGL(k_mfma_q8n, dim3(((blocks + 7) & ~7) * ((M + MFN_COLS - 1) / MFN_COLS)), dim3(MF_THREADS),
                           0, st, W[0], ws[0], N[0], K[0], (size_t)0, X[0], Xs[0], M, MfCols{}, out[0], out_stride[0],
                           jobs);
    } else {
        hipLaunchKernelGGL(k_mfma_q8, dim3(blocks, (M + MF_COLS - 1) / MF_COLS), dim3(MF_THREADS), 0, st, W[0], ws[0],
                           N[0], K[0], (size_t)0, X[0], Xs[0], M, MfCols{}, out[0], out_stride[0], jobs);
    }
    return (int)hipGetLastError();
}

// Dense: out[t][n] (row stride out_stride) for t < M over activation rows t.
extern "C" int l98k_mfma_gemm(const int8_t *W, const float *ws, int N, int K, const int8_t *X, const float *Xs, int M,
                              float *out, int out_stride, hipStream_t st) {
    return l98k_mfma_gemm_multi(1, &W, &ws, &N, &out, &out_stride, &K, &X, &Xs, M, st);
}

// Grouped (experts): group g (< *ng <= max_groups) multiplies bank rows of
// expert gexp[g] with its columns list[goff[g] ..], at most max_cols each.
// mean_cols, the caller's estimate of a group's columns, picks 16 or 32
// columns per tile; a group's tiles spread over the grid's y, about twice the
// mean's (blocks past a group's tiles exit at once, the tiles past the grid
// are walked).
static int mf_grouped_y(int max_cols, int mean_cols, int tc) {
    const int most = (max_cols + tc - 1) / tc, ys = 2 + 2 * mean_cols / tc;
    return ys < most ? ys : most;
}
// A grouped launch of any K: the bank, or `jobs` banks of the same N and K.  Up
// to 16 columns in a group (mean_cols) on k_mfma_q8n, but for launches of few
// tiles.  Its y is odd: with 2 or 4 blocks per row tile the ones past a group's
// columns, which exit at once, leave the same places of the chip empty in every
// row of tiles.  Measured (us, groups x rows x K at that many columns each:
// k_mfma_q8n with 3 or 5 / with 2 or 4 blocks / k_mfma_q8):
//     16 x  128 x   96 at  8:  4.1 /  4.1 /  3.7
//     64 x  128 x  704 at  2:  6.2 /  6.1 /  6.7
//     64 x  512 x  704 at  2:  8.8 / 11.7 / 18.0
//     64 x  512 x  704 at 16: 10.4 / 21.5 / 19.2
//    128 x 1024 x 1344 at  8: 38.4 / 57.5 / 98.9
static int mf_grouped(const int8_t *bank, const float *bank_s, int N, int K, const int8_t *X, const float *Xs,
                      const MfCols &c, int max_groups, int max_cols, int mean_cols, float *out, int out_stride,
                      MfJobs jobs, hipStream_t st) {
    const bool narrow = mean_cols <= 16 && (size_t)max_groups * ((N + MF_ROWS - 1) / MF_ROWS) >= 256;
    const int tr = narrow ? MFN_ROWS : MF_ROWS, nrt = (N + tr - 1) / tr;
    for (int j = 0; j < jobs.n; j++) jobs.j[j].blk0 = j * nrt;
    const int gx = nrt * (jobs.n ? jobs.n : 1);
    if (narrow)
        hipLaunchKernelGGL(k_mfma_q8n, dim3(gx, mf_grouped_y(max_cols, mean_cols, MFN_COLS) | 1, max_groups),
                           dim3(MF_THREADS), 0, st, bank, bank_s, N, K, (size_t)N * K, X, Xs, 0, c, out, out_stride,
                           jobs);
    else
        hipLaunchKernelGGL(k_mfma_q8, dim3(gx, 1, max_groups), dim3(MF_THREADS), 0, st, bank, bank_s, N, K,
                           (size_t)N * K, X, Xs, 0, c, out, out_stride, jobs);
    return (int)hipGetLastError();
}

extern "C" int l98k_mfma_gemm_grouped(const int8_t *bank, const float *bank_s, int N, int K, const int8_t *X,
                                      const float *Xs, const int *ng, int max_groups, const int *gexp,
                                      const int *goff, const int *gcnt, const int *list, const int *xmap,
                                      int max_cols, int mean_cols, float *out, int out_stride, hipStream_t st) {
    if (N < 1 || K < 32 || (K & 31) || max_groups < 1 || max_cols < 1 || out_stride < N) return -1;
    const MfCols c{gexp, goff, gcnt, list, xmap, ng};
    if (!mft_ok(N, K, max_cols * MAX_TOPK))
        return mf_grouped(bank, bank_s, N, K, X, Xs, c, max_groups, max_cols, mean_cols, out, out_stride, MfJobs{}, st);
    const int t = mean_cols <= 16 ? MFT_32x16 : MFT_32x32, tr = mft_tile_rows(t), tc = mft_tile_cols(t);
    mft_launch(t, dim3((N + tr - 1) / tr, mf_grouped_y(max_cols, mean_cols, tc), max_groups), bank, bank_s, N, K,
               (size_t)N * K, X, Xs, 0, c, out, out_stride, MfJobs{}, st);
    return (int)hipGetLastError();
}

// The experts' first half over `pairs` rows (group columns name them): silu(w1
// x) * w3 x, both banks N x K, quantized per 32 into q [pairs][N] and qs.  On
// the tiled kernel one launch (PAIR); else the two GEMMs as two jobs of one into
// h1 and h3 (scratch [pairs][N]) and the quantizing producer.  One launch instead
// of those two: 32 sessions of 4 rows at d = 2048, 24 +
// 5.3 -> 20.8 us per layer.
extern "C" int l98k_mfma_gemm_pair(const int8_t *bank1, const float *bank1_s, const int8_t *bank3,
                                   const float *bank3_s, int N, int K, const int8_t *X, const float *Xs, const int *ng,
                                   int max_groups, const int *gexp, const int *goff, const int *gcnt, const int *list,
                                   const int *xmap, int max_cols, int mean_cols, int pairs, float *h1, float *h3,
                                   int8_t *q, float *qs, hipStream_t st) {
    if (N < 32 || (N & 31) || K < 32 || (K & 31) || max_groups < 1 || max_cols < 1 || pairs < 1) return -1;
    const MfCols c{gexp, goff, gcnt, list, xmap, ng};
    if (mft_ok(N, K, max_cols * MAX_TOPK)) {
        const MfPair p{bank3, bank3_s, q, qs};
        const bool narrow = mean_cols <= 16;
        const dim3 grid(N / 32, mf_grouped_y(max_cols, mean_cols, narrow ? 16 : 32), max_groups);
        if (narrow)
            hipLaunchKernelGGL((k_mfma_q8t<2, 1, 2, 1, true>), grid, dim3(128), 0, st, bank1, bank1_s, N, K,
                               (size_t)N * K, X, Xs, 0, c, nullptr, 0, MfJobs{}, p);
        else
            hipLaunchKernelGGL((k_mfma_q8t<2, 1, 2, 2, true>), grid, dim3(256), 0, st, bank1, bank1_s, N, K,
                               (size_t)N * K, X, Xs, 0, c, nullptr, 0, MfJobs{}, p);
        return (int)hipGetLastError();
    }
    MfJobs jobs{};
    jobs.j[0] = MfJob{bank1, bank1_s, h1, X, Xs, N, N, 0, K};
    jobs.j[1] = MfJob{bank3, bank3_s, h3, X, Xs, N, N, 0, K};
    jobs.n = 2;
    const int rc = mf_grouped(bank1, bank1_s, N, K, X, Xs, c, max_groups, max_cols, mean_cols, h1, N, jobs, st);
    return rc ? rc : l98k_wide_pro(1, h1, h3, N, nullptr, nullptr, 0, N, pairs, q, qs, st);
}

static bool wide_pro_ok(int mode, int src_stride, const int *sel_idx, const float *sel_w, int topk, int n, int rows) {
    if (rows < 1 || n < 32 || (n & 31) || n > 4 * 64 * WP_MAXJ || mode < 0 || mode > 2) return false;
    if (mode < 2 && (src_stride < n || (src_stride & 3))) return false;
    if (mode == 2 && (topk < 1 || topk > MAX_TOPK || !sel_idx || !sel_w)) return false;
    return true;
}

// Two quantizing producers (modes as l98k_wide_pro) in one launch.
extern "C" int l98k_wide_pro2(int mode_a, const float *src_a, const float *src2_a, int stride_a, int n_a, int rows_a,
                              int8_t *xq_a, float *xqs_a, int mode_b, const float *src_b, const float *src2_b,
                              int stride_b, const int *sel_idx_b, const float *sel_w_b, int topk_b, int n_b,
                              int rows_b, int8_t *xq_b, float *xqs_b, hipStream_t st) {
    if (mode_a == 2 || !wide_pro_ok(mode_a, stride_a, nullptr, nullptr, 0, n_a, rows_a) ||
        !wide_pro_ok(mode_b, stride_b, sel_idx_b, sel_w_b, topk_b, n_b, rows_b) || !xq_a || !xqs_a || !xq_b || !xqs_b)
        return -1;
    const WideProArgs a{src_a, src2_a, nullptr, nullptr, xq_a, xqs_a, nullptr, mode_a, stride_a, 0, n_a};
    const WideProArgs b{src_b, src2_b, sel_idx_b, sel_w_b, xq_b, xqs_b, nullptr, mode_b, stride_b, topk_b, n_b};
    hipLaunchKernelGGL(k_wide_pro2, dim3(rows_a + rows_b), dim3(64), 0, st, a, rows_a, b);
    return (int)hipGetLastError();
}

extern "C" int l98k_wide_pro(int mode, const float *src, const float *src2, int src_stride, const int *sel_idx,
                             const float *sel_w, int topk, int n, int rows, int8_t *xq, float *xqs, hipStream_t st) {
    if (rows < 1 || n < 32 || (n & 31) || n > 4 * 64 * WP_MAXJ || mode < 0 || mode > 2) return -1;
    if (mode < 2 && (src_stride < n || (src_stride & 3))) return -1;
    if (mode == 2 && (topk < 1 || topk > MAX_TOPK || !sel_idx || !sel_w)) return -1;
    if (!xq || !xqs) return -1;
    hipLaunchKernelGGL(k_wide_pro, dim3(rows), dim3(64), 0, st, mode, src, src2, src_stride, sel_idx, sel_w, topk, n,
                       xq, xqs, (float *)nullptr);
    return (int)hipGetLastError();
}

// The same rows in float, unquantized (row stride n): the input of a norm
// that comes before the quantization.
extern "C" int l98k_wide_pro_f(int mode, const float *src, const float *src2, int src_stride, const int *sel_idx,
                               const float *sel_w, int topk, int n, int rows, float *fout, hipStream_t st) {
    if (rows < 1 || n < 32 || (n & 31) || n > 4 * 64 * WP_MAXJ || mode < 0 || mode > 2 || !fout) return -1;
    if (mode < 2 && (src_stride < n || (src_stride & 3))) return -1;
    if (mode == 2 && (topk < 1 || topk > MAX_TOPK || !sel_idx || !sel_w)) return -1;
    hipLaunchKernelGGL(k_wide_pro, dim3(rows), dim3(64), 0, st, mode, src, src2, src_stride, sel_idx, sel_w, topk, n,
                       (int8_t *)nullptr, (float *)nullptr, fout);
    return (int)hipGetLastError();
}
