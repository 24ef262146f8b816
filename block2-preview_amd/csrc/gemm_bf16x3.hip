// Segmented grouped GEMM in split-BF16 three-term arithmetic (gfx950) on
// pre-split operands.
//
// Every operand value a is split once into two BF16 numbers, hi = bf16(a)
// and lo = bf16(a - hi), so that a = hi + lo to about 2^-17 relative.  A
// product is then
//     a * b ~= a_hi * b_hi + a_hi * b_lo + a_lo * b_hi
// (the dropped a_lo * b_lo is ~2^-16 relative), each term one
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation.  Three BF16 MFMAs cost
// 3 * 16 cycles per 16x16x32 block against 8 * 32 cycles for the same block
// with FP32 16x16x4 MFMAs; the Davidson that uses them refines in FP64.
//
// Packed operands.  A GEMM operand is held as a row-major matrix whose rows
// run along the contraction index k, K rounded up to 32 with zeros; every 32
// k of a row are one aligned 128-byte line, the 32 hi values and then the 32
// lo values.  A k-step of a tile row is therefore one whole cache line: the
// loader reads it with eight lanes' 16-byte buffer loads and does no
// arithmetic.  (As two planes, a k-step read half of two lines, twice the
// requests between a compute unit's L1 and L2, whose number in flight bounds
// these kernels: H*psi at M=3000 with four right-hand sides 14.4 against
// 11.9 ms, L1 read requests of phase 2 8.8e8 against 3.4e8, matrix cores busy
// 33 against 49 % of it.)  The constant
// operators are packed once per plan (in the orientation each pair reads
// them), the wavefunction once per H*psi, and phase 1 writes its product W
// directly as packed W^T for phase 2.
//
// Task / segment semantics are those of seg_gemm_kernel (kernels.hip): a
// task is one TM x TN output tile accumulating sum_s alpha_s A_s B_s^T over
// its segments (A_s: M x K_s, B_s: N x K_s, both packed, lda / ldb the packed
// row stride in elements, hi and lo counted), the tile owned by exactly one
// task (no atomics).  alpha_s is applied to each segment's FP32
// partial sum when the segment ends.
#include "kernels.hpp"
#include "launch.hpp"

namespace b2g {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Lane l of v_mfma_f32_16x16x32_bf16 supplies A[l%16][8*(l/16) + i] and
// B[8*(l/16) + i][l%16] (i < 8); accumulator element r of lane l is
// D[4*(l/16) + r][l%16] (in-bounds probe of the builtin on gfx950).
__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Raw buffer resource over rows row0 .. row0 + tile of a packed matrix of
// `rows` rows and stride ld.  Rows from `rows` on lie past its end and read
// as zero.  (A packed matrix has rows * round8(K) < 2^28, so `tile` <= 128
// rows are fewer than 2^31 bytes.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t
pk_rsrc(const __bf16 *p, uint32_t row0, uint32_t rows, uint32_t ld, int tile) {
    const uint32_t n = min(rows - row0, (uint32_t)tile);
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<__bf16 *>(p + (uint64_t)row0 * ld), (short)0,
        (int)(2 * ld * n), 0x00020000);
}
__device__ __forceinline__ u32x4 pk_load(__amdgpu_buffer_rsrc_t r,
                                         uint32_t off, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0);
}

// element offset of the hi value (r, k) of a packed matrix of row stride ld;
// its lo value is 32 elements on
__device__ __forceinline__ uint64_t pk_offset(uint32_t r, uint32_t k,
                                              uint32_t ld) {
    return (uint64_t)r * ld + (k >> 5) * 64 + (k & 31);
}

// ------------------------------------------------------------------ packing
// One thread per 8-element group (8 consecutive k of one packed row).  The
// groups of a job are numbered matrix after matrix from each matrix's g0:
// row-major (row, k group) when the source runs along k, column-major
// (k group, row) for a transposed source, so that consecutive lanes read
// consecutive source addresses.  A workgroup takes 256 * kPackGPT
// consecutive groups; the group offsets of the matrices they span (at most
// one matrix per group) are staged in LDS for each thread's binary search.
constexpr int kPackGPT = 4;

__global__ __launch_bounds__(256) void pack_bf16_kernel(
    const double *__restrict__ src, __bf16 *__restrict__ dst,
    const PackMat *__restrict__ mats, int nmats, uint64_t ngroups,
    uint64_t src_rs, uint64_t dst_rs) {
    constexpr int G = 256 * kPackGPT;
    __shared__ uint64_t sg0[G + 1];
    __shared__ int sm[2];
    const int rhs = blockIdx.y;
    src += rhs * src_rs;
    dst += rhs * dst_rs;
    const uint64_t base = (uint64_t)blockIdx.x * G;
    if (base >= ngroups)
        return;
    const uint64_t last = (base + G < ngroups ? base + G : ngroups) - 1;
    if (threadIdx.x < 2) {
        // last matrix with g0 <= base (thread 0) / <= last (thread 1)
        const uint64_t key = threadIdx.x == 0 ? base : last;
        int a = 0, b = nmats - 1;
        while (a < b) {
            const int mid = (a + b + 1) >> 1;
            if (mats[mid].g0 <= key)
                a = mid;
            else
                b = mid - 1;
        }
        sm[threadIdx.x] = a;
    }
    __syncthreads();
    const int m0 = sm[0], nm = sm[1] - sm[0] + 1; // nm <= G
    for (int i = threadIdx.x; i < nm; i += 256)
        sg0[i] = mats[m0 + i].g0;
    __syncthreads();
    for (int it = 0; it < kPackGPT; it++) {
        const uint64_t g = base + (uint64_t)it * 256 + threadIdx.x;
        if (g > last)
            break;
        int a = 0, b = nm - 1;
        while (a < b) {
            const int mid = (a + b + 1) >> 1;
            if (sg0[mid] <= g)
                a = mid;
            else
                b = mid - 1;
        }
        const PackMat pm = mats[m0 + a];
        const uint32_t l = (uint32_t)(g - pm.g0);
        const uint32_t kg = pm.dst_ld >> 3;
        uint32_t r, k;
        if (pm.trans)
            k = (l / pm.rows) * 8, r = l % pm.rows;
        else
            r = l / kg, k = (l % kg) * 8;
        bf16x8 h, lw;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t kk = k + i;
            double v = 0.0;
            if (kk < pm.cols)
                v = src[pm.src + (pm.trans ? (uint64_t)kk * pm.src_ld + r
                                           : (uint64_t)r * pm.src_ld + kk)];
            const __bf16 vh = (__bf16)(float)v;
            h[i] = vh;
            lw[i] = (__bf16)(float)(v - (double)(float)vh);
        }
        __bf16 *o = dst + pm.dst + pk_offset(r, k, 2 * pm.dst_ld);
        *(bf16x8 *)o = h;
        *(bf16x8 *)(o + 32) = lw;
    }
}

hipError_t launch_pack_bf16(const double *src, __bf16 *dst,
                            const PackMat *mats, int nmats, uint64_t ngroups,
                            uint64_t src_rs, uint64_t dst_rs, int n_rhs,
                            int grid, hipStream_t st) {
    (void)grid;
    if (nmats <= 0 || ngroups == 0)
        return hipSuccess;
    const uint64_t g = (ngroups + 256 * kPackGPT - 1) / (256 * kPackGPT);
    if (g >= (1ull << 31))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(pack_bf16_kernel, dim3((unsigned)g, (unsigned)n_rhs),
                       dim3(256), 0, st, src, dst, mats, nmats, ngroups,
                       src_rs, dst_rs);
    return hipGetLastError();
}

// ------------------------------------------------------------- tile loader
// One workgroup = 4 waves (2x2); K staged through two LDS buffers in steps
// of 32 (one MFMA k-step).  An LDS row holds the 32 k values of one tile row
// (A) or tile column (B), so that a lane's 8 k values (a k group) are one
// 16-byte read; the k groups of a row are permuted by the row (slot) so that
// one k group of 16 consecutive rows falls on distinct banks without padding:
// two 128 x 128 workgroups fit a compute unit.
template <int TM, int TN> struct PkTile {
    static constexpr int TK = 32;
    static constexpr int VA = TM * 8, VB = TN * 8; // 16-byte vectors
    static_assert(VA % 256 == 0 && VB % 256 == 0, "whole loads per thread");
    static constexpr int GA = VA / 256, GB = VB / 256; // per thread
    static constexpr int ASZ = TM * TK, BSZ = TN * TK;
    static constexpr int BUF = 2 * ASZ + 2 * BSZ; // A hi, A lo, B hi, B lo
    u32x4 a[GA], b[GB];
    uint32_t va, vb, sa, sb;

    // element offset of k group g of a row
    static __device__ __forceinline__ int slot(int row, int g) {
        const int j = (row >> 2) & 3;
        return row * TK + 8 * (g ^ (((j ^ (j >> 1)) & 1) << 1 | j >> 1));
    }
    // Vector e of a tile: row e / 8, and part e % 8 of the row's line (hi
    // groups 0..3, lo groups 4..7).  Where it goes in LDS: the planes lie
    // one after the other; the lo plane reverses every four rows, so that
    // the eight lanes of a row, and the sixteen of two, meet no bank twice
    // (rows in their order: a third of the LDS cycles are conflicts).
    static __device__ __forceinline__ int place(int e, int plane) {
        const int row = e >> 3, g = e & 3;
        return (e & 4) ? plane + slot(row ^ 3, g) : slot(row, g);
    }
    // Offsets of one segment, in bytes from the tile's first row: the
    // thread's first vector, and 32 rows (a workgroup's reach).  Sums
    // saturate, so a row past the resource's end stays past it.
    __device__ __forceinline__ void setup(const Seg &sg, int tid) {
        va = sat32(2 * (uint64_t)sg.lda * (tid >> 3)) + 16 * (tid & 7);
        vb = sat32(2 * (uint64_t)sg.ldb * (tid >> 3)) + 16 * (tid & 7);
        sa = sat32(64 * (uint64_t)sg.lda), sb = sat32(64 * (uint64_t)sg.ldb);
    }
    static __device__ __forceinline__ uint32_t sat32(uint64_t v) {
        return v < 0xFFFFFF00u ? (uint32_t)v : 0xFFFFFF00u;
    }
    // k0 a multiple of 32: four bytes per k
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rA,
                                         __amdgpu_buffer_rsrc_t rB,
                                         uint32_t k0) {
#pragma unroll
        for (int g = 0; g < GA; g++)
            a[g] = pk_load(rA, reach(va, sa, g), 4 * k0);
#pragma unroll
        for (int g = 0; g < GB; g++)
            b[g] = pk_load(rB, reach(vb, sb, g), 4 * k0);
    }
    static __device__ __forceinline__ uint32_t reach(uint32_t v, uint32_t s,
                                                     int g) {
        for (int i = 0; i < g; i++)
            v = __builtin_elementwise_add_sat(v, s);
        return v;
    }

    __device__ __forceinline__ void store(__bf16 *buf, int tid) const {
#pragma unroll
        for (int g = 0; g < GA; g++)
            *(u32x4 *)(buf + place(tid + 256 * g, ASZ)) = a[g];
#pragma unroll
        for (int g = 0; g < GB; g++)
            *(u32x4 *)(buf + 2 * ASZ + place(tid + 256 * g, BSZ)) = b[g];
    }
};

// OUT 0: D0 is the packed transpose of the output (row n, k index m, of a
//        task's block at d_off, ldd the packed row stride; rows M <= m <
//        ldd / 2 receive the zeros of the masked A rows, so the padding of
//        W^T is rewritten by every launch), written through LDS as 16-byte
//        vectors along m;
// OUT 1: D0 is the FP64 output (row-major, ldd), D1 the FP64 split-K
//        partial buffer (task.beta bit 1), as in seg_gemm_kernel.
template <int TM, int TN, int OUT>
__global__ __launch_bounds__(256) void seg_gemm_pk_kernel(
    const __bf16 *__restrict__ A, const __bf16 *__restrict__ B,
    void *__restrict__ D0, void *__restrict__ D1,
    const Task *__restrict__ tasks, int ntasks, const Seg *__restrict__ segs,
    uint64_t a_rs, uint64_t b_rs, uint64_t d_rs, uint64_t p_rs, double scale,
    int beta0, int nrhs, XcdSplit xs) {
    typedef PkTile<TM, TN> T;
    constexpr int WM = TM / 2, WN = TN / 2;
    constexpr int FM = WM / 16, FN = WN / 16;
    __shared__ __attribute__((aligned(16))) __bf16 smem[2 * T::BUF];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lk = lane >> 4;
    T ld;
    for (TaskRange tr(ntasks, nrhs, xs); tr.more(); tr.next()) {
        const Task task = tasks[tr.task()];
        const int rhs = tr.rhs();
        const uint64_t ao = rhs * a_rs, bo = rhs * b_rs;
        // acc: the tile's sum; part: the running segment's unscaled sum
        // (phase 1 tasks have one segment with alpha = 1: part is the sum)
        f32x4 acc[FM][FN], part[FM][FN];
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                acc[i][j] = f32x4{0, 0, 0, 0};
                part[i][j] = f32x4{0, 0, 0, 0};
            }
        uint32_t s = task.seg_begin, k0 = 0;
        if (s < task.seg_end) {
            Seg cur = segs[s];
            Seg nxt = cur;
            if (s + 1 < task.seg_end)
                nxt = segs[s + 1];
            __amdgpu_buffer_rsrc_t rA =
                pk_rsrc(A + ao + cur.a_off, task.row0, task.M, cur.lda, TM);
            __amdgpu_buffer_rsrc_t rB =
                pk_rsrc(B + bo + cur.b_off, task.col0, task.N, cur.ldb, TN);
            int buf = 0;
            ld.setup(cur, tid);
            ld.load(rA, rB, 0);
            ld.store(smem, tid);
            __syncthreads();
            float alpha = (float)cur.alpha; // of the segment in LDS
            while (true) {
                k0 += T::TK;
                const bool seg_done = k0 >= cur.K;
                const float a_done = alpha;
                if (seg_done) {
                    k0 = 0;
                    s++;
                    cur = nxt;
                    if (s + 1 < task.seg_end)
                        nxt = segs[s + 1];
                    rA =
                pk_rsrc(A + ao + cur.a_off, task.row0, task.M, cur.lda, TM);
                    rB =
                pk_rsrc(B + bo + cur.b_off, task.col0, task.N, cur.ldb, TN);
                    alpha = (float)cur.alpha;
                    ld.setup(cur, tid);
                }
                const bool more = s < task.seg_end;
                if (more)
                    ld.load(rA, rB, k0);
                const __bf16 *sAh = smem + buf * T::BUF;
                const __bf16 *sAl = sAh + T::ASZ;
                const __bf16 *sBh = sAh + 2 * T::ASZ;
                const __bf16 *sBl = sBh + T::BSZ;
                bf16x8 fah[FM], fal[FM], fbh[FN], fbl[FN];
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    const int r = wm * WM + i * 16 + lr;
                    fah[i] = *(const bf16x8 *)(sAh + T::slot(r, lk));
                    fal[i] = *(const bf16x8 *)(sAl + T::slot(r ^ 3, lk));
                }
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    const int r = wn * WN + j * 16 + lr;
                    fbh[j] = *(const bf16x8 *)(sBh + T::slot(r, lk));
                    fbl[j] = *(const bf16x8 *)(sBl + T::slot(r ^ 3, lk));
                }
                // small cross terms first, then the leading term
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++) {
                        part[i][j] = mfma_bf16(fal[i], fbh[j], part[i][j]);
                        part[i][j] = mfma_bf16(fah[i], fbl[j], part[i][j]);
                        part[i][j] = mfma_bf16(fah[i], fbh[j], part[i][j]);
                    }
                if (OUT == 1 && seg_done) {
                    mfma_settle<f32x4, FM * FN>(&part[0][0]);
#pragma unroll
                    for (int i = 0; i < FM; i++)
#pragma unroll
                        for (int j = 0; j < FN; j++) {
                            acc[i][j] += a_done * part[i][j];
                            part[i][j] = f32x4{0, 0, 0, 0};
                        }
                }
                if (!more)
                    break;
                buf ^= 1;
                ld.store(smem + buf * T::BUF, tid);
                __syncthreads();
            }
            __syncthreads();
        }
        if constexpr (OUT == 0) {
            // W^T through LDS: the tile (row m, column n) lands in a float
            // [TM][TN] array in the (free) staging buffers (columns permuted
            // by the group of 8 rows, for the banks of the reads), then
            // every thread writes 8 consecutive m of one W^T row as a
            // 16-byte vector per plane (whole rows of 256 bytes per 16
            // lanes)
            mfma_settle<f32x4, FM * FN>(&part[0][0]);
            static_assert(TM * TN * 4 <= 2 * T::BUF * 2, "W^T staging");
            float *tile = (float *)smem;
            auto at = [](int m, int n) {
                return m * TN + (n ^ (((m >> 3) << 2) & (TN - 1)));
            };
            __syncthreads();
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        tile[at(wm * WM + i * 16 + 4 * lk + r,
                                wn * WN + j * 16 + lr)] = part[i][j][r];
            __syncthreads();
            __bf16 *W = (__bf16 *)D0 + rhs * d_rs;
            constexpr int MG = TM / 8;
            for (int v = tid; v < TN * MG; v += 256) {
                const int n = v / MG, m0 = 8 * (v % MG);
                const uint32_t row = task.row0 + m0, col = task.col0 + n;
                if (row < task.ldd / 2 && col < task.N) {
                    bf16x8 h, l;
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        const float x = tile[at(m0 + q, n)];
                        const __bf16 xh = (__bf16)x;
                        h[q] = xh;
                        l[q] = (__bf16)(x - (float)xh);
                    }
                    __bf16 *o = W + task.d_off + pk_offset(col, row, task.ldd);
                    *(bf16x8 *)o = h;
                    *(bf16x8 *)(o + 32) = l;
                }
            }
            __syncthreads(); // the staging buffers are the next task's
        } else {
            double *D = (double *)D0 + rhs * d_rs;
            double *P = (double *)D1 + rhs * p_rs;
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const uint32_t row =
                            task.row0 + wm * WM + i * 16 + 4 * lk + r;
                        const uint32_t col = task.col0 + wn * WN + j * 16 + lr;
                        if (row < task.M && col < task.N) {
                            const uint64_t idx =
                                task.d_off + (uint64_t)row * task.ldd + col;
                            const double v = scale * (double)acc[i][j][r];
                            if (task.beta & 2)
                                P[idx] = v;
                            else if ((task.beta | beta0) & 1)
                                D[idx] += v;
                            else
                                D[idx] = v;
                        }
                    }
        }
    }
}

template <int OUT>
hipError_t launch_seg_gemm_pk(int cfg, const __bf16 *A, const __bf16 *B,
                              void *D0, void *D1, const Task *tasks, int ntasks,
                              const Seg *segs, uint64_t a_rs, uint64_t b_rs,
                              uint64_t d_rs, uint64_t p_rs, double scale,
                              int beta0, int n_rhs, int grid, hipStream_t st,
                              XcdSplit xs) {
    if (ntasks <= 0)
        return hipSuccess;
    const dim3 g = task_grid(grid, ntasks, n_rhs);
#define B2G_LAUNCH(TM_, TN_)                                                   \
    hipLaunchKernelGGL((seg_gemm_pk_kernel<TM_, TN_, OUT>), g, dim3(256), 0,   \
                       st, A, B, D0, D1, tasks, ntasks, segs, a_rs,            \
                       b_rs, d_rs, p_rs, scale, beta0, n_rhs, xs)
    switch (cfg) {
    case 0: B2G_LAUNCH(32, 32); break;
    case 1: B2G_LAUNCH(32, 64); break;
    case 2: B2G_LAUNCH(32, 128); break;
    case 3: B2G_LAUNCH(64, 32); break;
    case 4: B2G_LAUNCH(64, 64); break;
    case 5: B2G_LAUNCH(64, 128); break;
    case 6: B2G_LAUNCH(128, 32); break;
    case 7: B2G_LAUNCH(128, 64); break;
    default: B2G_LAUNCH(128, 128); break;
    }
#undef B2G_LAUNCH
    return hipGetLastError();
}

template hipError_t launch_seg_gemm_pk<0>(int, const __bf16 *, const __bf16 *,
                                          void *, void *, const Task *, int,
                                          const Seg *, uint64_t, uint64_t,
                                          uint64_t, uint64_t, double, int, int,
                                          int, hipStream_t, XcdSplit);
template hipError_t launch_seg_gemm_pk<1>(int, const __bf16 *, const __bf16 *,
                                          void *, void *, const Task *, int,
                                          const Seg *, uint64_t, uint64_t,
                                          uint64_t, uint64_t, double, int, int,
                                          int, hipStream_t, XcdSplit);

} // namespace b2g
