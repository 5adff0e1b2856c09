// FP64 MFMA GEMM that gathers both operands straight from the tensors
// through LDS (gfx950): no pack pass and no panels.
//
// For GEMMs with one row block per operand and any number of k blocks
// (dense contractions, merged DPD irrep GEMMs, batch instances).  Element
// (r, k) of an operand is at tensor + rows[r] + kmap[k]: one 32-bit row offset and
// one 64-bit k offset (its k block's base included) from the plan's tables,
// so that scattered, strided, broadcast and multi-block k are one path.  Rows
// past the tile's valid rows re-read row 0 (their products go to rows of C
// that nobody stores) and k past the task's end is stored as zero.
//
// Per stage of BK k the 256 threads load the tile's A' (BM x BK) and B'
// (BN x BK) elements with lanes along whichever side of the operand is
// unit-stride (rows, or k; one kernel per combination), one element per
// load: a stage's loads are issued a whole stage of MFMAs before their
// values go to LDS, and the k offsets a stage before that.  LDS holds two
// stages as [k][row]: rows are padded by 16 doubles, which puts the k rows
// 2q and 2q + 1 that half a wave reads together on different halves of the
// banks, and XORed with 2 ((k / 2) % 8), which spreads the 16 k that half a
// wave of lanes along k writes over all of them; both accesses are then free
// of conflicts.  One barrier per stage.  v_mfma_f64_16x16x4 takes 64 cycles
// per SIMD, so the gather's address arithmetic and LDS traffic run beside it.
//
// KS > 1: the KS sets of waves take the stage's k steps in turn and their
// sums meet in LDS before the epilogue (small C tiles, all four waves busy).
// A task covers k in [kbeg, klen): a GEMM whose tiles do not fill the chip
// is cut along k into several tasks per tile, each storing its sums in a
// C panel of its own (c_ld > 0), which reduce_slices_kernel adds up.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace tblis_amd
{

namespace
{

typedef double v4d __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) char* GlobalBytes;

constexpr int kNT = 256;   // threads per workgroup
constexpr int kRowPad = 16;  // doubles between the k rows of a stage

__device__ __forceinline__ int row_swizzle(int k) { return ((k >> 1) & 7) << 1; }

// One operand of a task: this thread's elements of a stage of BK k x R rows.
//   KL == 0 (lanes along rows): row tid % R, k = NE (tid / R) + j
//   KL == 1 (lanes along k):    k = tid % BK, row tid / BK + (kNT / BK) j
// Addresses cost (next to) no vector instructions, which do not run beside
// FP64 MFMAs on a SIMD: rows and k are byte offsets, and where a wave's k are
// uniform (64 or more rows along lanes) the k offset is added to the base in
// scalar registers.
template <int R, int BK, int KL, bool SC, typename TC>
struct GatherSide
{
    static constexpr int NE = R * BK / kNT;
    static constexpr int NR = KL ? NE : 1, NK = KL ? 1 : NE;
    static constexpr bool UK = !KL && R % 64 == 0;
    static_assert(R * BK % kNT == 0 && kNT % R == 0 && kNT % BK == 0, "stage shape");

    const char* x;
    const int64_t* km;
    const double* ks;  // per-k scales (SC)
    uint32_t roff[NR];
    int64_t koff[NK], knext[NK];
    double kscale[SC ? NK : 1], snext[SC ? NK : 1], vscale[SC ? NK : 1];
    TC v[NE];
    int r0, k0;  // this thread's first row and k within the stage

    __device__ __forceinline__ void init(const TC* X, int64_t src, const int64_t* __restrict__ pool, int64_t rows,
                                         int64_t kmap, int64_t scales, int valid, int tid)
    {
        x = (const char*)(X + src);
        km = pool + kmap;
        ks = (const double*)(pool + scales);
        const int q = tid / R;
        r0 = KL ? tid / BK : tid % R;
        k0 = KL ? tid % BK : NE * (UK ? __builtin_amdgcn_readfirstlane(q) : q);
#pragma unroll
        for (int j = 0; j < NR; j++)
        {
            const int r = r0 + (KL ? kNT / BK * j : 0);
            roff[j] = (uint32_t)pool[rows + (r < valid ? r : 0)];
        }
    }
    // k offsets of the stage at k (the tables go on past the last k)
    __device__ __forceinline__ void fetch(int k)
    {
        const int64_t* m = km + k;
        const double* sc = ks + k;
#pragma unroll
        for (int j = 0; j < NK; j++)
        {
            knext[j] = UK ? m[k0 + j] : (int64_t)((const uint32_t*)m)[2 * (uint32_t)(k0 + j)];
            if constexpr (SC) snext[j] = sc[(uint32_t)(k0 + j)];
        }
    }
    __device__ __forceinline__ void load()
    {
#pragma unroll
        for (int j = 0; j < NE; j++)
        {
            if constexpr (UK)
            {
                // the base and k offset stay together in scalar registers
                GlobalBytes b = (GlobalBytes)x + koff[j];
                asm("" : "+s"(b));
                v[j] = *(const __attribute__((address_space(1))) TC*)(b + roff[0]);
            }
            else
                v[j] = *(const TC*)(x + (roff[KL ? j : 0] + (uint32_t)koff[KL ? 0 : j]));
        }
        if constexpr (SC)
#pragma unroll
            for (int j = 0; j < NK; j++) vscale[j] = kscale[j];
    }
    // the fetched offsets become those of the next load
    __device__ __forceinline__ void advance()
    {
#pragma unroll
        for (int j = 0; j < NK; j++)
        {
            koff[j] = knext[j];
            if constexpr (SC) kscale[j] = snext[j];
        }
    }
    // the loaded stage into LDS; TAIL: zeros from its left-th k on
    template <bool TAIL>
    __device__ __forceinline__ void store(double* __restrict__ lds, int left) const
    {
#pragma unroll
        for (int j = 0; j < NE; j++)
        {
            const int kk = k0 + (KL ? 0 : j), r = r0 + (KL ? kNT / BK * j : 0);
            double d = (double)v[j];
            if constexpr (SC) d *= vscale[KL ? 0 : j];
            if (TAIL) d = kk < left ? d : 0.0;
            lds[kk * (R + kRowPad) + (r ^ row_swizzle(kk))] = d;
        }
    }
};

// The tile's sums (the KS wave sets' together) into C with alpha / beta, or
// into a C panel.  red0, red1: LDS that no wave reads any more, 2 W MB NB KiB
// and W MB NB KiB times two (KS up to 4).
template <int MB, int NB, int W, int KS, typename TC>
__device__ __forceinline__ void finish_tile(const PanelTask& t, v4d (&acc)[MB][NB], v4d* red0, v4d* red1, int kw,
                                            int wave, int r0, int c0, int lane, const int64_t* __restrict__ pool,
                                            TC* __restrict__ C, double* __restrict__ cws, double alpha, double beta)
{
    if constexpr (KS > 1)
    {
        // partial sums of the other wave sets
        auto part = [&](int q) {
            return (q < 3 ? red0 + (q - 1) * W * MB * NB * 64 : red1 + (q - 3) * W * MB * NB * 64) +
                   wave * MB * NB * 64 + lane;
        };
        if (kw > 0)
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) part(kw)[(i * NB + j) * 64] = acc[i][j];
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int q = 1; q < KS; q++)
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] += part(q)[(i * NB + j) * 64];
    }
    // D register r of lane l holds D[l / 16 + 4 r][l % 16] of each block
    const int cl = lane & 15, rl = lane >> 4;
    if (t.c_ld > 0)
    {
        // unscaled sums into a C panel (leading dimension c_ld at c_src in
        // cws): one k slice's, or a timing run's
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 4; r++)
            {
                const int row = r0 + i * 16 + rl + 4 * r;
                if (row >= t.mlen) continue;
#pragma unroll
                for (int j = 0; j < NB; j++)
                {
                    const int col = c0 + j * 16 + cl;
                    if (col < t.nlen) cws[t.c_src + (int64_t)row * t.c_ld + col] = acc[i][j][r];
                }
            }
        return;
    }
    // c_ld == 0: C through its row and column offsets
    int64_t coff[NB];
#pragma unroll
    for (int j = 0; j < NB; j++)
    {
        const int col = c0 + j * 16 + cl;
        coff[j] = col < t.nlen ? pool[t.c_colmap + col] : 0;
    }
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
        {
            const int row = r0 + i * 16 + rl + 4 * r;
            if (row >= t.mlen) continue;
            const int64_t roff = t.c_src + pool[t.c_rowmap + row];
#pragma unroll
            for (int j = 0; j < NB; j++)
            {
                const int col = c0 + j * 16 + cl;
                if (col >= t.nlen) continue;
                TC* p = C + roff + coff[j];
                double v = alpha * acc[i][j][r];
                if (beta != 0.0) v += beta * (double)*p;
                *p = (TC)v;
            }
        }
}

template <int BM, int BN, int WGM, int WGN, int KS, int BK, typename TC, int AK, int BKL, bool SC>
__global__ __launch_bounds__(kNT, BM == 128 ? 2 : BM == 64 ? 4 : 3) void gemm_gather_kernel(const PanelTask* __restrict__ tasks, int ntasks,
                                                          const int64_t* __restrict__ pool, const TC* A,
                                                          const TC* B, TC* __restrict__ C,
                                                          double* __restrict__ cws, double alpha, double beta,
                                                          int use_k)
{
    static_assert(WGM * WGN * KS * 64 == kNT, "four waves");
    constexpr int WM = BM / WGM, WN = BN / WGN, MB = WM / 16, NB = WN / 16;
    constexpr int SA = BK * (BM + kRowPad), SB = BK * (BN + kRowPad);  // doubles per stage
    constexpr int RED = KS > 1 ? (KS - 1) * WGM * WGN * MB * NB * 64 * 4 : 0;
    __shared__ double lds[2 * (SA + SB) > RED ? 2 * (SA + SB) : RED];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave_all / (WGM * WGN), wave = wave_all % (WGM * WGN);
    const int wm = wave % WGM, wn = wave / WGM;
    const int lr = lane & 15, lk = lane >> 4;

    for (int ti = blockIdx.x; ti < ntasks; ti += gridDim.x)
    {
        const PanelTask t = tasks[ti];
        v4d acc[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

        const int kend = t.klen;
        const int nst = use_k && kend > t.kbeg ? (kend - t.kbeg + BK - 1) / BK : 0;
        if (nst > 0)
        {
            GatherSide<BM, BK, AK, SC, TC> a;
            GatherSide<BN, BK, BKL, false, TC> b;
            a.init(A, t.a_src, pool, t.a_rt, t.a_km, t.a_kt, t.mlen, tid);
            b.init(B, t.b_src, pool, t.b_rt, t.b_km, 0, t.nlen, tid);
            int k = t.kbeg;  // of the stage fetched next
            auto fetch = [&]() {
                a.fetch(k);
                b.fetch(k);
                k += BK;
            };
            auto load = [&]() {
                a.load();
                b.load();
                a.advance();
                b.advance();
            };
            fetch();
            a.advance();
            b.advance();
            fetch();
            load();
            const int left = kend - t.kbeg - (nst - 1) * BK;  // k of the last stage
            if (nst == 1)
            {
                a.template store<true>(lds, left);
                b.template store<true>(lds + SA, left);
            }
            else
            {
                a.template store<false>(lds, 0);
                b.template store<false>(lds + SA, 0);
            }
            fetch();
            load();
            __syncthreads();
            auto multiply = [&](const double* cur) {
                constexpr int Q = BK / 4 / KS;
                // 32 x 32 wave tiles read a step's operands ahead of the
                // previous step's MFMAs; 64 x 64 ones have no registers left
                // for it (16 MFMAs a step cover the reads of the other wave)
                constexpr int D = MB * NB <= 4 ? 2 : 1;
                double fa[D][MB], fb[D][NB];
                auto frags = [&](int q) {
                    const int kr = 4 * (KS * q + kw) + lk;
                    const double* pa = cur + kr * (BM + kRowPad) + wm * WM + (lr ^ row_swizzle(kr));
                    const double* pb = cur + SA + kr * (BN + kRowPad) + wn * WN + (lr ^ row_swizzle(kr));
#pragma unroll
                    for (int i = 0; i < MB; i++) fa[q % D][i] = pa[16 * i];
#pragma unroll
                    for (int j = 0; j < NB; j++) fb[q % D][j] = pb[16 * j];
                };
                if (D > 1) frags(0);
#pragma unroll
                for (int q = 0; q < Q; q++)
                {
                    if (D == 1)
                        frags(q);
                    else
                    {
                        if (q + 1 < Q) frags(q + 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++)
                            acc[i][j] =
                                __builtin_amdgcn_mfma_f64_16x16x4f64(fa[q % D][i], fb[q % D][j], acc[i][j], 0, 0, 0);
                    if (D > 1) __builtin_amdgcn_sched_barrier(0);
                }
            };
            // stage s from cur while stage s + 1 goes to nxt
            auto stage = [&](const double* cur, double* nxt) {
                fetch();
                a.template store<false>(nxt, 0);
                b.template store<false>(nxt + SA, 0);
                load();
                multiply(cur);
                __syncthreads();
            };
            // Two stages per pass, so that the LDS addresses of each are
            // constants; the last stage (the only one that may be short) and
            // the one that stores it come after the loop.  The loads go on
            // past the task's last stage (in bounds: the k tables' padding
            // repeats the last k), their values are not used.
            double* const buf0 = lds;
            double* const buf1 = lds + SA + SB;
            int s = 0;
            for (; s + 3 < nst; s += 2)
            {
                stage(buf0, buf1);
                stage(buf1, buf0);
            }
            if (s + 2 < nst)
            {
                stage(buf0, buf1);
                s++;
            }
            if (s + 1 < nst)
            {
                double* cur = lds + (s & 1) * (SA + SB);
                double* nxt = lds + (~s & 1) * (SA + SB);
                a.template store<true>(nxt, left);
                b.template store<true>(nxt + SA, left);
                multiply(cur);
                __syncthreads();
                s++;
            }
            multiply(lds + (s & 1) * (SA + SB));
            if constexpr (KS > 1) __syncthreads();  // the stages are read
        }
        finish_tile<MB, NB, WGM * WGN, KS>(t, acc, (v4d*)lds, (v4d*)lds + 2 * WGM * WGN * MB * NB * 64, kw, wave, wm * WM,
                                           wn * WN, lane, pool, C, cws, alpha, beta);
        // the next task's stages reuse the LDS
        __syncthreads();
    }
}

// ------------------------------------------------- 16-byte pieces, no registers
//
// The same product for FP64 operands whose elements come in aligned pairs
// (see vec_layout in panel.cpp): 16 bytes per lane go from memory straight
// to LDS, and every address of a stage is the stage's first k offset (a
// scalar) plus a per-thread constant.  Per 64 x 64 x 16 stage a wave issues
// 4 loads and 8 LDS reads for 16 MFMAs, where the element-wise kernel has 9
// loads, 8 LDS writes, 8 LDS reads and 16 address instructions; each of
// these takes about 8 cycles from the MFMAs of its SIMD.  Without staging
// registers NST stages can be in flight.
//
// Pieces in LDS, 16 bytes each:
//   lanes along rows: [k][row pair], pairs XORed with 8 ((k / 2) % 2)
//   lanes along k:    [row][k pair], pairs XORed with the row (/ 2)
// MFMA step h (0, 1) of an 8-k group takes k = 2 lk + h in lane quarter lk,
// so that a pair of k is one 16-byte read.  Half a wave's 8-byte reads of
// pairs (2 k, 16 rows) and a quarter's 16-byte reads (16 rows) touch every
// bank once.
template <int R, int BK, int KL>
struct PieceSide
{
    static constexpr int N = R * BK / 2 / kNT;  // pieces per thread
    static constexpr int U = BK / 2;            // k pairs per row
    static_assert(R * BK / 2 % kNT == 0, "stage shape");

    const char* x;
    const int64_t* km;
    uint32_t off[N];
    int64_t base;  // k offset of the stage loaded next

    static __device__ __forceinline__ int piece(int j, int wave, int lane) { return (j * (kNT / 64) + wave) * 64 + lane; }
    static __device__ __forceinline__ int kswz(int row) { return U == 8 ? (row >> 1) & 7 : row & (U - 1); }
    // first k within the stage of a piece
    static __device__ __forceinline__ int piece_k(int u)
    {
        return KL ? 2 * ((u % U) ^ kswz(u / U)) : u / (R / 2);
    }
    __device__ __forceinline__ void init(const double* X, int64_t src, const int64_t* __restrict__ pool, int64_t rows,
                                         int64_t kmap, int kbeg, int kend, int valid, int wave, int lane)
    {
        x = (const char*)(X + src);
        km = pool + kmap + kbeg;
#pragma unroll
        for (int j = 0; j < N; j++)
        {
            const int u = piece(j, wave, lane);
            const int k = piece_k(u);
            int r = KL ? u / U : 2 * ((u % (R / 2)) ^ (((k >> 1) & 1) << 3));
            r = r < valid ? r : 0;
            const int kk = k < kend - kbeg ? k : 0;  // short tasks: pieces past the end are not loaded
            off[j] = (uint32_t)pool[rows + r] + (uint32_t)(km[kk] - km[0]);
        }
    }
    __device__ __forceinline__ void fetch(int k) { base = km[k]; }
    // left: valid k of the stage (TAIL); pieces past it become zeros
    template <bool TAIL>
    __device__ __forceinline__ void load(double* lds, int left, int wave, int lane) const
    {
        GlobalBytes b = (GlobalBytes)x + base;
        asm("" : "+s"(b));
#pragma unroll
        for (int j = 0; j < N; j++)
        {
            const int u0 = piece(j, wave, 0);
            if (!TAIL || piece_k(u0 + lane) < left)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(b + off[j]),
                                                 (__attribute__((address_space(3))) void*)(lds + 2 * u0), 16, 0, 0);
            else
                *(double2*)(lds + 2 * (u0 + lane)) = double2{0.0, 0.0};
        }
    }
    // operand of the two MFMA steps of the 8-k group g: row r0 + lr
    static __device__ __forceinline__ void frag(double (&v)[2], const double* lds, int g, int r0, int lr, int lk)
    {
        if constexpr (KL)
        {
            const int row = r0 + lr;
            const double2 d = *(const double2*)(lds + 2 * (row * U + ((4 * g + lk) ^ kswz(lr))));
            v[0] = d.x;
            v[1] = d.y;
        }
        else
        {
            const int p = ((r0 + lr) >> 1) ^ ((lk & 1) << 3);
            const double* q = lds + 2 * ((8 * g + 2 * lk) * (R / 2) + p) + (lr & 1);
            v[0] = q[0];
            v[1] = q[R];
        }
    }
};

template <int VM>
__device__ __forceinline__ void wait_and_barrier()
{
    // at most VM loads of this wave in flight, its LDS accesses done
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | 7 << 4 | 0 << 8 | (VM >> 4) << 14);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int BM, int BN, int WGM, int WGN, int KS, int BK, int NST, int OCC, int AK, int BKL>
__global__ __launch_bounds__(kNT, OCC) void gemm_pieces_kernel(const PanelTask* __restrict__ tasks, int ntasks,
                                                               const int64_t* __restrict__ pool, const double* A,
                                                               const double* B, double* __restrict__ C,
                                                               double* __restrict__ cws, double alpha, double beta,
                                                               int use_k)
{
    static_assert(WGM * WGN * KS * 64 == kNT && NST >= 2 && NST <= 4, "four waves");
    constexpr int WM = BM / WGM, WN = BN / WGN, MB = WM / 16, NB = WN / 16;
    constexpr int SA = BK * BM, ST = BK * (BM + BN);  // doubles
    constexpr int G = BK / 8 / KS;                    // 8-k groups of a stage per wave set
    // one variable per stage: the compiler then knows which stage's loads an
    // LDS read has to wait for
    __shared__ double ring0[ST], ring1[ST], ring2[NST > 2 ? ST : 2], ring3[NST > 3 ? ST : 2];
    static_assert(KS == 1 || (KS <= 4 && 2 * WGM * WGN * MB * NB * 256 <= ST), "partial sums fit two stages");
    using PA = PieceSide<BM, BK, AK>;
    using PB = PieceSide<BN, BK, BKL>;
    constexpr int PER = PA::N + PB::N;  // loads of a wave per stage

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave_all / (WGM * WGN), wave = wave_all % (WGM * WGN);
    const int wm = wave % WGM, wn = wave / WGM;
    const int lr = lane & 15, lk = lane >> 4;

    for (int ti = blockIdx.x; ti < ntasks; ti += gridDim.x)
    {
        const PanelTask t = tasks[ti];
        v4d acc[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

        const int kend = t.klen;
        const int nst = use_k && kend > t.kbeg ? (kend - t.kbeg + BK - 1) / BK : 0;
        if (nst > 0)
        {
            PA a;
            PB b;
            a.init(A, t.a_src, pool, t.a_rt, t.a_km, t.kbeg, kend, t.mlen, wave_all, lane);
            b.init(B, t.b_src, pool, t.b_rt, t.b_km, t.kbeg, kend, t.nlen, wave_all, lane);
            const int left = kend - t.kbeg - (nst - 1) * BK;  // k of the last stage
            int k = 0;                                         // of the stage fetched next
            auto fetch = [&]() {
                a.fetch(k);
                b.fetch(k);
                k += BK;
            };
            auto whole = [&](double* st) {
                a.template load<false>(st, 0, wave_all, lane);
                b.template load<false>(st + SA, 0, wave_all, lane);
            };
            auto tail = [&](double* st) {
                a.template load<true>(st, left, wave_all, lane);
                b.template load<true>(st + SA, left, wave_all, lane);
            };
            auto multiply = [&](const double* cur) {
                double fa[2][MB][2], fb[2][NB][2];
                auto frags = [&](int g) {
                    const int gg = KS * g + kw;
#pragma unroll
                    for (int i = 0; i < MB; i++) PA::frag(fa[g & 1][i], cur, gg, wm * WM + 16 * i, lr, lk);
#pragma unroll
                    for (int j = 0; j < NB; j++) PB::frag(fb[g & 1][j], cur + SA, gg, wn * WN + 16 * j, lr, lk);
                };
                frags(0);
#pragma unroll
                for (int g = 0; g < G; g++)
                {
                    if (g + 1 < G) frags(g + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int i = 0; i < MB; i++)
#pragma unroll
                            for (int j = 0; j < NB; j++)
                                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[g & 1][i][h], fb[g & 1][j][h],
                                                                                 acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            auto ring = [&](int s) { return s == 0 ? ring0 : s == 1 ? ring1 : s == 2 ? ring2 : ring3; };
            // fill NST - 1 stages
            fetch();
#pragma unroll
            for (int s = 0; s < NST - 1; s++)
            {
                if (s + 1 < nst)
                    whole(ring(s));
                else if (s + 1 == nst)
                    tail(ring(s));
                fetch();  // (the k tables go on past the last k)
            }
            // stage s from cur; its successor NST - 1 stages on goes to nxt,
            // which the barrier has shown to be read
            auto stage = [&](const double* cur, double* nxt) {
                wait_and_barrier<(NST - 2) * PER>();
                whole(nxt);
                fetch();
                multiply(cur);
            };
            // whole stages in passes over the ring, so that LDS addresses
            // are constants
            int s = 0;
            for (; s + 2 * NST - 1 < nst; s += NST)
            {
                if constexpr (NST == 2)
                {
                    stage(ring0, ring1);
                    stage(ring1, ring0);
                }
                else if constexpr (NST == 3)
                {
                    stage(ring0, ring2);
                    stage(ring1, ring0);
                    stage(ring2, ring1);
                }
                else
                {
                    stage(ring0, ring3);
                    stage(ring1, ring0);
                    stage(ring2, ring1);
                    stage(ring3, ring2);
                }
            }
            // the remaining stages (fewer than two passes), the last of them short
            auto last = [&](const double* cur, double* nxt) {
                if (s >= nst) return;
                wait_and_barrier<0>();
                if (s + NST < nst)
                    whole(nxt);
                else if (s + NST == nst)
                    tail(nxt);
                fetch();
                multiply(cur);
                s++;
            };
            while (s < nst)
            {
                last(ring0, NST == 2 ? ring1 : NST == 3 ? ring2 : ring3);
                last(ring1, ring0);
                if constexpr (NST > 2) last(ring2, ring1);
                if constexpr (NST > 3) last(ring3, ring2);
            }
            if constexpr (KS > 1) __syncthreads();  // the stages are read
        }
        finish_tile<MB, NB, WGM * WGN, KS>(t, acc, (v4d*)ring0, (v4d*)ring1, kw, wave, wm * WM, wn * WN, lane, pool, C,
                                           cws, alpha, beta);
        __syncthreads();  // the next task's stages reuse the LDS
    }
}

struct LdsTile
{
    int bm, bn, wgm, wgn, ks, bk;
};

// id (after the register-fed tiles), BM, BN, waves WGM x WGN x KS (four), k
// per stage; pieces: stages in flight + 1, workgroups per CU
#define TBLIS_LDS_TILES(X)            \
    X(0, 128, 64, 2, 2, 1, 16, 3, 2)  \
    X(1, 64, 64, 2, 2, 1, 16, 2, 4)   \
    X(2, 32, 32, 1, 1, 4, 32, 2, 4)

constexpr LdsTile kLTiles[] = {
#define X(id, bm, bn, wgm, wgn, ks, bk, nst, occ) {bm, bn, wgm, wgn, ks, bk},
    TBLIS_LDS_TILES(X)
#undef X
};
constexpr int kNumLTiles = sizeof(kLTiles) / sizeof(kLTiles[0]);

template <int BM, int BN, int WGM, int WGN, int KS, int BK, int NST, int OCC, typename TC, bool SC>
hipError_t launch_gather_k(const PanelLaunch& L)
{
    auto go = [&](auto* k) {
        const dim3 grid(persistent_grid((const void*)k, kNT, L.ntasks));
        hipLaunchKernelGGL(k, grid, dim3(kNT), 0, L.stream, L.tasks, L.ntasks, L.pool, (const TC*)L.A, (const TC*)L.B,
                           (TC*)L.C, L.cws, L.alpha, L.beta, L.use_k);
        return hipGetLastError();
    };
    // 16-byte pieces: the plan's offsets allow them and the tensors start on 16 bytes
    if constexpr (sizeof(TC) == 8 && !SC)
        if (L.pieces && ((uintptr_t)L.A | (uintptr_t)L.B) % 16 == 0)
            switch (L.group)
            {
                case 0: return go(&gemm_pieces_kernel<BM, BN, WGM, WGN, KS, BK, NST, OCC, 0, 0>);
                case 1: return go(&gemm_pieces_kernel<BM, BN, WGM, WGN, KS, BK, NST, OCC, 1, 0>);
                case 2: return go(&gemm_pieces_kernel<BM, BN, WGM, WGN, KS, BK, NST, OCC, 0, 1>);
                case 3: return go(&gemm_pieces_kernel<BM, BN, WGM, WGN, KS, BK, NST, OCC, 1, 1>);
            }
    switch (L.group)
    {
        case 0: return go(&gemm_gather_kernel<BM, BN, WGM, WGN, KS, BK, TC, 0, 0, SC>);
        case 1: return go(&gemm_gather_kernel<BM, BN, WGM, WGN, KS, BK, TC, 1, 0, SC>);
        case 2: return go(&gemm_gather_kernel<BM, BN, WGM, WGN, KS, BK, TC, 0, 1, SC>);
        case 3: return go(&gemm_gather_kernel<BM, BN, WGM, WGN, KS, BK, TC, 1, 1, SC>);
    }
    return hipErrorInvalidValue;
}

template <typename TC, bool SC>
hipError_t launch_lds_t(const PanelLaunch& L, int lt)
{
    switch (lt)
    {
#define X(id, bm, bn, wgm, wgn, ks, bk, nst, occ) \
    case id: return launch_gather_k<bm, bn, wgm, wgn, ks, bk, nst, occ, TC, SC>(L);
        TBLIS_LDS_TILES(X)
#undef X
        default:
            return hipErrorInvalidValue;
    }
}

}  // namespace

int lds_num_tiles() { return kNumLTiles; }
int lds_tile_m(int lt) { return kLTiles[lt].bm; }
int lds_tile_n(int lt) { return kLTiles[lt].bn; }
int lds_tile_k(int lt) { return kLTiles[lt].bk; }

hipError_t launch_gemm_lds(const PanelLaunch& L, int lt)
{
    if (L.ntasks == 0) return hipSuccess;
    if (lt < 0 || lt >= kNumLTiles) return hipErrorInvalidValue;
    if (L.scaled) return L.dtype == 0 ? launch_lds_t<double, true>(L, lt) : launch_lds_t<float, true>(L, lt);
    return L.dtype == 0 ? launch_lds_t<double, false>(L, lt) : launch_lds_t<float, false>(L, lt);
}

}  // namespace tblis_amd
