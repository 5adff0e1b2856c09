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
        if constexpr (KS > 1)
        {
            // partial sums of the other wave sets, in the stage buffers
            v4d* red = (v4d*)lds;
            if (kw > 0)
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        red[(((kw - 1) * WGM * WGN + wave) * MB * NB + i * NB + j) * 64 + lane] = acc[i][j];
            __syncthreads();
            if (kw == 0)
#pragma unroll
                for (int q = 0; q < KS - 1; q++)
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++)
                            acc[i][j] += red[((q * WGM * WGN + wave) * MB * NB + i * NB + j) * 64 + lane];
        }

        // D register r of lane l holds D[l / 16 + 4 r][l % 16] of each block
        const int cl = lane & 15, rl = lane >> 4;
        if (KS > 1 && kw > 0)
        {
            // set 0 writes the tile
        }
        else if (t.c_ld > 0)
        {
            // unscaled sums into a C panel (leading dimension c_ld at c_src
            // in cws): one k slice's, or a timing run's
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                {
                    const int row = wm * WM + i * 16 + rl + 4 * r;
                    if (row >= t.mlen) continue;
#pragma unroll
                    for (int j = 0; j < NB; j++)
                    {
                        const int col = wn * WN + j * 16 + cl;
                        if (col < t.nlen) cws[t.c_src + (int64_t)row * t.c_ld + col] = acc[i][j][r];
                    }
                }
        }
        else
        {
            // c_ld == 0: C through its row and column offsets
            int64_t coff[NB];
#pragma unroll
            for (int j = 0; j < NB; j++)
            {
                const int col = wn * WN + j * 16 + cl;
                coff[j] = col < t.nlen ? pool[t.c_colmap + col] : 0;
            }
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                {
                    const int row = wm * WM + i * 16 + rl + 4 * r;
                    if (row >= t.mlen) continue;
                    const int64_t roff = t.c_src + pool[t.c_rowmap + row];
#pragma unroll
                    for (int j = 0; j < NB; j++)
                    {
                        const int col = wn * WN + j * 16 + cl;
                        if (col >= t.nlen) continue;
                        TC* p = C + roff + coff[j];
                        double v = alpha * acc[i][j][r];
                        if (beta != 0.0) v += beta * (double)*p;
                        *p = (TC)v;
                    }
                }
        }
        // the next task's stages reuse the LDS
        __syncthreads();
    }
}

struct LdsTile
{
    int bm, bn, wgm, wgn, ks, bk;
};

// id (after the register-fed tiles), BM, BN, waves WGM x WGN x KS (four), k per stage
#define TBLIS_LDS_TILES(X)    \
    X(0, 128, 128, 2, 2, 1, 16) \
    X(1, 64, 64, 2, 2, 1, 16)   \
    X(2, 32, 32, 1, 1, 4, 32)

constexpr LdsTile kLTiles[] = {
#define X(id, bm, bn, wgm, wgn, ks, bk) {bm, bn, wgm, wgn, ks, bk},
    TBLIS_LDS_TILES(X)
#undef X
};
constexpr int kNumLTiles = sizeof(kLTiles) / sizeof(kLTiles[0]);

template <int BM, int BN, int WGM, int WGN, int KS, int BK, typename TC, int AK, int BKL, bool SC>
hipError_t launch_gather_t(const PanelLaunch& L)
{
    auto* k = &gemm_gather_kernel<BM, BN, WGM, WGN, KS, BK, TC, AK, BKL, SC>;
    const dim3 grid(persistent_grid((const void*)k, kNT, L.ntasks));
    hipLaunchKernelGGL(k, grid, dim3(kNT), 0, L.stream, L.tasks, L.ntasks, L.pool, (const TC*)L.A, (const TC*)L.B,
                       (TC*)L.C, L.cws, L.alpha, L.beta, L.use_k);
    return hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN, int KS, int BK, typename TC, bool SC>
hipError_t launch_gather_k(const PanelLaunch& L)
{
    switch (L.group)
    {
        case 0: return launch_gather_t<BM, BN, WGM, WGN, KS, BK, TC, 0, 0, SC>(L);
        case 1: return launch_gather_t<BM, BN, WGM, WGN, KS, BK, TC, 1, 0, SC>(L);
        case 2: return launch_gather_t<BM, BN, WGM, WGN, KS, BK, TC, 0, 1, SC>(L);
        case 3: return launch_gather_t<BM, BN, WGM, WGN, KS, BK, TC, 1, 1, SC>(L);
    }
    return hipErrorInvalidValue;
}

template <typename TC, bool SC>
hipError_t launch_lds_t(const PanelLaunch& L, int lt)
{
    switch (lt)
    {
#define X(id, bm, bn, wgm, wgn, ks, bk) \
    case id: return launch_gather_k<bm, bn, wgm, wgn, ks, bk, TC, SC>(L);
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
