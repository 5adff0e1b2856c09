// Split-BF16 MFMA GEMM that gathers both FP32 operands straight from the
// tensors through LDS (gfx950): no pack pass and no panels.
//
// The products and sums are those of the panel kernel (gemm_panel_bf16.hip):
// x = hi + mid + lo in BF16, six products per block, FP32 sums restarted
// every 256 k.  Here each element is loaded as FP32 (4 bytes where the pack
// and the panels move 4 + 6 + 6), split once per workgroup in registers and
// put into LDS as the three terms, from where every wave reads MFMA operands.
//
// A thread's unit of a stage is 8 consecutive k of one row:
//   mode 0  lanes along rows: one 4-byte load per k, the k offset (uniform
//           over a wave) added to the base in scalar registers
//   mode 1  lanes along k, BK of them to a row: one 4-byte load per element of
//           8 rows, turned into units through the wave's own rows of the LDS
//           stage that the units then fill
//   mode 2  lanes along k, the unit one aligned run: two 16-byte loads
// Offsets are 32-bit bytes from the operand's lowest element (the plan's
// tables).  Loads go out a stage before their values are split, k offsets a
// stage before that.  LDS: two stages of [term][octet][row] with
// 16 bytes per (octet, row), rows XORed with the octet, so that neither the
// writes of lanes along k nor the reads conflict.  One barrier per stage.
//
// Per 16 k the 128 x 128 tile takes 768 cycles of MFMA, 560 of LDS (72 KiB)
// and about 440 of vector instructions; the 64 x 64 tile 192, 288 and 220.
// The splits, LDS round trips and MFMAs of a stage follow one another in a
// wave, so what overlaps them is the other workgroups of the CU (two, three):
// with more registers per thread for a second set of loads in flight the
// 1024-instance batch took 2955 us instead of 2289.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace tblis_amd
{

namespace
{

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float staged_f32 __attribute__((may_alias));  // FP32 values in the LDS of BF16 stages
typedef const __attribute__((address_space(1))) char* GlobalBytes;

// Two values rounded to BF16 in one word (the first in the low half), and
// what is left of them.
__device__ __forceinline__ uint32_t round_pair(float& a, float& b)
{
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
    a -= __builtin_bit_cast(float, w << 16);
    b -= __builtin_bit_cast(float, w & 0xffff0000u);
    return w;
}

// Orders this wave's LDS accesses before and after it, for lanes that read
// what other lanes of the wave wrote.  A wave's LDS accesses are carried out
// in order, so that only the compiler has to keep it: no instruction.
__device__ __forceinline__ void wave_exchange()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kNT = 256;  // threads per workgroup: one unit of A' and of B' per stage

// One operand of a task.
template <int R, int BK, int mode>
struct UnitSide
{
    static constexpr int O = BK / 8;
    static_assert(R * O == kNT && R % 64 == 0, "one unit per thread");
    static constexpr int TERM = O * R;             // pieces (16 bytes) of a term of a stage
    static constexpr int RW = 64 / O;              // rows of a wave's units
    static constexpr int RP = RW * 16 / (4 * BK);  // rows staged per (term, octet) run of RW pieces

    const char* x;
    const uint32_t* km;
    static constexpr int NR = mode == 1 ? 8 : 1, NK = mode == 0 ? 8 : 1;
    uint32_t roff[NR], koff[NK], knext[NK];
    float v[8];
    int row, oct;  // the unit
    int wrow, kk;  // the wave's first row; this lane's k (octet's first in mode 2)

    __device__ __forceinline__ void init(const float* X, int64_t src, const int64_t* __restrict__ pool,
                                         int64_t rows, int64_t kmap, int valid, int tid)
    {
        x = (const char*)(X + src);
        km = (const uint32_t*)(pool + kmap);
        row = mode ? tid / O : tid % R;
        oct = mode ? tid % O : __builtin_amdgcn_readfirstlane(tid / R);
        wrow = tid / 64 * RW;
        kk = mode == 1 ? tid % BK : 8 * oct;
#pragma unroll
        for (int j = 0; j < NR; j++)
        {
            const int r = mode == 1 ? wrow + 64 / BK * j + tid % 64 / BK : row;
            roff[j] = (uint32_t)pool[rows + (r < valid ? r : 0)];
        }
    }
    // k offsets of the stage at k (the tables go on past the last k)
    __device__ __forceinline__ void fetch(int k)
    {
        const uint32_t* m = km + k;
#pragma unroll
        for (int j = 0; j < NK; j++) knext[j] = m[(uint32_t)(kk + j)];
    }
    __device__ __forceinline__ void advance()
    {
#pragma unroll
        for (int j = 0; j < NK; j++) koff[j] = knext[j];
    }
    __device__ __forceinline__ void load()
    {
        if constexpr (mode == 2)
        {
            const f32x4* p = (const f32x4*)(x + (roff[0] + koff[0]));
            const f32x4 a = p[0], b = p[1];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = a[j], v[4 + j] = b[j];
        }
        else if constexpr (mode == 1)
        {
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = *(const float*)(x + (roff[j] + koff[0]));
        }
        else
        {
#pragma unroll
            for (int j = 0; j < 8; j++)
            {
                GlobalBytes b = (GlobalBytes)x + (uint32_t)__builtin_amdgcn_readfirstlane(koff[j]);
                asm("" : "+s"(b));
                v[j] = *(const __attribute__((address_space(1))) float*)(b + roff[0]);
            }
        }
    }
    // a loaded stage, split, into LDS; TAIL: zeros from its left-th k on
    template <bool TAIL>
    __device__ __forceinline__ void store(u32x4* __restrict__ lds, int left) const
    {
        float f[8];
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] = v[j];
        if constexpr (mode == 1)
        {
            // row r of the wave at the run r / RP of its rows' pieces, in
            // the (term, octet) order of the stage
            auto at = [&](int r) {
                const int c = r / RP;
                return (staged_f32*)(lds + (c / O) * TERM + (c % O) * R + wrow) + r % RP * BK;
            };
#pragma unroll
            for (int j = 0; j < 8; j++) at(64 / BK * j + (int)threadIdx.x % 64 / BK)[kk] = f[j];
            wave_exchange();  // the wave's lanes read one another's values
            const f32x4* p = (const f32x4*)(at(row - wrow) + 8 * oct);
            const f32x4 a = p[0], b = p[1];
#pragma unroll
            for (int j = 0; j < 4; j++) f[j] = a[j], f[4 + j] = b[j];
            wave_exchange();  // before the units overwrite them
        }
        u32x4 h, m, l;
#pragma unroll
        for (int j = 0; j < 4; j++)
        {
            float d = f[2 * j], e = f[2 * j + 1];
            if (TAIL) d = 8 * oct + 2 * j < left ? d : 0.0f, e = 8 * oct + 2 * j + 1 < left ? e : 0.0f;
            h[j] = round_pair(d, e);
            m[j] = round_pair(d, e);
            l[j] = round_pair(d, e);
        }
        u32x4* p = lds + oct * R + (row ^ (oct * (16 / O)));
        p[0] = h;
        p[TERM] = m;
        p[2 * TERM] = l;
    }
    // MFMA operand of the 16-k step q: rows r0 + lr, k octet 2 q + lh
    static __device__ __forceinline__ void frag(bf16x8 (&f)[3], const u32x4* lds, int q, int r0, int lr, int lh)
    {
        const int o = 2 * q + lh;
        const u32x4* p = lds + o * R + ((r0 + lr) ^ (o * (16 / O)));
#pragma unroll
        for (int t = 0; t < 3; t++) f[t] = __builtin_bit_cast(bf16x8, p[t * TERM]);
    }
};

template <int BM, int BN, int WGM, int WGN, int BK, int OCC, int AM, int BMODE>
__global__ __launch_bounds__(kNT, OCC) void gemm_gather_bf16_kernel(const PanelTask* __restrict__ tasks, int ntasks,
                                                                    const int64_t* __restrict__ pool, const float* A,
                                                                    const float* B, float* __restrict__ C,
                                                                    float* __restrict__ cws, double alpha,
                                                                    double beta, int use_k)
{
    static_assert(WGM * WGN * 64 == kNT, "four waves");
    constexpr int WM = BM / WGM, WN = BN / WGN, MB = WM / 32, NB = WN / 32;
    constexpr int SA = 3 * BM * BK / 8, ST = 3 * (BM + BN) * BK / 8;  // pieces of 16 bytes
    constexpr int CHUNK = 256 / BK;                                   // stages per accumulation chunk
    // 32 x 32 waves have the registers to sum the five small products apart
    // from hi hi, whose sum is then rounded once per 16 k and not six times:
    // they replace panel tiles that cut the sum over their waves (256 x 256 x
    // 256: error 2.4e-7 in one sum, 1.2e-7 in the panel tile's four)
    constexpr bool LOW = MB * NB == 1;
    using SideA = UnitSide<BM, BK, AM>;
    using SideB = UnitSide<BN, BK, BMODE>;
    __shared__ u32x4 ring0[ST], ring1[ST];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int lr = lane & 31, lh = lane >> 5;

    for (int ti = blockIdx.x; ti < ntasks; ti += gridDim.x)
    {
        const PanelTask t = tasks[ti];
        f32x16 acc[MB][NB], low[LOW ? MB : 1][LOW ? NB : 1], tot[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                for (int r = 0; r < 16; r++)
                {
                    acc[i][j][r] = tot[i][j][r] = 0.0f;
                    if constexpr (LOW) low[i][j][r] = 0.0f;
                }
        auto close_chunk = [&]() {
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
                {
                    if constexpr (LOW) acc[i][j] += low[i][j];
                    tot[i][j] += acc[i][j];
                    for (int r = 0; r < 16; r++)
                    {
                        acc[i][j][r] = 0.0f;
                        if constexpr (LOW) low[i][j][r] = 0.0f;
                    }
                }
        };

        const int kend = t.klen;
        const int nst = use_k && kend > t.kbeg ? (kend - t.kbeg + BK - 1) / BK : 0;
        if (nst > 0)
        {
            SideA a;
            SideB b;
            a.init(A, t.a_src, pool, t.a_rt, t.a_km, t.mlen, tid);
            b.init(B, t.b_src, pool, t.b_rt, t.b_km, t.nlen, tid);
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
            auto store = [&](u32x4* st) {
                a.template store<false>(st, 0);
                b.template store<false>(st + SA, 0);
            };
            auto store_last = [&](u32x4* st, int left) {
                a.template store<true>(st, left);
                b.template store<true>(st + SA, left);
            };
            const int left = kend - t.kbeg - (nst - 1) * BK;  // k of the last stage
            fetch();
            a.advance();
            b.advance();
            fetch();
            load();
            fetch();
            if (nst == 1)
                store_last(ring0, left);
            else
            {
                store(ring0);
                load();
            }
            __syncthreads();
            auto multiply = [&](const u32x4* cur) {
                constexpr int PA[6] = {1, 0, 2, 0, 1, 0};
                constexpr int PB[6] = {1, 2, 0, 1, 0, 0};
#pragma unroll
                for (int q = 0; q < BK / 16; q++)
                {
                    bf16x8 fb[NB][3];
#pragma unroll
                    for (int j = 0; j < NB; j++) SideB::frag(fb[j], cur + SA, q, wn * WN + 32 * j, lr, lh);
#pragma unroll
                    for (int i = 0; i < MB; i++)
                    {
                        bf16x8 fa[3];
                        SideA::frag(fa, cur, q, wm * WM + 32 * i, lr, lh);
#pragma unroll
                        for (int p = 0; p < 6; p++)
#pragma unroll
                            for (int j = 0; j < NB; j++)
                            {
                                f32x16& sum = LOW && p < 5 ? low[i][j] : acc[i][j];
                                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[PA[p]], fb[j][PB[p]], sum, 0, 0, 0);
                            }
                    }
                }
            };
            // stage s from cur while stage s + 1 is split into nxt and stage
            // s + 2 loaded
            auto stage = [&](const u32x4* cur, u32x4* nxt) {
                fetch();
                store(nxt);
                load();
                multiply(cur);
                // 64 x 64 wave tiles: split and address instructions between
                // the MFMAs (permuted 64/32 258 -> 236 us; 32 x 32 waves lose)
                if constexpr (MB * NB > 1)
#pragma unroll
                    for (int g = 0; g < 6 * MB * NB * (BK / 16); g++)
                    {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
                    }
                __syncthreads();
            };
            // two stages per pass (constant LDS addresses); the last stage and
            // the one that stores it, which may be short, come after the loop
            int s = 0;
            for (; s + 3 < nst; s += 2)
            {
                stage(ring0, ring1);
                stage(ring1, ring0);
                if ((s + 2) % CHUNK == 0) close_chunk();
            }
            if (s + 2 < nst)
            {
                stage(ring0, ring1);
                s++;
                if (s % CHUNK == 0) close_chunk();
            }
            if (s + 1 < nst)
            {
                store_last(s & 1 ? ring0 : ring1, left);
                multiply(s & 1 ? ring1 : ring0);
                __syncthreads();
                s++;
                if (s % CHUNK == 0) close_chunk();
            }
            multiply(s & 1 ? ring1 : ring0);
            close_chunk();
        }
        // D register r of lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
        int64_t coff[NB];
#pragma unroll
        for (int j = 0; j < NB; j++)
        {
            const int col = wn * WN + j * 32 + lr;
            coff[j] = t.c_ld == 0 && col < t.nlen ? pool[t.c_colmap + col] : 0;
        }
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++)
            {
                const int row = wm * WM + i * 32 + 8 * (r / 4) + 4 * lh + r % 4;
                if (row >= t.mlen) continue;
                const int64_t roff = t.c_ld == 0 ? t.c_src + pool[t.c_rowmap + row] : t.c_src + (int64_t)row * t.c_ld;
#pragma unroll
                for (int j = 0; j < NB; j++)
                {
                    const int col = wn * WN + j * 32 + lr;
                    if (col >= t.nlen) continue;
                    if (t.c_ld > 0)
                    {
                        cws[roff + col] = tot[i][j][r];  // a k slice's sums
                        continue;
                    }
                    float* p = C + roff + coff[j];
                    double v = alpha * (double)tot[i][j][r];
                    if (beta != 0.0) v += beta * (double)*p;
                    *p = (float)v;
                }
            }
        __syncthreads();  // the next task's stages reuse the LDS
    }
}

struct GatherTile
{
    int bm, bn, bk;
};

// id (after the panel tiles), BM, BN, waves WGM x WGN, k per stage, waves per SIMD
#define TBLIS_GATHER_BF16_TILES(X)   \
    X(0, 128, 128, 2, 2, 16, 2)      \
    X(1, 64, 64, 2, 2, 32, 3)

constexpr GatherTile kGTiles[] = {
#define X(id, bm, bn, wgm, wgn, bk, occ) {bm, bn, bk},
    TBLIS_GATHER_BF16_TILES(X)
#undef X
};
constexpr int kNumGTiles = sizeof(kGTiles) / sizeof(kGTiles[0]);

template <int BM, int BN, int WGM, int WGN, int BK, int OCC>
hipError_t launch_t(const PanelLaunch& L)
{
    auto go = [&](auto* k) {
        const dim3 grid(persistent_grid((const void*)k, kNT, L.ntasks));
        hipLaunchKernelGGL(k, grid, dim3(kNT), 0, L.stream, L.tasks, L.ntasks, L.pool, (const float*)L.A,
                           (const float*)L.B, (float*)L.C, (float*)L.cws, L.alpha, L.beta, L.use_k);
        return hipGetLastError();
    };
    switch (L.group)
    {
        case 0: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 0, 0>);
        case 1: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 1, 0>);
        case 2: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 2, 0>);
        case 3: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 0, 1>);
        case 4: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 1, 1>);
        case 5: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 2, 1>);
        case 6: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 0, 2>);
        case 7: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 1, 2>);
        case 8: return go(&gemm_gather_bf16_kernel<BM, BN, WGM, WGN, BK, OCC, 2, 2>);
    }
    return hipErrorInvalidValue;
}

}  // namespace

int gather_bf16_num_tiles() { return kNumGTiles; }
int gather_bf16_tile_m(int t) { return kGTiles[t].bm; }
int gather_bf16_tile_n(int t) { return kGTiles[t].bn; }
int gather_bf16_tile_k(int t) { return kGTiles[t].bk; }

hipError_t launch_gemm_gather_bf16(const PanelLaunch& L, int t)
{
    if (L.ntasks == 0) return hipSuccess;
    if (L.dtype != 1 || L.scaled) return hipErrorInvalidValue;
    switch (t)
    {
#define X(id, bm, bn, wgm, wgn, bk, occ) \
    case id: return launch_t<bm, bn, wgm, wgn, bk, occ>(L);
        TBLIS_GATHER_BF16_TILES(X)
#undef X
        default:
            return hipErrorInvalidValue;
    }
}

}  // namespace tblis_amd
