// npu_weight_quant_batchmatmul on int4 / int8 NZ and int8 [N, K] weights for 16 < M rows: batches and prompts whose
// output has too few 128 x 256 tiles to fill the chip, and prefill on an N of no whole 256-column tiles.
//
// A workgroup of 8 waves owns 16 * TM rows x 256 columns and one range of K steps (128 rows of an int4 weight, 64 of
// an int8 one).  Per step the activation rows, the column block's sixteen 1 KB weight blocks and its scale / offset
// rows come into a ring of LDS stages by direct-to-LDS loads, as many steps ahead as the ring holds; wave w multiplies
// all rows by columns 32w .. 32w+31.  The group algebra is the other kernels',
//   acc += s * sum_k x*(w + BASE) + s*(offset - BASE) * sum_k x,
// on exact operands (BASE = 0 for an int8 weight).  The group sums of x are taken in the kernel: wave i sums row tile i
// on the matrix cores (against ones) and hands it to the others through LDS, so a group (128 or 512 rows of it, if it is
// longer) is folded one step later, row tile by row tile between the next step's first MFMAs.  K is split over
// workgroups where the tiles alone leave CUs idle: each split stores its fp32 sums in the MFMA layout (whole KB per
// store) and nz_mid_reduce adds them in split order.
//
// What bounds it: per step and CU the LDS reads (8 waves x the activation stage: 160 KB at 80 rows), the MFMAs and
// the fold take about the same time; on few rows the weight stream.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace qk {
namespace {

namespace nm {
constexpr int BN = 256, NT = 512, TN = 2;
constexpr int W_BYTES = 16 * 1024;  // a step's 16 weight blocks
constexpr int SC_BYTES = 2 * 1024;  // two groups' scale rows, two groups' offset rows (512 bytes each)
constexpr int OROWB = 2 * BN + 16;  // padded output staging row (bytes)
constexpr int ksw(bool w8) { return w8 ? 64 : 128; }  // K rows per step
constexpr int x_bytes(int tm, bool w8) { return 16 * tm * ksw(w8) * 2; }
constexpr int stage(int tm, bool w8) { return x_bytes(tm, w8) + W_BYTES + SC_BYTES; }
constexpr int xs_bytes(int tm) { return 2 * 16 * tm * 4; }
constexpr int stages(int tm, bool w8) { return std::min(6, (160 * 1024 - xs_bytes(tm)) / stage(tm, w8)); }
}  // namespace nm

// a lane offset past any buffer here (each is below 2^31 bytes): the load returns zeros and reads no memory
constexpr uint32_t kMidOutside = 0x80000000u;

template <uint32_t MAGIC>
__device__ __forceinline__ u32x4 mid_op4(uint32_t w) {  // the eight nibbles of an NZ word as magic 16-bit values
    const uint32_t mask = __builtin_amdgcn_readfirstlane(0x000f000fu);
    const uint32_t magic = __builtin_amdgcn_readfirstlane(MAGIC | 0x00080008u);
    return (u32x4){(w & mask) ^ magic, ((w >> 4) & mask) ^ magic, ((w >> 8) & mask) ^ magic, ((w >> 12) & mask) ^ magic};
}

template <int N, int MOST>
__device__ __forceinline__ void mid_wait(int later) {  // at most `later` steps' loads (N each, 0 <= later <= MOST <= 4) left
    if (later == MOST) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(MOST * N));
        return;
    }
    switch (later) {
    case 0: __builtin_amdgcn_s_waitcnt(vmcnt_imm(0)); break;
    case 1: __builtin_amdgcn_s_waitcnt(vmcnt_imm(N)); break;
    case 2: __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * N)); break;
    default: __builtin_amdgcn_s_waitcnt(vmcnt_imm(3 * N)); break;
    }
}

// HALF: an int4 step holds two 64-row groups; each is folded within its step, every wave summing x itself (row tiles
// of at most 64 rows: more would spill, and a spill's memory operations would break the hand-counted waits).
// Otherwise a group is one step or several (or all of K).

// wblk / wstep: bytes from one 16-column weight block to the next and from one step to the next; nk: the weight is
// int8 [N, K] rows (the 16 bytes a lane takes from an NZ block are contiguous in row 16*block + lane%16).
template <int DT, int TM, bool W8, bool HALF>
__global__ __launch_bounds__(nm::NT) void nz_mid(WqbmmArgs p, int tiles_m, int tiles_n, int nsplit, uint32_t wblk,
                                                 uint32_t wstep, int nk, float* __restrict__ part) {
    using namespace nm;
    typedef Mfma<DT> MM;
    constexpr int KSW = ksw(W8), NKT = KSW / 32, BM = 16 * TM;
    constexpr int XB = x_bytes(TM, W8), STG = stage(TM, W8), NSTG = stages(TM, W8);
    constexpr int XN = XB / 1024, XPW = (XN + 7) / 8;  // activation DMAs per step, and per wave
    constexpr float BASE = W8 ? 0.0f : MM::BASE;
    static_assert(NSTG >= 3 && NSTG * STG + xs_bytes(TM) <= 160 * 1024 && BM * OROWB <= NSTG * STG, "LDS");
    static_assert(TM <= 6, "one wave sums each row tile; taller tiles would spill, and a spill's memory operations "
                           "would break the hand-counted waits");
    __shared__ __attribute__((aligned(1024))) char smem[NSTG * STG + xs_bytes(TM)];
    float* const xsbuf = reinterpret_cast<float*>(smem + NSTG * STG);  // [step parity][row]

    const int M = (int)p.M, N = (int)p.N, K = (int)p.K, G = (int)p.group;
    const int ntiles = tiles_m * tiles_n;
    const int id = xcd_swizzle(blockIdx.x, gridDim.x);  // a split's row tiles of one column block side by side
    const int split = id / ntiles, tile = id % ntiles;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const int m0 = tm * BM, n0 = tn * BN;
    const int rows = M - m0 < BM ? M - m0 : BM;
    const int S = K / KSW;
    const int s0 = (int)((int64_t)split * S / nsplit), s1 = (int)((int64_t)(split + 1) * S / nsplit);

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, g4 = lane >> 4;
    const uint32_t sbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const uint32_t ldx = (uint32_t)K * 2u;
    // rows past M (their row offset is in the lane offset) read zeros
    const __amdgpu_buffer_rsrc_t rx =
        make_rsrc(static_cast<const char*>(p.x) + (size_t)m0 * ldx, (uint32_t)rows * ldx);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, (uint32_t)K * (uint32_t)N / (W8 ? 1u : 2u));
    const uint32_t nsb = (uint32_t)(K / G) * (uint32_t)N * 2u, ng = (uint32_t)(K / G);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.scale, nsb);
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.offset ? p.offset : p.scale, nsb);
    const bool has_off = p.offset != nullptr;

    // activations: int4 rows of 256 bytes, DMA q covers rows 4q..4q+3 (chunk c of row r at LDS chunk c ^ (r & 15));
    // int8 rows of 128 bytes, rows 8q..8q+7 (chunk c ^ (r & 7)).  A wave with no row of its own left repeats the last.
    uint32_t vx[XPW], xl[XPW];
#pragma unroll
    for (int u = 0; u < XPW; ++u) {
        const int q = wave + 8 * u < XN ? wave + 8 * u : XN - 1;
        const int row = W8 ? 8 * q + (lane >> 3) : 4 * q + (lane >> 4);
        vx[u] = (uint32_t)row * ldx + 16u * (uint32_t)(W8 ? (lane & 7) ^ (row & 7) : (lane & 15) ^ (row & 15));
        xl[u] = 1024u * (uint32_t)q;
    }
    // weight blocks wave and wave + 8 of the column block; blocks past N are outside the buffer
    uint32_t vw[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int b = tn * 16 + wave + 8 * u;
        const uint32_t l = nk ? (uint32_t)fr * (uint32_t)K + 16u * (uint32_t)g4 : 16u * (uint32_t)lane;
        vw[u] = b < N / 16 ? (uint32_t)b * wblk + l : kMidOutside;
    }
    // scale / offset rows of a step's first group (lanes 0..31) and the next one (32..63): 16 bytes of 8 columns each
    const int scol = n0 + 8 * (lane & 31);

    // Steps run in order, so the group and the ring slot of the next step to issue, and to multiply, are counted along.
    const int gsteps = HALF ? 1 : G / KSW;
    int ig = HALF ? 2 * s0 : s0 / gsteps, ileft = gsteps - s0 % gsteps, islot = 0;
    auto issue = [&](int s) {
        const uint32_t base = sbase + (uint32_t)islot * STG;
#pragma unroll
        for (int u = 0; u < XPW; ++u) dma16(rx, base + xl[u], vx[u], (uint32_t)s * (uint32_t)(KSW * 2));
#pragma unroll
        for (int u = 0; u < 2; ++u) dma16(rw, base + XB + 1024u * (uint32_t)(wave + 8 * u), vw[u], (uint32_t)s * wstep);
        if (wave < 2) {  // the scale rows, the offset rows (the scales again when there are none: not used)
            uint32_t g = (uint32_t)ig + (uint32_t)(lane >> 5);
            g = g < ng ? g : ng - 1;
            const uint32_t v = scol < N ? (g * (uint32_t)N + (uint32_t)scol) * 2u : kMidOutside;
            dma16(wave == 0 ? rs : ro, base + XB + W_BYTES + 1024u * (uint32_t)wave, v, 0);
        }
        if (--ileft == 0) {
            ileft = gsteps;
            ig += HALF ? 2 : 1;
        }
        islot = islot + 1 < NSTG ? islot + 1 : 0;
    };

    f32x4 acc[TM][TN], ag[TM][TN];
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = ag[i][j] = zero4;
    float sf[TN], sx[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) sf[j] = sx[j] = 0.0f;
    const int xt = wave % TM;  // the row tile whose sum of x this wave takes: no branch around the MFMAs
    f32x4 xsum = zero4;        // since the last fold
    for (int e = tid; e < 2 * BM; e += NT) xsbuf[e] = 0.0f;  // what the first fold (of nothing) reads
    const u32x4 ones = {MM::ONES, MM::ONES, MM::ONES, MM::ONES};
    // lane parts of the LDS addresses: a_at[kt] of an activation fragment (row tile i adds i * 16 rows)
    int a_at[NKT];
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
        a_at[kt] = W8 ? fr * 128 + 16 * ((2 * g4 + kt) ^ (fr & 7)) : fr * 256 + 16 * ((4 * kt + g4) ^ fr);
    constexpr int ROWT = W8 ? 2048 : 4096;  // LDS bytes of 16 rows

    // Raw sums are folded at a group's end and inside a longer group: an int4 one every 128 rows, since at BASE times the
    // size of the products they would lose what the base's share takes off again (one fp16 group of 5120 rows, positive
    // x, M = 200, N = 13696: 9.8e-4 off the 64-bit result, folded 2.1e-4, which is the output's rounding).  int8 operands
    // carry no base: every 512 rows keeps the rounding of the long chain low (8192 rows of one group, M = 100, N = 28672:
    // the 32-bit sums are 1.7e-7 off, at one fold 5.8e-7) for 2-3 % of the time (M = 400, K = 11008, N = 4096: 67.6 us,
    // one fold 65.2, every 128 rows 72.4).
    constexpr int FSTEPS = (W8 ? 512 : 128) / KSW;
    int gleft = gsteps - s0 % gsteps, fleft = 0;  // steps left of the group being multiplied, and to its next fold
    int cslot = 0;
    for (int s = s0; s < s0 + NSTG - 1 && s < s1; ++s) issue(s);
    for (int s = s0; s < s1; ++s) {
        // stage s has landed once at most the later steps' loads are outstanding
        const int later = s1 - 1 - s < NSTG - 2 ? s1 - 1 - s : NSTG - 2;
        if (wave < 2) mid_wait<XPW + 3, NSTG - 2>(later);
        else mid_wait<XPW + 2, NSTG - 2>(later);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();  // stage s visible to every wave; every wave is done with stage s-1
        __builtin_amdgcn_sched_barrier(0);
        const char* As = smem + cslot * STG;
        const char* Bs = As + XB;
        const char* sc = As + XB + W_BYTES;
        cslot = cslot + 1 < NSTG ? cslot + 1 : 0;
        const bool first = FSTEPS == 1 || fleft == 0;  // new sums start with this step
        if (FSTEPS > 1) {
            if (first) fleft = gleft < FSTEPS ? gleft : FSTEPS;
            --fleft;
            if (--gleft == 0) gleft = gsteps;
        }
        // LDS reads go out ahead of their use: the weight, the factors' raw values, the row tile whose x this wave sums,
        // then each row tile's fragments one tile before its MFMAs.  Row tiles run one after the other over the whole
        // step, so a tile's fold of the previous group (VALU) runs under the MFMAs of the tile before it.
        u32x4 bw[TN], af[2][NKT];
        f32x4 xs[2];
#pragma unroll
        for (int j = 0; j < TN; ++j) bw[j] = *reinterpret_cast<const u32x4*>(Bs + (TN * wave + j) * 1024 + 16 * lane);
        const float* xsp = xsbuf + ((s - 1) & 1) * BM + 4 * g4;  // the previous step's sums of x
        auto load_tile = [&](int i) {
            if (!HALF) xs[i & 1] = *reinterpret_cast<const f32x4*>(xsp + 16 * i);
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) af[i & 1][kt] = *reinterpret_cast<const u32x4*>(As + a_at[kt] + i * ROWT);
        };
        load_tile(0);
        constexpr int NU = HALF ? 2 : 1;
        uint16_t rf[NU][TN], rof[NU][TN];  // raw scale and offset of the step's groups
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int at = 512 * u + 2 * (16 * TN * wave + 16 * j + fr);
                rf[u][j] = *reinterpret_cast<const uint16_t*>(sc + at);
                rof[u][j] = *reinterpret_cast<const uint16_t*>(sc + 1024 + at);
            }
        __builtin_amdgcn_sched_barrier(0);
        if (s + NSTG - 1 < s1) issue(s + NSTG - 1);  // into the buffer of stage s-1
        u32x4 b[NKT][TN];
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (W8) b[kt][j] = i8_operand<DT>(bw[j][2 * kt], bw[j][2 * kt + 1]);
                else b[kt][j] = mid_op4<MM::MAGIC>(bw[j][kt]);
            }
        auto factors = [&](int u, float (&f)[TN], float (&x)[TN]) {  // s and s * (offset - BASE) of the step's group u
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f[j] = load_half_bits(rf[u][j], p.s_dtype);
                x[j] = f[j] * ((has_off ? load_half_bits(rof[u][j], p.s_dtype) : 0.0f) - BASE);
            }
        };
        // acc += s * sums + s * (offset - BASE) * sum of x, pinned where it stands
        auto fold = [&](int i, const f32x4 (&a)[TN], const f32x4& x, const float (&f)[TN], const float (&fx)[TN]) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    acc[i][j][q] = __builtin_fmaf(f[j], a[j][q], __builtin_fmaf(fx[j], x[q], acc[i][j][q]));
                    asm volatile("" : "+v"(acc[i][j][q]));
                }
        };
        if constexpr (HALF) {
            float f[2][TN], fx[2][TN];
            factors(0, f[0], fx[0]);
            factors(1, f[1], fx[1]);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                if (i + 1 < TM) load_tile(i + 1);
                __builtin_amdgcn_sched_barrier(0);
                f32x4 a[2][TN], x[2];
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    const int u = kt >> 1;
                    x[u] = MM::mma(af[i & 1][kt], ones, (kt & 1) ? x[u] : zero4);
#pragma unroll
                    for (int j = 0; j < TN; ++j) a[u][j] = MM::mma(af[i & 1][kt], b[kt][j], (kt & 1) ? a[u][j] : zero4);
                }
                fold(i, a[0], x[0], f[0], fx[0]);
                fold(i, a[1], x[1], f[1], fx[1]);
            }
        } else {
            auto tiles = [&](auto fresh) {  // fresh: new sums start, so those before them are folded
                constexpr bool F = decltype(fresh)::value;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (i + 1 < TM) load_tile(i + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    if (F) {
                        fold(i, ag[i], xs[i & 1], sf, sx);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            ag[i][j] = MM::mma(af[i & 1][kt], b[kt][j], F && kt == 0 ? zero4 : ag[i][j]);
                }
            };
            if (first) {
                tiles(std::true_type());
                factors(0, sf, sx);
                xsum = zero4;
            } else if constexpr (FSTEPS > 1) {
                tiles(std::false_type());
            }
            // this step's sum of x of row tile xt, for the next step's fold (waves past TM write the same again)
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
                xsum = MM::mma(*reinterpret_cast<const u32x4*>(As + a_at[kt] + xt * ROWT), ones, xsum);
            if (fr == 0) *reinterpret_cast<f32x4*>(xsbuf + (s & 1) * BM + 16 * xt + 4 * g4) = xsum;
        }
    }
    __syncthreads();  // the last step's sums of x are visible; every wave is past its last reads of the ring
    if constexpr (!HALF) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const f32x4 xs = *reinterpret_cast<const f32x4*>(xsbuf + ((s1 - 1) & 1) * BM + 16 * (i) + 4 * g4);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[i][j][q] = __builtin_fmaf(sf[j], ag[i][j][q], __builtin_fmaf(sx[j], xs[q], acc[i][j][q]));
        }
    }

    if (nsplit > 1) {  // this range's sums in the MFMA layout, read once by nz_mid_reduce
        f32x4* dst = reinterpret_cast<f32x4*>(part) + (((int64_t)split * ntiles + tile) * 8 + wave) * (TM * TN * 64) + lane;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) __builtin_nontemporal_store(acc[i][j], dst + (i * TN + j) * 64);
        return;
    }
    // + bias, cast, staged through LDS for 16-byte row stores
    float bv[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + 16 * (TN * wave + j) + fr;
        bv[j] = p.bias_dtype && n < N ? load_scalar(p.bias, n, p.bias_dtype) : 0.0f;
    }
    uint16_t* ot = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float v = acc[i][j][q] + bv[j];
                ot[(16 * (i) + 4 * g4 + q) * (OROWB / 2) + 16 * (TN * wave + j) + fr] =
                    (uint16_t)(p.out_dtype == QK_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v));
            }
    __syncthreads();
    constexpr int CPRO = 2 * BN / 16;  // 16-byte chunks per output row
    for (int q = tid; q < BM * CPRO; q += NT) {
        const int row = q / CPRO, c = q % CPRO;
        if (row >= rows) break;
        if (n0 + 8 * c >= N) continue;  // the last column tile of a ragged N
        const u32x4 v = *reinterpret_cast<const u32x4*>(smem + row * OROWB + 16 * c);
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.out) +
                                                                (size_t)(m0 + row) * N + n0 + 8 * c));  // written once
    }
}

// The splits of nz_mid: one thread per 16-byte piece (rows 4g..4g+3 of one column of one 16 x 16 fragment) adds the
// splits' pieces in split order, adds the bias and casts.  All of a thread's loads go out before the first add.
__global__ __launch_bounds__(256) void nz_mid_reduce(WqbmmArgs p, int tm_frags, int tiles_m, int tiles_n,
                                                     int nsplit, const f32x4* __restrict__ part) {
    const int pieces = 16 * tm_frags * 64;
    const int64_t per_split = (int64_t)tiles_m * tiles_n * pieces;
    const int N = (int)p.N, M = (int)p.M;
    for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < per_split; idx += (int64_t)gridDim.x * 256) {
        const int lane = (int)(idx & 63), tile = (int)(idx / pieces), rest = (int)(idx % pieces) >> 6;
        const int f = rest % (tm_frags * nm::TN), wave = rest / (tm_frags * nm::TN);
        const int m = (tile % tiles_m) * 16 * tm_frags + 16 * (f / nm::TN) + 4 * (lane >> 4);
        const int n = (tile / tiles_m) * nm::BN + 16 * (nm::TN * wave + f % nm::TN) + (lane & 15);
        if (n >= N || m >= M) continue;
        f32x4 v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (k < nsplit) v[k] = __builtin_nontemporal_load(part + (int64_t)k * per_split + idx);
        const float b = p.bias_dtype ? load_scalar(p.bias, n, p.bias_dtype) : 0.0f;
        f32x4 sum = v[0];
#pragma unroll
        for (int k = 1; k < 16; ++k)
            if (k < nsplit) sum += v[k];
        uint16_t* dst = static_cast<uint16_t*>(p.out) + (size_t)m * N + n;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float o = sum[r] + b;
            const uint32_t h = p.out_dtype == QK_BF16 ? f32_to_bf16_bits(o) : f32_to_f16_bits(o);
            if (m + r < M) dst[(size_t)r * N] = (uint16_t)h;
        }
    }
}

}  // namespace

NzMidPlan nz_mid_plan(const WqbmmArgs& p) {
    NzMidPlan z;
    const int64_t G = p.group == 0 ? p.K : p.group;
    const bool w8 = p.w_dtype == QK_I8_NZ || p.w_dtype == QK_I8_NK;
    const int ks = nm::ksw(w8);
    const PlanOverride& ov = plan_override();
    if (!(w8 || p.w_dtype == QK_I4_NZ) || ov.nz_mid == 0 || ov.w4nz_off || p.M <= 0 || p.N <= 0 || p.K <= 0) return z;
    if (p.N % 16 != 0 || p.K % ks != 0 || G <= 0 || p.K % G != 0) return z;
    z.half = !w8 && G == 64;
    if (!z.half && G % ks != 0) return z;
    if (p.M * p.K * 2 >= ((int64_t)1 << 31) || p.K * p.N >= ((int64_t)1 << 31) || (p.K / G) * p.N * 2 >= ((int64_t)1 << 31) ||
        p.M * p.N >= ((int64_t)1 << 31))
        return z;
    if (((uintptr_t)p.x | (uintptr_t)p.w | (uintptr_t)p.scale | (uintptr_t)p.out |
         (uintptr_t)(p.offset ? p.offset : p.scale)) % 16 != 0)
        return z;
    const int S = (int)(p.K / ks);
    z.tiles_n = (int)((p.N + 255) / 256);
    if ((p.M + 31) / 32 * z.tiles_n >= ((int64_t)1 << 20)) return z;
    // Row tiles of at most 96 rows (64 with half-step groups), all of one height, and the K split: the pair with the
    // lowest estimate in us, from steps timed at N = 11008, K = 4096 without a split (int4, 128 rows of K: 0.96 / 1.26
    // / 1.58 with 2 / 4 / 6 row tiles of 16; int8, 64 rows: 0.82 / 0.96): rounds of workgroups x steps, about 5 of
    // launch, first loads and epilogue, and for a split another launch and the partials written and read.
    const int most = z.half ? 4 : 6;
    const int t16 = (int)((p.M + 15) / 16), tm_lo = (t16 + most - 1) / most;
    for (int tm = tm_lo; tm <= tm_lo + 2 && tm <= t16; ++tm) {
        const int h = std::max(2, (t16 + tm - 1) / tm);
        const double step = w8 ? 0.72 + 0.045 * h : 0.65 + 0.155 * h;
        const int tiles = tm * z.tiles_n;  // below 2^22
        for (int ns = 1; ns <= 16 && ns <= S; ++ns) {
            if (ov.nz_mid > 0 && ov.nz_mid < 17 && ns != ov.nz_mid) continue;
            const double part = (double)ns * (double)tiles * h * 16 * 256 * 4;
            if (ns > 1 && part > 512e6) break;
            const double t = (double)((tiles * ns + 255) / 256) * (double)((S + ns - 1) / ns) * step + 5.0 +
                             (ns > 1 ? 1.0 + 2 * part / 5e6 : 0.0);
            if (z.ok && t >= z.us) continue;
            z.us = t;
            z.tm = h;
            z.tiles_m = tm;
            z.nsplit = ns;
            z.ok = true;
        }
    }
    // [N, K] rows come in slower than NZ blocks (N = 8192 K = 8192, M = 20 / 64 24.2 / 29.1 us against 22.8 / 27.4)
    if (p.w_dtype == QK_I8_NK) z.us *= 1.12;
    return z;
}

namespace {

template <int DT, int TM, bool W8>
void launch_mode(const WqbmmArgs& p, const NzMidPlan& z, float* part, hipStream_t stream) {
    const bool nk = p.w_dtype == QK_I8_NK;
    const uint32_t wblk = nk ? 16u * (uint32_t)p.K : (uint32_t)(p.K / nm::ksw(W8)) * 1024u, wstep = nk ? 64u : 1024u;
    const dim3 grid((uint32_t)(z.tiles_m * z.tiles_n * z.nsplit)), block(nm::NT);
    if constexpr (!W8 && TM <= 4)
        if (z.half) {
            nz_mid<DT, TM, W8, true><<<grid, block, 0, stream>>>(p, z.tiles_m, z.tiles_n, z.nsplit, wblk, wstep, 0, part);
            return;
        }
    nz_mid<DT, TM, W8, false><<<grid, block, 0, stream>>>(p, z.tiles_m, z.tiles_n, z.nsplit, wblk, wstep, (int)nk, part);
}

template <int DT, bool W8>
void launch_tm(const WqbmmArgs& p, const NzMidPlan& z, float* part, hipStream_t stream) {
    switch (z.tm) {
    case 2: launch_mode<DT, 2, W8>(p, z, part, stream); break;
    case 3: launch_mode<DT, 3, W8>(p, z, part, stream); break;
    case 4: launch_mode<DT, 4, W8>(p, z, part, stream); break;
    case 5: launch_mode<DT, 5, W8>(p, z, part, stream); break;
    default: launch_mode<DT, 6, W8>(p, z, part, stream); break;
    }
}

}  // namespace

// [split counters, unused][partials fp32 [split][tile][rows x 256]]
size_t nz_mid_workspace(const NzMidPlan& z) {
    if (!z.ok || z.nsplit == 1) return 0;
    return QK_SPLIT_COUNTER_BYTES + (size_t)z.nsplit * z.tiles_m * z.tiles_n * z.tm * 16 * 256 * sizeof(float);
}

hipError_t launch_nz_mid(const WqbmmArgs& p, const NzMidPlan& z, void* workspace, size_t ws_bytes, hipStream_t stream) {
    if (!z.ok) return hipErrorInvalidValue;
    float* part = nullptr;
    if (z.nsplit > 1) {
        if (!workspace || ws_bytes < nz_mid_workspace(z) || (uintptr_t)workspace % 16 != 0) return hipErrorInvalidValue;
        part = reinterpret_cast<float*>(static_cast<char*>(workspace) + QK_SPLIT_COUNTER_BYTES);
    }
    const bool w8 = p.w_dtype != QK_I4_NZ;
    if (p.x_dtype == QK_BF16) {
        if (w8) launch_tm<QK_BF16, true>(p, z, part, stream);
        else launch_tm<QK_BF16, false>(p, z, part, stream);
    } else {
        if (w8) launch_tm<QK_F16, true>(p, z, part, stream);
        else launch_tm<QK_F16, false>(p, z, part, stream);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || z.nsplit == 1) return e;
    const int64_t pieces = (int64_t)z.tiles_m * z.tiles_n * 16 * z.tm * 64;
    const int64_t blocks = std::min<int64_t>((pieces + 255) / 256, 65536);
    nz_mid_reduce<<<dim3((uint32_t)blocks), dim3(256), 0, stream>>>(p, z.tm, z.tiles_m, z.tiles_n, z.nsplit,
                                                                   reinterpret_cast<const f32x4*>(part));
    return hipGetLastError();
}

}  // namespace qk
