// iq_gemmw.hip -- the prefill GEMM on wide tiles, for whole 128-column groups
// and matrices and T large enough to fill the card with them (launch_gemm in
// iq_gemm.hip compares the two estimates).
//
// y[t,n] = sum_k x[t,k] * dequant(W,n,k) (+ bias[n]) on 8 waves (2 along the
// rows, 4 along the columns) of v_mfma_f32_16x16x32: 256 x 256 tiles for
// bf16 activations (a wave 128 x 64), 128 x 256 for bf16 at short T and for
// fp32 activations prepared as fp16 hi + lo (a wave 64 x 64, two products
// per weight operand).  One workgroup per CU (its LDS).
//
// What bounds the narrower tiles of iq_gemm.hip is LDS: 64 x 64 of a wave
// fed by both operands from LDS in 16 bits takes a read of LDS's full rate,
// besides the converted weights' way into it.  Here
//  - the weights of a group lie in LDS as the packed codes; a wave converts
//    its 64 columns once per group into registers (64 of them), where they
//    serve all of its rows, so LDS carries the activations and half or a
//    quarter of the weights' bytes, and the conversion (1.5 VALU ops per
//    int8 code to bf16) is shared by 128 rows;
//  - a whole group (K = 128) of activations is in LDS, so the group's
//    products of 16 rows x 64 columns finish in 16 registers and are scaled
//    from there (acc += s * P), instead of holding a second accumulator set
//    over two steps;
//  - both arrive by buffer loads straight into LDS, one instruction a step
//    while the previous group is multiplied (in a burst at the group's start
//    they held up every wave's products: 1024 x 16384 x 4096 bf16 x int8
//    170 -> 144 us), in an order of chunks that spreads a read's
//    lanes over the banks (conflicts 3-7 % of the busy cycles).
// The next group's codes are converted behind the last 16-row block of a
// group, each operand where it has been used for the last time, so one set
// of registers and one LDS buffer of codes suffice: 250 of 256 registers and
// 160 KiB of LDS at 256 x 256 x int8.
//
// Measured (one MI355X, T = 1024, eight calls in a graph on one set of
// weights, the narrow tiles -> these): bf16 activations, 7B gate 18944 x 3584
// int8 / int4 190 / 203 -> 156 / 168 us (892 / 828 TFLOP/s), down 3584 x
// 18944 241 / 260 -> 157 / 175; fp32 activations with their preparation,
// gate 362 / 344 -> 281 / 282 us, down 350 / 355 -> 299 / 305.  1024 x 16384
// x 4096, which fills one round of tiles: 958 TFLOP/s of bf16 products, 1030
// of fp16 ones; a dense bf16 library product of that size reaches about
// 1000, and zero activations run 13 % faster than random ones, so power is
// part of what bounds it.
#include <algorithm>

#include "iq_gemm.h"
#include "iq_internal.h"
#include "iq_limbs.h"
#include "iq_plan.h"

namespace iq {

namespace {

constexpr int kWThreads = 512;

typedef int rsrc4_t __attribute__((ext_vector_type(4)));

// A buffer resource in scalar registers, for the asm below (base and size
// are the same in every lane).
__device__ __forceinline__ rsrc4_t rsrc4(const void* base, int64_t bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    rsrc4_t r;
    r[0] = int(__builtin_amdgcn_readfirstlane(uint32_t(b)));
    r[1] = int(__builtin_amdgcn_readfirstlane(uint32_t(b >> 32)));
    r[2] = __builtin_amdgcn_readfirstlane(int(bytes));
    r[3] = 0x00020000;
    return r;
}

// One wave's copy of 64 x 16 bytes from memory straight into LDS at
// lds .. lds + 1023 (lane i's 16 bytes at lds + 16 i; lanes past the
// resource's end bring zeros).  The whole offset is the lane's: rows past the
// operand's last begin inside a tile, and a scalar offset is documented to be
// outside the resource's range check.  In asm, because the compiler waits for
// every such load before any read of LDS; wait_vm_barrier is what orders
// them here.  No register is written, so nothing is in flight that the
// compiler could reuse.
__device__ __forceinline__ void dma16(rsrc4_t r, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 :: "v"(voff), "s"(r), "s"(lds) : "memory", "m0");
}

// Waits until at most the wave's N latest memory operations are in flight
// (and its LDS reads are done), then for the other waves.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm_only_barrier() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(N) : "memory");
}

__device__ __forceinline__ float4_t mfma16b(bf16x8_t a, bf16x8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// KIND 0 int8 / 1 int4; LO: fp16 hi + lo operands, else bf16; MB: 16-row
// blocks of a wave (tile 32 MB x 256).
template <int KIND, bool LO, int MB>
__global__ __launch_bounds__(kWThreads, 2) void gemmw_kernel(const GemmwParams p) {
    constexpr int BM = 32 * MB, BN = 256;
    constexpr int PARTS = LO ? 2 : 1;
    constexpr uint32_t APART = BM * 256;         // bytes of one operand part of a stage
    constexpr uint32_t ASTAGE = APART * PARTS;
    constexpr int NA = BM / 4 / 8;               // DMA instructions per wave, stage and part
    constexpr uint32_t WROW = KIND == 1 ? 64 : 128;  // weight bytes of a row and group
    constexpr int NW = KIND == 1 ? 2 : 4;        // DMA instructions per wave and group
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t lds0 = uint32_t(uintptr_t((__attribute__((address_space(3))) uint8_t*)lds));
    constexpr uint32_t WBASE = 2 * ASTAGE;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int l15 = lane & 15, kq = lane >> 4;

    // Workgroups [0, full): whole tiles; then the K ranges of the others.
    const int ntiles = p.tiles_m * p.tiles_n, tail = ntiles - p.full;
    const bool whole = int(blockIdx.x) < p.full;
    const int split = whole ? 0 : (int(blockIdx.x) - p.full) / tail;
    const int tt = whole ? 0 : int(blockIdx.x) - p.full - split * tail;
    // Workgroup b runs on XCD b % 8: each XCD takes a contiguous run of the
    // whole tiles, and of a range's.
    const int n = whole ? p.full : tail, b = whole ? int(blockIdx.x) : tt;
    const int xcd = b % 8, base = n / 8, extra = n % 8;
    const int ti = xcd * base + (xcd < extra ? xcd : extra) + b / 8;
    const int t = whole ? ti : p.full + ti;
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
    const int64_t row_bytes = KIND == 1 ? p.K / 2 : p.K;
    const int gbeg = split * p.gch, gend = whole ? int(p.G) : std::min(int(p.G), gbeg + p.gch);
    const bool direct = whole || p.splits == 1;

    const int64_t xrows = std::min<int64_t>(p.T - m0, BM), nrows = std::min<int64_t>(p.N - n0, BN);
    const rsrc4_t ra = rsrc4(p.a + m0 * p.K, xrows * p.K * 2);
    const rsrc4_t ral = rsrc4(LO ? p.al + m0 * p.K : p.a, LO ? xrows * p.K * 2 : 0);
    const rsrc4_t rw = rsrc4(p.q + n0 * row_bytes, nrows * row_bytes);
    const rsrc_t rsc = make_rsrc(p.scales + n0 * p.G, nrows * p.G * 2);
    const rsrc_t rzp = make_rsrc(KIND == 1 ? p.zeros + n0 * p.G : nullptr, KIND == 1 ? nrows * p.G : 0);

    // Copy sources.  Activation instruction j covers rows 4j .. 4j + 3, 16
    // chunks of 16 bytes each; row r's chunk c lies at chunk c ^ (r & 15).
    // Weight instruction j covers 8 (int8) or 16 (int4) rows; row n's chunk
    // c at c ^ ((n >> 1) & 7) (int8) or c ^ ((n >> 2) & 3) (int4).  With
    // these orders no read below meets a bank twice.
    const uint32_t avoff = uint32_t((lane >> 4) * p.K * 2) + uint32_t(((lane & 15) ^ (lane >> 4)) << 4);
    const uint32_t wvoff = KIND == 1 ? uint32_t((lane >> 2) * row_bytes) + uint32_t(((lane & 3) ^ (lane >> 4)) << 4)
                                     : uint32_t((lane >> 3) * row_bytes) + uint32_t(((lane & 7) ^ (lane >> 4)) << 4);
    auto dma_w = [&](int g, int i) {
        const int j = wave * NW + i;
        dma16(rw, (KIND == 1 ? wvoff : wvoff ^ uint32_t((i & 1) << 6)) +
                      uint32_t(j * (1024 / WROW) * row_bytes + int64_t(g) * WROW), lds0 + WBASE + uint32_t(j) * 1024);
    };
    auto dma_a = [&](int g, uint32_t stage, int i) {
        const int part = i / NA, j = wave * NA + i % NA;
        dma16(part ? ral : ra, (avoff ^ uint32_t((i & 3) << 6)) + uint32_t(int64_t(j) * 8 * p.K + int64_t(g) * 256),
              lds0 + stage + part * APART + uint32_t(j) * 1024);
    };
    constexpr int NAT = NA * PARTS;

    // LDS read addresses
    const uint32_t aaddr = uint32_t(wm * 16 * MB + l15) * 256 + uint32_t((kq ^ l15) << 4);
    const uint32_t waddr =
        KIND == 1 ? WBASE + uint32_t(wn * 64 + l15) * 64 + uint32_t((l15 >> 2) << 4) + 4 * kq
                  : WBASE + uint32_t(wn * 64 + l15) * 128 + uint32_t(((kq >> 1) ^ (l15 >> 1)) << 4) + 8 * (kq & 1);

    int64_t ncol[4];
    bool nval[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
        const int c = wn * 64 + nb * 16 + l15;
        ncol[nb] = n0 + c;
        nval[nb] = ncol[nb] < p.N;
    }
    const uint32_t soff = uint32_t((wn * 64 + l15) * p.G);
    auto load_scales = [&](int g, uint16_t (&s)[4]) {
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
            s[nb] = __builtin_amdgcn_raw_buffer_load_b16(rsc, (soff + uint32_t(nb * 16 * p.G + g)) * 2, 0, 0);
    };
    auto load_zeros = [&](int g, uint32_t (&z)[4]) {
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
            z[nb] = KIND == 1 ? __builtin_amdgcn_raw_buffer_load_b8(rzp, soff + uint32_t(nb * 16 * p.G + g), 0, 0) : 0u;
    };

    // Converted weights of the current group: [16-column block][32-column k step]
    u32x4_t wc[4][4];
    // a lane's raw codes of one k step (8 codes: 8 bytes, or one dword of
    // nibbles) of 16-column block nb
    struct Raw {
        uint32_t d[KIND == 1 ? 1 : 2];
    };
    auto raw_at = [&](int nb, int s) {
        Raw r;
        if (KIND == 1) {
            r.d[0] = *reinterpret_cast<const uint32_t*>(lds + (waddr ^ uint32_t(s << 4)) + nb * 16 * WROW);
        } else {
            const uint2 v = *reinterpret_cast<const uint2*>(lds + (waddr ^ uint32_t(s << 5)) + nb * 16 * WROW);
            r.d[0] = v.x;
            r.d[KIND == 1 ? 0 : 1] = v.y;
        }
        return r;
    };
    auto convert = [&](const Raw& w, uint32_t z) {
        uint32_t o0, o1, o2, o3;
        if (KIND == 0) {
            const uint32_t d0 = w.d[0], d1 = w.d[KIND == 1 ? 0 : 1];
            if (LO) {
                dq_int8_x4(d0, o0, o1);
                dq_int8_x4(d1, o2, o3);
            } else {
                bf16_int8_x4(d0, o0, o1);
                bf16_int8_x4(d1, o2, o3);
            }
        } else {
            if (LO) dq_int4_x8(w.d[0], zpair_1024(z), zpair_64(z), o0, o1, o2, o3);
            else bf16_int4_x8(w.d[0], z, o0, o1, o2, o3);
        }
        return u32x4_t{o0, o1, o2, o3};
    };

    float4_t acc[MB][4];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int nb = 0; nb < 4; nb++) acc[i][nb] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // Scales of the current group (fp32) and the requests for the next
    // one's; zero points one group further ahead (the next group's weights
    // are converted during this one).
    uint16_t sn[4];
    uint32_t zn[4], zz = 0;
    float sc[4];
    // The compiler does not count the copies into LDS among the memory
    // operations in flight, so a wait it places for an ordinary load issued
    // before them would wait for the copies too: the loads of one group are
    // taken over at its end, where everything has arrived.
    auto take = [&]() {
#pragma unroll
        for (int nb = 0; nb < 4; nb++) sc[nb] = __uint_as_float(uint32_t(sn[nb]) << 16);
        if (KIND == 1) zz = zn[0] | zn[1] << 8 | zn[2] << 16 | zn[3] << 24;
        asm volatile("" : "+v"(sc[0]), "+v"(sc[1]), "+v"(sc[2]), "+v"(sc[3]), "+v"(zz));
    };
    auto zero_of = [&](int nb) { return KIND == 1 ? (zz >> (8 * nb)) & 0xFFu : 0u; };
    load_scales(gbeg, sn);
    load_zeros(gbeg, zn);
#pragma unroll
    for (int i = 0; i < NW; i++) dma_w(gbeg, i);
#pragma unroll
    for (int i = 0; i < NAT; i++) dma_a(gbeg, 0, i);
    wait_vm_barrier<0>();
    take();
    load_zeros(gbeg + 1 < gend ? gbeg + 1 : gbeg, zn);
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int s = 0; s < 4; s++) wc[nb][s] = convert(raw_at(nb, s), zero_of(nb));
    wait_vm_barrier<0>();
    take();

    constexpr int NS = 4 * MB;      // steps of a group: 16 rows x 32 columns each
    constexpr int SB = NS - 4;      // the first step that reads the next group's weights
    // The copies of the next group go out one instruction a step: the
    // weights in the first steps, then the activations.
    static_assert(NW + NAT <= SB, "copies outlast the group");
    constexpr int LEAD = LO ? 2 : 1; // steps an activation read is ahead of its use
    // 16-row blocks of this wave that hold rows of x.  In the last tile along
    // the rows a wave may have fewer than MB: it leaves out the others'
    // products, and its SIMD's other wave has the matrix core to itself (7B
    // gate int8, fp32 activations at T = 201: 105 -> 103 us).  128-row tiles
    // only: a loop beside the one below; in one loop with it, or on 256-row
    // tiles, the accumulators of both forms do not fit the registers.
    const int live = int(std::min<int64_t>(MB, (std::max<int64_t>(xrows - wm * 16 * MB, 0) + 15) / 16));
    const bool less = MB == 4 && live < MB;
    uint32_t stage = 0;
    for (int g = gbeg; less && g < gend; g++) {
        const int gn = g + 1 < gend ? g + 1 : g, gz = g + 2 < gend ? g + 2 : gend - 1;
        load_scales(gn, sn);
        load_zeros(gz, zn);
        const uint32_t ab = aaddr + stage;
        // the copies, sums, conversions and barriers of the loop below, in a
        // plain order: these waves have time to spare
#pragma unroll
        for (int i = 0; i < NW; i++) dma_w(gn, i);
#pragma unroll
        for (int i = 0; i < NAT; i++) dma_a(gn, stage ^ ASTAGE, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mb = 0; mb < MB - 1; mb++) {
            if (mb >= live) continue;
            float4_t P[4], Q[4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint32_t ad = (ab ^ uint32_t(s << 6)) + mb * 4096;
                const u32x4_t hi = *reinterpret_cast<const u32x4_t*>(lds + ad);
                const u32x4_t lo = LO ? *reinterpret_cast<const u32x4_t*>(lds + ad + APART) : hi;
                const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int nb = 0; nb < 4; nb++) {
                    const float4_t c = s == 0 ? zero : P[nb];
                    if (LO) P[nb] = mfma16(__builtin_bit_cast(half8_t, hi), __builtin_bit_cast(half8_t, wc[nb][s]), c);
                    else P[nb] = mfma16b(__builtin_bit_cast(bf16x8_t, hi), __builtin_bit_cast(bf16x8_t, wc[nb][s]), c);
                    if (LO)
                        Q[nb] = mfma16(__builtin_bit_cast(half8_t, lo), __builtin_bit_cast(half8_t, wc[nb][s]),
                                       s == 0 ? zero : Q[nb]);
                }
            }
#pragma unroll
            for (int nb = 0; nb < 4; nb++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    acc[mb][nb][r] = __builtin_fmaf(sc[nb], LO ? P[nb][r] + Q[nb][r] : P[nb][r], acc[mb][nb][r]);
        }
        wait_vm_only_barrier<NAT>();
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int nb = 0; nb < 4; nb++) wc[nb][s] = convert(raw_at(nb, s), zero_of(nb));
        wait_vm_barrier<0>();
        take();
        stage ^= ASTAGE;
    }
    for (int g = gbeg; !less && g < gend; g++) {
        const int gn = g + 1 < gend ? g + 1 : g, gz = g + 2 < gend ? g + 2 : gend - 1;
        load_scales(gn, sn);
        load_zeros(gz, zn);
        const uint32_t ab = aaddr + stage;
        u32x4_t af[LEAD + 1][PARTS];
        Raw raw[4];
        float4_t P[4], Q[4];  // the sums of the hi (or bf16) and lo products
        auto read_a = [&](int i) {
            u32x4_t(&a)[PARTS] = af[i % (LEAD + 1)];
            const uint32_t ad = (ab ^ uint32_t((i & 3) << 6)) + (i >> 2) * 4096;
            a[0] = *reinterpret_cast<const u32x4_t*>(lds + ad);
            if (LO) a[PARTS - 1] = *reinterpret_cast<const u32x4_t*>(lds + ad + APART);
        };
        auto scale = [&](int mb, int nb) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                acc[mb][nb][r] = __builtin_fmaf(sc[nb], LO ? P[nb][r] + Q[nb][r] : P[nb][r], acc[mb][nb][r]);
        };
#pragma unroll
        for (int i = 0; i < LEAD; i++) read_a(i);
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const int mb = i >> 2, s = i & 3;
            if (i == SB) wait_vm_only_barrier<NAT>();
            if (i + LEAD < NS) read_a(i + LEAD);
            if (mb == MB - 1)
#pragma unroll
                for (int nb = 0; nb < 4; nb++) raw[nb] = raw_at(nb, s);
            if (i < NW) dma_w(gn, i);
            else if (i - NW < NAT) dma_a(gn, stage ^ ASTAGE, i - NW);
            __builtin_amdgcn_sched_barrier(0);
            const u32x4_t(&a)[PARTS] = af[i % (LEAD + 1)];
#pragma unroll
            for (int nb = 0; nb < 4; nb++) {
                // a 16-row block's sums are scaled just before the next
                // block's first product takes their place
                if (s == 0 && mb > 0) {
                    scale(mb - 1, nb);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const float4_t c = s == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : P[nb];
                if (LO) P[nb] = mfma16(__builtin_bit_cast(half8_t, a[0]), __builtin_bit_cast(half8_t, wc[nb][s]), c);
                else P[nb] = mfma16b(__builtin_bit_cast(bf16x8_t, a[0]), __builtin_bit_cast(bf16x8_t, wc[nb][s]), c);
                if (s == 0 && mb > 0) __builtin_amdgcn_sched_barrier(0);
            }
            if (LO) {
#pragma unroll
                for (int nb = 0; nb < 4; nb++)
                    Q[nb] = mfma16(__builtin_bit_cast(half8_t, a[PARTS - 1]), __builtin_bit_cast(half8_t, wc[nb][s]),
                                   s == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : Q[nb]);
            }
            if (mb == MB - 1)
#pragma unroll
                for (int nb = 0; nb < 4; nb++) wc[nb][s] = convert(raw[nb], zero_of(nb));
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int nb = 0; nb < 4; nb++) scale(MB - 1, nb);
        wait_vm_barrier<0>();
        take();
        stage ^= ASTAGE;
    }

    float* dst = direct ? p.y + m0 * p.N + n0 : p.part + (int64_t(split) * tail + ti) * (BM * BN);
    const int64_t pitch = direct ? p.N : BN;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const int row = wm * 16 * MB + mb * 16 + 4 * kq;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (m0 + row + r >= p.T) continue;
            const float rsv = LO ? p.rs[m0 + row + r] : 1.0f;
#pragma unroll
            for (int nb = 0; nb < 4; nb++) {
                if (!nval[nb]) continue;
                const float bv = p.bias && direct ? bf16_to_f32(p.bias[ncol[nb]]) : 0.0f;
                dst[(row + r) * pitch + (ncol[nb] - n0)] = LO ? acc[mb][nb][r] * rsv + bv : acc[mb][nb][r] + bv;
            }
        }
    }
}

// The split tiles' outputs: their range sums in range order, plus the bias.
// Four consecutive columns per thread (VEC: y rows are 16-byte aligned).
template <bool VEC>
__global__ __launch_bounds__(256) void gemmw_reduce_kernel(const GemmwParams p, int bm, int tail) {
    constexpr int BN = 256;
    const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;  // in [tail][bm][BN]
    const int ti = int(i / (bm * BN)), row = int(i / BN) % bm, col = int(i % BN);
    const int t = p.full + ti;
    const int64_t m = int64_t(t % p.tiles_m) * bm + row, n = int64_t(t / p.tiles_m) * BN + col;
    if (m >= p.T || n >= p.N) return;
    const int64_t stride = int64_t(tail) * bm * BN;
    float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < p.splits; s0 += 8) {
        float4_t v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int s = s0 + j < p.splits ? s0 + j : p.splits - 1;
            v[j] = *reinterpret_cast<const float4_t*>(p.part + s * stride + i);
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (s0 + j < p.splits) sum += v[j];
    }
    float* dst = p.y + m * p.N + n;
    if (VEC) {
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] += p.bias ? bf16_to_f32(p.bias[n + e]) : 0.0f;
        *reinterpret_cast<float4_t*>(dst) = sum;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < p.N) dst[e] = sum[e] + (p.bias ? bf16_to_f32(p.bias[n + e]) : 0.0f);
    }
}

template <int KIND, bool LO, int MB>
void launch_t(const GemmwParams& p, hipStream_t stream) {
    constexpr size_t lds = size_t(2) * 32 * MB * 256 * (LO ? 2 : 1) + 256 * (KIND == 1 ? 64 : 128);
    allow_big_lds<gemmw_kernel<KIND, LO, MB>>();
    const int tail = p.tiles_m * p.tiles_n - p.full;
    gemmw_kernel<KIND, LO, MB><<<unsigned(p.full + tail * p.splits), kWThreads, lds, stream>>>(p);
    if (p.splits > 1) {
        const unsigned grid = unsigned(tail * (32 * MB * 256 / 4 / 256));
        if (p.N % 4 == 0 && reinterpret_cast<uintptr_t>(p.y) % 16 == 0)
            gemmw_reduce_kernel<true><<<grid, 256, 0, stream>>>(p, 32 * MB, tail);
        else
            gemmw_reduce_kernel<false><<<grid, 256, 0, stream>>>(p, 32 * MB, tail);
    }
}

}  // namespace

hipError_t launch_gemmw(GemmwParams p, int kind, const GemmwPlan& pl, hipStream_t stream) {
    p.tiles_m = pl.tiles_m;
    p.tiles_n = pl.tiles_n;
    p.full = pl.full;
    p.splits = pl.splits;
    p.gch = pl.gch;
    if (p.al) {
        if (kind == 1) launch_t<1, true, 4>(p, stream);
        else launch_t<0, true, 4>(p, stream);
    } else if (pl.bm == 256) {
        if (kind == 1) launch_t<1, false, 8>(p, stream);
        else launch_t<0, false, 8>(p, stream);
    } else {
        if (kind == 1) launch_t<1, false, 4>(p, stream);
        else launch_t<0, false, 4>(p, stream);
    }
    return hipGetLastError();
}

}  // namespace iq
