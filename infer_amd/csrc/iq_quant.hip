// iq_quant.hip -- on-device quantize + pack and the quantised embedding
// gather for gfx950.
//
// quantize: bit-exact to llm::quantize (src/quant.cpp:34-84): one wave64
// covers eight 128-column groups of one row, 8 lanes per group, each lane 16
// consecutive columns (two 16-byte loads of bf16).
// The group's absmax (int8) or [min,max] widened to 0 (int4) is reduced
// inside the group's lanes; every lane then derives the same bf16 scale and
// writes its codes, so stores stay coalesced.  Groups whose scale is
// ordinary (finite, not tiny) take a rounding path without per-value range
// tests; a wave holding any other group takes the general path.
// Arithmetic follows the reference operation by operation: fp32 correctly
// rounded division, round-half-even (std::lrint under the default mode),
// the reference's clamps, and its comparison forms for max/min so that NaN
// inputs are skipped the same way (the file is built without fast-math and
// with -ffp-contract=off).
//
// embedding: out[t,i] = s * float(q - z) exactly as dequant()
// (src/quant.cpp:86-93; kernels/ops/quant.cu:304-309).
#include <algorithm>

#include "iq_internal.h"
#include "iq_limbs.h"

namespace iq {

namespace {

constexpr int kQThreads = 256;

// Reference clamp (std::max(lo, std::min(hi, v))).
__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// lrint(w / s) of the reference (fp32 division rounded to nearest, then
// round-half-even to an integer), for bf16 w and a bf16 scale s > 0 given
// with r = 1 / s (correctly rounded).  Both w and s carry 8-bit
// significands, W 2^a and S 2^b, so the exact quotient q* = (W / S) 2^(a-b)
// is either a half-integer or at least 2^(a-b) / (2 S) away from every
// half-integer, while both fl(q*) (what the reference rounds) and t = w * r
// are within 2^-22 |q*| <= 2^-22 (255 / S) 2^(a-b) of q*: far inside that
// gap.  So rint(t) equals lrint(fl(q*)) except at exact ties q* = h, which
// fma(h, s, -w) == 0 detects exactly (h has 9 and s 8 significant bits, so
// h * s is exact), and there rint(h) rounds half to even as lrint does.
// Non-finite t (s = 0 or infinite, or a NaN input) gives 0, as int(lrint)
// does on x86-64 for such quotients (lrint yields LONG_MIN, int(long) keeps
// its low 32 bits); |q*| < 2^31 otherwise, since s is w's group maximum / 127
// (or the range / 15) rounded to bf16.
__device__ __forceinline__ int qdiv(float w, float s, float r) {
    const float t = w * r;
    if (!(__builtin_fabsf(t) < 9.2233720368547758e18f)) return 0;
    const float h = __builtin_floorf(t) + 0.5f;
    const bool tie = __builtin_fmaf(h, s, -w) == 0.0f;
    return int(__builtin_rintf(tie ? h : t));
}

// qdiv for a group whose scale is finite, at least 2^-64 (not moved) and
// positive, and whose values are finite or NaN: |w / s| <= 127 (int8) or
// <= 15 (int4 range) so t is finite, and a NaN w gives 0, the reference's
// result for it.  No per-value range test, no scaling by `up`, and no tie
// test: with r within one ulp of 1 / s (v_rcp_f32), t = w r and one
// correction q = fma(fma(-t, s, w), r, t) give exactly the correctly
// rounded fp32 quotient w / s for every pair of bf16 values whose ratio
// lies in [2^-30, 2^10) (checked exhaustively over all significand pairs,
// both signs and the three candidate reciprocals: tests/cpp/
// quant_div_check.c); smaller ratios round to 0 either way.  rint(q) is
// then lrint of the reference's quotient, ties to even included.
__device__ __forceinline__ int qdiv_fast(float w, float s, float r) {
    const float t = w * r;
    const float q = __builtin_fmaf(__builtin_fmaf(-t, s, w), r, t);
    // v_cvt_i32_f32 converts NaN to 0 (and saturates, which |q| <= 128 never
    // reaches): the reference's code for a NaN value
    int c;
    __asm__("v_cvt_i32_f32 %0, %1" : "=v"(c) : "v"(__builtin_rintf(q)));
    return c;
}

// Scale and reciprocal used by qdiv: very small scales (bf16 subnormals
// included) are moved up by 2^64 together with the values (exact powers of
// two), so that 1 / s stays finite.
struct QScale {
    float s, up;  // scale (moved), factor applied to w
    // correctly rounded reciprocal (qdiv); the fast path uses v_rcp_f32
    __device__ float r() const { return 1.0f / s; }
};
__device__ __forceinline__ QScale qscale(float s) {
    QScale q;
    q.up = s < 5.421010862427522e-20f ? 1.8446744073709552e19f : 1.0f;  // 2^-64, 2^64
    q.s = s * q.up;
    return q;
}

// Max / min over the 8 lanes of a half DPP row (one quantisation group of
// quantize8_kernel): half-row mirror, then two quad permutations.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float oct_maxf(float v) {
    v = __builtin_fmaxf(v, dpp_f<0x141>(v));  // row_half_mirror
    v = __builtin_fmaxf(v, dpp_f<0x4E>(v));   // quad_perm 2,3,0,1
    return __builtin_fmaxf(v, dpp_f<0xB1>(v));  // quad_perm 1,0,3,2
}
__device__ __forceinline__ float oct_minf(float v) {
    v = __builtin_fminf(v, dpp_f<0x141>(v));
    v = __builtin_fminf(v, dpp_f<0x4E>(v));
    return __builtin_fminf(v, dpp_f<0xB1>(v));
}

// Max over the 8 lanes of a half DPP row of non-negative values compared
// as unsigned integers (bf16 / fp32 magnitude bits: the order of the
// values).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t oct_maxu(uint32_t v) {
    v = max(v, dpp_u<0x141>(v));
    v = max(v, dpp_u<0x4E>(v));
    return max(v, dpp_u<0xB1>(v));
}

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// Largest magnitude among a lane's 16 bf16 values (8 words), as bf16 bits:
// magnitudes compare as unsigned integers; a result above 0x7F80 means the
// lane holds a NaN.
__device__ __forceinline__ uint32_t absmax16_bits(const uint32_t (&wd)[8]) {
    u16x2_t m[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        m[i] = __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, wd[2 * i] & 0x7FFF7FFFu),
                                         __builtin_bit_cast(u16x2_t, wd[2 * i + 1] & 0x7FFF7FFFu));
    m[0] = __builtin_elementwise_max(m[0], m[1]);
    m[2] = __builtin_elementwise_max(m[2], m[3]);
    m[0] = __builtin_elementwise_max(m[0], m[2]);
    return max(uint32_t(m[0][0]), uint32_t(m[0][1]));
}

// Bytes 0 of c0..c3 in one word (two's complement int8 codes).
__device__ __forceinline__ uint32_t pack4_b0(int c0, int c1, int c2, int c3) {
    const uint32_t lo = __builtin_amdgcn_perm(uint32_t(c1), uint32_t(c0), 0x0C0C0400u);  // c0.b0 c1.b0 0 0
    const uint32_t hi = __builtin_amdgcn_perm(uint32_t(c3), uint32_t(c2), 0x0C0C0400u);  // c2.b0 c3.b0 0 0
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// The quantiser: 8 lanes per group and 16 columns per lane (two 16-byte
// loads), so the per-group work (reductions, the scale's two divisions and
// its bf16 rounding, addresses) is spread over many values.  Items are (row,
// 8 groups); rows whose group count is not a multiple of 8 leave the
// surplus lanes of their last item idle.  A wave walks its items in grid
// strides with three register sets: the values of the next two items are
// in flight while one is converted (each set is refilled right after its
// item is converted, so no wait covers a newer request), and the item
// cursor is wave-uniform (scalar arithmetic).  Group statistics: the
// magnitudes of groups without NaN are compared as unsigned bf16 bits
// (packed 16-bit maxima), the int4 range with fp32 min / max; a wave
// holding a NaN takes the reference's comparison loop.
// RAGGED (cols % 128 != 0): the same requests and stores at any byte offset;
// columns past the row's end (the next row's values) count as zero, which
// no group statistic sees, and the lane they begin in stores its codes one
// byte at a time.  Bound by HBM like the whole-group form (element by
// element loads and byte stores in all lanes: 15872 x 2146 int4 52.5 ->
// 28.0 us, 15872 x 2147 int8 56.5 -> 26.9).
// SHARED: ragged rows of up to 4 groups, 8, 4 or 2 of them an item (`sh`: the
// log2 of the group slots that a row takes of the item's 8).  With one row an
// item half of the lanes or more idled, and inputs in the last-level cache
// took longer than with the element loads (per row / shared: 200000 x 100
// int4 104 -> 20 us, 40000 x 200 int8 23.3 -> 10.7, 263000 x 258 int8 120 ->
// 68, 150000 x 400 int4 80 -> 44; element loads 95, 20.7, 116 and 78).
template <int KIND, bool RAGGED, bool SHARED>
__global__ __launch_bounds__(kQThreads) void quantize8_kernel(const uint16_t* __restrict__ w, int64_t rows,
                                                              int64_t cols, int64_t G, int64_t octs, int sh,
                                                              uint8_t* __restrict__ q, uint16_t* __restrict__ scales,
                                                              uint8_t* __restrict__ zeros) {
    const int lane = threadIdx.x & 63, sub = lane & 7;
    // this lane's group of an item, and (SHARED) its row
    const int gl = SHARED ? (lane >> 3) & ((1 << sh) - 1) : lane >> 3, rl = SHARED ? lane >> (3 + sh) : 0;
    const int per = SHARED ? 8 >> sh : 1;  // rows of an item
    const int64_t blocks = SHARED ? (rows + per - 1) / per : rows;
    const int64_t items = blocks * octs;
    const int64_t stride = int64_t(gridDim.x) * (kQThreads / 64);
    const int64_t first0 = int64_t(blockIdx.x) * (kQThreads / 64) + (threadIdx.x >> 6);
    const int64_t first = (int64_t(__builtin_amdgcn_readfirstlane(uint32_t(first0 >> 32))) << 32) |
                          int64_t(__builtin_amdgcn_readfirstlane(uint32_t(first0)));
    if (first >= items) return;
    const int64_t sr = stride / octs, so = stride % octs;
    struct Cursor {
        int64_t r, o;  // row block, 8 groups of it
    };
    auto advance = [&](Cursor& c) {
        c.r += sr;
        c.o += so;
        if (c.o >= octs) {
            c.o -= octs;
            c.r += 1;
        }
    };
    struct Raw {
        uint4 a, b;
    };
    auto fetch = [&](const Cursor& c) {
        const bool rok = c.r < blocks;
        // RAGGED: a resource over the item's columns, whose last chunk runs
        // into the next row
        const int64_t r = rok ? c.r * per : 0, col0 = c.o * (8 * kGroup);
        const int64_t span = SHARED ? per * cols + 16 : 8 * kGroup + 16;
        const int64_t avail = RAGGED ? std::min<int64_t>((rows - r) * cols - col0, span) : cols;
        const rsrc_t rw = make_rsrc(w + r * cols + (RAGGED ? col0 : 0), rok ? avail * 2 : 0);
        const int64_t g = c.o * 8 + gl;
        uint32_t off;
        if (SHARED)
            off = r + rl < rows && gl * kGroup + sub * 16 < int(cols) ? uint32_t(rl * int(cols) + gl * kGroup + sub * 16) * 2
                                                                      : kOob;
        else if (RAGGED) off = col0 + lane * 16 < cols ? uint32_t(lane * 32) : kOob;
        else off = g < G ? uint32_t((g * kGroup + sub * 16) * 2) : kOob;
        Raw x;
        x.a = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0));
        // (added to the lane's offset, not as the scalar offset, which is
        // documented to be outside the range check: these 16 bytes can be
        // the first past the matrix)
        x.b = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, off + 16, 0, 0));
        return x;
    };
    auto process = [&](const Cursor& cc, const Raw& cur) {
        const int64_t r = SHARED ? cc.r * per + rl : cc.r;
        const int64_t g = cc.o * 8 + gl;
        const bool gvalid = g < G && (!SHARED || r < rows);
        uint32_t wd[8] = {cur.a.x, cur.a.y, cur.a.z, cur.a.w, cur.b.x, cur.b.y, cur.b.z, cur.b.w};
        const int64_t c0 = g * kGroup + sub * 16;
        const int64_t left = cols - c0;  // columns of the row from this lane's first on
        const bool edge = RAGGED && (cc.o + 1) * 8 * kGroup > cols;  // wave-uniform: the row ends here
        if (edge) {
            if ((cols & 1) && (cc.r + 1) * per >= rows) {
                // the matrix ends inside a 4-byte word, which the buffer
                // resource cuts off whole: its last value on its own
                const uint32_t e = w[rows * cols - 1];
#pragma unroll
                for (int i = 0; i < 8; i++) wd[i] = r + 1 == rows && left == 2 * i + 1 ? e : wd[i];
            }
#pragma unroll
            for (int i = 0; i < 8; i++) wd[i] = left >= 2 * i + 2 ? wd[i] : (left == 2 * i + 1 ? wd[i] & 0xFFFFu : 0u);
        }
        float v[16];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[2 * i] = __uint_as_float(wd[i] << 16);
            v[2 * i + 1] = __uint_as_float(wd[i] & 0xFFFF0000u);
        }
        const uint32_t mb = absmax16_bits(wd);
        const bool nan = __builtin_amdgcn_ballot_w64(mb > 0x7F80u) != 0;  // wave-uniform
        if (KIND == 0) {
            // amax = std::max(amax, fabs(v)) over the group: without NaN the
            // largest magnitude (exact); with one, the reference's loop
            // (comparisons skip NaN, quiet or signalling)
            float amax;
            if (!nan) {
                amax = __uint_as_float(oct_maxu(mb) << 16);
            } else {
                amax = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float a = __builtin_fabsf(v[i]);
                    amax = amax < a ? a : amax;
                }
                amax = oct_maxf(amax);
            }
            const uint16_t sb = f32_to_bf16(amax > 0.0f ? amax / 127.0f : 1.0f);
            const QScale qs = qscale(bf16_to_f32(sb));
            uint32_t d[4];
            const bool plain = qs.up == 1.0f && qs.s < 3.0e38f;
            if (__builtin_amdgcn_ballot_w64(!plain) == 0) {
                const float rf = __builtin_amdgcn_rcpf(qs.s);
                int c[16];
#pragma unroll
                for (int i = 0; i < 16; i++) c[i] = clampi(qdiv_fast(v[i], qs.s, rf), -127, 127);
#pragma unroll
                for (int j = 0; j < 4; j++) d[j] = pack4_b0(c[4 * j], c[4 * j + 1], c[4 * j + 2], c[4 * j + 3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) d[j] = 0;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int c = clampi(qdiv(v[i] * qs.up, qs.s, qs.r()), -127, 127);
                    d[i / 4] |= uint32_t(uint8_t(int8_t(c))) << (8 * (i % 4));
                }
            }
            if (!gvalid) return;
            if (sub == 0) scales[r * G + g] = sb;
            uint8_t* const dst = q + r * cols + c0;
            if (!RAGGED) {
                *reinterpret_cast<uint4*>(dst) = make_uint4(d[0], d[1], d[2], d[3]);
            } else if (!edge || left >= 16) {
                __builtin_memcpy(dst, d, 16);
            } else {
#pragma unroll
                for (int i = 0; i < 15; i++)
                    if (i < left) dst[i] = uint8_t(d[i / 4] >> (8 * (i % 4)));
            }
        } else {
            // lo = min(0, min w), hi = max(0, max w) over the group, NaN
            // skipped: without NaN fp32 min / max in any order (the zero's
            // sign, which maxNum may pick either way, reaches no output)
            float mn = 0.0f, mx = 0.0f;
            if (!nan) {
                float a[8], b[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    a[i] = __builtin_fminf(v[2 * i], v[2 * i + 1]);
                    b[i] = __builtin_fmaxf(v[2 * i], v[2 * i + 1]);
                }
#pragma unroll
                for (int s2 = 4; s2 >= 1; s2 >>= 1)
#pragma unroll
                    for (int i = 0; i < s2; i++) {
                        a[i] = __builtin_fminf(a[i], a[i + s2]);
                        b[i] = __builtin_fmaxf(b[i], b[i + s2]);
                    }
                mn = __builtin_fminf(a[0], 0.0f);
                mx = __builtin_fmaxf(b[0], 0.0f);
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    mn = v[i] < mn ? v[i] : mn;
                    mx = mx < v[i] ? v[i] : mx;
                }
            }
            mn = oct_minf(mn);
            mx = oct_maxf(mx);
            const uint16_t sb = f32_to_bf16(mx > mn ? (mx - mn) / 15.0f : 1.0f);
            const QScale qs = qscale(bf16_to_f32(sb));
            uint32_t d[2] = {0, 0};
            int z;
            const bool plain = qs.up == 1.0f && qs.s < 3.0e38f;
            if (__builtin_amdgcn_ballot_w64(!plain) == 0) {
                const float rf = __builtin_amdgcn_rcpf(qs.s);
                z = clampi(qdiv_fast(-mn, qs.s, rf), 0, 15);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int c = clampi(qdiv_fast(v[i], qs.s, rf) + z, 0, 15);
                    d[i / 8] |= uint32_t(c) << (4 * (i % 8));
                }
            } else {
                z = clampi(qdiv(-mn * qs.up, qs.s, qs.r()), 0, 15);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int c = clampi(qdiv(v[i] * qs.up, qs.s, qs.r()) + z, 0, 15);
                    d[i / 8] |= uint32_t(c) << (4 * (i % 8));
                }
            }
            if (!gvalid) return;
            if (sub == 0) {
                scales[r * G + g] = sb;
                zeros[r * G + g] = uint8_t(z);
            }
            uint8_t* const dst = q + (r * cols + c0) / 2;  // (cols is even)
            if (!RAGGED) {
                *reinterpret_cast<uint2*>(dst) = make_uint2(d[0], d[1]);
            } else if (!edge || left >= 16) {
                __builtin_memcpy(dst, d, 8);
            } else {
#pragma unroll
                for (int i = 0; i < 7; i++)
                    if (2 * i < left) dst[i] = uint8_t(d[i / 4] >> (8 * (i % 4)));
            }
        }
    };
    Cursor c0{first / octs, first % octs}, c1 = c0, c2;
    advance(c1);
    c2 = c1;
    advance(c2);
    Raw ra = fetch(c0), rb = fetch(c1), rc;
    // three items per iteration: sets a, b, c hold items c0, c1, c2
    for (;;) {
        rc = fetch(c2);
        process(c0, ra);
        Cursor n = c2;
        advance(n);  // c0 + 3 strides
        if (c1.r >= blocks) break;
        ra = fetch(n);
        process(c1, rb);
        if (c2.r >= blocks) break;
        Cursor n1 = n;
        advance(n1);
        rb = fetch(n1);
        process(c2, rc);
        if (n.r >= blocks) break;
        c0 = n;
        c1 = n1;
        c2 = n1;
        advance(c2);
    }
}

template <bool FAST>
__global__ __launch_bounds__(256) void embedding_kernel(QView t, const int64_t* __restrict__ ids,
                                                        int64_t T, int64_t H, float* __restrict__ out) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;  // one thread per 4 outputs
    const int64_t per_row = (H + 3) / 4;
    if (idx >= T * per_row) return;
    const int64_t tk = idx / per_row, c0 = (idx % per_row) * 4;
    const int64_t id = ids[tk];
    float* o = out + tk * H + c0;
    const int n = int(H - c0 < 4 ? H - c0 : 4);
    if (id < 0 || id >= t.rows) {
        for (int i = 0; i < n; i++) o[i] = __builtin_nanf("");
        return;
    }
    for (int i = 0; i < n; i++) {
        const int64_t c = c0 + i, g = c / kGroup;
        const float s = bf16_to_f32(t.scales[id * t.groups + g]);
        float val;
        if (t.kind == 0) {
            val = s * float(int8_t(t.q[id * t.cols + c]));
        } else {
            const uint8_t byte = t.q[(id * t.cols + c) / 2];
            const int nib = (c & 1) ? (byte >> 4) : (byte & 0xF);
            val = s * float(nib - int(t.zeros[id * t.groups + g]));
        }
        o[i] = val;
    }
}

}  // namespace

hipError_t launch_quantize(const uint16_t* w, int64_t rows, int64_t cols, int kind, uint8_t* q,
                           uint16_t* scales, uint8_t* zeros, hipStream_t stream) {
    const int64_t G = (cols + kGroup - 1) / kGroup;
    // enough resident waves to stream; each walks items in strides of the grid
    const int64_t cap = int64_t(device_cu_count()) * 8;
    const int64_t octs = (G + 7) / 8;
    // ragged rows of up to 4 groups share items (from 5 on more than half of
    // an item's lanes have work: 100000 x 514 int8 51 us, element loads 109)
    const bool ragged = cols % kGroup != 0, shared = ragged && G <= 4;
    const int sh = !shared ? 3 : (G > 2 ? 2 : int(G) - 1);
    const int64_t items = (rows + (8 >> sh) - 1) / (8 >> sh) * octs;
    const unsigned grid = unsigned(std::min<int64_t>((items + 3) / 4, cap));
    auto launch = [&](auto kernel) { kernel<<<grid, kQThreads, 0, stream>>>(w, rows, cols, G, octs, sh, q, scales, zeros); };
    if (shared) kind == 0 ? launch(quantize8_kernel<0, true, true>) : launch(quantize8_kernel<1, true, true>);
    else if (ragged) kind == 0 ? launch(quantize8_kernel<0, true, false>) : launch(quantize8_kernel<1, true, false>);
    else kind == 0 ? launch(quantize8_kernel<0, false, false>) : launch(quantize8_kernel<1, false, false>);
    return hipGetLastError();
}

hipError_t launch_embedding(const QView& t, const int64_t* ids, int64_t T, int64_t H, float* out,
                            hipStream_t stream) {
    const int64_t n = T * ((H + 3) / 4);
    const unsigned grid = unsigned((n + 255) / 256);
    embedding_kernel<true><<<grid, 256, 0, stream>>>(t, ids, T, H, out);
    return hipGetLastError();
}

}  // namespace iq
