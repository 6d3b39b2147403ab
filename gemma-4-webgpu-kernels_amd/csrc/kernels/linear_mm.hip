// Quantised projections of many activation rows on the fp16 matrix cores
// (gfx950), x split once ahead of them: y = x . W^T with packed 2/4/8-bit W.
// The semantics are those of linear_q.hip (rust/src/backend_cpu.rs:174-222).
//
// x is cut into 32-token x 256-k segments (64 k in linear_mm_few); each token's
// segment is scaled by the power of two that puts its largest |x| in [2^14, 2^15)
// and split into hi = fp16(x'), lo = fp16(2^11 (x' - hi)). hi + 2^-11 lo is x' to 2^-23
// of its value for every element within 2^-27 of the segment's largest (one f32
// significand in four is rounded, in its last bit) and to 2^-50 of the largest for
// smaller ones. lo's own scale is what keeps elements beside an outlier: without it
// they are held to 2^-39 of the largest, and where the outlier meets a weight of 0 that
// is the output's error. The weight fields are integers of at most 8 bits, exact in
// fp16 also times 2^-11, so each product with hi or lo is exact in f32 and a segment's
// sum is one v_mfma_f32_32x32x16_f16 chain, folded into the f32 total with the segment's
// scale by one fma. Against 64 bits that is closer than the three bf16 parts of
// linear_q_mfma, which hold all of x (two thirds of the accumulated terms, in chains of
// 256 k): 6.3e-7 -> 1.8e-7 relative through a 2048-row 4-bit MLP.
#include "g4a_math.h"
#include "g4a_params.h"

namespace {

typedef _Float16 mm_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 mm_h8 __attribute__((ext_vector_type(8)));
typedef float mm_f16v __attribute__((ext_vector_type(16)));
constexpr int MM_SEG = 256;  // k of one scale
constexpr float MM_LO = 2048.0f;  // 2^11: lo's own scale

// The order of the 8 k's of chunk c (k = 8c ..) in an operand: which k of the
// chunk's 8 (4-, 8-bit) or of its pair's 16 (2-bit) sits at position pos. It is
// the order in which the fields come out of a word by masks (mm_frag); the sum
// over k does not depend on it.
template <int BITS>
__device__ __forceinline__ constexpr int mm_k(int c, int pos) {
    if (BITS == 4) return 8 * c + pos / 2 + 4 * (pos & 1);
    if (BITS == 2) return 16 * (c / 2) + 4 * (c & 1) + pos / 2 + 8 * (pos & 1);
    return 8 * c + pos;
}

// The exponent a of a segment's scale 2^a from its largest |x|: not below the f32
// normal range (it would flush), and an infinity counts as the largest float, so
// that the finite values beside it stay finite.
__device__ __forceinline__ int mm_scale_exp(float mx) {
    return max(__builtin_amdgcn_frexp_expf(fminf(mx, 3.40282347e38f)) - 15, -126);
}
__device__ __forceinline__ mm_h8 mm_all(float v) {
    const _Float16 c = (_Float16)v;
    return mm_h8{c, c, c, c, c, c, c, c};
}
// x = +-inf leaves lo = inf - inf: any number of the weight's sign keeps the product's
// infinity, as in f32 (a finite lo is at most 2^14; an x that is NaN is NaN in hi).
__device__ __forceinline__ mm_h8 mm_lo(mm_h8 lo) { return __builtin_elementwise_min(lo, mm_all(32768.0f)); }
__device__ __forceinline__ mm_h2 mm_pair(uint32_t v) {
    mm_h2 r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}
// The parts of eight x' = x 2^-a: hi = fp16(x'), lo = fp16(2^11 (x' - hi)). hi is converted
// in pairs, once: the barrier keeps the compiler from converting each value again for lo.
__device__ __forceinline__ void mm_split(const float (&x)[8], int a, mm_h8& hi, mm_h8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const mm_h2 h = {(_Float16)ldexpf(x[i], -a), (_Float16)ldexpf(x[i + 1], -a)};
        uint32_t u;
        __builtin_memcpy(&u, &h, 4);
        asm("" : "+v"(u));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            hi[i + j] = mm_pair(u)[j];
            lo[i + j] = (_Float16)__builtin_fmaf((float)hi[i + j], -MM_LO, ldexpf(x[i + j], 11 - a));
        }
    }
    lo = mm_lo(lo);
}
// The weight operand against lo: w / MM_LO, exact.
__device__ __forceinline__ mm_h8 mm_frag_lo(mm_h8 w) { return w * mm_all(1.0f / MM_LO); }

// x -> xs: token block tb of 32, chunk c, part p (hi, lo), token t: 8 fp16 at
// (((tb * K/8 + c) * 2 + p) * 32 + t) * 8, so a matrix operand is 512 contiguous
// bytes; xscale[(tb * segments + seg) * 32 + t] = 2^a. Workgroup = (segment, token
// block), thread = 32 k of one token; tokens past M are zeros. Bound by the copy:
// x read once, as much written.
template <int BITS>
__device__ __forceinline__ void split_x(const G4aSplitXParams& p) {
    const uint32_t tok = threadIdx.x >> 3, part = threadIdx.x & 7, seg = blockIdx.x, tb = blockIdx.y;
    const uint32_t m = tb * 32 + tok, k0 = seg * MM_SEG + 32 * part;
    const bool on = m < p.M && k0 < p.K;
    const float* __restrict__ src = p.x + (size_t)min(m, p.M - 1) * p.K + min(k0, p.K - 32);
    float x[32];
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float4 v = *reinterpret_cast<const float4*>(src + 4 * i);
        x[4 * i] = on ? v.x : 0.0f;
        x[4 * i + 1] = on ? v.y : 0.0f;
        x[4 * i + 2] = on ? v.z : 0.0f;
        x[4 * i + 3] = on ? v.w : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) mx = fmaxf(mx, fabsf(x[i]));
    mx = g4a_max8(mx);  // the token's 8 threads
    const int a = mm_scale_exp(mx);
    if (part == 0) p.xscale[((size_t)tb * gridDim.x + seg) * 32 + tok] = ldexpf(1.0f, a);
    if (k0 >= p.K) return;
    mm_h8* const dst = reinterpret_cast<mm_h8*>(p.xs) + ((size_t)tb * (p.K / 8) + k0 / 8) * 64 + tok;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        mm_h8 hi, lo;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = x[mm_k<BITS>(c, i)];
        mm_split(v, a, hi, lo);
        dst[c * 64] = hi;
        dst[c * 64 + 32] = lo;
    }
}

// (1024 + u * 2^s) per half -> u - z: one packed fma, exact
__device__ __forceinline__ mm_h2 mm_fix(uint32_t v, float scale, float off) {
    const mm_h2 m = {(_Float16)scale, (_Float16)scale}, o = {(_Float16)off, (_Float16)off};
    return __builtin_elementwise_fma(mm_pair(v), m, o);
}

// The 8 fields of MFMA step i (0 .. 3) from a lane's BITS words (32 k of a row)
// as fp16 integers: a field masked into the low bits of 0x6400 is 1024 + u exactly.
// x & m | 0x64006400 in one instruction (m in a register: no second literal).
__device__ __forceinline__ uint32_t mm_bits(uint32_t x, uint32_t m) {
    uint32_t c = 0x64006400u;
    asm("" : "+v"(m), "+s"(c));  // held in registers, where v_and_or_b32 can take them
    return (x & m) | c;
}
template <int BITS>
__device__ __forceinline__ mm_h8 mm_frag(const uint32_t (&w)[BITS], int i, uint32_t xm) {
    mm_h2 q[4];
    if constexpr (BITS == 4) {
        const uint32_t v = w[i], u = v >> 8;
        q[0] = mm_fix(mm_bits(v, 0x000F000Fu), 1.0f, -1032.0f);
        q[1] = mm_fix(mm_bits(v, 0x00F000F0u), 0.0625f, -72.0f);
        q[2] = mm_fix(mm_bits(u, 0x000F000Fu), 1.0f, -1032.0f);
        q[3] = mm_fix(mm_bits(u, 0x00F000F0u), 0.0625f, -72.0f);
    } else if constexpr (BITS == 2) {
        const uint32_t v = (i & 1) ? w[i >> 1] >> 8 : w[i >> 1];
        q[0] = mm_fix(mm_bits(v, 0x00030003u), 1.0f, -1026.0f);
        q[1] = mm_fix(mm_bits(v, 0x000C000Cu), 0.25f, -258.0f);
        q[2] = mm_fix(mm_bits(v, 0x00300030u), 0.0625f, -66.0f);
        q[3] = mm_fix(mm_bits(v, 0x00C000C0u), 0.015625f, -18.0f);
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t v = w[2 * i + j] ^ xm;  // offset binary
            q[2 * j] = mm_fix(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u), 1.0f, -1152.0f);
            q[2 * j + 1] = mm_fix(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u), 1.0f, -1152.0f);
        }
    }
    mm_h8 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        r[2 * j] = q[j][0];
        r[2 * j + 1] = q[j][1];
    }
    return r;
}

// A lane's words of one 64-k step (rows start on 8 bytes: 4-bit and 8-bit steps
// are then 16-byte loads at 8-byte alignment, which global loads take).
template <int BITS>
__device__ __forceinline__ void mm_load_w(const uint8_t* src, uint32_t (&w)[BITS]) {
    if constexpr (BITS == 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(src);
        w[0] = v.x;
        w[1] = v.y;
    } else {
        typedef uint32_t u4a8 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
        for (int j = 0; j < BITS / 4; ++j) {
            const u4a8 v = *reinterpret_cast<const u4a8*>(src + 16 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * j + e] = v[e];
        }
    }
}

// A step's offset kept in scalar registers, so that the address is a scalar base plus a
// lane offset (the compiler would keep a vector address per lane and advance it: eight
// registers more than the 8-bit blocks have, which then spilled: [1536, 6144] M = 120
// 27.6 us, 22.6 without).
__device__ __forceinline__ size_t mm_scalar(size_t offset) {
    asm("" : "+s"(offset));
    return offset;
}

// One output (or four along n): the epilogue of modes 0, 1, 2 as in linear_q.hip.
template <int MODE>
__device__ __forceinline__ float mm_out(float v, float v2, float bcol) {
    if (MODE == 1) return g4a_gelu_tanh(v) * v2;
    if (MODE == 2) return g4a_gelu_tanh(v) * bcol;
    return v;
}

// Stores the 16 outputs a lane holds of a 32 x 32 block: rows n0 + 8 (v / 4) + 4 h + v % 4
// of token m (v the register, h = lane / 32).
template <int MODE>
__device__ __forceinline__ void mm_store(const G4aLinearMmParams& p, const float (&a)[16], const float (&a2)[16],
                                         uint32_t n0, uint32_t m, int h) {
    const bool vec = (p.N & 3) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0;
    float s[16], s2[16], bv[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const uint32_t n = min(n0 + 8 * (v >> 2) + 4 * h + (v & 3), p.N - 1);
        s[v] = p.s[n];
        s2[v] = MODE == 1 ? p.s2[n] : 0.0f;
        bv[v] = MODE == 2 ? p.b[(size_t)min(m, p.M - 1) * p.b_stride + p.b_off + n] : 0.0f;
    }
    // every load in before the first store (vmcnt(0)): y may alias them as far as the
    // compiler knows, so a load after a store would wait for it
    __builtin_amdgcn_s_waitcnt(0x0F70);
    if (m >= p.M) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t n = n0 + 8 * q + 4 * h;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int v = 4 * q + e;
            o[e] = mm_out<MODE>(a[v] * s[v], a2[v] * s2[v], bv[v]);
        }
        float* const dst = p.y + (size_t)m * p.N + n;
        if (vec && n < p.N) {
            *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < p.N) dst[e] = o[e];
        }
    }
}

// 4 bytes per lane straight to LDS (lane i at dst + i); see copy16s_to_lds.
__device__ __forceinline__ void copy4s_to_lds(const void* sbase, uint32_t voff, float* lds_dst) {
    const uint32_t m0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) float*)lds_dst);
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(m0) : "memory");
}

// Many rows: workgroup = 64 TB tokens x 32 NW weight rows (mode 1: half of them of
// each weight), NW waves of 64 rows x 32 TB tokens. Per 64-k step the split x tile (8
// KiB per token block), the packed weights and the scales stream into a 2-slot LDS
// ring by global->LDS copies: once every wave holds a step's last operands in
// registers (at its third of four MFMA steps) its slot takes the step after next. At
// TB = 2 a wave issues 32 MFMAs (1024 cycles) per step with one operand set being read
// and unpacked ahead of them; with the reads placed where used, a step took 1.3 us
// instead of 0.8 (4 waves, one workgroup). Bound by the MFMAs and the vector
// instructions between them, which do not overlap: of the cycles with every CU busy the
// matrix pipe works 0.53 and the other vector instructions issue in 0.40 (counters), at a
// clock that falls from 2.4 to 1.8 GHz. Gate + up 4-bit [6144, 1536] at M = 2048 takes 152
// us (1020 TFLOP/s of fp16 products), 235 with three bf16 parts; 7 more with 64-bit copy
// addresses per lane and the sums cleared after a fold.
template <int BITS, int MODE, int NW, int TB>
__device__ __forceinline__ void linear_mm_tile(const G4aLinearMmParams& p) {
    constexpr int XF = 4096 * TB;                // floats of a step's x tile (2 TB token blocks)
    constexpr int CX = 16 * TB / NW;             // x copies per wave and step
    constexpr int CW = BITS == 4 ? 1 : 2;        // weight copies (4 bytes a lane at 2 bits, else 16)
    constexpr int WL = BITS == 2 ? 64 : 256;     // floats per weight copy
    constexpr int NV = CX + CW + 1;              // copies per step
    // the sums over hi and lo apart, scaled at a segment's end, or at TB = 2, which has no
    // registers for that, weights times 2^-11 against lo: 8 packed multiplies per 8 MFMAs
    // (gate + up of 2048 tokens 153 -> 156 us)
    constexpr int NP = TB == 1 ? 2 : 1;
    constexpr int SLOT = XF + NW * CW * WL + 64 * TB;
    __shared__ __attribute__((aligned(16))) float lds[2][SLOT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w >> 1, wt = w & 1, h = lane >> 5, rl = lane & 31;
    const uint32_t nblk = (p.M + 31) / 32, tb0 = blockIdx.y * 2 * TB;
    const uint32_t nsteps = p.K / 64, nseg = (p.K + MM_SEG - 1) / MM_SEG;
    const uint32_t n0 = blockIdx.x * (MODE == 1 ? 16 : 32) * NW;
    // row block b of the workgroup's NW (wave row r holds blocks 2r, 2r + 1): mode 1
    // alternates the two weights
    auto block_row = [&](int b) { return MODE == 1 ? n0 + 32 * (b >> 1) : n0 + 32 * b; };
    // every copy is addressed as a scalar base, which the step moves, plus a lane offset
    // (64-bit lane addresses were a fifth of the loop's vector instructions, and those do
    // not run beside the MFMAs)
    const uint32_t wrow = min(block_row(w), p.N - 1);  // a block past N re-reads the last row
    const uint8_t* const wsrc = (MODE == 1 && (w & 1) ? p.wb2 : p.wb) + (size_t)wrow * p.row_bytes;
    const uint32_t woff = min((uint32_t)rl, p.N - 1 - wrow) * p.row_bytes + h * 4 * BITS;
    // x copy i of this wave: 1 KiB piece w * CX + i of the step's 8 KiB token blocks
    constexpr int WPB = NW / (2 * TB);  // waves per token block
    const float* const xsrc = reinterpret_cast<const float*>(p.xs) +
                              (size_t)min(tb0 + w / WPB, nblk - 1) * p.K * 32 + (w % WPB) * CX * 256;
    const uint32_t xoff = 16 * lane;
    // scales of two token blocks (at TB = 2 of this wave's two)
    const uint32_t sb = min(tb0 + (TB == 2 ? 2 * (w & 1) : 0), nblk - 1);
    const float* const ssrc = p.xscale + (size_t)sb * nseg * 32;
    const uint32_t soff = 4 * (min((uint32_t)h, nblk - 1 - sb) * nseg * 32 + rl);
    // copy c (< NV) of step st
    auto issue_one = [&](uint32_t st, float* d, int c) {
        if (c < CX) {
            copy16s_to_lds(xsrc + (size_t)st * 2048 + 256 * c, xoff, d + 256 * (w * CX + c));
        } else if (c < CX + CW) {
            const int j = c - CX;
            float* const wd = d + XF + (w * CW + j) * WL;
            const uint8_t* src = wsrc + (size_t)st * 8 * BITS;
            if constexpr (BITS == 2) copy4s_to_lds(src + 4 * j, woff, wd);
            else copy16s_to_lds(src + 16 * j, woff, wd);
        } else {
            copy4s_to_lds(ssrc + (st >> 2) * 32, soff, d + XF + NW * CW * WL + (TB == 2 ? 64 * (w & 1) : 0));
        }
    };
    auto issue = [&](uint32_t st, int slot) {
#pragma unroll
        for (int c = 0; c < NV; ++c) issue_one(st, lds[slot], c);
    };
    mm_f16v tot[2][TB], acc[NP][2][TB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int v = 0; v < 16; ++v) tot[rb][tb][v] = 0.0f;
    uint32_t wc[2][BITS];
    // operands of two MFMA steps: [step & 1][row block], against lo, [step & 1][part][token block]
    mm_h8 a[2][2], al[2], bx[2][2][TB];
    auto read_w = [&](const float* d) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int j = 0; j < CW; ++j) {
                const float* const ws = d + XF + ((2 * wr + rb) * CW + j) * WL;
                if constexpr (BITS == 2) {
                    wc[rb][j] = reinterpret_cast<const uint32_t*>(ws)[lane];
                } else {
                    const uint4 v = reinterpret_cast<const uint4*>(ws)[lane];
                    wc[rb][4 * j] = v.x;
                    wc[rb][4 * j + 1] = v.y;
                    wc[rb][4 * j + 2] = v.z;
                    wc[rb][4 * j + 3] = v.w;
                }
            }
    };
    auto read_x = [&](const float* d, int i) {
        const float* const xb = d + 2048 * TB * wt + 1024 * h + 4 * rl;
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
                bx[i & 1][part][tb] = *reinterpret_cast<const mm_h8*>(xb + 2048 * tb + (2 * i + part) * 128);
    };
    auto unpack_w = [&](int i) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) a[i & 1][rb] = mm_frag<BITS>(wc[rb], i, p.xm);
    };
    auto scale_w = [&](int i, int rb) {  // step i's weights for lo
        al[rb] = NP == 2 ? a[i & 1][rb] : mm_frag_lo(a[i & 1][rb]);
    };
    auto mfma = [&](int i, int n, bool zero) {  // the n-th of step i's 4 TB; zero: onto 0
        const int part = n / (2 * TB), tb = (n >> 1) % TB, rb = n & 1;
        mm_f16v& sum = acc[part % NP][rb][tb];
        mm_f16v c = sum;
        if (zero) {
#pragma unroll
            for (int v = 0; v < 16; ++v) c[v] = 0.0f;
        }
        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(part ? al[rb] : a[i & 1][rb], bx[i & 1][part][tb], c, 0, 0, 0);
    };
    issue(0, 0);
    if (nsteps > 1) issue(1, 1);
    if (nsteps > 1) wait_vm<NV>();
    else wait_vm<0>();
    barrier_lds();
    read_w(lds[0]);
    read_x(lds[0], 0);
    unpack_w(0);
    for (uint32_t st0 = 0; st0 < nsteps; st0 += 4) {  // a segment of x's scales
        float sc[TB];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t st = st0 + u;
            if (u > 0 && st >= nsteps) break;
            float* const d = lds[u & 1];
            const float* const dn = lds[(u & 1) ^ 1];
            if (u == 0) {
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) sc[tb] = d[XF + NW * CW * WL + 32 * (TB * wt + tb) + rl];
            }
            // operands come one MFMA step ahead, their LDS reads and unpacking spread over
            // the MFMAs in flight
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                read_x(d, i + 1);
                unpack_w(i + 1);
#pragma unroll
                for (int n = 0; n < 4 * TB; ++n) {
                    if (n < 2) scale_w(i, n);
                    mfma(i, n, u == 0 && i == 0 && n < 2 * TB * NP);
                }
#pragma unroll
                for (int j = 0; j < 4 * TB; ++j) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                  // an MFMA
                    if (j < 2 * TB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
                    __builtin_amdgcn_sched_group_barrier(0x002, 8 / TB, 0);             // vector ALU
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (st + 1 < nsteps) {
                wait_vm<0>();   // step st + 1's copies, issued a step ago
                barrier_lds();  // every wave's; every wave has read slot u & 1 for the last time
                read_w(dn);
                read_x(dn, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < 4 * TB; ++n) {
                mfma(3, n, false);
                __builtin_amdgcn_sched_barrier(0);
                if (n < 2) scale_w(3, n);
                if (st + 2 < nsteps) {
#pragma unroll
                    for (int c = n; c < NV; c += 4 * TB) issue_one(st + 2, d, c);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (st + 1 < nsteps) unpack_w(0);
        }
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float t = acc[0][rb][tb][v];
                    if (NP == 2) t = __builtin_fmaf(acc[NP - 1][rb][tb][v], 1.0f / MM_LO, t);
                    tot[rb][tb][v] = __builtin_fmaf(t, sc[tb], tot[rb][tb][v]);
                }
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const uint32_t m = (tb0 + TB * wt + tb) * 32 + rl;
        float a[2][16];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int v = 0; v < 16; ++v) a[rb][v] = tot[rb][tb][v];
        if (MODE == 1) {
            mm_store<1>(p, a[0], a[1], block_row(2 * wr), m, h);
        } else {
            mm_store<MODE>(p, a[0], a[0], block_row(2 * wr), m, h);
            __builtin_amdgcn_sched_barrier(0);  // not both blocks' loads at once
            mm_store<MODE>(p, a[1], a[1], block_row(2 * wr + 1), m, h);
        }
    }
}

// Fewer rows: workgroup = 32 RB weight rows (of each weight) x 32 TB tokens, its 8
// waves taking every eighth 64-k step, operands straight from memory (x from L2),
// the waves' sums added through LDS in order. The tiles above would leave most CUs
// idle here: [1536, 6144] at M = 120 takes 20 us, 100 as 128 x 128 tiles, 91 with
// three bf16 parts and no k split. Bound by the round trips of a wave's few steps: at
// [2048, 1536] M = 120 the waves wait for loads in 43 % of their cycles and to issue in
// 38 %, vector instructions take 12 % (counters); the 59 MB that come through L2 in 6.5 us
// are a quarter of what it gives.
template <int BITS, int MODE, int RB, int TB>
__device__ __forceinline__ void linear_mm_ksplit(const G4aLinearMmParams& p) {
    constexpr int NWT = MODE == 1 ? 2 : 1;  // weights
    constexpr int NR = NWT * RB;            // 32-row blocks
    constexpr int NB = NR * TB;             // 32 x 32 blocks
    constexpr int AHEAD = 1;                // steps in flight ahead of the one computing
    __shared__ float red[8][NB][16][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, rl = lane & 31;
    const uint32_t nblk = (p.M + 31) / 32, tb0 = blockIdx.y * TB;
    const uint32_t nsteps = p.K / 64, nseg = (p.K + MM_SEG - 1) / MM_SEG;
    const uint32_t n0 = blockIdx.x * 32 * RB;
    // scalar bases, which the step moves, and lane offsets (as linear_mm_tile)
    const uint8_t* wp[NR];
    uint32_t woff[RB];
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        const uint32_t row = min(n0 + 32 * (q % RB), p.N - 1);
        wp[q] = (q >= RB ? p.wb2 : p.wb) + (size_t)row * p.row_bytes;
        woff[q % RB] = min((uint32_t)rl, p.N - 1 - row) * p.row_bytes + h * 4 * BITS;
    }
    const uint8_t* xp[TB];
    const uint8_t* scp[TB];
    const uint32_t xoff = 16 * (256 * h + rl), soff = 4 * rl;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const uint32_t b = min(tb0 + tb, nblk - 1);
        xp[tb] = reinterpret_cast<const uint8_t*>(p.xs) + (size_t)b * p.K * 128;
        scp[tb] = reinterpret_cast<const uint8_t*>(p.xscale + (size_t)b * nseg * 32);
    }
    struct Step {
        uint32_t w[NR][BITS];
        mm_h8 x[TB][4][2];
        float sc[TB];
    };
    auto load = [&](Step& s, uint32_t st) {
        if (st >= nsteps) return;  // (the step index is the wave's: no divergence)
#pragma unroll
        for (int q = 0; q < NR; ++q) mm_load_w<BITS>(wp[q] + mm_scalar((size_t)st * 8 * BITS) + woff[q % RB], s.w[q]);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const uint8_t* const xs = xp[tb] + mm_scalar((size_t)st * 8192);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int part = 0; part < 2; ++part)
                    s.x[tb][i][part] = *reinterpret_cast<const mm_h8*>(xs + xoff + (2 * i + part) * 512);
            s.sc[tb] = *reinterpret_cast<const float*>(scp[tb] + mm_scalar((size_t)(st >> 2) * 128) + soff);
        }
    };
    float tot[NB][16];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[b][v] = 0.0f;
    auto compute = [&](const Step& s) {
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            mm_f16v acc[TB];
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[tb][v] = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                mm_h8 a = mm_frag<BITS>(s.w[q], i, p.xm);
#pragma unroll
                for (int part = 0; part < 2; ++part) {
                    if (part) a = mm_frag_lo(a);
#pragma unroll
                    for (int tb = 0; tb < TB; ++tb)
                        acc[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, s.x[tb][i][part], acc[tb], 0, 0, 0);
                }
            }
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    tot[q * TB + tb][v] = __builtin_fmaf(acc[tb][v], s.sc[tb], tot[q * TB + tb][v]);
        }
    };
    // a wave's steps w, w + 8, .. in a ring of 1 + AHEAD register sets
    Step s[1 + AHEAD];
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) load(s[d], w + 8 * d);
    for (uint32_t st = w; st < nsteps; st += 8 * (1 + AHEAD)) {
#pragma unroll
        for (int d = 0; d <= AHEAD; ++d) {
            load(s[(d + AHEAD) % (1 + AHEAD)], st + 8 * (d + AHEAD));
            __builtin_amdgcn_sched_barrier(0);
            if (st + 8 * d < nsteps) compute(s[d]);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) red[w][b][v][lane] = tot[b][v];
    __syncthreads();
    // each wave sums registers 4 q4 .. + 3 of some row x token blocks over the waves
    for (int item = w; item < RB * TB * 4; item += 8) {
        const int rt = item >> 2, q4 = item & 3, tb = rt % TB, rb = rt / TB;
        float o[NWT][4];
#pragma unroll
        for (int q = 0; q < NWT; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float t = 0.0f;
#pragma unroll
                for (int k = 0; k < 8; ++k) t += red[k][(q * RB + rb) * TB + tb][4 * q4 + e][lane];
                o[q][e] = t;
            }
        const uint32_t m = (tb0 + tb) * 32 + rl;
        const uint32_t n = n0 + 32 * rb + 8 * q4 + 4 * h;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (m >= p.M || n + e >= p.N) continue;
            const float v2 = MODE == 1 ? o[NWT - 1][e] * p.s2[n + e] : 0.0f;
            const float bc = MODE == 2 ? p.b[(size_t)m * p.b_stride + p.b_off + n + e] : 0.0f;
            o[0][e] = mm_out<MODE>(o[0][e] * p.s[n + e], v2, bc);
        }
        if (m >= p.M) continue;
        float* const dst = p.y + (size_t)m * p.N + n;
        if ((p.N & 3) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0) {
            if (n < p.N) *reinterpret_cast<float4*>(dst) = make_float4(o[0][0], o[0][1], o[0][2], o[0][3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < p.N) dst[e] = o[0][e];
        }
    }
}

// A lane's words of a 64-k step for v_mfma_f32_16x16x32_f16 (16 k of a row), and
// the 8 fields of its MFMA step i (0, 1) in the order of mm_k.
template <int BITS>
__device__ __forceinline__ void mm_load_w16(const uint8_t* src, uint32_t (&w)[BITS / 2]) {
    if constexpr (BITS == 2) {
        w[0] = *reinterpret_cast<const uint32_t*>(src);
    } else if constexpr (BITS == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(src);
        w[0] = v.x;
        w[1] = v.y;
    } else {
        typedef uint32_t u4a8 __attribute__((ext_vector_type(4), aligned(8)));
        const u4a8 v = *reinterpret_cast<const u4a8*>(src);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = v[e];
    }
}
// Four lanes of a row (g = lane / 16) hold 16 adjacent k each, while x is read with
// four adjacent k per lane (whole 64-byte pieces per load): trade words across the
// lanes so that lane g holds k = 16 j + 4 g .. + 3 for j = 0 .. 3. Fields of the
// result: 8-bit word j; else word i holds j = i in its lower and i + 2 in its upper half.
__device__ __forceinline__ void mm_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void mm_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
template <int BITS>
__device__ __forceinline__ void mm_spread(const uint32_t (&w)[BITS / 2], uint32_t (&o)[BITS == 8 ? 4 : 2]) {
    if constexpr (BITS == 8) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = w[e];
        mm_swap32(o[0], o[2]);
        mm_swap32(o[1], o[3]);
        mm_swap16(o[0], o[1]);
        mm_swap16(o[2], o[3]);
    } else if constexpr (BITS == 4) {
        uint32_t a = w[0], b = w[1];
        mm_swap32(a, b);
        o[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);  // lower halves
        o[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // upper halves
        mm_swap16(o[0], o[1]);
    } else {
        uint32_t a = w[0], b = w[0] >> 16;
        mm_swap32(a, b);
        o[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        o[1] = o[0] >> 8;
        mm_swap16(o[0], o[1]);
    }
}
// The 8 fields of MFMA step i (0, 1) of a 64-k step: position pos holds j, e as mm_few_x.
template <int BITS>
__device__ __forceinline__ mm_h8 mm_few_frag(const uint32_t (&o)[BITS == 8 ? 4 : 2], int i, uint32_t xm) {
    uint32_t t[BITS];
#pragma unroll
    for (int e = 0; e < BITS; ++e) t[e] = o[e % (BITS == 8 ? 4 : 2)];
    return mm_frag<BITS>(t, BITS == 2 ? 2 * i : i, xm);
}
// Index 4 j + e of that position's x.
template <int BITS>
__device__ __forceinline__ constexpr int mm_few_x(int i, int pos) {
    return BITS == 8 ? 8 * i + pos : 4 * (i + 2 * (pos & 1)) + pos / 2;
}

// 16 rows of x or fewer (a serving batch's step): workgroup = 16 RB weight rows (of
// each weight), NW waves taking every NW-th 64-k step, x split in registers by the
// wave that uses it (a launch ahead for it would cost 3 us), one scale per token and
// step; the waves' sums added through LDS in order. Bound by each wave's chain of
// steps: at [1536, 6144] M = 12 its cycles are half waits for loads, a quarter waits to
// issue and a quarter vector instructions (counters; L2 delivers 33 MB in 14.6 us, no
// limit). Three steps' loads are in flight and none past the last step is made (those
// loads alone were 5 of 12 us at M = 16). [2048, 1536] at M = 12 takes 5.8 us, gate + up
// [6144, 1536] 9.8, [1536, 6144] 14.7 (7.2, 19.0 and 19.3 as words; NW = 8).
// NW = 16 halves the chain of a row of 16 .. 32 steps: [2048, 1536] M = 12 5.5 -> 5.1,
// M = 2 4.4 -> 4.0, [1536, 2048] M = 4 5.2 -> 4.8. Longer rows lose ([1536, 4096] M = 8
// 8.4 against 9.0), shorter ones have no step for each wave.
template <int BITS, int MODE, int RB, int NW>
__device__ __forceinline__ void linear_mm_few(const G4aLinearMmParams& p) {
    constexpr int NWT = MODE == 1 ? 2 : 1;
    constexpr int NR = NWT * RB;  // 16-row blocks
    constexpr int D = 3;          // steps in flight
    __shared__ float red[NW][NR][4][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, rl = lane & 15;
    const uint32_t nsteps = p.K / 64, n0 = blockIdx.x * 16 * RB;
    const uint8_t* wp[NR];
#pragma unroll
    for (int q = 0; q < NR; ++q)
        wp[q] = (q >= RB ? p.wb2 : p.wb) + (size_t)min(n0 + 16 * (q % RB) + rl, p.N - 1) * p.row_bytes + g * 2 * BITS;
    const float* const xp = p.x + (size_t)min((uint32_t)rl, p.M - 1) * p.K + 4 * g;
    struct Step {
        uint32_t w[NR][BITS / 2];
        float4 x[4];
    };
    auto load = [&](Step& s, uint32_t st) {
        if (st >= nsteps) return;  // (the step index is the wave's: no divergence)
#pragma unroll
        for (int q = 0; q < NR; ++q) mm_load_w16<BITS>(wp[q] + (size_t)st * 8 * BITS, s.w[q]);
#pragma unroll
        for (int i = 0; i < 4; ++i) s.x[i] = *reinterpret_cast<const float4*>(xp + (size_t)st * 64 + 16 * i);
    };
    typedef float f4v_ __attribute__((ext_vector_type(4)));
    float tot[NR][4];
#pragma unroll
    for (int q = 0; q < NR; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) tot[q][v] = 0.0f;
    auto compute = [&](const Step& s) {
        float x[16], mx = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[4 * i] = s.x[i].x;
            x[4 * i + 1] = s.x[i].y;
            x[4 * i + 2] = s.x[i].z;
            x[4 * i + 3] = s.x[i].w;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(x[i]));
        mx = g4a_col_max4(mx);  // the token's 64 k
        const int a = mm_scale_exp(mx);
        mm_h8 hi[2], lo[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = x[mm_few_x<BITS>(c, i)];
            mm_split(v, a, hi[c], lo[c]);
        }
        const float sc = ldexpf(1.0f, a);
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            f4v_ acc = {0.0f, 0.0f, 0.0f, 0.0f};
            uint32_t o[BITS == 8 ? 4 : 2];
            mm_spread<BITS>(s.w[q], o);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const mm_h8 f = mm_few_frag<BITS>(o, i, p.xm);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(f, hi[i], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(mm_frag_lo(f), lo[i], acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) tot[q][v] = __builtin_fmaf(acc[v], sc, tot[q][v]);
        }
    };
    Step s[D];
#pragma unroll
    for (int d = 0; d + 1 < D; ++d) load(s[d], w + NW * d);
    for (uint32_t st = w; st < nsteps; st += NW * D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(s[(d + D - 1) % D], st + NW * (d + D - 1));
            __builtin_amdgcn_sched_barrier(0);
            if (st + NW * d < nsteps) compute(s[d]);
        }
    }
#pragma unroll
    for (int q = 0; q < NR; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[w][q][v][lane] = tot[q][v];
    __syncthreads();
    // output (token m, row nn of the workgroup), rows next to each other across threads
    for (uint32_t e = tid; e < 16 * 16 * RB; e += 64 * NW) {
        const uint32_t m = e / (16 * RB), nn = e % (16 * RB), n = n0 + nn;
        if (m >= p.M || n >= p.N) continue;
        const int rb = nn >> 4, src = 16 * ((nn >> 2) & 3) + m;
        float o = 0.0f, o2 = 0.0f;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            o += red[k][rb][nn & 3][src];
            if (MODE == 1) o2 += red[k][NR - RB + rb][nn & 3][src];
        }
        p.y[(size_t)m * p.N + n] = mm_out<MODE>(o * p.s[n], MODE == 1 ? o2 * p.s2[n] : 0.0f,
                                                MODE == 2 ? p.b[(size_t)m * p.b_stride + p.b_off + n] : 0.0f);
    }
}

}  // namespace

// Forms 0, 1, 4: tiles of 128 tokens x 256 / 128 rows and 64 tokens x 128 rows; 2, 3:
// k-split blocks of 32 tokens x 64 / 32 rows (in mode 1 the tiles share their rows
// between the weights, the blocks hold as many of each). At 8 bits form 1, whose two
// workgroups a CU the weights' LDS rules out, and form 2 of two weights, which spills,
// are not built (linear_mm_choose).
#define G4A_MM(B, MODE)                                                                                           \
    extern "C" __global__ __launch_bounds__(512) void g4a_linear_mm_0_b##B##_mode##MODE(G4aLinearMmParams p) {    \
        linear_mm_tile<B, MODE, 8, 2>(p);                                                                         \
    }                                                                                                             \
    extern "C" __global__ __launch_bounds__(512, MODE == 1 ? 2 : 4) void g4a_linear_mm_3_b##B##_mode##MODE(       \
        G4aLinearMmParams p) {                                                                                    \
        linear_mm_ksplit<B, MODE, 1, 1>(p);                                                                       \
    }
#define G4A_MM_1(B, MODE)                                                                                         \
    extern "C" __global__ __launch_bounds__(256, 2) void g4a_linear_mm_1_b##B##_mode##MODE(G4aLinearMmParams p) { \
        linear_mm_tile<B, MODE, 4, 2>(p);                                                                         \
    }
#define G4A_MM_2(B, MODE)                                                                                         \
    extern "C" __global__ __launch_bounds__(512) void g4a_linear_mm_2_b##B##_mode##MODE(G4aLinearMmParams p) {    \
        linear_mm_ksplit<B, MODE, 2, 1>(p);                                                                       \
    }
#define G4A_MM_T64(B, MODE)                                                                                       \
    extern "C" __global__ __launch_bounds__(256, 3) void g4a_linear_mm_4_b##B##_mode##MODE(G4aLinearMmParams p) {   \
        linear_mm_tile<B, MODE, 4, 1>(p);                                                                         \
    }
#define G4A_MM_FEW(B, MODE, RB)                                                                                   \
    extern "C" __global__ __launch_bounds__(512) void g4a_linear_mm_few_r##RB##_b##B##_mode##MODE(              \
        G4aLinearMmParams p) {                                                                                    \
        linear_mm_few<B, MODE, RB, 8>(p);                                                                         \
    }
#define G4A_MM_FEW16(B)                                                                                           \
    extern "C" __global__ __launch_bounds__(1024) void g4a_linear_mm_few_w16_b##B##_mode0(G4aLinearMmParams p) {    \
        linear_mm_few<B, 0, 1, 16>(p);                                                                            \
    }
#define G4A_MM_SET(B)                                                                                             \
    G4A_MM(B, 0) G4A_MM(B, 1) G4A_MM(B, 2) G4A_MM_T64(B, 0) G4A_MM_T64(B, 1) G4A_MM_T64(B, 2)                       \
    G4A_MM_FEW(B, 0, 1) G4A_MM_FEW(B, 0, 2) G4A_MM_FEW(B, 1, 1) G4A_MM_FEW(B, 1, 2) G4A_MM_FEW(B, 2, 1)             \
    G4A_MM_FEW(B, 2, 2) G4A_MM_FEW16(B)                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void g4a_split_x_b##B(G4aSplitXParams p) { split_x<B>(p); }
G4A_MM_SET(2)
G4A_MM_SET(4)
G4A_MM_SET(8)
G4A_MM_1(2, 0) G4A_MM_1(2, 1) G4A_MM_1(2, 2) G4A_MM_1(4, 0) G4A_MM_1(4, 1) G4A_MM_1(4, 2)
G4A_MM_2(2, 0) G4A_MM_2(2, 1) G4A_MM_2(2, 2) G4A_MM_2(4, 0) G4A_MM_2(4, 1) G4A_MM_2(4, 2)
G4A_MM_2(8, 0) G4A_MM_2(8, 2)
