// lm_head_split.h — the LM head for B > 1 on the bf16 matrix cores, with f32
// results: logits[b][v] = dot(hidden[b], W[v]) (src/model.rs:317-325,
// src/quant.rs:121-161).
//
// Every f32 operand is the exact sum of three bf16 parts (each the
// round-to-nearest of what the parts before it leave: 8 + 8 + 8 bits).  A
// product of two parts is exact in f32, and v_mfma_f32_32x32x16_bf16 sums
// them in f32.  int8 and int4 codes are bf16 integers already, so their
// products with the three parts of x are all of the product; for f32 weights
// the six products down to 2^-18 of the largest are taken and the three left
// out are below 2^-26 of it.  The f32 matrix instructions this replaces run
// at 1/16 of the bf16 rate and round after every 4 products instead of 16:
// measured against 64-bit sums the relative error is 1.2e-7 (256 x 768 x 50257
// f32; 3.6e-7 before) and 1.4e-7 (64 x 2048 x 128256 int8; 5.8e-7 before).
//
// What bounds it: three (codes) or six (f32) bf16 MFMAs per tile step at the
// 1.8-1.9 GHz that the card holds under them, the splitting beside them, and
// the weights' stream from HBM.  Measured against the f32 matrix-core kernel:
// 256 x 768 x 50257 f32 244 -> 146 us (six products at that clock: 82);
// 64 x 2048 x 128256 int8 337 -> 130; 17 x 768 x 50257 int8, groups of 64,
// 81 -> 29.5; 32 x 4096 x 32000 int4 196 -> 88.
//
// Layout.  v_mfma_f32_32x32x16_bf16, A = 32 hidden rows, B = 32 vocab rows: lane
// l holds row l % 32 of each operand at h = 8 (l / 32) .. + 7 of the step's 16.
// A workgroup of NW waves covers 32 NB hidden rows and 32 NV NW vocab rows; each
// wave holds NB x NV accumulator tiles.  h goes in chunks of 16 KT.
//   - x: loaded XD chunks ahead, split by the workgroup while the chunk before it
//     is multiplied, its parts put into LDS in fragment order
//     ([tile][step][part][lane], 16 bytes a lane; two buffers, one barrier a
//     chunk), where stores and ds_read_b128 are conflict-free.  Splitting it
//     once per workgroup is why the tile is wide in v.
//   - W: each row belongs to one wave, which loads WD chunks ahead with 2 to 8
//     neighbouring lanes per row (a lane per row kept the address unit busy for
//     64 cache lines an instruction) and turns the rows into fragments through
//     LDS of its own, 16-byte blocks xor-swizzled by row.  A lane's values of a
//     chunk are contiguous (its steps use them 8 at a time; x is staged in the
//     same order).  Codes whose groups are no multiple of 64, or whose rows are
//     none of 32, are loaded straight into fragments, each step's 16 together.
//   - Each tile's sum over a chunk starts from zero and joins the f32 total once,
//     times the group's scale (the reference scales each group's own sum).
// Loads need 4-byte alignment only (buffer loads); every offset is bounded by
// the tile's buffer descriptor, and positions past H read zeros.
//
// A result that is not finite is computed again by plain f32 sums: infinities
// and NaNs in the operands have no three finite parts, and a value whose bf16
// rounding overflows would turn into one.
#pragma once
#include <type_traits>

#include "lm_head.h"
#include "row_common.h"

namespace nis {

typedef __bf16 lh_b8 __attribute__((ext_vector_type(8)));
typedef float lh_f16 __attribute__((ext_vector_type(16)));

constexpr int kLsMaxH = 1 << 16;         // (a tile's bytes stay below 2^31)

__device__ u4v nis_buffer_load_u4(i4v rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.buffer.load.v4i32");
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
__device__ u2v nis_buffer_load_u2(i4v rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.buffer.load.v2i32");
__device__ uint32_t nis_buffer_load_u1(i4v rsrc, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.raw.buffer.load.i32");

// Two f32 to packed bf16, rounded to nearest even.
__device__ __forceinline__ uint32_t ls_pk_bf16(float a, float b) {
    uint32_t r;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// The three bf16 parts of 8 floats.
__device__ __forceinline__ void ls_split8(const float (&x)[8], u4v (&p)[3]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float a = x[2 * e], b = x[2 * e + 1];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const uint32_t k = ls_pk_bf16(a, b);
            p[i][e] = k;
            if (i < 2) {  // exact: the rest has at most 16 (then 8) significant bits
                a -= __uint_as_float(k << 16);
                b -= __uint_as_float(k & 0xFFFF0000u);
            }
        }
    }
}

// A lane's weights of one chunk and one 32-row tile, as loaded: 8 KT values.
template <int FMT, int KT>
struct LsRaw {
    static constexpr int kWords = FMT == kLhF32 ? 8 * KT : (FMT == kLhInt8 ? 2 * KT : KT);
    uint32_t u[kWords];
};

// Step s of a chunk as bf16 parts (one part for codes, which are exact).
template <int FMT, int KT>
__device__ __forceinline__ void ls_parts(const LsRaw<FMT, KT>& r, int s, u4v (&p)[FMT == kLhF32 ? 3 : 1]) {
    if constexpr (FMT == kLhF32) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(r.u[8 * s + e]);
        ls_split8(x, p);
    } else if constexpr (FMT == kLhInt8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t c = r.u[2 * s + h];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float a = (float)((c >> (16 * e)) & 255u) - 128.0f;
                const float b = (float)((c >> (16 * e + 8)) & 255u) - 128.0f;
                p[0][2 * h + e] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
            }
        }
    } else {
        uint32_t lo = r.u[s] & 0x0F0F0F0Fu, hi = (r.u[s] >> 4) & 0x0F0F0F0Fu;
        asm("" : "+v"(lo), "+v"(hi));  // (the masks hidden: byte conversions, not bit extracts)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = (float)((lo >> (8 * e)) & 255u) - 8.0f;
            const float b = (float)((hi >> (8 * e)) & 255u) - 8.0f;
            p[0][e] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
        }
    }
}

// One logit by plain f32 sums (results that are not finite).
template <int FMT>
__device__ __noinline__ float ls_plain(const LmHeadArgs& a, int64_t b, int64_t v) {
    const float* x = a.x + b * a.ldx;
    float s = 0.f;
    for (int g = 0; g < a.groups; ++g) {
        float t = 0.f;
        for (int h = g * a.group; h < (g + 1) * a.group; ++h) {
            const int64_t i = v * (int64_t)a.H + h;
            const float wv = FMT == kLhF32 ? ((const float*)a.w)[i] : lh_code(a, i, FMT);
            t = fmaf(x[h], wv, t);
        }
        s += a.groups > 1 ? t * a.scales[v * a.groups + g] : t;
    }
    return s;
}

template <int FMT, int NB, int NV, int KT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void lm_head_split_kernel(LmHeadArgs a) {
    constexpr int T = 64 * NW;
    constexpr int C = 16 * KT;                   // h per chunk
    constexpr int NP = FMT == kLhF32 ? 3 : 1;    // parts of a weight
    // chunks in flight: more while the accumulators leave registers.  (Loads
    // return in order: x is asked for as far ahead as W, or the wait for a
    // chunk's x would be one for the W asked for before it.)
    constexpr int WD = NB <= 2 && (NV == 1 || (NB == 1 && FMT != kLhF32)) ? 4 : (FMT == kLhF32 ? 1 : 2);
    constexpr int XD = NB <= 2 ? WD : 1;
    constexpr int kWords = LsRaw<FMT, KT>::kWords;
    constexpr int kLpr = kWords / 2;             // 16-byte blocks of a row's chunk (lanes per row)
    __shared__ u4v xs[2][NB][KT][3][64];
    __shared__ u4v ws[NW][FMT == kLhF32 && NB == 8 ? 1 : 32 * kLpr];
    const int tid = (int)threadIdx.x, l = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(wave_id());
    const int r32 = l & 31, q = l >> 5;
    const int64_t b0 = (int64_t)blockIdx.y * (32 * NB);
    const int64_t v0 = ((int64_t)blockIdx.x * NW + w) * (32 * NV);
    const int H = a.H, nc = (H + C - 1) / C;
    const bool grouped = FMT != kLhF32 && a.groups > 1;
    // each lane's values of a chunk contiguous, or each step's 16 together
    const bool runs = FMT == kLhF32 || ((H & 31) == 0 && !(grouped && (a.group & 63) != 0));
    // (a lane's 8 values of step s start at h = 8 (KT q + s) of the chunk, or at
    // 16 s + 8 q)

    // the wave's rows of W; a wave past V reads nothing
    const int row_bytes = FMT == kLhF32 ? H * 4 : (FMT == kLhInt8 ? H : H / 2);
    const int64_t vleft = a.V - v0;
    const int rows = (int)(vleft < 0 ? 0 : (vleft < 32 * NV ? vleft : 32 * NV));
    const uint64_t wp = (uint64_t)(uintptr_t)a.w + (uint64_t)(rows > 0 ? v0 * row_bytes : 0);
    const i4v wr = {(int32_t)(uint32_t)wp, (int32_t)(uint32_t)((wp >> 32) & 0xFFFFu), rows * row_bytes, 0x00020000};
    constexpr int kOut = 0x7FFFFFF0;  // (reads nothing)
    constexpr int kRpi = 64 / kLpr;   // rows of one load instruction
    constexpr int kBpw = FMT == kLhF32 ? 4 : 1;                // 16-byte block -> h: 4 floats, 16 or 32 codes
    constexpr int kHpb = FMT == kLhF32 ? 4 : (FMT == kLhInt8 ? 16 : 32);
    // (8 tiles of f32 are bound by their MFMAs: there a lane loads its own run
    // of its own row, and neither LDS nor more registers are spent on W)
    constexpr bool kDirect = FMT == kLhF32 && NB == 8;
    const int lrow = kDirect ? r32 : l / kLpr, lblk = kDirect ? q * (kLpr / 2) : l % kLpr;
    auto load_w = [&](int c, int j, LsRaw<FMT, KT>& r) {  // tile j of chunk c
        const int k0 = c * C;
        if (runs) {
            const int off = (FMT == kLhInt4 ? k0 >> 1 : k0 * kBpw) + 16 * lblk;
#pragma unroll
            for (int i = 0; i < kLpr / 2; ++i) {
                const int row = 32 * j + lrow + (kDirect ? 0 : kRpi * i);
                const int bi = kDirect ? i : 0;
                const bool in = row < rows && k0 + kHpb * (lblk + bi) < H;
                const u4v t = nis_buffer_load_u4(wr, in ? row * row_bytes + off + 16 * bi : kOut, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) r.u[4 * i + e] = t[e];
            }
        } else {
            const int rb = 32 * j + r32 < rows ? (32 * j + r32) * row_bytes : kOut;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int k = k0 + 16 * s + 8 * q;
                const bool in = rb != kOut && k < H;
                if constexpr (FMT == kLhInt8) {
                    const u2v t = nis_buffer_load_u2(wr, in ? rb + k : kOut, 0, 0);
                    r.u[2 * s] = t.x;
                    r.u[2 * s + 1] = t.y;
                } else if constexpr (FMT == kLhInt4) {
                    r.u[s] = nis_buffer_load_u1(wr, in ? rb + (k >> 1) : kOut, 0, 0);
                }
            }
        }
    };
    // a tile's rows, as loaded by rows, into each lane's run of its own row
    auto turn_w = [&](LsRaw<FMT, KT>& r) {
        if (!runs || kDirect) return;
        static_assert(kLpr == 2 || kLpr == 4 || kLpr == 8, "lanes per row");
        auto swz = [](int row) { return kLpr == 8 ? (row >> 1) & 7 : (kLpr == 4 ? (row >> 2) & 3 : 0); };
#pragma unroll
        for (int i = 0; i < kLpr / 2; ++i) {
            const int row = kRpi * i + lrow;
            ws[w][row * kLpr + (lblk ^ swz(row))] = u4v{r.u[4 * i], r.u[4 * i + 1], r.u[4 * i + 2], r.u[4 * i + 3]};
        }
        lds_wave_fence();
#pragma unroll
        for (int i = 0; i < kLpr / 2; ++i) {
            const u4v t = ws[w][r32 * kLpr + ((q * (kLpr / 2) + i) ^ swz(r32))];
#pragma unroll
            for (int e = 0; e < 4; ++e) r.u[4 * i + e] = t[e];
        }
        lds_wave_fence();
    };

    // x: slot i = tid + T u stages 8 floats, block i % (2 KT) of row i / (2 KT)
    // (neighbouring lanes on one row's cache line); its place in LDS is the
    // fragment lane that uses it, xor-swizzled by the block so that the stores
    // of 8 neighbouring lanes meet different banks
    constexpr int kXb = 2 * KT, kXr = T / kXb;  // blocks of a row's chunk, rows per load
    constexpr int SPT = 32 * NB > kXr ? 32 * NB / kXr : 1;  // (some lanes idle at one tile of 8 waves)
    const int64_t bl = (int64_t)a.B - b0;
    const int brows = (int)(bl < 32 * NB ? bl : 32 * NB);
    const uint64_t xb = (uint64_t)(uintptr_t)(a.x + b0 * a.ldx);
    const int ldx4 = (int)(4 * a.ldx);
    const i4v xd = {(int32_t)(uint32_t)xb, (int32_t)(uint32_t)((xb >> 32) & 0xFFFFu),
                    (brows - 1) * ldx4 + 4 * H, 0x00020000};
    // (kDirect: a wave per tile and step instead, each lane its own fragment's
    // 8 floats; more cache lines per load, but no swizzle to hold in registers)
    const int xblk = kDirect ? KT * q + (tid >> 6) % KT : tid % kXb;
    const int xrow = kDirect ? 32 * ((tid >> 6) / KT) + r32 : tid / kXb;
    auto swx = [](int blk) { return kDirect ? 0 : blk * (4 / KT); };
    u4v* const xdst = &xs[0][0][runs ? xblk % KT : xblk >> 1][0][32 * (runs ? xblk / KT : xblk & 1)];
    int xsw[KT];  // the lane's place in the fragments of step s
#pragma unroll
    for (int s = 0; s < KT; ++s) xsw[s] = 32 * q + (r32 ^ swx(runs ? KT * q + s : 2 * s + q));
    f4v xr[XD][SPT][2];
    auto load_x = [&](int c, int u, f4v (&r)[2]) {
        const int row = xrow + kXr * u;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = c * C + 8 * xblk + 4 * h;
            r[h] = nis_buffer_load_f4(xd, k < H && row < brows ? row * ldx4 + 4 * k : kOut, 0, 0);
        }
    };
    auto stage_x = [&](int u, int buf, const f4v (&r)[2]) {
        const int row = xrow + kXr * u;
        if (32 * NB < kXr && row >= 32 * NB) return;
        const float x8[8] = {r[0].x, r[0].y, r[0].z, r[0].w, r[1].x, r[1].y, r[1].z, r[1].w};
        u4v p[3];
        ls_split8(x8, p);
        u4v* const d = xdst + buf * (NB * KT * 3 * 64) + (row >> 5) * (KT * 3 * 64) + ((row & 31) ^ swx(xblk));
#pragma unroll
        for (int k = 0; k < 3; ++k) d[64 * k] = p[k];
    };

    lh_f16 tot[NB][NV];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) tot[i][j][r] = 0.f;

    // The products of steps [S0, S1) for every tile: each tile's sum starts
    // from zero with the smallest products (which round at their own size),
    // and joins the total once, times its group's scale.  (One accumulator
    // for the whole row rounded each of its MFMAs at full size: error 4.2e-7
    // where this form has 1.1e-7.)
    // The next step's fragments of x are read while a step's MFMAs run; side(p,
    // n) is the rest of the chunk's work, in n parts between the MFMAs.
    constexpr bool kUpFront = FMT == kLhF32 && NB == 8;  // (all of side before the MFMAs: no registers left for it)
    auto products = [&](auto s0c, auto s1c, int buf, const u4v (&wf)[KT][NV][NP], const float (&sc)[NV], auto side) {
        constexpr int S0 = decltype(s0c)::value, S = decltype(s1c)::value - S0;
        u4v xf[2][3];
        auto frag = [&](int p) {
#pragma unroll
            for (int k = 2; k >= 0; --k) xf[p & 1][k] = xs[buf][p / S][S0 + p % S][k][xsw[S0 + p % S]];
        };
        // (two sets of sums where registers allow: one joins the total while the
        // next tile's MFMAs run)
        constexpr int NA = FMT == kLhF32 && NB == 8 ? 2 : 1;
        lh_f16 acc[NA][NV];
        auto add = [&](int i) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    tot[i][j][r] = FMT == kLhF32 ? tot[i][j][r] + acc[i % NA][j][r]
                                                 : fmaf(acc[i % NA][j][r], sc[j], tot[i][j][r]);
        };
        if (kUpFront) {
            side(-1, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        frag(0);
#pragma unroll
        for (int p = 0; p < NB * S; ++p) {
            const int i = p / S, s = p % S;
            if (p + 1 < NB * S) frag(p + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (s == 0)
#pragma unroll
                for (int j = 0; j < NV; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i % NA][j][r] = 0.f;
#pragma unroll
            for (int o = 2; o >= 0; --o)  // parts k of x and m of W, k + m = o
#pragma unroll
                for (int k = o; k >= 0; --k) {
                    if (o - k >= NP) continue;
#pragma unroll
                    for (int j = 0; j < NV; ++j)
                        acc[i % NA][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(lh_b8, xf[p & 1][k]), __builtin_bit_cast(lh_b8, wf[S0 + s][j][o - k]),
                            acc[i % NA][j], 0, 0, 0);
                }
            side(p, NB * S);
            if (NA == 2 && s == 0 && i > 0) add(i - 1);
            if (NA == 1 && s == S - 1) add(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (NA == 2) add(NB - 1);
    };
    // each vocab row's scale of the group of h (1 without groups)
    auto scales = [&](int h, float (&sc)[NV]) {
#pragma unroll
        for (int j = 0; j < NV; ++j) sc[j] = 1.0f;
        if (grouped) {
            const int g = lh_group_of(a, min(h, H - 1));
#pragma unroll
            for (int j = 0; j < NV; ++j) sc[j] = a.scales[min(v0 + 32 * j + r32, a.V - 1) * a.groups + g];
        }
    };

    // Each workgroup begins its walk over h at another chunk: in step, all of
    // them would read one chunk's column of the rows, 64 or 128 bytes every
    // row_bytes, which lie in a fraction of the memory channels (50257 x 768
    // f32, 4 waves a workgroup: 208 us in step, 166 apart).  Past the last chunk: an h that reads nothing.
    const int rot = (int)(((blockIdx.x >> 3) * 5 + blockIdx.y) % (unsigned)nc);
    auto at = [&](int c) { return c >= nc ? nc : (c + rot >= nc ? c + rot - nc : c + rot); };
    LsRaw<FMT, KT> raw[WD][NV];
    // (x of chunk c is in xr[c % XD] until it is staged, a chunk ahead of its use)
#pragma unroll
    for (int d = 0; d < (XD > WD ? XD : WD); ++d) {
        if (d < XD)
#pragma unroll
            for (int u = 0; u < SPT; ++u) load_x(at(d), u, xr[d][u]);
        if (d < WD)
#pragma unroll
            for (int j = 0; j < NV; ++j) load_w(at(d), j, raw[d][j]);
    }
#pragma unroll
    for (int u = 0; u < SPT; ++u) {
        stage_x(u, 0, xr[0][u]);
        load_x(at(XD), u, xr[0][u]);
    }
    for (int c0 = 0; c0 < nc; c0 += WD) {
#pragma unroll
        for (int d = 0; d < WD; ++d) {
            const int c = c0 + d;
            if (c >= nc) break;
            float sc[KT / 2][NV];
#pragma unroll
            for (int s = 0; s < KT / 2; ++s) scales(at(c) * C + 32 * s, sc[s]);
            u4v wf[KT][NV][NP];
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                turn_w(raw[d][j]);
#pragma unroll
                for (int s = 0; s < KT; ++s) ls_parts<FMT, KT>(raw[d][j], s, wf[s][j]);
            }
            // (one barrier a chunk: chunk c is staged, and chunk c - 1 is no
            // longer read, so its buffer takes chunk c + 1)
            lds_barrier();
            // chunk c + 1 staged, x of chunk c + 1 + XD and W of chunk c + WD asked for
            const int xc = at(c + 1 + XD), wc = at(c + WD);
            auto side = [&](int p, int n) {
#pragma unroll
                for (int u = 0; u < SPT + NV; ++u) {
                    if (kUpFront ? p >= 0 : u * n / (SPT + NV) != p) continue;
                    if (u < NV) {
                        load_w(wc, u, raw[d][u]);
                    } else {
                        stage_x(u - NV, (c + 1) & 1, xr[(d + 1) % XD][u - NV]);
                        load_x(xc, u - NV, xr[(d + 1) % XD][u - NV]);
                    }
                }
            };
            using std::integral_constant;
            if (runs || KT == 2) {
                products(integral_constant<int, 0>{}, integral_constant<int, KT>{}, c & 1, wf, sc[0], side);
            } else if constexpr (KT == 4) {  // (groups of 32, 96, ...: two steps each at least)
                products(integral_constant<int, 0>{}, integral_constant<int, 2>{}, c & 1, wf, sc[0], side);
                products(integral_constant<int, 2>{}, integral_constant<int, 4>{}, c & 1, wf, sc[1], [](int, int) {});
            }
        }
    }

#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int64_t v = v0 + 32 * j + r32;
        if (v >= a.V) continue;
        const float sc = (FMT != kLhF32 && !grouped) ? a.scales[v] : 1.0f;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t b = b0 + 32 * i + 8 * (r >> 2) + 4 * q + (r & 3);
                if (b < a.B) {
                    float y = tot[i][j][r];
                    if (FMT != kLhF32) y *= sc;  // dot * scale (quant.rs:128)
                    if (!(fabsf(y) < INFINITY)) {
                        y = ls_plain<FMT>(a, b, v);
                        if (FMT != kLhF32) y *= sc;
                    }
                    a.out[b * a.ld + v] = y;
                }
            }
    }
}

}  // namespace nis
