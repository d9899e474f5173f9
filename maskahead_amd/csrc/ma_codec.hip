// Packed-KV codec kernels: whole-prefix dequant, gather of selected entries, and the
// 4-bit quantizers of the append path.  All integer/byte work, bit-exact against the
// reference's torch codec (reference.py:35-268).
#include <algorithm>

#include "ma_common.h"
#include "ma_quant.h"

namespace {

constexpr int KG = 32;  // key token group (the only one shipped configs use)
constexpr int VG = 32;  // value channel group

struct PrefixArgs {
    const uint8_t *kq;
    const uint16_t *ks, *kz;
    const uint8_t *vq;
    const uint16_t *vs, *vz;
    const void *kf, *vf;
    int64_t skq[4], sks[3], svq[4], svs[3], skf[3], svf[3];
    int nq, nf, fdtype;
};

PrefixArgs make_args(const ma_prefix *p) {
    PrefixArgs a;
    a.kq = (const uint8_t *)p->kq;
    a.ks = (const uint16_t *)p->ks;
    a.kz = (const uint16_t *)p->kz;
    a.vq = (const uint8_t *)p->vq;
    a.vs = (const uint16_t *)p->vs;
    a.vz = (const uint16_t *)p->vz;
    a.kf = p->kf;
    a.vf = p->vf;
    for (int i = 0; i < 4; ++i) {
        a.skq[i] = p->skq[i];
        a.svq[i] = p->svq[i];
    }
    for (int i = 0; i < 3; ++i) {
        a.sks[i] = p->sks[i];
        a.svs[i] = p->svs[i];
        a.skf[i] = p->skf[i];
        a.svf[i] = p->svf[i];
    }
    a.nq = p->nq;
    a.nf = p->nf;
    a.fdtype = p->fdtype;
    return a;
}

// ---------------------------------------------------------------- dequant_prefix
// Grid (tiles of DQ_TOK tokens, B*H, 2): keys (z = 0) or values (z = 1) of a tile.  Bound by
// bytes, nearly all of them the rows it writes, so every store instruction writes whole rows:
//   packed keys    thread = 8 channels of 8 tokens of a key group: a code word per channel
//                  in, 8 values per token out, D/8 threads a row; groups start at different
//                  tokens, or every wave would be writing at the same offset of an 8 KB
//                  stride, into the same memory channels
//   packed values  thread = 8 channels of a token: a code word in, 8 values out, D/8 a row
//   16-bit part    thread = 8 channels of a token, converted
// 8 192 tokens x 4 heads of D 128 to f16, 22 MB: 10.3 us cold, 6.3 repeated; 35.3 cold with
// stores of one element.
constexpr int DQ_TOK = 128, DQ_VB = 8;

// x or y, by value (`c ? x : y` on two fields of the kernel's arguments selects an address,
// which puts the whole argument struct in scratch memory)
template <class T>
__device__ __forceinline__ T pick(bool c, T x, T y) {
    return c ? x : y;
}

// 8 consecutive values at element `off` of an output of dtype DT
template <int DT, bool VEC>
__device__ __forceinline__ void put8(void *base, int64_t off, const float (&x)[8]) {
    if constexpr (!VEC) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ma_store_f(base, off + i, DT, x[i]);
    } else if constexpr (DT == MA_F32) {
        typedef __attribute__((ext_vector_type(4))) float f32x4;
#pragma unroll
        for (int i = 0; i < 8; i += 4) *(f32x4 *)((float *)base + off + i) = f32x4{x[i], x[i + 1], x[i + 2], x[i + 3]};
    } else {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (DT == MA_BF16) {
                w[i] = ma_pack_bf16x2(x[2 * i], x[2 * i + 1]);
            } else {
                w[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x[2 * i]) |
                       ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x[2 * i + 1]) << 16);
            }
        }
        *(uint4 *)((uint16_t *)base + off) = uint4{w[0], w[1], w[2], w[3]};
    }
}

template <int DT, bool VEC>
__device__ __forceinline__ void dequant_tile(const PrefixArgs &a, int b, int h, int D, void *out, int64_t ob,
                                             int64_t on, int kv, int t0) {
    const int n = a.nq + a.nf;
    const int q1 = min(t0 + DQ_TOK, a.nq);   // packed tokens [t0, q1) of the tile
    if (kv == 0) {
        const int tpt = D / 8, d = (threadIdx.x % tpt) * 8;
        for (int i = threadIdx.x / tpt; t0 + i * 8 < q1; i += 256 / tpt) {
            const int g = t0 / KG + i / 4, o = i % 4;   // tokens 8o .. 8o + 7 of group g
            const uint8_t *row = a.kq + b * a.skq[0] + h * a.skq[1] + (int64_t)g * a.skq[2] +
                                 (int64_t)d * a.skq[3] + o * 4;
            uint32_t w[8];
            uint16_t sc[8], zp[8];
            const int64_t so = b * a.sks[0] + h * a.sks[1] + (int64_t)g * a.sks[2] + d;
#pragma unroll
            for (int c = 0; c < 8; ++c) w[c] = *(const uint32_t *)(row + c * a.skq[3]);
#pragma unroll
            for (int c = 0; c < 8; c += 2) {
                const uint32_t s2 = *(const uint32_t *)(a.ks + so + c), z2 = *(const uint32_t *)(a.kz + so + c);
                sc[c] = (uint16_t)s2;
                sc[c + 1] = (uint16_t)(s2 >> 16);
                zp[c] = (uint16_t)z2;
                zp[c + 1] = (uint16_t)(z2 >> 16);
            }
            const int64_t og = ob + (int64_t)(g * KG + o * 8) * on + d;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int tr = (t + g) & 7;
                float x[8];
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    x[c] = ma_dq((w[c] >> (tr * 4)) & 15u, ma_f16_to_f32(sc[c]), ma_f16_to_f32(zp[c]));
                put8<DT, VEC>(out, og + tr * on, x);
            }
        }
    } else {
        // DQ_VB tokens' loads in flight together (tokens past the end read the last one)
        const int tpt = D / 8, per = 256 / tpt, oct = threadIdx.x % tpt;
        const uint8_t *vq = a.vq + b * a.svq[0] + h * a.svq[1] + (int64_t)(oct / 4) * a.svq[3] + (oct % 4) * 4;
        const int64_t so = b * a.svs[0] + h * a.svs[1] + oct / 4;
        for (int j0 = t0 + threadIdx.x / tpt; j0 < q1; j0 += DQ_VB * per) {
            uint32_t w[DQ_VB];
            uint16_t sc[DQ_VB], zp[DQ_VB];
#pragma unroll
            for (int u = 0; u < DQ_VB; ++u) {
                const int j = min(j0 + u * per, q1 - 1);
                w[u] = *(const uint32_t *)(vq + (int64_t)j * a.svq[2]);
                sc[u] = a.vs[so + (int64_t)j * a.svs[2]];
                zp[u] = a.vz[so + (int64_t)j * a.svs[2]];
            }
#pragma unroll
            for (int u = 0; u < DQ_VB; ++u) {
                const int j = j0 + u * per;
                float x[8];
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    x[c] = ma_dq((w[u] >> (4 * c)) & 15u, ma_f16_to_f32(sc[u]), ma_f16_to_f32(zp[u]));
                if (j < q1) put8<DT, VEC>(out, ob + (int64_t)j * on + oct * 8, x);
            }
        }
    }
    // 16-bit part (residual tail, or the whole prefix of a bf16 cache)
    const void *src = pick(kv, a.vf, a.kf);
    const int64_t s0 = pick(kv, a.svf[0], a.skf[0]), s1 = pick(kv, a.svf[1], a.skf[1]),
                  s2 = pick(kv, a.svf[2], a.skf[2]);
    const int tpt = D / 8, oct = threadIdx.x % tpt;
    for (int j = max(t0, a.nq) + threadIdx.x / tpt; j < min(t0 + DQ_TOK, n); j += 256 / tpt) {
        const int64_t so = b * s0 + h * s1 + (int64_t)(j - a.nq) * s2 + oct * 8;
        float x[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) x[c] = ma_load_f(src, so + c, a.fdtype);
        put8<DT, VEC>(out, ob + (int64_t)j * on + oct * 8, x);
    }
}

template <bool VEC>
__global__ void __launch_bounds__(256) dequant_prefix_kernel(PrefixArgs a, int H, int D, ma_tensor4 ko,
                                                             ma_tensor4 vo) {
    const int b = blockIdx.y / H, h = blockIdx.y % H, kv = blockIdx.z, t0 = blockIdx.x * DQ_TOK;
    void *out = pick(kv, vo.ptr, ko.ptr);
    const int dtype = pick(kv, vo.dtype, ko.dtype);
    const int64_t ob = b * pick(kv, vo.s[0], ko.s[0]) + h * pick(kv, vo.s[1], ko.s[1]), on = pick(kv, vo.s[2], ko.s[2]);
    if (dtype == MA_BF16) dequant_tile<MA_BF16, VEC>(a, b, h, D, out, ob, on, kv, t0);
    else if (dtype == MA_F16) dequant_tile<MA_F16, VEC>(a, b, h, D, out, ob, on, kv, t0);
    else dequant_tile<MA_F32, VEC>(a, b, h, D, out, ob, on, kv, t0);
}

// ---------------------------------------------------------------- gather
// grid (ceil(k / TPB_TOK), B*H), 256 threads; D/4 threads per selected entry, 4
// channels each.  Indices outside [0, n) produce zeros (never an out-of-bounds read).
// vec: the 4 key scales / zeros of a thread are one 8-byte load each and bf16 outputs are
// written 8 bytes at a time (the host checks the alignment this needs).
__global__ void __launch_bounds__(256) gather_kernel(PrefixArgs a, int H, int D, const int64_t *idx, int64_t sib,
                                                     int64_t sih, int k, ma_tensor4 ko, ma_tensor4 vo, int vec) {
    const int bh = blockIdx.y, b = bh / H, h = bh % H;
    const int tpt = D / 4;               // threads per token
    const int toks = 256 / tpt;
    const int i = blockIdx.x * toks + threadIdx.x / tpt;
    const int c0 = (threadIdx.x % tpt) * 4;
    if (i >= k) return;
    const int n = a.nq + a.nf;
    const int64_t j64 = idx[b * sib + h * sih + i];
    float kx[4] = {0.f, 0.f, 0.f, 0.f}, vx[4] = {0.f, 0.f, 0.f, 0.f};
    if (j64 >= 0 && j64 < n) {
        const int j = (int)j64;
        if (j < a.nq) {
            const int g = j / KG, tt = j % KG;
            const uint8_t *krow = a.kq + b * a.skq[0] + h * a.skq[1] + (int64_t)g * a.skq[2] + (int64_t)c0 * a.skq[3];
            uint32_t kb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) kb[e] = krow[(int64_t)e * a.skq[3] + (tt >> 1)];
            const int64_t so = b * a.sks[0] + h * a.sks[1] + (int64_t)g * a.sks[2] + c0;
            uint16_t ks[4], kz[4];
            if (vec) {
                const uint2 sv = *(const uint2 *)&a.ks[so], zv = *(const uint2 *)&a.kz[so];
                ks[0] = sv.x & 0xffffu; ks[1] = sv.x >> 16; ks[2] = sv.y & 0xffffu; ks[3] = sv.y >> 16;
                kz[0] = zv.x & 0xffffu; kz[1] = zv.x >> 16; kz[2] = zv.y & 0xffffu; kz[3] = zv.y >> 16;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ks[e] = a.ks[so + e];
                    kz[e] = a.kz[so + e];
                }
            }
            const int cg = c0 / VG, w = c0 % VG;
            const uint8_t *src = a.vq + b * a.svq[0] + h * a.svq[1] + (int64_t)j * a.svq[2] + (int64_t)cg * a.svq[3];
            const uint32_t two = (uint32_t)src[w >> 1] | ((uint32_t)src[(w >> 1) + 1] << 8);
            const int64_t vso = b * a.svs[0] + h * a.svs[1] + (int64_t)j * a.svs[2] + cg;
            const float vsc = ma_f16_to_f32(a.vs[vso]), vzp = ma_f16_to_f32(a.vz[vso]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t code = (tt & 1) ? (kb[e] >> 4) : (kb[e] & 15u);
                kx[e] = ma_dq(code, ma_f16_to_f32(ks[e]), ma_f16_to_f32(kz[e]));
                vx[e] = ma_dq((two >> (4 * e)) & 15u, vsc, vzp);
            }
        } else {
            const int jf = j - a.nq;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                kx[e] = ma_load_f(a.kf, b * a.skf[0] + h * a.skf[1] + (int64_t)jf * a.skf[2] + c0 + e, a.fdtype);
                vx[e] = ma_load_f(a.vf, b * a.svf[0] + h * a.svf[1] + (int64_t)jf * a.svf[2] + c0 + e, a.fdtype);
            }
        }
    }
    const int64_t ok = b * ko.s[0] + h * ko.s[1] + (int64_t)i * ko.s[2] + c0;
    const int64_t ov = b * vo.s[0] + h * vo.s[1] + (int64_t)i * vo.s[2] + c0;
    if (vec && ko.dtype == MA_BF16 && vo.dtype == MA_BF16) {
        uint2 kw, vw;
        kw.x = (uint32_t)ma_f32_to_bf16(kx[0]) | ((uint32_t)ma_f32_to_bf16(kx[1]) << 16);
        kw.y = (uint32_t)ma_f32_to_bf16(kx[2]) | ((uint32_t)ma_f32_to_bf16(kx[3]) << 16);
        vw.x = (uint32_t)ma_f32_to_bf16(vx[0]) | ((uint32_t)ma_f32_to_bf16(vx[1]) << 16);
        vw.y = (uint32_t)ma_f32_to_bf16(vx[2]) | ((uint32_t)ma_f32_to_bf16(vx[3]) << 16);
        *(uint2 *)((uint16_t *)ko.ptr + ok) = kw;
        *(uint2 *)((uint16_t *)vo.ptr + ov) = vw;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            ma_store_f(ko.ptr, ok + e, ko.dtype, kx[e]);
            ma_store_f(vo.ptr, ov + e, vo.dtype, vx[e]);
        }
    }
}

// Rows of a 16-bit prefix into outputs of the same dtype: copied as they are, 16 bytes a
// thread, D/8 threads a row, GR_ROWS rows of K and V in flight per thread.  Bound by bytes:
// 8 192 of 65 536 rows of 32 lanes (D 128, 268 MB) took 94.9 us through gather_kernel's
// element loads.
constexpr int GR_ROWS = 4;
template <int D>
__global__ void __launch_bounds__(256) gather_rows_kernel(PrefixArgs a, int H, const int64_t *idx, int64_t sib,
                                                          int64_t sih, int k, ma_tensor4 ko, ma_tensor4 vo) {
    constexpr int TPT = D / 8, PER = 256 / TPT;
    const int b = blockIdx.y / H, h = blockIdx.y % H;
    const int c0 = (threadIdx.x % TPT) * 8;
    const int i0 = blockIdx.x * PER * GR_ROWS + threadIdx.x / TPT;
    const int64_t *ix = idx + b * sib + h * sih;
    int64_t j[GR_ROWS];
#pragma unroll
    for (int u = 0; u < GR_ROWS; ++u) j[u] = ix[min(i0 + u * PER, k - 1)];
    const uint16_t *ks = (const uint16_t *)a.kf + b * a.skf[0] + h * a.skf[1] + c0;
    const uint16_t *vs = (const uint16_t *)a.vf + b * a.svf[0] + h * a.svf[1] + c0;
    uint4 kw[GR_ROWS], vw[GR_ROWS];
#pragma unroll
    for (int u = 0; u < GR_ROWS; ++u) {   // an index outside the prefix reads row 0 and gives zeros
        const bool ok = j[u] >= 0 && j[u] < a.nf;
        const int64_t r = ok ? j[u] : 0;
        kw[u] = *(const uint4 *)(ks + r * a.skf[2]);
        vw[u] = *(const uint4 *)(vs + r * a.svf[2]);
    }
    uint16_t *kd = (uint16_t *)ko.ptr + b * ko.s[0] + h * ko.s[1] + c0;
    uint16_t *vd = (uint16_t *)vo.ptr + b * vo.s[0] + h * vo.s[1] + c0;
#pragma unroll
    for (int u = 0; u < GR_ROWS; ++u) {
        const int i = i0 + u * PER;
        if (i >= k) break;
        const bool ok = j[u] >= 0 && j[u] < a.nf;
        *(uint4 *)(kd + (int64_t)i * ko.s[2]) = ok ? kw[u] : uint4{0u, 0u, 0u, 0u};
        *(uint4 *)(vd + (int64_t)i * vo.s[2]) = ok ? vw[u] : uint4{0u, 0u, 0u, 0u};
    }
}

// ---------------------------------------------------------------- quantizers
// The source of a quantizer: token rows 0 .. na-1 from `a`, the rest from `b` (row i - na)
// -- [residual | new tokens] of an append without building that tensor; na = 0 reads `b`
// alone.  a and b have the same dtype.
struct TwoSrc {
    ma_tensor4 a, b;
    int na;
};

// One append in one launch.  kv 0 = keys, 1 = values; a workgroup
// belongs to one (lane, kv) and is one of
//   head  the residual rows and, before a barrier, the key groups (the first gh) that read
//         what these replace: in place, so one workgroup does both
//   bulk  BULK tokens of the other groups
//   copy  COPY residual rows where nothing that is overwritten is read (na = 0: the rows of
//         `a` are free; move = 0: its rows stay and `b`'s follow them)
// What bounds it: a block's append (32 residual + 32 new tokens, 4 lanes of D 128) is one
// load-to-store latency, 6.4 us; an 8 192-token prompt's is latency and the quantizer's VALU
// work (about 13 operations a value, 3.4 us of it), 12.3 us for 22 MB.  As three launches --
// two quantizers with 2-byte loads, and two workgroups a lane copying the residual an
// element at a time -- they took 28.1 and 34.4 us, 20 us of each the residual's copy.
// A residual far longer than what is kept of it (blocks staged unquantized, then quantized) is
// mostly bulk: 2 048 rows 64.1 -> 8.2 us, 8 192 rows 246.9 -> 11.3, with every group that reads
// `a` in the head.
constexpr int AP_NT = 256;
constexpr int BULK = 128;     // tokens of a bulk workgroup: a key group per wave at D = 128
constexpr int COPY = 64;      // rows of a copy workgroup, and of a head's pass

struct AppendArgs {
    TwoSrc src[2];
    uint8_t *q[2];
    int64_t sq[2][4];
    _Float16 *s[2], *z[2];
    int64_t ss[2][3];
    int H, D, lanes;
    int ntok;                    // tokens quantized
    int keep, first;             // residual rows [first, keep) written from source rows r + ntok
    int gh, nhead, nbulk;        // head groups; head (0 or 1) and bulk workgroups per (lane, kv)
};

// the source rows of one lane
struct RowSrc {
    const char *a, *b;
    int64_t sa, sb;   // bytes per row
    int na;
};

template <int DT>
__device__ __forceinline__ RowSrc row_src(const TwoSrc &s, int b, int h) {
    constexpr int ES = DT == MA_F32 ? 4 : 2;
    RowSrc r;
    r.a = (const char *)s.a.ptr + (b * s.a.s[0] + h * s.a.s[1]) * ES;
    r.b = (const char *)s.b.ptr + (b * s.b.s[0] + h * s.b.s[1]) * ES;
    r.sa = s.a.s[2] * ES;
    r.sb = s.b.s[2] * ES;
    r.na = s.na;
    return r;
}

__device__ __forceinline__ const char *src_row(const RowSrc &r, int i) {
    return i < r.na ? r.a + i * r.sa : r.b + (int64_t)(i - r.na) * r.sb;
}

// N consecutive elements at p as f32; VEC: p is aligned to N elements
template <int DT, int N, bool VEC>
__device__ __forceinline__ void load_n(const char *p, float (&x)[N]) {
    if constexpr (!VEC) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = ma_load_f(p, i, DT);
    } else if constexpr (DT == MA_F32) {
        typedef __attribute__((ext_vector_type(N < 4 ? N : 4))) float fv;
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const fv v = *(const fv *)(p + 4 * i);
#pragma unroll
            for (int e = 0; e < (N < 4 ? N : 4); ++e) x[i + e] = v[e];
        }
    } else {
        typedef __attribute__((ext_vector_type(N / 2))) uint32_t uv;
        uint32_t w[N / 2];
        if constexpr (N == 2) {
            w[0] = *(const uint32_t *)p;
        } else {
            const uv v = *(const uv *)p;
#pragma unroll
            for (int i = 0; i < N / 2; ++i) w[i] = v[i];
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint16_t h = (uint16_t)(w[i / 2] >> ((i & 1) * 16));
            x[i] = DT == MA_BF16 ? ma_bf16_to_f32(h) : ma_f16_to_f32(h);
        }
    }
}

// key groups g0, g0 + step, ... below g1 of one lane: thread c of a group's D / 2 = two
// channels of its 32 tokens, all loads in flight, no exchange between threads
template <int DT, bool VEC>
__device__ __forceinline__ void quant_keys(const AppendArgs &A, const RowSrc &R, int b, int h, int g0, int g1) {
    const int tpg = A.D / 2;
    const int d = (threadIdx.x % tpg) * 2;
    constexpr int ES = DT == MA_F32 ? 4 : 2;
    for (int g = g0 + threadIdx.x / tpg; g < g1; g += AP_NT / tpg) {
        float x[KG][2];
        float lo[2] = {INFINITY, INFINITY}, hi[2] = {-INFINITY, -INFINITY};
#pragma unroll
        for (int t = 0; t < KG; ++t) load_n<DT, 2, VEC>(src_row(R, g * KG + t) + d * ES, x[t]);
#pragma unroll
        for (int t = 0; t < KG; ++t)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                lo[c] = fminf(lo[c], x[t][c]);
                hi[c] = fmaxf(hi[c], x[t][c]);
            }
        const int64_t so = b * A.ss[0][0] + h * A.ss[0][1] + (int64_t)g * A.ss[0][2] + d;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const QuantGroup qp = quant_params(lo[c], hi[c], DT);
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < KG; ++t) w[t >> 3] |= quant_code(x[t][c], qp, DT) << ((t & 7) * 4);
            *(uint4 *)(A.q[0] + b * A.sq[0][0] + h * A.sq[0][1] + (int64_t)g * A.sq[0][2] +
                       (int64_t)(d + c) * A.sq[0][3]) = uint4{w[0], w[1], w[2], w[3]};
            A.s[0][so + c] = (_Float16)qp.step;
            A.z[0][so + c] = (_Float16)qp.lo;
        }
    }
}

// value tokens [t0, t1) of one lane: thread = 8 channels of a token, a group's range from
// its 4 adjacent threads; VB tokens' loads in flight per thread
template <int DT, bool VEC>
__device__ __forceinline__ void quant_values(const AppendArgs &A, const RowSrc &R, int b, int h, int t0, int t1) {
    constexpr int VB = 4;
    constexpr int ES = DT == MA_F32 ? 4 : 2;
    const int tpt = A.D / 8, per = AP_NT / tpt;
    const int oct = threadIdx.x % tpt, cg = oct / 4;
    for (int j0 = t0 + threadIdx.x / tpt; j0 < t1; j0 += VB * per) {
        float x[VB][8];
#pragma unroll
        for (int u = 0; u < VB; ++u)   // tokens past the end read the last one and are not written
            load_n<DT, 8, VEC>(src_row(R, min(j0 + u * per, t1 - 1)) + oct * 8 * ES, x[u]);
#pragma unroll
        for (int u = 0; u < VB; ++u) {
            const int j = j0 + u * per;
            float lo = x[u][0], hi = x[u][0];
#pragma unroll
            for (int c = 1; c < 8; ++c) {
                lo = fminf(lo, x[u][c]);
                hi = fmaxf(hi, x[u][c]);
            }
            lo = fminf(lo, ma_quad<0xB1>(lo));   // lanes ^ 1, then ^ 2
            lo = fminf(lo, ma_quad<0x4E>(lo));
            hi = fmaxf(hi, ma_quad<0xB1>(hi));
            hi = fmaxf(hi, ma_quad<0x4E>(hi));
            const QuantGroup qp = quant_params(fminf(INFINITY, lo), fmaxf(-INFINITY, hi), DT);
            uint32_t w = 0;
#pragma unroll
            for (int c = 0; c < 8; ++c) w |= quant_code(x[u][c], qp, DT) << (c * 4);
            if (j < t1) {
                *(uint32_t *)(A.q[1] + b * A.sq[1][0] + h * A.sq[1][1] + (int64_t)j * A.sq[1][2] +
                              (int64_t)cg * A.sq[1][3] + (oct % 4) * 4) = w;
                const int64_t so = b * A.ss[1][0] + h * A.ss[1][1] + (int64_t)j * A.ss[1][2] + cg;
                if (oct % 4 == 0) A.s[1][so] = (_Float16)qp.step;
                if (oct % 4 == 1) A.z[1][so] = (_Float16)qp.lo;
            }
        }
    }
}

// A pass of at most COPY residual rows, from r0: the loads, then (after whatever must come
// between) the stores.  A thread holds 8 elements of a row.
template <int DT, bool VEC>
struct ResidualPass {
    static constexpr int ES = DT == MA_F32 ? 4 : 2, NW = 2 * ES;
    static constexpr int MAXR = COPY * 256 / 8 / AP_NT;   // rows per thread at the largest D (256)
    uint32_t w[MAXR][NW];

    __device__ __forceinline__ void load(const AppendArgs &A, const RowSrc &R, int r0) {
        const int tpt = A.D / 8, per = AP_NT / tpt, oct = threadIdx.x % tpt, rt = threadIdx.x / tpt;
#pragma unroll
        for (int e = 0; e < MAXR; ++e) {
            const int r = r0 + rt + e * per;
            if (e * per < COPY && r < A.keep) {
                const char *p = src_row(R, r + A.ntok) + oct * 8 * ES;
                if constexpr (VEC) {
#pragma unroll
                    for (int i = 0; i < NW; i += 4) {
                        const uint4 v = *(const uint4 *)(p + 4 * i);
                        w[e][i] = v.x;
                        w[e][i + 1] = v.y;
                        w[e][i + 2] = v.z;
                        w[e][i + 3] = v.w;
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < NW; ++i)
                        w[e][i] = ES == 4 ? *(const uint32_t *)(p + 4 * i)
                                          : (uint32_t) * (const uint16_t *)(p + 4 * i) |
                                                ((uint32_t) * (const uint16_t *)(p + 4 * i + 2) << 16);
                }
            }
        }
    }
    __device__ __forceinline__ void store(const AppendArgs &A, const RowSrc &R, int r0) {
        const int tpt = A.D / 8, per = AP_NT / tpt, oct = threadIdx.x % tpt, rt = threadIdx.x / tpt;
#pragma unroll
        for (int e = 0; e < MAXR; ++e) {
            const int r = r0 + rt + e * per;
            if (e * per < COPY && r < A.keep) {
                char *p = (char *)R.a + r * R.sa + oct * 8 * ES;
                if constexpr (VEC) {
#pragma unroll
                    for (int i = 0; i < NW; i += 4)
                        *(uint4 *)(p + 4 * i) = uint4{w[e][i], w[e][i + 1], w[e][i + 2], w[e][i + 3]};
                } else {
#pragma unroll
                    for (int i = 0; i < NW; ++i) {
                        if constexpr (ES == 4) {
                            *(uint32_t *)(p + 4 * i) = w[e][i];
                        } else {
                            *(uint16_t *)(p + 4 * i) = (uint16_t)w[e][i];
                            *(uint16_t *)(p + 4 * i + 2) = (uint16_t)(w[e][i] >> 16);
                        }
                    }
                }
            }
        }
    }
};

template <int DT, bool VEC>
__global__ void __launch_bounds__(AP_NT) append_packed_kernel(AppendArgs A) {
    const int units = A.lanes * 2;
    const int u = blockIdx.x / units, y = blockIdx.x % units;
    const int kv = y / A.lanes, bh = y % A.lanes, b = bh / A.H, h = bh % A.H;
    const RowSrc R = row_src<DT>(A.src[kv], b, h);
    ResidualPass<DT, VEC> pass;
    if (u < A.nhead) {
        // the residual's first rows are on their way while the groups are quantized; nothing
        // is stored to `a` before every thread has read what it needs of it
        pass.load(A, R, A.first);
        if (kv == 0) quant_keys<DT, VEC>(A, R, b, h, 0, A.gh);
        else quant_values<DT, VEC>(A, R, b, h, 0, A.gh * KG);
        __syncthreads();
        pass.store(A, R, A.first);
        // further rows, each pass read whole before any of it is written: its destinations lie
        // below the sources of every later pass
        for (int r0 = A.first + COPY; r0 < A.keep; r0 += COPY) {
            __syncthreads();
            pass.load(A, R, r0);
            __syncthreads();
            pass.store(A, R, r0);
        }
    } else if (u < A.nhead + A.nbulk) {
        const int t0 = A.gh * KG + (u - A.nhead) * BULK, t1 = min(t0 + BULK, A.ntok);
        if (kv == 0) quant_keys<DT, VEC>(A, R, b, h, t0 / KG, t1 / KG);
        else quant_values<DT, VEC>(A, R, b, h, t0, t1);
    } else {
        const int r0 = A.first + (u - A.nhead - A.nbulk) * COPY;
        pass.load(A, R, r0);
        pass.store(A, R, r0);
    }
}

// Fills in the workgroups of an append of ntok quantized tokens and residual rows
// [first, keep), and launches it (D divides 256 and is a multiple of 32).
int launch_append(AppendArgs &A, int dtype, hipStream_t st, const char *who) {
    const int na = A.src[0].na;
    // the residual replaces rows that are read: those of quantized groups below row `keep`, and
    // its own (rows of `a` from `keep` on are written by nobody)
    const bool in_place = A.ntok > 0 && na > 0 && A.keep > 0;
    A.gh = in_place ? std::min((std::min(na, A.keep) + KG - 1) / KG, A.ntok / KG) : 0;
    A.nhead = in_place ? 1 : 0;
    A.nbulk = (A.ntok - A.gh * KG + BULK - 1) / BULK;
    const int ncopy = in_place ? 0 : std::max(0, (A.keep - A.first + COPY - 1) / COPY);
    const int64_t wgs = (int64_t)(A.nhead + A.nbulk + ncopy) * A.lanes * 2;
    if (wgs == 0) return MA_OK;
    // 16-byte loads and stores: aligned bases and rows of whole 16-byte pieces
    bool vec = true;
    for (int kv = 0; kv < 2; ++kv) {
        const ma_tensor4 *ts[2] = {&A.src[kv].a, &A.src[kv].b};
        for (const ma_tensor4 *t : ts) {
            const int64_t m = dtype == MA_F32 ? 4 : 8;
            if (t->ptr && (((uintptr_t)t->ptr & 15) || t->s[0] % m || t->s[1] % m || t->s[2] % m)) vec = false;
        }
    }
    const dim3 grid((unsigned)wgs);
#define MA_APPEND(DT_)                                                                                           \
    do {                                                                                                         \
        if (vec) hipLaunchKernelGGL((append_packed_kernel<DT_, true>), grid, dim3(AP_NT), 0, st, A);             \
        else hipLaunchKernelGGL((append_packed_kernel<DT_, false>), grid, dim3(AP_NT), 0, st, A);                \
    } while (0)
    if (dtype == MA_BF16) MA_APPEND(MA_BF16);
    else if (dtype == MA_F16) MA_APPEND(MA_F16);
    else MA_APPEND(MA_F32);
#undef MA_APPEND
    return ma_check_launch(who);
}

// ---- the quantizers alone (append_packed_kernel serves appends).  Bound by latency up to a few
// thousand tokens: 4 heads of D 128 x 8 192, keys 5.1 us and values 5.1 (7.2 and 6.8 as a launch
// of that kernel, whose workgroups are fewer and hold a residual pass's registers); 512 tokens
// 4.6 and 4.2 (6.6 and 6.4), 32 768 12.0 and 12.0 (14.5 and 15.6), D 256 x 512 5.0 and 4.0 (10.0
// and 9.8).
// DT: the dtype, a compile-time constant so that a thread's loads are straight-line code
// (all of them in flight at once) instead of one branch per element
// keys: a workgroup of D threads a token group; thread = one channel of it.
template <int DT>
__global__ void quantize_keys_kernel(ma_tensor4 src, int ng, int H, int D, uint8_t *kq, int64_t q0, int64_t q1,
                                     int64_t q2, int64_t q3, _Float16 *ks, _Float16 *kz, int64_t s0, int64_t s1,
                                     int64_t s2) {
    const int bh = blockIdx.x / ng, b = bh / H, h = bh % H;
    const int g = blockIdx.x % ng;
    const int d = threadIdx.x;
    if (d >= D) return;
    float x[KG];
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int t = 0; t < KG; ++t) {
        x[t] = ma_load_f(src.ptr, b * src.s[0] + h * src.s[1] + (int64_t)(g * KG + t) * src.s[2] + d, DT);
        lo = fminf(lo, x[t]);
        hi = fmaxf(hi, x[t]);
    }
    QuantGroup qp = quant_params(lo, hi, DT);
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < KG; ++t) w[t >> 3] |= quant_code(x[t], qp, DT) << ((t & 7) * 4);
    uint4 out = {w[0], w[1], w[2], w[3]};
    *(uint4 *)(kq + b * q0 + h * q1 + (int64_t)g * q2 + (int64_t)d * q3) = out;
    int64_t so = b * s0 + h * s1 + (int64_t)g * s2 + d;
    ks[so] = (_Float16)qp.step;
    kz[so] = (_Float16)qp.lo;
}

// values: one thread per (token, channel group); grid-stride over B*H*T*(D/VG) items.
template <int DT>
__global__ void __launch_bounds__(256) quantize_values_kernel(ma_tensor4 src, int BH, int H, int T, int D,
                                                              uint8_t *vq, int64_t q0, int64_t q1, int64_t q2,
                                                              int64_t q3, _Float16 *vs, _Float16 *vz, int64_t s0,
                                                              int64_t s1, int64_t s2) {
    const int ncg = D / VG;
    const int64_t total = (int64_t)BH * T * ncg;
    for (int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x; it < total; it += (int64_t)gridDim.x * 256) {
        int cg = (int)(it % ncg);
        int64_t rest = it / ncg;
        int j = (int)(rest % T);
        int bh = (int)(rest / T), b = bh / H, h = bh % H;
        float x[VG];
        float lo = INFINITY, hi = -INFINITY;
#pragma unroll
        for (int c = 0; c < VG; ++c) {
            x[c] = ma_load_f(src.ptr, b * src.s[0] + h * src.s[1] + (int64_t)j * src.s[2] + cg * VG + c, DT);
            lo = fminf(lo, x[c]);
            hi = fmaxf(hi, x[c]);
        }
        QuantGroup qp = quant_params(lo, hi, DT);
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < VG; ++c) w[c >> 3] |= quant_code(x[c], qp, DT) << ((c & 7) * 4);
        uint4 out = {w[0], w[1], w[2], w[3]};
        *(uint4 *)(vq + b * q0 + h * q1 + (int64_t)j * q2 + (int64_t)cg * q3) = out;
        int64_t so = b * s0 + h * s1 + (int64_t)j * s2 + cg;
        vs[so] = (_Float16)qp.step;
        vz[so] = (_Float16)qp.lo;
    }
}

// the head dims whose rows the append kernel's 256 threads share evenly
bool append_dim(int D) { return D > 0 && D % VG == 0 && D <= AP_NT && AP_NT % D == 0; }

}  // namespace

// ---------------------------------------------------------------- validation helpers
int ma_validate_prefix(const ma_prefix *p, int D, const char *who) {
    if (!p) {
        ma_set_error("%s: prefix is NULL", who);
        return MA_EINVAL;
    }
    if (D != 64 && D != 128) {
        ma_set_error("%s: head_dim %d not built (64, 128)", who, D);
        return MA_EUNSUPPORTED;
    }
    if (p->nq < 0 || p->nf < 0) {
        ma_set_error("%s: negative prefix length", who);
        return MA_EINVAL;
    }
    if (p->nq > 0) {
        if (p->kbits != 4 || p->vbits != 4) {
            ma_set_error("%s: packed bit widths k=%d v=%d not built (4/4)", who, p->kbits, p->vbits);
            return MA_EUNSUPPORTED;
        }
        if (p->kgroup != KG || p->vgroup != VG) {
            ma_set_error("%s: groups k=%d v=%d not built (32/32)", who, p->kgroup, p->vgroup);
            return MA_EUNSUPPORTED;
        }
        if (p->nq % KG) {
            ma_set_error("%s: quantized length %d is not a multiple of %d", who, p->nq, KG);
            return MA_EINVAL;
        }
        if (!p->kq || !p->ks || !p->kz || !p->vq || !p->vs || !p->vz) {
            ma_set_error("%s: packed prefix pointers missing", who);
            return MA_EINVAL;
        }
        if ((((uintptr_t)p->kq | (uintptr_t)p->vq) & 15) || ((p->skq[2] | p->skq[3] | p->svq[2] | p->svq[3]) & 15)) {
            ma_set_error("%s: packed payload rows must be 16-byte aligned", who);
            return MA_EINVAL;
        }
        // key scale/zero are read as f16 pairs (two channels per 32-bit load)
        if ((((uintptr_t)p->ks | (uintptr_t)p->kz) & 3) || ((p->sks[0] | p->sks[1] | p->sks[2]) & 1)) {
            ma_set_error("%s: key scale/zero must be 4-byte aligned with even strides", who);
            return MA_EINVAL;
        }
    }
    if (p->nf > 0) {
        if (!p->kf || !p->vf) {
            ma_set_error("%s: 16-bit prefix pointers missing", who);
            return MA_EINVAL;
        }
        if (p->fdtype != MA_BF16 && p->fdtype != MA_F16 && p->fdtype != MA_F32) {
            ma_set_error("%s: bad prefix dtype %d", who, p->fdtype);
            return MA_EINVAL;
        }
    }
    return MA_OK;
}

static bool out_dtype_ok(int dt) { return dt == MA_BF16 || dt == MA_F32 || dt == MA_F16; }

extern "C" int ma_dequant_prefix(const ma_prefix *p, int B, int H, int D, ma_tensor4 k_out, ma_tensor4 v_out,
                                 void *stream) {
    int rc = ma_validate_prefix(p, D, "ma_dequant_prefix");
    if (rc) return rc;
    if (B <= 0 || H <= 0 || !k_out.ptr || !v_out.ptr || !out_dtype_ok(k_out.dtype) || !out_dtype_ok(v_out.dtype)) {
        ma_set_error("ma_dequant_prefix: bad sizes or outputs");
        return MA_EINVAL;
    }
    int n = p->nq + p->nf;
    if (n == 0) return MA_OK;
    dim3 grid((n + DQ_TOK - 1) / DQ_TOK, B * H, 2);
    // 16-byte stores: aligned bases and rows of whole 16-byte pieces
    auto al16 = [](const ma_tensor4 &t) {
        const int64_t m = t.dtype == MA_F32 ? 4 : 8;
        return ((uintptr_t)t.ptr & 15) == 0 && t.s[0] % m == 0 && t.s[1] % m == 0 && t.s[2] % m == 0;
    };
    if (al16(k_out) && al16(v_out))
        hipLaunchKernelGGL(dequant_prefix_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, make_args(p), H, D,
                           k_out, v_out);
    else
        hipLaunchKernelGGL(dequant_prefix_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, make_args(p), H, D,
                           k_out, v_out);
    return ma_check_launch("ma_dequant_prefix");
}

extern "C" int ma_gather_kv(const ma_prefix *p, int B, int H, int D, const int64_t *idx, const int64_t sidx[2], int k,
                            ma_tensor4 k_out, ma_tensor4 v_out, void *stream) {
    int rc = ma_validate_prefix(p, D, "ma_gather_kv");
    if (rc) return rc;
    if (B <= 0 || H <= 0 || k < 0 || !idx || !sidx || !k_out.ptr || !v_out.ptr || !out_dtype_ok(k_out.dtype) ||
        !out_dtype_ok(v_out.dtype)) {
        ma_set_error("ma_gather_kv: bad sizes or outputs");
        return MA_EINVAL;
    }
    if (k == 0) return MA_OK;
    // a 16-bit prefix gathered in its own dtype, every row of whole 16-byte pieces: copied
    auto rows16 = [](const void *ptr, const int64_t *s) {
        return ((uintptr_t)ptr & 15) == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0;
    };
    if (p->nq == 0 && p->nf > 0 && p->fdtype != MA_F32 && k_out.dtype == p->fdtype && v_out.dtype == p->fdtype &&
        rows16(p->kf, p->skf) && rows16(p->vf, p->svf) && rows16(k_out.ptr, k_out.s) && rows16(v_out.ptr, v_out.s)) {
        const int rows = 256 / (D / 8) * GR_ROWS;
        const dim3 rgrid((k + rows - 1) / rows, B * H);
        if (D == 128)
            hipLaunchKernelGGL(gather_rows_kernel<128>, rgrid, dim3(256), 0, (hipStream_t)stream, make_args(p), H, idx,
                               sidx[0], sidx[1], k, k_out, v_out);
        else
            hipLaunchKernelGGL(gather_rows_kernel<64>, rgrid, dim3(256), 0, (hipStream_t)stream, make_args(p), H, idx,
                               sidx[0], sidx[1], k, k_out, v_out);
        return ma_check_launch("ma_gather_kv");
    }
    int toks = 256 / (D / 4);
    dim3 grid((k + toks - 1) / toks, B * H);
    // 8-byte scale / zero loads and output stores: 8-byte aligned bases, strides in whole
    // groups of 4 elements
    auto al8 = [](const void *ptr) { return ((uintptr_t)ptr & 7) == 0; };
    const int vec = al8(p->ks) && al8(p->kz) && p->sks[0] % 4 == 0 && p->sks[1] % 4 == 0 && p->sks[2] % 4 == 0 &&
                    al8(k_out.ptr) && al8(v_out.ptr) && k_out.s[0] % 4 == 0 && k_out.s[1] % 4 == 0 &&
                    k_out.s[2] % 4 == 0 && v_out.s[0] % 4 == 0 && v_out.s[1] % 4 == 0 && v_out.s[2] % 4 == 0;
    hipLaunchKernelGGL(gather_kernel, grid, dim3(256), 0, (hipStream_t)stream, make_args(p), H, D, idx, sidx[0],
                       sidx[1], k, k_out, v_out, vec);
    return ma_check_launch("ma_gather_kv");
}

extern "C" int ma_quantize_keys(ma_tensor4 src, int B, int H, int T, int D, int group, void *kq, const int64_t skq[4],
                                void *ks, void *kz, const int64_t sks[3], void *stream) {
    if (group != KG) {
        ma_set_error("ma_quantize_keys: token group %d not built (32)", group);
        return MA_EUNSUPPORTED;
    }
    if (B <= 0 || H <= 0 || T < 0 || T % KG || D <= 0 || D > 1024 || !src.ptr || !kq || !ks || !kz || !skq || !sks ||
        ((uintptr_t)kq & 15) || ((skq[2] | skq[3]) & 15) || !out_dtype_ok(src.dtype)) {
        ma_set_error("ma_quantize_keys: bad geometry (T %% 32, 16-byte aligned payload rows)");
        return MA_EINVAL;
    }
    if (T == 0) return MA_OK;
    const int ng = T / KG;
    const dim3 grid((unsigned)((int64_t)ng * B * H));
#define MA_QK(DT_)                                                                                                    \
    hipLaunchKernelGGL(quantize_keys_kernel<DT_>, grid, dim3(D), 0, (hipStream_t)stream, src, ng, H, D, (uint8_t *)kq, \
                       skq[0], skq[1], skq[2], skq[3], (_Float16 *)ks, (_Float16 *)kz, sks[0], sks[1], sks[2])
    if (src.dtype == MA_BF16) MA_QK(MA_BF16);
    else if (src.dtype == MA_F16) MA_QK(MA_F16);
    else MA_QK(MA_F32);
#undef MA_QK
    return ma_check_launch("ma_quantize_keys");
}

extern "C" int ma_quantize_values(ma_tensor4 src, int B, int H, int T, int D, int group, void *vq,
                                  const int64_t svq[4], void *vs, void *vz, const int64_t svs[3], void *stream) {
    if (group != VG) {
        ma_set_error("ma_quantize_values: channel group %d not built (32)", group);
        return MA_EUNSUPPORTED;
    }
    if (B <= 0 || H <= 0 || T < 0 || D <= 0 || D % VG || !src.ptr || !vq || !vs || !vz || !svq || !svs ||
        ((uintptr_t)vq & 15) || ((svq[2] | svq[3]) & 15) || !out_dtype_ok(src.dtype)) {
        ma_set_error("ma_quantize_values: bad geometry (D %% 32, 16-byte aligned payload rows)");
        return MA_EINVAL;
    }
    if (T == 0) return MA_OK;
    int64_t items = (int64_t)B * H * T * (D / VG);
    int blocks = (int)((items + 255) / 256);
    if (blocks > 65535) blocks = 65535;
#define MA_QV(DT_)                                                                                                    \
    hipLaunchKernelGGL(quantize_values_kernel<DT_>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, src, B * H, H,   \
                       T, D, (uint8_t *)vq, svq[0], svq[1], svq[2], svq[3], (_Float16 *)vs, (_Float16 *)vz, svs[0],   \
                       svs[1], svs[2])
    if (src.dtype == MA_BF16) MA_QV(MA_BF16);
    else if (src.dtype == MA_F16) MA_QV(MA_F16);
    else MA_QV(MA_F32);
#undef MA_QV
    return ma_check_launch("ma_quantize_values");
}

extern "C" int ma_append_packed(ma_tensor4 k_res, ma_tensor4 v_res, int old_res, ma_tensor4 k_new, ma_tensor4 v_new,
                                int B, int H, int T, int D, int move, int keep, void *kq, const int64_t skq[4],
                                void *ks, void *kz, const int64_t sks[3], void *vq, const int64_t svq[4], void *vs,
                                void *vz, const int64_t svs[3], void *stream) {
    const char *who = "ma_append_packed";
    if (B <= 0 || H <= 0 || T <= 0 || old_res < 0 || move < 0 || keep < 0 || move % KG || move + keep != old_res + T ||
        !append_dim(D) || !k_new.ptr || !v_new.ptr ||
        ((old_res > 0 || keep > 0) && (!k_res.ptr || !v_res.ptr))) {
        ma_set_error("%s: bad geometry (move %% 32, move + keep = old_res + T, D | 256)", who);
        return MA_EINVAL;
    }
    if (k_new.dtype != v_new.dtype || !out_dtype_ok(k_new.dtype) ||
        ((old_res > 0 || keep > 0) && (k_res.dtype != k_new.dtype || v_res.dtype != k_new.dtype))) {
        ma_set_error("%s: the residual and the new tokens must share one 16-bit or f32 dtype", who);
        return MA_EINVAL;
    }
    AppendArgs A{};
    if (move) {
        if (!kq || !ks || !kz || !skq || !sks || !vq || !vs || !vz || !svq || !svs || ((uintptr_t)kq & 15) ||
            ((uintptr_t)vq & 15) || ((skq[2] | skq[3] | svq[2] | svq[3]) & 15)) {
            ma_set_error("%s: packed planes missing or payload rows not 16-byte aligned", who);
            return MA_EINVAL;
        }
        A.q[0] = (uint8_t *)kq;
        A.q[1] = (uint8_t *)vq;
        A.s[0] = (_Float16 *)ks;
        A.z[0] = (_Float16 *)kz;
        A.s[1] = (_Float16 *)vs;
        A.z[1] = (_Float16 *)vz;
        std::copy(skq, skq + 4, A.sq[0]);
        std::copy(svq, svq + 4, A.sq[1]);
        std::copy(sks, sks + 3, A.ss[0]);
        std::copy(svs, svs + 3, A.ss[1]);
    }
    A.src[0] = TwoSrc{k_res, k_new, old_res};
    A.src[1] = TwoSrc{v_res, v_new, old_res};
    A.H = H;
    A.D = D;
    A.lanes = B * H;
    A.ntok = move;
    A.keep = keep;
    A.first = move ? 0 : old_res;   // nothing quantized: the residual's rows stay, the new ones follow
    return launch_append(A, k_new.dtype, (hipStream_t)stream, who);
}
