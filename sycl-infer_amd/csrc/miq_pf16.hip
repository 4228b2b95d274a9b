// Batched GEMM for Q4_K / Q5_K / Q6_K beyond the decode sizes, on fp16 MFMA
// with exact integer arithmetic: out[t][n] = alpha * sum_k W[n][k] * act_t[k]
// (+ residual), for one or several matrices of one activation.
//
// Why fp16 and still exact.  Per 32-value group g the reference forms the
// int32 dot I = sum q*x8 and adds sx*(d*sc*I - dmin*m*xsum) (i8.cpp:40-61,
// 96-121).  Here the weight operand is the integer q*sc (at most 31*63 = 1953)
// put as it is into an fp16's bits -- below 2048 the fp16 with bits n is
// exactly n * 2^-24 -- and the activation operand is x8 (exact in fp16); every
// product is exact in fp32 and every partial sum of a group is an integer
// below 2^24 times 2^-24, so one v_mfma_f32_16x16x32_f16 (K = 32 = one group)
// returns 2^-24 * sc*I exactly.  The epilogue is then one fp32 fma per output
// and group (ab += (2^24 sx) * C), the block's d and dmin are applied once per
// 256 values (acc += d*ab - dmin*T), and T = sum_g m_g * (sx*xsum)_g runs on
// bf16 MFMA with sx*xsum split into three bf16 terms (24 significant bits)
// against the exact m.
//
// Structure.  A pre-pass writes the quantized activation as records in MFMA
// operand order.  A workgroup (one per CU) owns 256 rows x 16*TT tokens, TT
// chosen so that the token tiles cover the batch; each of its eight waves owns
// 32 rows and all tokens, and decodes its own weights straight into operand
// registers (two permlane swaps spread a row's 16-byte pieces over the four
// lanes of the operand), so no weight passes through LDS and a decoded weight
// serves 16*TT tokens.  The records stream into an LDS ring by direct loads issued
// two 128-value stages ahead, one barrier per stage; weights are loaded one block
// ahead into registers.  At a block's end the compiler waits for the weights
// (vmcnt(0), for the copies of the loop-carried ones; every Q4_K and Q5_K form, Q6_K
// from TT = 8 on), and so for the stages in flight too: the ring is worth about one
// stage there.
//
// What bounds it: the instruction issue of the two waves per SIMD -- per
// 32-value group a wave issues 8*TT fp32 fmas and 2*TT MFMAs, and the two
// overlap only in part -- with the decode (about 24 VALU per group) and LDS
// operand reads (1 KiB per two MFMAs) next.  Where the time went, and what was
// done: the loads of a stage issued together stalled every wave 1600 to 3000
// clocks in the address queue, so they are dealt out over the tiles; weights
// are held in their load registers to the block's start (hold()); 128-row tiles
// of 4 waves, two workgroups per CU, let the older one run ahead and leave the
// younger alone at the end.  17408 x 5120 Q4_K, pre-pass included: 128 / 256 /
// 512 / 1024 tokens 56 / 83 / 143 / 269 us; the form that decoded through LDS
// with two barriers per 64 values took 91 / 125 / 190 us at 128 / 256 / 512.
// Q6_K 5120 x 17408 (two planes, two MFMAs per group): 512 tokens 210 us, before
// 273; 128 tokens 100 us, before 149; at TT = 6, 7 and 8 it spills 2 to 13 registers.
#include <type_traits>
#include <utility>

#include "miq_internal.h"
#include "miq_units.h"
#include "miq_xq.h"

namespace miq {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint16_t us2 __attribute__((ext_vector_type(2)));

constexpr int kPW = 8;        // waves per workgroup
constexpr int kPT = 64 * kPW;
constexpr int kPN = 32 * kPW; // weight rows per workgroup: each wave owns 32
constexpr int kPfSegs = 8;    // matrices of one launch
constexpr int kPfRing = 3;    // activation stages in LDS
// Partial sums of the matrices of one launch at most (one matrix takes up to
// 64 MiB); more matrices go out in further launches that use the same memory.
constexpr size_t kPfPartBytes = (size_t)256 << 20;

// One activation record per (token tile of 16*TT tokens, 256-value block):
//   X   [8 groups][TT][64 lanes][16 B]  fp16 codes in MFMA operand order: lane
//       (token li = l % 16, h = l / 16) holds codes 8h + {0,2,1,3,4,6,5,7}
//   SX  [8 groups][16 li][TT] fp32      2^24 * the group scale of token 16*tt + li
//   U   [TT][64 lanes][16 B]            bf16 terms of sx*xsum: lane (li, lq) term
//       lq (hi, mid, lo, 0) of the eight groups
constexpr size_t pf_x_bytes(int TT) { return (size_t)8 * TT * 1024; }
constexpr size_t pf_aux_bytes(int TT) { return ((size_t)TT * 512 + (size_t)TT * 1024 + 1023) / 1024 * 1024; }
constexpr size_t pf_rec_bytes(int TT) { return pf_x_bytes(TT) + pf_aux_bytes(TT); }
constexpr int pf_lds_bytes(int TT) { return kPfRing * 4 * TT * 1024 + 2 * (int)pf_aux_bytes(TT) + kPN * 8; }

struct PfSeg {
    const uint8_t *w;
    float *out;
    const float *residual;
    uint32_t w_bytes;
    int n_rows;
    int out_stride;
    float alpha;
    int vec_out;     // out / residual allow 16-byte row stores
    int nt;          // row tiles
    int P;           // workgroups that share its tiles (the first P of the launch)
    int rounds;      // data-parallel rounds of one tile per workgroup
    int xmap;        // stream-K ranges are dealt to the 8 XCDs
    uint32_t poff;   // its partial slots, from part + poff
    uint32_t coff;   // its arrival counters, from cnt + coff
};

struct PfArgs {
    const uint8_t *rec;  // activation records [token tile][block]
    uint32_t row_bytes;
    int K;
    int TB;
    int mt;        // token tiles
    int nseg;
    float *part;   // per matrix [2 * workgroups] slots of [2*TT][512 threads][4] partial sums (stream-K)
    uint64_t *cnt; // per matrix [tile] arrival counters (xcd_arrival), zero between launches
    int32_t *dots; // parity form: [TB][n_rows][K/32] MFMA group results
    int astray;    // a test: every second workgroup of an XCD takes itself for one on another
    PfSeg seg[kPfSegs];
};

// ---------------------------------------------------------------- pre-pass
__device__ __forceinline__ uint16_t bf16_trunc(float f) { return (uint16_t)(__builtin_bit_cast(uint32_t, f) >> 16); }
__device__ __forceinline__ float bf16_val(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

// Quantized activation -> records.  One thread per 16-byte X operand piece
// (the first nx threads), then one per (record, token) for SX and U.  Tokens
// past TB are written as zeros.
template <int TT>
__global__ __launch_bounds__(256) void pf_prep_kernel(const int8_t *x8, const float *xmeta, const int32_t *xsumq, int TB,
                                                      int nb, uint32_t nx, uint32_t na, uint8_t *rec) {
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e < nx) {
        const int lane = (int)(e & 63);
        uint32_t r = e >> 6;
        const int tt = (int)(r % TT);
        r /= TT;
        const int g = (int)(r & 7);
        r >>= 3;  // record: token tile * nb + block
        const int b = (int)(r % nb), t = (int)(r / nb) * 16 * TT + 16 * tt + (lane & 15), h = lane >> 4;
        uint2 v = make_uint2(0, 0);
        if (t < TB) v = *reinterpret_cast<const uint2 *>(x8 + ((size_t)(8 * b + g) * TB + t) * 32 + 8 * h);
        constexpr int order[8] = {0, 2, 1, 3, 4, 6, 5, 7};
        h8 o;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t w = order[i] < 4 ? v.x : v.y;
            o[i] = (_Float16)(int)(int8_t)(w >> (8 * (order[i] & 3)));
        }
        *reinterpret_cast<h8 *>(rec + (size_t)r * pf_rec_bytes(TT) + (size_t)((g * TT + tt) * 64 + lane) * 16) = o;
        return;
    }
    const uint32_t a = e - nx;
    if (a >= na) return;
    const int li = (int)(a & 15);
    uint32_t r = a >> 4;
    const int tt = (int)(r % TT);
    r /= TT;
    const int b = (int)(r % nb), t = (int)(r / nb) * 16 * TT + 16 * tt + li;
    uint8_t *aux = rec + (size_t)r * pf_rec_bytes(TT) + pf_x_bytes(TT);
    uint32_t term[3][4] = {};
#pragma unroll
    for (int g = 0; g < 8; g++) {
        float sv = 0.0f, u = 0.0f;
        if (t < TB) {
            const size_t gi = (size_t)(8 * b + g) * TB + t;
            sv = xmeta[gi * 2];
            u = sv * (float)(xsumq[gi * 2] + xsumq[gi * 2 + 1]);
        }
        reinterpret_cast<float *>(aux)[(g * 16 + li) * TT + tt] = sv * 16777216.0f;
        const uint16_t hi = bf16_trunc(u);
        const float r1 = u - bf16_val(hi);
        const uint16_t mid = bf16_trunc(r1);
        const uint16_t lo = bf16_trunc(r1 - bf16_val(mid));
        term[0][g >> 1] |= (uint32_t)hi << (16 * (g & 1));
        term[1][g >> 1] |= (uint32_t)mid << (16 * (g & 1));
        term[2][g >> 1] |= (uint32_t)lo << (16 * (g & 1));
    }
    uint4 *ub = reinterpret_cast<uint4 *>(aux + TT * 512) + tt * 64 + li;
#pragma unroll
    for (int q = 0; q < 3; q++) ub[16 * q] = make_uint4(term[q][0], term[q][1], term[q][2], term[q][3]);
    ub[48] = make_uint4(0, 0, 0, 0);
}

// The quantizer and the records in one pass: a workgroup takes one 256-value
// block of 16 tokens, eight lanes per (token, group) as xq_kernel, writes the
// activation buffers and collects the records' pieces in LDS, from where they
// go out in runs of 1 KiB.  One launch and one pass over the codes less than
// xq_kernel + pf_prep_kernel (7.8 + 6.0 us at 512 x 5120).
template <int TT>
__global__ __launch_bounds__(1024) void pf_quant_kernel(const float *__restrict__ x, const float *__restrict__ up, int stride,
                                                        int8_t *__restrict__ x8, float *__restrict__ xmeta,
                                                        int32_t *__restrict__ xsumq, int TB, int nb, uint8_t *__restrict__ rec) {
    __shared__ __align__(16) uint2 lx[8][4][16][2];  // X operand pieces: [group][h][token][half]
    __shared__ float ls[8][16], lu[8][16];
    const int tid = threadIdx.x, l = tid & 7, g = (tid >> 3) & 7, li = tid >> 6;
    const int b = blockIdx.x % nb, tile = blockIdx.x / nb, t = 16 * tile + li;
    const bool live = t < TB;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (live) {
        const size_t o = (size_t)t * stride + 256 * b + 32 * g + 4 * l;
        const float4 a = *reinterpret_cast<const float4 *>(x + o);
        v[0] = a.x;
        v[1] = a.y;
        v[2] = a.z;
        v[3] = a.w;
        if (up) {
            const float4 c = *reinterpret_cast<const float4 *>(up + o);
            v[0] = silu(v[0]) * c.x;
            v[1] = silu(v[1]) * c.y;
            v[2] = silu(v[2]) * c.z;
            v[3] = silu(v[3]) * c.w;
        }
    }
    uint32_t word;
    int sq, s1;
    float sc;
    xq_lane4(v, word, sq, s1, sc);
    if (live) {
        const size_t gi = (size_t)(8 * b + g) * TB + t;
        reinterpret_cast<uint32_t *>(x8 + gi * 32)[l] = word;
        if (l == 0) {
            reinterpret_cast<float2 *>(xmeta)[gi] = make_float2(sc, 0.0f);
            reinterpret_cast<int2 *>(xsumq)[gi] = make_int2(sq, s1);
        }
    }
    constexpr int order[4] = {0, 2, 1, 3};
    uint16_t hv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) hv[i] = __builtin_bit_cast(uint16_t, (_Float16)(int)(int8_t)(word >> (8 * order[i])));
    lx[g][l >> 1][li][l & 1] = make_uint2(hv[0] | (uint32_t)hv[1] << 16, hv[2] | (uint32_t)hv[3] << 16);
    if (l == 0) {
        ls[g][li] = sc * 16777216.0f;
        lu[g][li] = sc * (float)(sq + s1);
    }
    __syncthreads();
    uint8_t *R = rec + ((size_t)(tile / TT) * nb + b) * pf_rec_bytes(TT);
    const int tt = tile % TT;
    if (tid < 512) {
        const int gg = tid >> 6, lane = tid & 63;
        *reinterpret_cast<uint4 *>(R + (size_t)((gg * TT + tt) * 64 + lane) * 16) = *reinterpret_cast<const uint4 *>(&lx[gg][lane >> 4][lane & 15][0]);
    } else if (tid < 640) {
        const int gg = (tid - 512) >> 4, i = tid & 15;
        reinterpret_cast<float *>(R + pf_x_bytes(TT))[(gg * 16 + i) * TT + tt] = ls[gg][i];
    } else if (tid < 704) {
        const int q = (tid - 640) >> 4, i = tid & 15;
        uint32_t w[4] = {0, 0, 0, 0};
        if (q < 3)
#pragma unroll
            for (int gg = 0; gg < 8; gg++) {
                float r = lu[gg][i];
                for (int k = 0; k < q; k++) r -= bf16_val(bf16_trunc(r));
                w[gg >> 1] |= (uint32_t)bf16_trunc(r) << (16 * (gg & 1));
            }
        reinterpret_cast<uint4 *>(R + pf_x_bytes(TT) + TT * 512)[tt * 64 + q * 16 + i] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// ---------------------------------------------------------------- weights
// Raw bytes of one 256-value block of row li for lane (li, h): Q4_K/Q5_K dword
// h of the header and the code bytes [16h, 16h+16) and [64+16h, ...) (the
// permlane swaps of split() give each lane bytes 8h..8h+7 of every 32-byte
// pair), Q5_K also qh bytes 8h..8h+7.
template <uint32_t TYPE> struct PfRaw {
    uint32_t hw;
    u4v qa, qb;
    u2v qh;
    template <int part> __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rw, uint32_t boff, int h) {
        constexpr uint32_t qoff = TYPE == MIQ_TYPE_Q4_K ? 16 : 48;
        if constexpr (part == 0) hw = bload4(rw, boff + 4 * h);
        if constexpr (part == 1) qa = __builtin_bit_cast(u4v, bload16(rw, boff + qoff + 16 * h));
        if constexpr (part == 2) qb = __builtin_bit_cast(u4v, bload16(rw, boff + qoff + 64 + 16 * h));
        if constexpr (part == 3) qh = __builtin_bit_cast(u2v, __builtin_amdgcn_raw_buffer_load_b64(rw, boff + 16 + 8 * h, 0, 0));
    }
    // The loaded registers stay as they are up to here: without this the
    // compiler copies parts of them right after the loads are issued, which
    // waits for them a whole block early.
    __device__ __forceinline__ void hold() {
        asm volatile("" : "+v"(hw), "+v"(qa), "+v"(qb));
        if constexpr (TYPE == MIQ_TYPE_Q5_K) asm volatile("" : "+v"(qh));
    }
};
// Q6_K: lane (li, h) takes ql bytes [16h, 16h+16) and [64+16h, ...), qh bytes
// [16h, ...) and dword h of the scales.  Blocks are 210 bytes (2-byte aligned),
// so each piece is the dword-aligned bytes around it, realigned by sh at the
// block's start.
template <> struct PfRaw<MIQ_TYPE_Q6_K> {
    u4v qa, qb, qh;
    u2v sw;
    uint32_t ea, eb, eh, dw, sh;
    template <int part> __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rw, uint32_t boff, int h) {
        const uint32_t o = (boff & ~3u) + 16 * h;
        if constexpr (part == 0) qa = __builtin_bit_cast(u4v, bload16(rw, o));
        if constexpr (part == 1) ea = bload4(rw, o + 16);
        if constexpr (part == 2) qb = __builtin_bit_cast(u4v, bload16(rw, o + 64));
        if constexpr (part == 3) eb = bload4(rw, o + 80);
        if constexpr (part == 4) qh = __builtin_bit_cast(u4v, bload16(rw, o + 128));
        if constexpr (part == 5) eh = bload4(rw, o + 144);
        if constexpr (part == 6) sw = __builtin_bit_cast(u2v, __builtin_amdgcn_raw_buffer_load_b64(rw, (boff & ~3u) + 192 + 4 * h, 0, 0));
        if constexpr (part == 7) {
            dw = bload4(rw, (boff & ~3u) + 208);
            sh = boff & 3u;
        }
    }
    __device__ __forceinline__ void hold() {
        asm volatile("" : "+v"(qa), "+v"(qb), "+v"(qh), "+v"(sw), "+v"(ea), "+v"(eb), "+v"(eh), "+v"(dw));
    }
};
// its load instructions
template <uint32_t TYPE> constexpr int pf_raw_loads() { return TYPE == MIQ_TYPE_Q4_K ? 3 : TYPE == MIQ_TYPE_Q5_K ? 4 : 8; }

// header dword h of row li in lane (li, h) -> all four dwords in every lane
__device__ __forceinline__ uint4 gather4(uint32_t w) {
    const auto a = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    return make_uint4(b[0], b[1], c[0], c[1]);
}
// 16-byte pieces [16h, 16h+16) of lanes h = 0..3 -> bytes 8h..8h+7 of the two 32-byte pairs
__device__ __forceinline__ void split_pairs(const u4v &q, uint2 &p0, uint2 &p1) {
    const auto s0 = __builtin_amdgcn_permlane16_swap(q.x, q.z, false, false);
    const auto s1 = __builtin_amdgcn_permlane16_swap(q.y, q.w, false, false);
    const auto t0 = __builtin_amdgcn_permlane32_swap(s0[0], s0[1], false, false);
    const auto t1 = __builtin_amdgcn_permlane32_swap(s1[0], s1[1], false, false);
    p0 = make_uint2(t0[0], t1[0]);
    p1 = make_uint2(t0[1], t1[1]);
}
// byte k of w in both 16-bit halves
template <int k> __device__ __forceinline__ us2 dup_byte(uint32_t w) {
    return __builtin_bit_cast(us2, __builtin_amdgcn_perm(w, w, 0x0C000C00u | k | (k << 16)));
}
__device__ __forceinline__ uint32_t pf_bf16_pair(uint32_t w, int k) {
    const float a = (float)((w >> (8 * k)) & 0xFFu), b = (float)((w >> (8 * k + 8)) & 0xFFu);
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}

// Weight operand of one group: one fp16 plane, two for Q6_K (hi, lo).
template <uint32_t TYPE> struct PfOp {
    h8 p[TYPE == MIQ_TYPE_Q6_K ? 2 : 1];
};
// which of a half block's two 32-byte pairs holds its group gl
template <uint32_t TYPE> constexpr int pf_pair(int gl) { return TYPE == MIQ_TYPE_Q6_K ? gl & 1 : gl >> 1; }

// The block a wave works on, one row tile: its codes by pair and its scales.
template <uint32_t TYPE> struct PfBlk {
    u4v qa, qb;
    u2v qh;
    uint32_t sc[2];  // the eight 6-bit scales as bytes
    uint32_t mn[2];  // and mins
    float d, dm;
    __device__ __forceinline__ void take(const PfRaw<TYPE> &R, int) {
        const uint4 hd = gather4(R.hw);
        qa = R.qa;
        qb = R.qb;
        if constexpr (TYPE == MIQ_TYPE_Q5_K) qh = R.qh;
        sc[0] = hd.y & 0x3F3F3F3Fu;
        sc[1] = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
        mn[0] = hd.z & 0x3F3F3F3Fu;
        mn[1] = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
        d = h2f(hd.x);
        dm = h2f(hd.x >> 16);
    }
    template <int hf> __device__ __forceinline__ void split(uint2 (&q)[2]) { split_pairs(hf == 0 ? qa : qb, q[0], q[1]); }
    // A operand of group g from its pair of the codes: q * sc as fp16 bits
    template <int g> __device__ __forceinline__ PfOp<TYPE> op(const uint2 &q) const {
        constexpr uint32_t M = 0x000F000Fu;
        const us2 s = dup_byte<(g & 3)>(sc[g >> 2]);
        uint32_t e[4];
        if constexpr (g & 1) {
            e[0] = (q.x >> 4) & M;
            e[1] = (q.x >> 12) & M;
            e[2] = (q.y >> 4) & M;
            e[3] = (q.y >> 12) & M;
        } else {
            e[0] = q.x & M;
            e[1] = (q.x >> 8) & M;
            e[2] = q.y & M;
            e[3] = (q.y >> 8) & M;
        }
        if constexpr (TYPE == MIQ_TYPE_Q5_K) {
            constexpr uint32_t B = 0x00100010u;
            const uint32_t tx = g < 4 ? qh.x << (4 - (g & 3) - (g & 4)) : qh.x >> (g & 3);
            const uint32_t ty = g < 4 ? qh.y << (4 - (g & 3) - (g & 4)) : qh.y >> (g & 3);
            e[0] |= tx & B;
            e[1] |= (tx >> 8) & B;
            e[2] |= ty & B;
            e[3] |= (ty >> 8) & B;
        }
        uint4 o;
        o.x = __builtin_bit_cast(uint32_t, (us2)(__builtin_bit_cast(us2, e[0]) * s));
        o.y = __builtin_bit_cast(uint32_t, (us2)(__builtin_bit_cast(us2, e[1]) * s));
        o.z = __builtin_bit_cast(uint32_t, (us2)(__builtin_bit_cast(us2, e[2]) * s));
        o.w = __builtin_bit_cast(uint32_t, (us2)(__builtin_bit_cast(us2, e[3]) * s));
        return {{__builtin_bit_cast(h8, o)}};
    }
    // bf16 A operand of the dmin term: the row's eight mins against each of the three terms
    __device__ __forceinline__ b8 mins(int lq) const {
        uint4 m = make_uint4(pf_bf16_pair(mn[0], 0), pf_bf16_pair(mn[0], 2), pf_bf16_pair(mn[1], 0), pf_bf16_pair(mn[1], 2));
        if (lq == 3) m = make_uint4(0, 0, 0, 0);
        return __builtin_bit_cast(b8, m);
    }
};

// Q6_K: group g = 4*(128-value half) + p takes nibble p/2 of pair p%2 of the
// half and bits 2p of its qh bytes; its two 16-value sub-groups have signed
// 8-bit scales, lanes h < 2 in the first.  (q-32)*sc reaches 4096 and odd
// values above 2048 are no fp16, so there are two planes: with sc = 2*s2 + s1
// (s1 = sc & 1), hi = v * 2*s2 (even, exact) and lo = s1 ? v : 0, v = q - 32,
// all in units of 2^-24 (the code put as it is into an fp16's bits).  The lo
// plane's MFMA accumulates onto the hi plane's: sc0*I0 + sc1*I1 exactly.
template <> struct PfBlk<MIQ_TYPE_Q6_K> {
    u4v qa, qb;
    uint2 qh[2];
    uint32_t sc[4];  // this lane's sub-group scale of group g: byte 2*(g & 1) of sc[g >> 1]
    float d, dm;
    __device__ __forceinline__ static u4v align(const u4v &v, uint32_t e, uint32_t sh) {
        u4v o;
        o.x = __builtin_amdgcn_alignbyte(v.y, v.x, sh);
        o.y = __builtin_amdgcn_alignbyte(v.z, v.y, sh);
        o.z = __builtin_amdgcn_alignbyte(v.w, v.z, sh);
        o.w = __builtin_amdgcn_alignbyte(e, v.w, sh);
        return o;
    }
    __device__ __forceinline__ void take(const PfRaw<MIQ_TYPE_Q6_K> &R, int h) {
        qa = align(R.qa, R.ea, R.sh);
        qb = align(R.qb, R.eb, R.sh);
        split_pairs(align(R.qh, R.eh, R.sh), qh[0], qh[1]);
        const uint4 s = gather4(__builtin_amdgcn_alignbyte(R.sw.y, R.sw.x, R.sh));
        const uint32_t b = 8 * (h >> 1);
        sc[0] = s.x >> b;
        sc[1] = s.y >> b;
        sc[2] = s.z >> b;
        sc[3] = s.w >> b;
        d = h2f(R.dw >> (8 * R.sh));
        dm = 0.0f;
    }
    template <int hf> __device__ __forceinline__ void split(uint2 (&q)[2]) { split_pairs(hf == 0 ? qa : qb, q[0], q[1]); }
    template <int g> __device__ __forceinline__ PfOp<MIQ_TYPE_Q6_K> op(const uint2 &q) const {
        constexpr int p = g & 3, nib = p >= 2 ? 4 : 0;
        constexpr uint32_t M = 0x000F000Fu, B = 0x00300030u;
        const int s = (int)(int8_t)(sc[g >> 1] >> (16 * (g & 1)));
        const _Float16 m = (_Float16)(s & ~1);
        const h2 m2 = h2{m, m};
        const uint32_t odd = 0u - (uint32_t)(s & 1);
        const uint2 hq = qh[g >> 2];
        const uint32_t tx = p < 2 ? hq.x << (4 - 2 * (p & 1)) : hq.x >> (2 * (p & 1));
        const uint32_t ty = p < 2 ? hq.y << (4 - 2 * (p & 1)) : hq.y >> (2 * (p & 1));
        const uint32_t e[4] = {((q.x >> nib) & M) | (tx & B), ((q.x >> (nib + 8)) & M) | ((tx >> 8) & B),
                               ((q.y >> nib) & M) | (ty & B), ((q.y >> (nib + 8)) & M) | ((ty >> 8) & B)};
        const h2 off = __builtin_bit_cast(h2, 0x80208020u);  // -32 * 2^-24
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const h2 v = __builtin_bit_cast(h2, e[i]) + off;
            hi[i] = __builtin_bit_cast(uint32_t, v * m2);
            lo[i] = __builtin_bit_cast(uint32_t, v) & odd;
        }
        return {{__builtin_bit_cast(h8, make_uint4(hi[0], hi[1], hi[2], hi[3])),
                 __builtin_bit_cast(h8, make_uint4(lo[0], lo[1], lo[2], lo[3]))}};
    }
};

// f(0), f(1), ..., f(N - 1) with the index as a constant
template <class F, int... I> __device__ __forceinline__ void static_for_(F &f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &f) { static_for_(f, std::make_integer_sequence<int, N>{}); }

// ---------------------------------------------------------------- LDS DMA
// 1 KiB from base + soff + 16*lane straight into LDS at lds_addr + 16*lane.
// Inline asm, so that the compiler does not track it: its tracking of a load
// into LDS waits for every such load before the next LDS read.  The caller
// orders it with an explicit vmcnt and a barrier.
__device__ __forceinline__ void pf_dma(__amdgpu_buffer_rsrc_t r, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
    const uint32_t la = __builtin_amdgcn_readfirstlane(lds_addr), so = __builtin_amdgcn_readfirstlane(soff);
    uint32_t keep;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(keep)
        : "s"(la), "v"(voff), "s"(r), "s"(so)
        : "memory");
}
// this wave's loads down to the N youngest and its LDS reads are done, then the workgroup meets
template <int N> __device__ __forceinline__ void pf_sync() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// ---------------------------------------------------------------- GEMM
// DOTS: the parity form -- every group's MFMA result (2^-24 * sc * I) goes to
// A.dots as sc * I instead of the epilogue; one tile per workgroup.
template <uint32_t TYPE, int TT, bool DOTS = false>
__global__ __launch_bounds__(kPT, 2) void pf16_kernel(PfArgs A) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ int lflag;
    constexpr int kStage = 4 * TT * 1024;                // X bytes of a 128-value stage
    constexpr int kAux = (int)pf_aux_bytes(TT);
    constexpr int kLAux = kPfRing * kStage;              // aux, two blocks
    constexpr int kLD = kLAux + 2 * kAux;                // [wave][row tile][d, dmin][16]
    constexpr int kXn = (4 * TT + kPW - 1) / kPW;        // X DMA instructions per wave and stage (the last may be idle)
    constexpr int kAn = (kAux / 1024 + kPW - 1) / kPW;   // aux DMA instructions per wave (the last may be idle)
    constexpr int kRl = 2 * pf_raw_loads<TYPE>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int K = A.K, nkb = K / 256;
    const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t voff = lane * 16;
    f4 acc[2][TT], ab[2][TT];

    // Blocks [kb0, kb1) of row tile n0 (matrix S) and token tile tg into acc.
    auto run = [&](const PfSeg &S, int n0, int tg, int kb0, int kb1) {
        const __amdgpu_buffer_rsrc_t rw = make_rsrc(S.w, S.w_bytes);
        const __amdgpu_buffer_rsrc_t rr =
            make_rsrc(A.rec + (size_t)tg * nkb * pf_rec_bytes(TT), (uint32_t)(nkb * pf_rec_bytes(TT)));
        const int s0 = 2 * kb0, s1 = 2 * kb1;
        const uint32_t wend = __builtin_amdgcn_readfirstlane(S.w_bytes);
        uint32_t wb[2];
        bool ok[2];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            const int row = n0 + 32 * wave + 16 * rt + li;
            ok[rt] = row < S.n_rows;
            wb[rt] = (uint32_t)row * A.row_bytes;
        }
        PfRaw<TYPE> R[2];
        PfBlk<TYPE> B[2];
        // One load instruction each: part i of a block's weights (a row past the end
        // reads zeros, past the buffer), piece i of a stage's X and of a block's aux.
        // Past the range they fetch the last stage or block again, so that every wave
        // has issued the same number of loads wherever it waits.
        auto load_w = [&](auto i_c, int kb) {
            constexpr int i = decltype(i_c)::value, rt = i / pf_raw_loads<TYPE>();
            const uint32_t o = (uint32_t)(kb < kb1 ? kb : kb1 - 1) * block_bytes(TYPE);
            R[rt].template load<i % pf_raw_loads<TYPE>()>(rw, ok[rt] ? wb[rt] + o : wend, lq);
        };
        uint32_t slot = 0;  // ring slot of the stage being issued (bytes)
        auto load_x = [&](int i, int s) {
            const int sc = s < s1 ? s : s1 - 1;
            const uint32_t so = (uint32_t)(sc >> 1) * (uint32_t)pf_rec_bytes(TT) + (uint32_t)(sc & 1) * kStage;
            int p = wave * kXn + i;
            if (p >= 4 * TT) p = 0;  // no piece left (odd TT): one that is fetched anyway
            pf_dma(rr, lbase + slot + p * 1024, voff, so + p * 1024);
            if (i == kXn - 1) slot = slot == (kPfRing - 1) * kStage ? 0 : slot + kStage;
        };
        auto load_aux = [&](int i, int kb) {
            const uint32_t so = (uint32_t)(kb < kb1 ? kb : kb1 - 1) * (uint32_t)pf_rec_bytes(TT) + (uint32_t)pf_x_bytes(TT);
            int c = wave + kPW * i;
            if (c >= kAux / 1024) c = wave < kAux / 1024 ? wave : 0;  // no piece left: one that is there again
            pf_dma(rr, lbase + kLAux + (kb & 1) * kAux + c * 1024, voff, so + c * 1024);
        };
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < TT; b++) acc[a][b] = f4{0, 0, 0, 0};
        // The previous range is done with every LDS buffer: its reads, and the loads
        // that it issued past its end.  A wave without a piece of its own fetches one
        // of another wave's again (load_x, load_aux), so a late one of those loads
        // and this range's own would meet in one place with nothing to order them.
        pf_sync<0>();
        // in the order that the loop keeps: aux, X(s), weights, X(s + 1)
#pragma unroll
        for (int i = 0; i < kAn; i++) load_aux(i, kb0);
#pragma unroll
        for (int i = 0; i < kXn; i++) load_x(i, s0);
        auto first_w = [&](auto i_c) { load_w(i_c, kb0); };
        static_for<kRl>(first_w);
#pragma unroll
        for (int i = 0; i < kXn; i++) load_x(i, s0 + 1);
        uint32_t xs = 0;  // ring slot being read (bytes)

        for (int kb = kb0; kb < kb1; kb++) {
            const uint8_t *aux = lds + kLAux + (kb & 1) * kAux;
            auto stage = [&](auto hf_c) {
                constexpr int hf = decltype(hf_c)::value;
                const int s = 2 * kb + hf;
                // The first group's weight operand, ready before the barrier.
                uint2 q[2][2];
                PfOp<TYPE> a[2][2];
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    if constexpr (hf == 0) {
                        R[rt].hold();
                        B[rt].take(R[rt], lq);
                        if (lq == 0) {
                            float *D = reinterpret_cast<float *>(lds + kLD) + (wave * 2 + rt) * 32 + li;
                            D[0] = B[rt].d;
                            D[16] = B[rt].dm;
                        }
                    }
                    B[rt].template split<hf>(q[rt]);
                    a[0][rt] = B[rt].template op<4 * hf>(q[rt][0]);
                }
                // X(s) (and the block's aux before it) is in LDS when at most the loads
                // issued after it are outstanding: in the first half the weights and
                // X(s+1), in the second the next block's aux, X(s+1) and weights.
                pf_sync<hf ? kAn + kXn + kRl : kRl + kXn>();
                const uint8_t *X = lds + xs + lane * 16;
                xs = xs == (kPfRing - 1) * kStage ? 0 : xs + kStage;
                h8 b[3];  // X operands, read two tiles ahead
                float sx[2][TT];
                auto read_x = [&](auto i_c) {
                    constexpr int i = decltype(i_c)::value;
                    if constexpr (i < 4 * TT) b[i % 3] = *reinterpret_cast<const h8 *>(X + i * 1024);
                };
                auto read_sx = [&](auto gl_c) {
                    constexpr int gl = decltype(gl_c)::value;
                    const float *p = reinterpret_cast<const float *>(aux) + ((4 * hf + gl) * 16 + li) * TT;
                    if constexpr (TT % 2) {
#pragma unroll
                        for (int i = 0; i < TT; i++) sx[gl & 1][i] = p[i];
                    } else {
                        using V = std::conditional_t<TT % 4 == 0, f4, f2>;
                        constexpr int n = sizeof(V) / 4;
#pragma unroll
                        for (int i = 0; i < TT / n; i++)
#pragma unroll
                            for (int v = 0; v < n; v++) sx[gl & 1][n * i + v] = reinterpret_cast<const V *>(p)[i][v];
                    }
                };
                read_x(std::integral_constant<int, 0>{});
                read_x(std::integral_constant<int, 1>{});
                read_sx(std::integral_constant<int, 0>{});
                // The loads of this stage (first half: the next block's aux, X(s+2) and
                // the next block's weights; second half: X(s+2)), dealt out over the
                // tiles below: issued together they fill the CU's address queue and
                // stall every wave in turn (1600 to 3000 clocks a stage).
                constexpr int kOps = hf ? kXn : kAn + kXn + kRl;
                auto load_op = [&](auto j_c) {
                    constexpr int j = decltype(j_c)::value;
                    if constexpr (hf) load_x(j, s + 2);
                    else if constexpr (j < kAn) load_aux(j, kb + 1);
                    else if constexpr (j < kAn + kXn) load_x(j - kAn, s + 2);
                    else load_w(std::integral_constant<int, j - kAn - kXn>{}, kb + 1);
                };
                // Group gl: tile tt's MFMAs are issued one tile ahead of its
                // epilogue; the next group's first X operands, scales and weight
                // operand are fetched and decoded on the way.
                auto group = [&](auto gl_c) {
                    constexpr int gl = decltype(gl_c)::value, g = 4 * hf + gl;
                    f4 c[2][2];
                    auto mm = [&](int tt) {
#pragma unroll
                        for (int rt = 0; rt < 2; rt++)
                            c[tt & 1][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[gl & 1][rt].p[0], b[(gl * TT + tt) % 3], f4{0, 0, 0, 0}, 0, 0, 0);
                        if constexpr (TYPE == MIQ_TYPE_Q6_K)
#pragma unroll
                            for (int rt = 0; rt < 2; rt++)
                                c[tt & 1][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[gl & 1][rt].p[1], b[(gl * TT + tt) % 3], c[tt & 1][rt], 0, 0, 0);
                    };
                    mm(0);
                    auto tile = [&](auto tt_c) {
                        constexpr int tt = decltype(tt_c)::value;
                        read_x(std::integral_constant<int, gl * TT + tt + 2>{});
                        auto op_here = [&](auto j_c) {
                            constexpr int j = decltype(j_c)::value;
                            if constexpr ((hf ? 1 + 2 * j : j * 4 * TT / kOps) == gl * TT + tt) load_op(j_c);
                        };
                        static_for<kOps>(op_here);
                        if constexpr (tt + 1 < TT) mm(tt + 1);
                        if constexpr (gl < 3 && tt < 2)
                            a[(gl + 1) & 1][tt] = B[tt].template op<(g + 1) & 7>(q[tt][pf_pair<TYPE>((gl + 1) & 3)]);
                        if constexpr (gl < 3 && tt == TT - 2) read_sx(std::integral_constant<int, gl + 1>{});
#pragma unroll
                        for (int rt = 0; rt < 2; rt++) {
                            if constexpr (DOTS) {
                                const int t = (tg * TT + tt) * 16 + li;
#pragma unroll
                                for (int v = 0; v < 4; v++) {
                                    const int row = n0 + 32 * wave + 16 * rt + 4 * lq + v;
                                    if (t < A.TB && row < S.n_rows)
                                        A.dots[((size_t)t * S.n_rows + row) * (K / 32) + 8 * kb + g] =
                                            (int32_t)(c[tt & 1][rt][v] * 16777216.0f);
                                }
                            } else {
#pragma unroll
                                for (int v = 0; v < 4; v++) {
                                    if constexpr (g == 0) ab[rt][tt][v] = sx[gl & 1][tt] * c[tt & 1][rt][v];
                                    else ab[rt][tt][v] = __builtin_fmaf(sx[gl & 1][tt], c[tt & 1][rt][v], ab[rt][tt][v]);
                                }
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    static_for<TT>(tile);
                };
                static_for<4>(group);
            };
            static_for<2>(stage);
            if constexpr (!DOTS && TYPE == MIQ_TYPE_Q6_K) {
                // block end: acc += d * ab
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const f4 d4 = *reinterpret_cast<const f4 *>(reinterpret_cast<const float *>(lds + kLD) + (wave * 2 + rt) * 32 + 4 * lq);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[rt][tt][v] = __builtin_fmaf(d4[v], ab[rt][tt][v], acc[rt][tt][v]);
                }
            } else if constexpr (!DOTS) {
                // block end: acc += d * ab - dmin * (m . sx*xsum); the bf16 MFMA's K
                // slots are (m, m, m, 0) x (hi, mid, lo, 0)
                const uint8_t *U = aux + TT * 512 + lane * 16;
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const float *D = reinterpret_cast<const float *>(lds + kLD) + (wave * 2 + rt) * 32 + 4 * lq;
                    const f4 d4 = *reinterpret_cast<const f4 *>(D), dm4 = *reinterpret_cast<const f4 *>(D + 16);
                    const b8 mv = B[rt].mins(lq);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) {
                        const b8 uv = *reinterpret_cast<const b8 *>(U + tt * 1024);
                        const f4 T = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mv, uv, f4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            acc[rt][tt][v] = __builtin_fmaf(d4[v], ab[rt][tt][v], acc[rt][tt][v]);
                            acc[rt][tt][v] = __builtin_fmaf(-dm4[v], T[v], acc[rt][tt][v]);
                        }
                    }
                }
            }
        }
    };

    // C[row][token]: lane holds rows 4*lq .. 4*lq+3 of each row tile for one token
    auto store = [&](const PfSeg &S, int n0, int tg) {
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            const int row = n0 + 32 * wave + 16 * rt + 4 * lq;
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                const int t = (tg * TT + tt) * 16 + li;
                if (t >= A.TB) continue;
                const size_t o = (size_t)t * S.out_stride + row;
                if (S.vec_out && row + 3 < S.n_rows) {
                    f4 v = acc[rt][tt] * S.alpha;
                    if (S.residual) v += *reinterpret_cast<const f4 *>(S.residual + o);
                    *reinterpret_cast<f4 *>(S.out + o) = v;
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        if (row + v >= S.n_rows) break;
                        float val = S.alpha * acc[rt][tt][v];
                        if (S.residual) val += S.residual[o + v];
                        S.out[o + v] = val;
                    }
                }
            }
        }
    };

    // Schedule, matrix after matrix, each with the tiles and ranges that it has
    // alone (so its results are its own launch's bit for bit); nothing but a
    // tile's partials orders the workgroups, so one matrix's fix-up runs beside
    // the next one's tiles.  Tile t is row tile t / mt, token tile t % mt, so the token
    // tiles of a row tile are neighbours and read its weights from L2.
    // `rounds` data-parallel rounds: in round k workgroup w takes tile
    // k*P + (P/8)*(w % 8) + w/8, i.e. each XCD (dealt by blockIdx % 8) a run of
    // consecutive tiles; tiles past T are skipped.  The remaining `sk` tiles
    // are then split along K over all workgroups (stream-K): XCD x owns sk
    // tiles [x*sk/G, (x+1)*sk/G) and cuts their K blocks into P/G equal
    // contiguous ranges, one per workgroup of the XCD.  A tile covered by one
    // range is stored directly; otherwise each range writes a partial (slot 2v
    // for the tile it starts in, 2v+1 for the one it ends in), and the last
    // contributor to arrive adds the partials in range order (the result does
    // not depend on timing) and stores.  With G == 1 the partials go through
    // memory, else those of a tile stay in their XCD's L2; where its ranges were on
    // several XCDs all the same (see xcd_arrival), the last to arrive computes the
    // whole tile, in one sum.
    constexpr int kPart = 2 * TT * kPT;  // f4 of one partial tile
    const int w = blockIdx.x;
    for (int si = 0; si < A.nseg; si++) {
    const PfSeg &S = A.seg[si];
    const int P = S.P;
    if (w >= P) continue;
    const int T = S.nt * A.mt;
    const int F = S.rounds * P, sk = T > F ? T - F : 0;  // no stream-K tiles where the last round is not full (DOTS)
    const bool xmap = S.xmap;
    const int G = xmap ? 8 : 1, x = xmap ? w % 8 : 0, Pg = P / G, vl = xmap ? w / 8 : w;
    f4 *part = reinterpret_cast<f4 *>(A.part) + (size_t)S.poff * kPart;
    uint64_t *cnt = A.cnt + S.coff;
    // XCD x's tiles [tx0, tx0 + ntx): the first sk % G XCDs hold one more; range u of
    // its ntx * nkb blocks starts at u*rq + min(u, rr) (the first rr ranges hold one more)
    const int ntx = sk / G + (x < sk % G), tx0 = F + x * (sk / G) + (x < sk % G ? x : sk % G);
    const int total = ntx * nkb, rq = total / Pg, rr = total - rq * Pg;
    auto rstart = [&](int u) { return u * rq + (u < rr ? u : rr); };
    auto owner = [&](int blk) { return blk < rr * (rq + 1) ? blk / (rq + 1) : rr + (blk - rr * (rq + 1)) / rq; };
    const int bs = rstart(vl), be = rstart(vl + 1);
    const int v = x * Pg + vl;  // global range id (partial slots)
    // Added to b0 (at most 2^30 blocks): compute the last piece's tile again.  A
    // variable of its own cost up to 1.5 % of the launch.
    constexpr int kAgain = 1 << 30;
    int k = 0, b0 = bs;
    for (;;) {
        // next segment: a data-parallel tile, else the next piece of this
        // workgroup's stream-K range
        int t, kb0, kb1;
        bool dp;
        if (k < S.rounds) {
            dp = true;
            t = k * P + (w % 8) * (P / 8) + w / 8;
            k++;
            if (t >= T) continue;
            kb0 = 0;
            kb1 = nkb;
        } else if (b0 < be) {
            dp = false;
            const int lt = b0 / nkb;
            t = tx0 + lt;
            kb0 = b0 - lt * nkb;
            kb1 = be - lt * nkb < nkb ? be - lt * nkb : nkb;
        } else if (__builtin_expect(b0 >= kAgain, 0)) {
            dp = true;
            b0 -= kAgain;
            t = tx0 + (b0 - 1) / nkb;
            kb0 = 0;
            kb1 = nkb;
        } else {
            break;
        }
        const int n0 = t / A.mt * kPN, tg = t % A.mt;
        run(S, n0, tg, kb0, kb1);
        if (dp) {  // a whole tile
            if constexpr (!DOTS) store(S, n0, tg);
            continue;
        }
        const bool head = b0 == bs;
        b0 = (t - tx0) * nkb + kb1;
        if (kb0 == 0 && kb1 == nkb) {
            store(S, n0, tg);
            continue;
        }
        const int tb0 = (t - tx0) * nkb, tb1 = tb0 + nkb;
        const int v_lo = owner(tb0), v_hi = owner(tb1 - 1);
        int n_contrib = 0;  // ranges of the tile that hold a block (with few blocks some are empty)
        for (int u = v_lo; u <= v_hi; u++) n_contrib += rstart(u) < rstart(u + 1);
        const uint64_t one = xmap ? xcd_arrival(A.astray & vl) : 1;
        // A range that finds every other one arrived keeps its sums in registers.
        if (tid == 0)
            lflag = xcd_last(__hip_atomic_load(cnt + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), one, (uint32_t)n_contrib) == 1;
        __syncthreads();
        int fl = __builtin_amdgcn_readfirstlane(lflag);
        const bool own = fl;
        if (own) {
            if (tid == 0) __hip_atomic_store(cnt + t, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            f4 *mine = part + (size_t)(2 * v + (head ? 0 : 1)) * kPart + tid;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int c = 0; c < TT; c++)
                    mine[(a * TT + c) * kPT] = acc[a][c];
            if (!xmap) __threadfence();  // a reader on any XCD: write the partial back past the L2
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (tid == 0) {
                const uint64_t prev = __hip_atomic_fetch_add(cnt + t, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lflag = xcd_last(prev, one, (uint32_t)n_contrib);
                if (lflag) __hip_atomic_store(cnt + t, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            fl = __builtin_amdgcn_readfirstlane(lflag);
        }
        if (!fl) continue;
        if (__builtin_expect(fl == 2, 0)) {
            b0 += kAgain;
            continue;
        }
        if (!xmap) __threadfence();  // drop stale L2 lines first
        f4 sum[2][TT];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < TT; c++) sum[a][c] = f4{0, 0, 0, 0};
        for (int u = v_lo; u <= v_hi; u++) {
            const int us = rstart(u);
            if (us == rstart(u + 1)) continue;
            if (own && u == vl) {
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int c = 0; c < TT; c++) sum[a][c] += acc[a][c];
                continue;
            }
            const int sl = 2 * (x * Pg + u) + (us >= tb0 ? 0 : 1);  // range u starts in tile t, or ends in it
            const __amdgpu_buffer_rsrc_t rp = make_rsrc(part + (size_t)sl * kPart, kPart * 16);
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int c = 0; c < TT; c++)
                    sum[a][c] += __builtin_bit_cast(
                        f4, __builtin_amdgcn_raw_buffer_load_b128(rp, (uint32_t)(((a * TT + c) * kPT + tid) * 16), 0, 1));
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < TT; c++) acc[a][c] = sum[a][c];
        store(S, n0, tg);
    }
    }
    __builtin_amdgcn_s_waitcnt(0);  // no load into LDS is in flight when the workgroup's LDS is given back
}

static size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

template <int TT> static const void *pf_fn(uint32_t type, bool dots) {
    if (type == MIQ_TYPE_Q4_K) return dots ? (const void *)pf16_kernel<MIQ_TYPE_Q4_K, TT, true> : (const void *)pf16_kernel<MIQ_TYPE_Q4_K, TT>;
    if (type == MIQ_TYPE_Q5_K) return dots ? (const void *)pf16_kernel<MIQ_TYPE_Q5_K, TT, true> : (const void *)pf16_kernel<MIQ_TYPE_Q5_K, TT>;
    return dots ? (const void *)pf16_kernel<MIQ_TYPE_Q6_K, TT, true> : (const void *)pf16_kernel<MIQ_TYPE_Q6_K, TT>;
}
static const void *pf_fn(uint32_t type, int TT, bool dots) {
    switch (TT) {
    case 2: return pf_fn<2>(type, dots);
    case 3: return pf_fn<3>(type, dots);
    case 4: return pf_fn<4>(type, dots);
    case 5: return pf_fn<5>(type, dots);
    case 6: return pf_fn<6>(type, dots);
    case 7: return pf_fn<7>(type, dots);
    default: return pf_fn<8>(type, dots);
    }
}
template <int TT> static const void *pf_pre_fn(bool quant) {
    return quant ? (const void *)pf_quant_kernel<TT> : (const void *)pf_prep_kernel<TT>;
}
static const void *pf_pre_fn(int TT, bool quant) {
    switch (TT) {
    case 2: return pf_pre_fn<2>(quant);
    case 3: return pf_pre_fn<3>(quant);
    case 4: return pf_pre_fn<4>(quant);
    case 5: return pf_pre_fn<5>(quant);
    case 6: return pf_pre_fn<6>(quant);
    case 7: return pf_pre_fn<7>(quant);
    default: return pf_pre_fn<8>(quant);
    }
}

// more than 64 KiB of dynamic LDS (TT = 8)
static int pf_lds_limit() {
    static bool lds_set[64] = {false};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        set_error("miq prefill: no current device");
        return MIQ_EHIP;
    }
    if (!lds_set[dev]) {
        for (uint32_t type : {MIQ_TYPE_Q4_K, MIQ_TYPE_Q5_K, MIQ_TYPE_Q6_K})
            for (int TT = 2; TT <= 8; TT++)
                for (bool dots : {false, true})
                    if (hipFuncSetAttribute(pf_fn(type, TT, dots), hipFuncAttributeMaxDynamicSharedMemorySize, pf_lds_bytes(TT)) != hipSuccess) {
                        set_error("miq prefill: cannot raise the LDS limit to %d bytes", pf_lds_bytes(TT));
                        return MIQ_EHIP;
                    }
        lds_set[dev] = true;
    }
    return MIQ_OK;
}

bool pf16_serves(const miq_seg *s) { return s->type == MIQ_TYPE_Q4_K || s->type == MIQ_TYPE_Q5_K || s->type == MIQ_TYPE_Q6_K; }

// Token tiles of 16*TT tokens: the fewest, and of those the narrowest, that cover TB.
static int pf_tile(int TB, int *mt) {
    *mt = (TB + 127) / 128;
    const int per = (TB + *mt - 1) / *mt;
    return per <= 32 ? 2 : (per + 15) / 16;
}

// This GEMM against the split-K 16-token kernel, by a model of measured times
// (us; 32..1024 tokens, rows x K from 3584 x 1024 to 17408 x 5120 and
// 5120 x 17408; NK = rows * K in millions):
//   16-token kernel  8 + c16 * ceil(TB / 16) * NK   (weights once per 16 tokens)
//   this kernel      a + (t0 + t1 * TT) * B + TT / 4 * C
// B = 256-value blocks of 256 x 16*TT tiles per workgroup, C = workgroups that
// share a tile (2 where the tiles outnumber them), each but the last leaving a
// partial that the last adds.  At 17408 x 5120 Q4_K the lines cross at 32 tokens
// (29.8 against 30.4 us; 33 tokens 33.5 / 52.7), at 7168 x 5120 Q5_K between 128
// (one tile that nine workgroups share, 47.2 / 45.5) and 129 (two, 38.5 / 49.7), at
// 3584 x 1024 past 512 (30.1 / 26.3).
bool pf16_prefers(const miq_seg *s, int TB) {
    int n_cu = 0, mt = 0;
    if (device_cus(&n_cu) != MIQ_OK) n_cu = 256;
    const int TT = pf_tile(TB, &mt);
    const bool q6 = s->type == MIQ_TYPE_Q6_K;
    const double nkb = s->K / 256, T = (double)((s->n_rows + kPN - 1) / kPN) * mt;
    const double P = T * nkb < n_cu ? T * nkb : n_cu;
    const double C = T >= P ? 2.0 : P / T;
    const double nk = (double)s->n_rows * s->K * 1e-6;
    const double t = q6 ? 0.9 + 0.9 * TT : 1.15 + 0.57 * TT;
    return (q6 ? 22.0 : 18.0) + t * T * nkb / P + 0.25 * TT * C < 8.0 + (q6 ? 0.203 : 0.112) * ((TB + 15) / 16) * nk;
}

// The batches that miq_i8_gemm_noalloc refuses (they run on a kernel that needs
// a workspace) are fixed by this rule, whatever pf16_prefers() says, so that no
// shape it serves is lost when the cross-over moves; without a workspace
// (stream capture before the shape was run) the batches outside it fall back
// to the 16-token kernel.
bool pf16_refuses_noalloc(const miq_seg *s, int TB) {
    double c16, a0, ac, cpf;
    switch (s->type) {
    case MIQ_TYPE_Q4_K: c16 = 0.15; a0 = 44.0; ac = 4.3; cpf = 0.49; break;
    case MIQ_TYPE_Q5_K: c16 = 0.157; a0 = 44.0; ac = 4.3; cpf = 0.52; break;
    default: c16 = 0.255; a0 = 56.0; ac = 3.6; cpf = 0.70; break;  // Q6_K
    }
    int n_cu = 0;
    if (device_cus(&n_cu) != MIQ_OK) n_cu = 256;
    const double P = 2.0 * n_cu, mt = (TB + 127) / 128;
    const double T = (double)((s->n_rows + 127) / 128) * mt;
    const double C = T >= P ? 2.0 : P / T;
    const double nk = (double)s->n_rows * s->K * 1e-6;
    return a0 + ac * C + cpf * mt * nk < c16 * ((TB + 15) / 16) * nk;
}

static int launch(hipStream_t stream, const miq_seg *segs, int n_segs, int TB, int32_t *dots, bool quant, bool *no_ws) {
    const miq_seg *s = segs;
    const int K = s->K;
    const long nkb = K / 256;
    if ((size_t)TB * K * 2 >= 0xFFFFFFF0u) {
        set_error("miq prefill: activation of %d x %d exceeds the 4 GiB buffer window", TB, K);
        return MIQ_UNSUPPORTED;
    }
    PfArgs A{};
    const int TT = pf_tile(TB, &A.mt);
    A.row_bytes = (uint32_t)miq_row_bytes(s->type, K);
    A.K = K;
    A.TB = TB;
    A.dots = dots;
    A.astray = sw(kSwXcdAstray);
    int n_cu = 0;
    if (const int rc = device_cus(&n_cu)) return rc;
    if (const int rc = pf_lds_limit()) return rc;
    PfSeg seg[kPfSegs];
    int first[kPfSegs + 1] = {0}, n_launch = 1;  // launch l: segments [first[l], first[l + 1])
    uint32_t slots = 0, tiles = 0, max_slots = 0, max_tiles = 0;
    const size_t slot_bytes = (size_t)2 * TT * kPT * 16;
    for (int i = 0; i < n_segs; i++) {
        PfSeg &g = seg[i];
        g.w = (const uint8_t *)segs[i].w;
        g.w_bytes = dword_span((size_t)segs[i].n_rows * A.row_bytes);
        g.out = segs[i].out;
        g.residual = segs[i].residual;
        g.n_rows = segs[i].n_rows;
        g.out_stride = segs[i].out_stride;
        g.alpha = segs[i].alpha;
        g.vec_out = ((uintptr_t)g.out % 16 == 0) && (g.out_stride % 4 == 0) && (!g.residual || (uintptr_t)g.residual % 16 == 0);
        // One round of workgroups, one per CU, each taking an equal share of the
        // tiles' K blocks (stream-K); data-parallel rounds of one tile per
        // workgroup where the tiles divide evenly.
        g.nt = (g.n_rows + kPN - 1) / kPN;
        const long T = (long)g.nt * A.mt;
        long P = (long)n_cu / 8 * 8, rounds = T / P, sk = T % P;
        if (sk > 0) {
            rounds = 0;
            sk = T;
        }
        if (rounds == 0 && sk * nkb < P) P = sk * nkb >= 8 ? sk * nkb / 8 * 8 : sk * nkb;
        if (dots) {  // tile (w % 8) * (P / 8) + w / 8 of workgroup w is a permutation when 8 divides P
            rounds = 1;
            P = (T + 7) / 8 * 8;
            sk = 0;
        }
        g.P = (int)P;
        g.rounds = (int)rounds;
        g.xmap = !dots && sk >= 8 && P % 8 == 0;
        const uint32_t need = sk ? (uint32_t)(2 * P) : 0;
        if (i > first[n_launch - 1] && (slots + need) * slot_bytes > kPfPartBytes) {
            first[n_launch++] = i;
            slots = tiles = 0;
        }
        g.poff = slots;
        g.coff = tiles;
        slots += need;
        tiles += (uint32_t)T;
        max_slots = slots > max_slots ? slots : max_slots;
        max_tiles = tiles > max_tiles ? tiles : max_tiles;
    }
    first[n_launch] = n_segs;
    const size_t rec_bytes = align_up((size_t)A.mt * nkb * pf_rec_bytes(TT), 256);
    void *ws = nullptr, *cw = nullptr;
    *no_ws = true;
    if (const int rc = workspace_get(stream, kWsPrefill, rec_bytes + max_slots * slot_bytes, &ws)) return rc;
    if (const int rc = workspace_get(stream, kWsPrefillCnt, (size_t)max_tiles * 8, &cw, true)) return rc;
    *no_ws = false;
    A.rec = reinterpret_cast<const uint8_t *>(ws);
    A.part = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(ws) + rec_bytes);
    A.cnt = reinterpret_cast<uint64_t *>(cw);
    int nb = (int)nkb, tb = TB, stride = s->x_stride;
    uint8_t *rec = reinterpret_cast<uint8_t *>(ws);
    hipError_t e;
    if (quant) {
        void *pa[] = {(void *)&s->x, (void *)&s->act_up, &stride, (void *)&s->x8, (void *)&s->xmeta, (void *)&s->xsumq, &tb, &nb, &rec};
        e = hipLaunchKernel(pf_pre_fn(TT, true), dim3((unsigned)(A.mt * TT * nkb)), dim3(1024), pa, 0, stream);
    } else {
        uint32_t nx = (uint32_t)(A.mt * nkb * 8 * TT * 64), na = (uint32_t)(A.mt * nkb * TT * 16);
        void *pa[] = {(void *)&s->x8, (void *)&s->xmeta, (void *)&s->xsumq, &tb, &nb, &nx, &na, &rec};
        e = hipLaunchKernel(pf_pre_fn(TT, false), dim3((nx + na + 255) / 256), dim3(256), pa, 0, stream);
    }
    if (e != hipSuccess) return check_launch("miq prefill");
    void *ka[] = {&A};
    for (int l = 0; l < n_launch; l++) {
        int grid = 0;
        A.nseg = first[l + 1] - first[l];
        for (int i = 0; i < A.nseg; i++) {
            A.seg[i] = seg[first[l] + i];
            grid = A.seg[i].P > grid ? A.seg[i].P : grid;
        }
        if (hipLaunchKernel(pf_fn(s->type, TT, dots != nullptr), dim3((unsigned)grid), dim3(kPT), ka, pf_lds_bytes(TT), stream) != hipSuccess)
            return check_launch("miq prefill");
    }
    return check_launch("miq prefill");
}

int launch_pf16(hipStream_t stream, const miq_seg *segs, int n_segs, int TB, bool quant, bool *no_ws) {
    *no_ws = false;
    return launch(stream, segs, n_segs, TB, nullptr, quant, no_ws);
}

// Parity form (miq_group_dots path 2): one tile per workgroup with every
// 32-group's MFMA result written to `out`: sc * I, for Q6_K the two planes' sum
// sc0 * I0 + sc1 * I1 of the group's 16-value sub-groups, I = sum (q - 32) * x8.
int launch_pf16_dots(hipStream_t stream, const miq_seg *s, int TB, int32_t *out) {
    if (!pf16_serves(s)) {
        set_error("miq_group_dots: path 2 (the fp16 prefill decoder) serves Q4_K, Q5_K and Q6_K");
        return MIQ_UNSUPPORTED;
    }
    bool no_ws;
    return launch(stream, s, 1, TB, out, false, &no_ws);
}

}  // namespace miq
