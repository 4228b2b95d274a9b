// Chunked-prefill GEMM on int8 MFMA (v_mfma_i32_32x32x32_i8, full rate on
// gfx950): out[t][n] = alpha * sum_k W[n][k] * act_t[k] (+ residual) for many
// tokens.
//
// Workgroup tile: 64 tokens x 128 rows, 4 waves in a 2x2 arrangement, each
// wave 32 tokens x 64 rows = 1x2 MFMA tiles.  The K loop walks one 256-value
// block per step.  Each step the workgroup decodes its 128 rows' Q4_K/Q5_K/
// Q8_0 bytes once into int8 codes in LDS (plus per-(row, group) fp32 scales)
// and copies the 128 tokens' codes and scales next to them; the next step's
// raw bytes are fetched into registers while the current step computes.  A tile's
// K range may be cut into slices on several workgroups (m32_slices).
//
// One MFMA K step is one 32-value group, so every MFMA result is the exact
// int32 group dot of the reference (i8.cpp:49-57,109-118; q4exp.cpp:457-467);
// the fp32 epilogue applies sx*d*sc per (token, row, group) on the VALU and the
// rank-G dmin*m*xsum term (i8.cpp:60,120) runs on fp32 MFMA
// (v_mfma_f32_32x32x2_f32: tokens x 2 groups times 2 groups x rows).
// MFMA C layout (32x32): lane l, register v -> row 8*(v/4) + 4*(l/32) + v%4
// (tokens), column l%32 (weight rows).
#include "miq_internal.h"
#include "miq_units.h"

namespace miq {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u32 __attribute__((ext_vector_type(4)));

constexpr int kBM = 64;   // tokens per workgroup
constexpr int kBN = 128;  // weight rows per workgroup
// LDS rows of 256 codes; the 16-byte chunk c of row r lives at chunk c ^ (r & 15),
// so the 32 rows a b128 operand read touches hit distinct banks.
__device__ __forceinline__ int swz(int r, int chunk) { return r * 256 + ((chunk ^ (r & 15)) << 4); }

struct M32Args {
    const uint8_t *w;
    uint32_t w_bytes;
    uint32_t row_bytes;
    int K;
    int n_rows;
    int TB;
    const int8_t *x8;
    const float *xmeta;
    const int32_t *xsumq;
    float *out;
    int out_stride;
    const float *residual;
    float alpha;
    int32_t *dots;  // parity form: [TB][n_rows][K/32] int32 group dots
    int nt, T;      // row tiles, tiles
    int S;          // K slices per tile
    float *part;    // [tile][slice][8][256 threads][4] partial sums (S > 1)
    uint64_t *cnt;  // [tile] arrival counters (xcd_arrival), zero between launches
    int astray;     // a test: every second slice takes itself for one on another XCD
};

// LDS layout of one step
struct M32Lds {
    uint8_t wq[kBN * 256];        // weight codes [row][256], swizzled chunks
    uint8_t xq[kBM * 256];        // activation codes [token][256], swizzled chunks
    float dsc[8][kBN];            // d*sc per (group, row)
    float dmm[8][kBN];            // dmin*m per (group, row)
    float sx[8][kBM];             // activation scale per (group, token)
    float u[8][kBM];              // sx * (s0 + s1) per (group, token)
};

// Raw bytes one thread fetches for a step: two weight units (Q4_K/Q5_K:
// 16 B header + 32 B qs (+ 32 B qh for Q5_K) of a quarter block; Q8_0: a
// quarter of the 8-block step), four 16-byte activation chunks and one
// chunk each of xmeta / xsumq.
template <uint32_t TYPE> struct M32Raw {
    uint4 w[2][TYPE == MIQ_TYPE_Q5_K ? 5 : (TYPE == MIQ_TYPE_Q8_0 ? 5 : 3)];
    FetchQ6K f6[2];  // Q6_K: unit (row, blk2, half) as fetch_q6k loads it
    uint32_t sh6[2];  // and its block offset's byte shift
    uint4 x[4];
    uint4 m, q;
};

template <uint32_t TYPE>
__device__ __forceinline__ void m32_fetch(M32Raw<TYPE> &R, const M32Args &A, __amdgpu_buffer_rsrc_t rw,
                                          __amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t rm,
                                          __amdgpu_buffer_rsrc_t rq, int n0, int t0, int kb) {
    const int tid = threadIdx.x;
    // weights: unit = (row r, quarter c), 512 units, two per thread
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int unit = tid + 256 * i;
        const int r = unit >> 2, c = unit & 3;
        const int row = n0 + r;
        const uint32_t base = row < A.n_rows ? (uint32_t)row * A.row_bytes : A.w_bytes;
        if constexpr (TYPE == MIQ_TYPE_Q4_K) {
            const uint32_t b = base + (uint32_t)kb * kQ4KBytes;
            R.w[i][0] = bload16(rw, b);
            R.w[i][1] = bload16(rw, b + 16 + 32 * c);
            R.w[i][2] = bload16(rw, b + 32 + 32 * c);
        } else if constexpr (TYPE == MIQ_TYPE_Q5_K) {
            const uint32_t b = base + (uint32_t)kb * kQ5KBytes;
            R.w[i][0] = bload16(rw, b);
            R.w[i][1] = bload16(rw, b + 48 + 32 * c);
            R.w[i][2] = bload16(rw, b + 64 + 32 * c);
            R.w[i][3] = bload16(rw, b + 16);
            R.w[i][4] = bload16(rw, b + 32);
        } else if constexpr (TYPE == MIQ_TYPE_Q6_K) {  // c = blk2 * 2 + half (2-byte aligned blocks)
            R.f6[i] = fetch_q6k(rw, base + (uint32_t)kb * kQ6KBytes, c);
            R.sh6[i] = (base + (uint32_t)kb * kQ6KBytes) & 3u;
        } else {  // Q8_0: quarter c = blocks 2c, 2c+1 of the step (68 bytes, 4-byte aligned)
            const uint32_t b = base + (uint32_t)kb * 272u + 68u * c;
            R.w[i][0] = bload16(rw, b);
            R.w[i][1] = bload16(rw, b + 16);
            R.w[i][2] = bload16(rw, b + 32);
            R.w[i][3] = bload16(rw, b + 48);
            R.w[i][4] = make_uint4(bload4(rw, b + 64), 0, 0, 0);
        }
    }
    // activations: group g, token tt, half hf -> 16-byte chunk; 1024 chunks, 4 per thread
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ch = tid + 256 * i;
        const int g = ch >> 7, rest = ch & 127, tt = rest >> 1, hf = rest & 1;
        const int t = t0 + tt;
        const uint32_t off = t < A.TB ? ((uint32_t)(kb * 8 + g) * A.TB + t) * 32 + 16 * hf : 0xFFFFFFF0u;
        R.x[i] = bload16(rx, off);
    }
    // scales and sums: group g, token pair p -> 16 bytes of xmeta and of xsumq; 256 chunks
    {
        const int g = tid >> 5, p = tid & 31;
        const int t = t0 + 2 * p;
        const uint32_t off = t < A.TB ? ((uint32_t)(kb * 8 + g) * A.TB + t) * 8 : 0xFFFFFFF0u;
        R.m = bload16(rm, off);
        R.q = bload16(rq, off);
    }
}

template <uint32_t TYPE>
__device__ __forceinline__ void m32_store(const M32Raw<TYPE> &R, M32Lds &L, const M32Args &A, int n0, int t0) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int unit = tid + 256 * i;
        const int r = unit >> 2, c = unit & 3;
        const bool ok = n0 + r < A.n_rows;
        if constexpr (TYPE == MIQ_TYPE_Q4_K || TYPE == MIQ_TYPE_Q5_K) {
            const uint4 hdr = R.w[i][0];
            const uint32_t q[8] = {R.w[i][1].x, R.w[i][1].y, R.w[i][1].z, R.w[i][1].w,
                                   R.w[i][2].x, R.w[i][2].y, R.w[i][2].z, R.w[i][2].w};
            uint32_t lo[8], hi[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                lo[k] = q[k] & 0x0F0F0F0Fu;
                hi[k] = (q[k] >> 4) & 0x0F0F0F0Fu;
            }
            if constexpr (TYPE == MIQ_TYPE_Q5_K) {
                const uint32_t h[8] = {R.w[i][3].x, R.w[i][3].y, R.w[i][3].z, R.w[i][3].w,
                                       R.w[i][4].x, R.w[i][4].y, R.w[i][4].z, R.w[i][4].w};
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    lo[k] |= ((h[k] >> (2 * c)) & 0x01010101u) << 4;
                    hi[k] |= ((h[k] >> (2 * c + 1)) & 0x01010101u) << 4;
                }
            }
            // group 2c codes -> chunks 4c, 4c+1; group 2c+1 -> chunks 4c+2, 4c+3
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 0)) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 1)) = make_uint4(lo[4], lo[5], lo[6], lo[7]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 2)) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 3)) = make_uint4(hi[4], hi[5], hi[6], hi[7]);
            const float d = h2f(hdr.x), dm = h2f(hdr.x >> 16);
            int sc0, m0, sc1, m1;
            scale_min_k4(2 * c, hdr.y, hdr.z, hdr.w, sc0, m0);
            scale_min_k4(2 * c + 1, hdr.y, hdr.z, hdr.w, sc1, m1);
            L.dsc[2 * c][r] = ok ? d * (float)sc0 : 0.0f;
            L.dsc[2 * c + 1][r] = ok ? d * (float)sc1 : 0.0f;
            L.dmm[2 * c][r] = ok ? dm * (float)m0 : 0.0f;
            L.dmm[2 * c + 1][r] = ok ? dm * (float)m1 : 0.0f;
        } else if constexpr (TYPE == MIQ_TYPE_Q6_K) {
            // unit c = (blk2, half): plane p's 16 codes are sub-group s = 8*blk2 + 2p + half,
            // LDS chunk s; MFMA group g = 4*blk2 + p takes half 0 / 1 on its two lane halves,
            // whose scales go to dsc[g] / dmm[g]
            const RawQ6K u = dec_q6k(R.f6[i], R.sh6[i]);
            const int blk2 = c >> 1, half = c & 1;
            const uint32_t l0[4] = {u.l0.x, u.l0.y, u.l0.z, u.l0.w};
            const uint32_t l1[4] = {u.l1.x, u.l1.y, u.l1.z, u.l1.w};
            const uint32_t hh[4] = {u.h.x, u.h.y, u.h.z, u.h.w};
            const float d = h2f(u.dbits);
#pragma unroll
            for (int p = 0; p < 4; p++) {
                uint32_t q[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t src = (p & 1) ? l1[k] : l0[k];
                    q[k] = q6_signed(((p >= 2 ? (src >> 4) : src) & 0x0F0F0F0Fu) | (((hh[k] >> (2 * p)) & 0x03030303u) << 4));
                }
                *reinterpret_cast<uint4 *>(L.wq + swz(r, 8 * blk2 + 2 * p + half)) = make_uint4(q[0], q[1], q[2], q[3]);
                const float ds = ok ? d * (float)q6k_scale(u, c, p) : 0.0f;
                if (half) L.dmm[4 * blk2 + p][r] = ds;
                else L.dsc[4 * blk2 + p][r] = ds;
            }
        } else {  // Q8_0 blocks 2c, 2c+1: 68 bytes
            const uint32_t w[17] = {R.w[i][0].x, R.w[i][0].y, R.w[i][0].z, R.w[i][0].w, R.w[i][1].x, R.w[i][1].y,
                                    R.w[i][1].z, R.w[i][1].w, R.w[i][2].x, R.w[i][2].y, R.w[i][2].z, R.w[i][2].w,
                                    R.w[i][3].x, R.w[i][3].y, R.w[i][3].z, R.w[i][3].w, R.w[i][4].x};
            uint32_t a[8], b[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                a[k] = __builtin_amdgcn_alignbyte(w[k + 1], w[k], 2);
                b[k] = w[9 + k];
            }
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 0)) = make_uint4(a[0], a[1], a[2], a[3]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 1)) = make_uint4(a[4], a[5], a[6], a[7]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 2)) = make_uint4(b[0], b[1], b[2], b[3]);
            *reinterpret_cast<uint4 *>(L.wq + swz(r, 4 * c + 3)) = make_uint4(b[4], b[5], b[6], b[7]);
            L.dsc[2 * c][r] = ok ? h2f(w[0]) : 0.0f;
            L.dsc[2 * c + 1][r] = ok ? h2f(w[8] >> 16) : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ch = tid + 256 * i;
        const int g = ch >> 7, rest = ch & 127, tt = rest >> 1, hf = rest & 1;
        *reinterpret_cast<uint4 *>(L.xq + swz(tt, 2 * g + hf)) = R.x[i];
    }
    {
        const int g = tid >> 5, p = tid & 31;
        const int t = t0 + 2 * p;
        const float s0 = t < A.TB ? __builtin_bit_cast(float, R.m.x) : 0.0f;
        const float s1 = t + 1 < A.TB ? __builtin_bit_cast(float, R.m.z) : 0.0f;
        L.sx[g][2 * p] = s0;
        L.sx[g][2 * p + 1] = s1;
        L.u[g][2 * p] = s0 * (float)((int)R.q.x + (int)R.q.y);
        L.u[g][2 * p + 1] = s1 * (float)((int)R.q.z + (int)R.q.w);
    }
}

// DOTS: the parity form -- every MFMA result (the exact int32 group dot)
// goes to A.dots and nothing else is computed
// The forms: a workgroup takes a whole tile; a K slice of one; a whole tile in
// the parity form.  The first is an instance of its own because the slices'
// bookkeeping in its loop's registers costs 2 to 3 % (17408 x 5120 Q8_0 at 333
// tokens 163 us, 167 with S == 1 as a run-time case of the second).
enum M32Form { kM32Whole, kM32Sliced, kM32Dots };
template <uint32_t TYPE, M32Form FORM>
__global__ __launch_bounds__(256, 2) void mfma32_kernel(M32Args A) {
    constexpr bool DOTS = FORM == kM32Dots;
    extern __shared__ __align__(16) uint8_t lds_raw[];
    M32Lds &L = *reinterpret_cast<M32Lds *>(lds_raw);
    // Slices of one tile run on one XCD (the dispatcher deals by blockIdx % 8):
    // blockIdx = 8 * (tile / 8 * S + slice) + tile % 8.
    int slice = 0, tile = blockIdx.x;
    if constexpr (FORM == kM32Sliced) {
        const int bb = blockIdx.x >> 3;
        slice = bb % A.S;
        tile = bb / A.S * 8 + (blockIdx.x & 7);
        if (tile >= A.T) return;
    }
    const int n0 = tile % A.nt * kBN, t0 = tile / A.nt * kBM;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wt = (wave >> 1) * 32, wn = (wave & 1) * 64;  // wave tile origin (tokens, rows)
    const int l32 = lane & 31, hk = lane >> 5;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(A.w, A.w_bytes);
    const uint32_t xbytes = (uint32_t)(A.K / 32) * A.TB * 32, mbytes = (uint32_t)(A.K / 32) * A.TB * 8;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(A.x8, xbytes);
    const __amdgpu_buffer_rsrc_t rm = make_rsrc(A.xmeta, mbytes), rq = make_rsrc(A.xsumq, mbytes);

    v16f acc[2];
    const int steps = A.K / 256;
    int kb0 = 0, nkb = steps;  // this workgroup's steps of the tile
    if constexpr (FORM == kM32Sliced) {
        kb0 = slice * steps / A.S;
        nkb = (slice + 1) * steps / A.S;
    }
    v16f t2[2];
sum_steps:
#pragma unroll
    for (int j = 0; j < 2; j++) {
        acc[j] = v16f{};
        t2[j] = v16f{};
    }

    M32Raw<TYPE> R;
    m32_fetch<TYPE>(R, A, rw, rx, rm, rq, n0, t0, kb0);
    for (int kb = kb0; kb < nkb; kb++) {
        __syncthreads();  // the previous step's LDS reads are done
        m32_store<TYPE>(R, L, A, n0, t0);
        __syncthreads();
        if (kb + 1 < nkb) m32_fetch<TYPE>(R, A, rw, rx, rm, rq, n0, t0, kb + 1);
#pragma unroll 2
        for (int g = 0; g < 8; g++) {
            // operands: A = tokens (rows i), B = weight rows (columns j); lane half hk takes k 16*hk..16*hk+15
            const v4i32 av = *reinterpret_cast<const v4i32 *>(L.xq + swz(wt + l32, 2 * g + hk));
            v4i32 bv[2];
#pragma unroll
            for (int j = 0; j < 2; j++) bv[j] = *reinterpret_cast<const v4i32 *>(L.wq + swz(wn + 32 * j + l32, 2 * g + hk));
            if constexpr (TYPE == MIQ_TYPE_Q6_K) {
                // two 16-value sub-groups with their own scales: one MFMA per
                // sub-group, the other lane half's weights zeroed
                const v4i32 zero{0, 0, 0, 0};
                v16i I0[2], I1[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    I0[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, hk ? zero : bv[j], v16i{}, 0, 0, 0);
                    I1[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, hk ? bv[j] : zero, v16i{}, 0, 0, 0);
                }
                if constexpr (DOTS) {  // the unsigned-code sums wd = I + 32 * xsum of the half (i8.cpp:149)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int row = n0 + wn + 32 * j + l32;
#pragma unroll
                        for (int v = 0; v < 16; v++) {
                            const int t = t0 + wt + 8 * (v >> 2) + 4 * hk + (v & 3);
                            if (t < A.TB && row < A.n_rows) {
                                const int32_t *xs = A.xsumq + ((size_t)(8 * kb + g) * A.TB + t) * 2;
                                int32_t *o = A.dots + ((size_t)t * A.n_rows + row) * (A.K / 16) + 2 * (8 * kb + g);
                                o[0] = I0[j][v] + 32 * xs[0];
                                o[1] = I1[j][v] + 32 * xs[1];
                            }
                        }
                    }
                    continue;
                }
                float sxr[16];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4 sv = *reinterpret_cast<const float4 *>(&L.sx[g][wt + 8 * q + 4 * hk]);
                    sxr[4 * q + 0] = sv.x;
                    sxr[4 * q + 1] = sv.y;
                    sxr[4 * q + 2] = sv.z;
                    sxr[4 * q + 3] = sv.w;
                }
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float ds0 = L.dsc[g][wn + 32 * j + l32], ds1 = L.dmm[g][wn + 32 * j + l32];
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        acc[j][v] += sxr[v] * (ds0 * (float)I0[j][v]);
                        acc[j][v] += sxr[v] * (ds1 * (float)I1[j][v]);
                    }
                }
                continue;
            }
            v16i I[2];
#pragma unroll
            for (int j = 0; j < 2; j++) I[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv[j], v16i{}, 0, 0, 0);
            if constexpr (DOTS) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int row = n0 + wn + 32 * j + l32;
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const int t = t0 + wt + 8 * (v >> 2) + 4 * hk + (v & 3);
                        if (t < A.TB && row < A.n_rows)
                            A.dots[((size_t)t * A.n_rows + row) * (A.K / 32) + 8 * kb + g] = I[j][v];
                    }
                }
                continue;
            }
            // token scales of this lane's C rows: tokens 8*(v/4) + 4*hk + v%4
            float sxr[16];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 sv = *reinterpret_cast<const float4 *>(&L.sx[g][wt + 8 * q + 4 * hk]);
                sxr[4 * q + 0] = sv.x;
                sxr[4 * q + 1] = sv.y;
                sxr[4 * q + 2] = sv.z;
                sxr[4 * q + 3] = sv.w;
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float dsc = L.dsc[g][wn + 32 * j + l32];
#pragma unroll
                for (int v = 0; v < 16; v++) acc[j][v] += sxr[v] * (dsc * (float)I[j][v]);
            }
        }
        if constexpr (TYPE != MIQ_TYPE_Q8_0 && TYPE != MIQ_TYPE_Q6_K && !DOTS) {
            // dmin*m*xsum: A = u (tokens x 2 groups), B = dmin*m (2 groups x rows)
#pragma unroll
            for (int gp = 0; gp < 4; gp++) {
                const int g = 2 * gp + hk;
                const float a = L.u[g][wt + l32];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float b = L.dmm[g][wn + 32 * j + l32];
                    t2[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, t2[j], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 2; j++) acc[j] -= t2[j];
    if constexpr (DOTS) return;
    if (FORM == kM32Sliced && nkb - kb0 < steps) {
        // The last slice of a tile to arrive adds the slices in slice order (the
        // result does not depend on timing); one that finds every other one
        // arrived keeps its sums in registers.  The partials meet in the XCD's
        // L2 (stores drained before the arrival is counted, L1-bypassing
        // loads); where the slices were on several XCDs (see xcd_arrival), the last
        // to arrive computes the whole tile instead, in one sum.
        __shared__ int lflag;
        const __amdgpu_buffer_rsrc_t rp = make_rsrc(reinterpret_cast<v4f32 *>(A.part) + (size_t)tile * A.S * 2048, (uint32_t)A.S * 32768u);
        uint64_t *cnt = A.cnt + tile;
        if (threadIdx.x == 0)
            lflag = xcd_last(__hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), xcd_arrival(A.astray & slice), (uint32_t)A.S) == 1;
        __syncthreads();
        int fl = __builtin_amdgcn_readfirstlane(lflag);
        const bool own = fl;
        if (own) {
            if (threadIdx.x == 0) __hip_atomic_store(cnt, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                __builtin_amdgcn_raw_buffer_store_b128(
                    __builtin_bit_cast(v4u32, v4f32{acc[i >> 2][4 * (i & 3)], acc[i >> 2][4 * (i & 3) + 1], acc[i >> 2][4 * (i & 3) + 2], acc[i >> 2][4 * (i & 3) + 3]}),
                    rp, threadIdx.x * 16, (slice * 8 + i) * 4096, 0);
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (threadIdx.x == 0) {
                const uint64_t one = xcd_arrival(A.astray & slice);
                const uint64_t prev = __hip_atomic_fetch_add(cnt, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lflag = xcd_last(prev, one, (uint32_t)A.S);
                if (lflag) __hip_atomic_store(cnt, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            fl = __builtin_amdgcn_readfirstlane(lflag);
        }
        if (!fl) return;
        if (fl == 2) {
            kb0 = 0;
            nkb = steps;
            goto sum_steps;
        }
        v16f sum[2] = {};
        for (int k = 0; k < A.S; k++) {
            if (own && k == slice) {
#pragma unroll
                for (int j = 0; j < 2; j++) sum[j] += acc[j];
                continue;
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const v4f32 q = __builtin_bit_cast(v4f32, __builtin_amdgcn_raw_buffer_load_b128(rp, threadIdx.x * 16, (k * 8 + i) * 4096, 1));
#pragma unroll
                for (int v = 0; v < 4; v++) sum[i >> 2][4 * (i & 3) + v] += q[v];
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j] = sum[j];
    }
    // write: C[token][row]
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = n0 + wn + 32 * j + l32;
        if (row >= A.n_rows) continue;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int t = t0 + wt + 8 * (v >> 2) + 4 * hk + (v & 3);
            if (t < A.TB) {
                const size_t o = (size_t)t * A.out_stride + row;
                float val = A.alpha * acc[j][v];
                if (A.residual) val += A.residual[o];
                A.out[o] = val;
            }
        }
    }
}

bool mfma32_serves(const miq_seg *s) {
    // Q8_0 rows whose K is not a whole number of 256-value steps go to the 16-token kernel
    return s->type == MIQ_TYPE_Q4_K || s->type == MIQ_TYPE_Q5_K || s->type == MIQ_TYPE_Q6_K ||
           (s->type == MIQ_TYPE_Q8_0 && s->K % 256 == 0);
}

bool mfma32_fills(const miq_seg *s, int TB) {
    if (s->type != MIQ_TYPE_Q6_K || sw(kSwM32Fill) == 0) return true;  // M32_FILL=0: the tiled kernel at any size
    int cus = 0;
    if (device_cus(&cus) != MIQ_OK) return true;
    // measured (Q6_K, K 5120/17408): 136 or 80 tiles lose to the 16-token kernel by 1.4-2.3x, 272 / 320 tiles win by 1.1-1.7x
    return (long)((s->n_rows + kBN - 1) / kBN) * ((TB + kBM - 1) / kBM) >= cus;
}

// K slices per tile: as many as two workgroups per CU hold, of at least four
// steps.  A step lasts about 3.4 us, mostly its own latency (decode, two
// barriers), and a second workgroup on the CU makes it only 1.2 times longer:
// 5120 x 5120 Q8_0 took 70 us at any batch from 48 to 333 tokens (40 to 240
// tiles of 20 steps); sliced 25 us at 48, 31 at 128 and 52 at 333.
static int m32_slices(const miq_seg *s, int TB, int n_cu) {
    const int T = ((s->n_rows + kBN - 1) / kBN) * ((TB + kBM - 1) / kBM), nkb = s->K / 256;
    const int S = 2 * n_cu / T, most = nkb / 4;
    return S < 1 || most < 1 ? 1 : S < most ? S : most;
}

// Q8_0: this kernel against the split-K 16-token kernel, by a model of measured
// times (us; 48..512 tokens, 1024 / 5120 / 17408 x 5120; NK in millions).  Checked
// at K = 1024 to 17408, 1024 to 17408 rows and 8 to 512 tokens: nowhere more than
// 1.2 us (3 %) slower than this kernel unsliced from 48 tokens on.
// 16-token kernel 8 + 0.355 * ceil(TB / 16) * NK; this kernel 3.4 us a step,
// 1.2 times that with two workgroups per CU, 1.63 for each 2 * n_cu tiles
// beyond, and about 1.2 us per slice that the last one adds.
bool mfma32_prefers(const miq_seg *s, int TB) {
    if (s->type != MIQ_TYPE_Q8_0) return true;
    int n_cu = 0;
    if (device_cus(&n_cu) != MIQ_OK) n_cu = 256;
    const int S = m32_slices(s, TB, n_cu), nkb = s->K / 256;
    const double W = (double)((s->n_rows + kBN - 1) / kBN) * ((TB + kBM - 1) / kBM) * S;
    const double f = W <= n_cu ? 1.0 : W <= 2 * n_cu ? 1.2 : 1.63 * W / (2 * n_cu);
    return 6.0 + 3.4 * nkb / S * f + 1.2 * (S - 1) < 8.0 + 0.355 * ((TB + 15) / 16) * (double)s->n_rows * s->K * 1e-6;
}

template <uint32_t TYPE> static void m32_start(const M32Args &A, M32Form form, dim3 grid, hipStream_t stream) {
    constexpr size_t lds = sizeof(M32Lds);
    if (form == kM32Sliced) hipLaunchKernelGGL((mfma32_kernel<TYPE, kM32Sliced>), grid, dim3(256), lds, stream, A);
    else if (form == kM32Dots) hipLaunchKernelGGL((mfma32_kernel<TYPE, kM32Dots>), grid, dim3(256), lds, stream, A);
    else hipLaunchKernelGGL((mfma32_kernel<TYPE, kM32Whole>), grid, dim3(256), lds, stream, A);
}

int launch_mfma32(hipStream_t stream, const miq_seg *s, int TB, int32_t *dots) {
    M32Args A{};
    A.w = (const uint8_t *)s->w;
    A.row_bytes = (uint32_t)miq_row_bytes(s->type, s->K);
    A.w_bytes = dword_span((size_t)s->n_rows * A.row_bytes);
    A.K = s->K;
    A.n_rows = s->n_rows;
    A.TB = TB;
    A.x8 = s->x8;
    A.xmeta = s->xmeta;
    A.xsumq = s->xsumq;
    A.out = s->out;
    A.out_stride = s->out_stride;
    A.residual = s->residual;
    A.alpha = s->alpha;
    A.nt = (s->n_rows + kBN - 1) / kBN;
    A.T = A.nt * ((TB + kBM - 1) / kBM);
    int n_cu = 0;
    if (const int rc = device_cus(&n_cu)) return rc;
    A.S = dots ? 1 : m32_slices(s, TB, n_cu);
    // no scratch for the partials (a stream that captures a graph or has none of
    // its own, miq_i8_gemm_noalloc): unsliced
    if (A.S > 1 && scratch_get(stream, (size_t)A.T * A.S * 32768, A.T, &A.part, &A.cnt) != MIQ_OK) A.S = 1;
    A.astray = sw(kSwXcdAstray);
    const M32Form form = dots ? kM32Dots : A.S > 1 ? kM32Sliced : kM32Whole;
    const dim3 grid((unsigned)(form == kM32Sliced ? (A.T + 7) / 8 * 8 * A.S : A.T));
    A.dots = dots;  // the parity form is miq_group_dots path 3
    switch (s->type) {
    case MIQ_TYPE_Q4_K: m32_start<MIQ_TYPE_Q4_K>(A, form, grid, stream); break;
    case MIQ_TYPE_Q5_K: m32_start<MIQ_TYPE_Q5_K>(A, form, grid, stream); break;
    case MIQ_TYPE_Q6_K: m32_start<MIQ_TYPE_Q6_K>(A, form, grid, stream); break;
    default: m32_start<MIQ_TYPE_Q8_0>(A, form, grid, stream); break;
    }
    return check_launch(dots ? "miq_group_dots" : "miq mfma32");
}

}  // namespace miq
