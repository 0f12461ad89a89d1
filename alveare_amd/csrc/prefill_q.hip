// Prefill products on registered (tiled) weights for gfx950: the path of
// alv_gemv, alv_gemv_bf16 (but where gemm_q.hip's lds_tiles_faster says
// otherwise), alv_ffn_fused and alv_ffn_fused_bf16 from 17 (bf16 activations) or
// 33 (fp32) tokens.
//
// C[M, N] = X[M, K] * dequant(W)[N, K]^T in two launches:
//   1. pack_x_kernel lays the activations out once in MFMA operand order
//      (below), splitting fp32 values exactly into three bf16 terms; the FFN's
//      gate/up launch writes its activation in that order itself.
//   2. prefill_kernel: 4 or 8 waves per workgroup; a wave owns RB = 2 16-row
//      tiles of weights (for the GLU one gate, one up) against all TB x 16
//      tokens of the workgroup.
//
// Weights never touch LDS: lane (g, j) of v_mfma_f32_16x16x32_bf16's B operand
// holds 8 consecutive k of row j, one dword of nibbles, so each wave
// dequantizes its own rows straight into operand registers
// (q4_device.h::dequant8_mix), once per workgroup. (Dequantizing into LDS and
// reading back, as gemm_q.hip does, moves 256 KiB per 256 x 256 x 64 step through
// the 128 B per clock of LDS: as long as its matrix instructions take.)
// Activations go from memory straight into LDS (buffer_load ... lds), whole
// operand fragments of 1 KiB, and are read without bank conflicts.
//
// What bounds it: up to 128 tokens waiting, for the L2 (a substep's activations
// are asked for one substep ahead) and for issue. Gate/up of 3840 <-> 15360 at 45
// tokens, 33.8 us: the matrix cores busy 21 % of the time and the vector ALUs
// 36 % (68 clocks of dequantization per 16 x 32 weights a wave, 6.4 us of it),
// a wave's time 38 % at s_waitcnt or a barrier and 27 % at an instruction that is
// ready. Above, LDS reads (every wave reads all of the workgroup's
// activations, 512 KiB per 256 x 256 x 128 substep: 4096 clocks, as many as its
// matrix instructions) at 1.1-1.2 PFLOP/s of the 1.45 that a large bf16 product
// reaches on this card. Eight waves of two row tiles, two per SIMD, rather than
// four of four: a wave alone on its SIMD does not overlap its dequantization
// with its own matrix instructions (512 tokens 194 against 185 us, 3001: 954
// against 880). FFN 3840 <-> 15360, bf16, us per call, gemm_q.hip before and
// this kernel: 17 tokens 70 -> 48, 45: 72 -> 60, 128: 111 -> 77, 200: 146 -> 105,
// 512: 207 -> 183, 1024: 392 -> 323, 3001: 1224 -> 880.
//
// The order of k. A super-step of the tiled layout (512 columns, 16 blocks) is
// taken in T = 4 substeps of 128: substep t multiplies block T g + t in lane
// group g, so a lane's blocks are those its 80-byte run of the tile holds. The
// last super-step of nbl blocks takes T = ceil(nbl / 4) substeps the same way.
// Fragment (16 tokens tb, substep s, octet kk) is 64 x 16 bytes: lane (g, i)
// has token 16 tb + i, the eight columns of octet kk of its block.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "q4_device.h"
#include "q4_host.h"

namespace alv {

namespace {

constexpr int kFragBytes = 1024;
constexpr int kStepBytes = 4 * kFragBytes;  // 16 tokens x one substep

// Substeps of K columns, and the last super-step's.
struct PackGeom {
    int nss;   // super-steps
    int T;     // substeps of the last one
    int nbl;   // its blocks
    int S;     // substeps in all
};

__host__ __device__ inline PackGeom pack_geom(int K) {
    PackGeom p;
    const int nb = K / kBlockK;
    p.nss = (nb + 15) / 16;
    p.nbl = nb - 16 * (p.nss - 1);
    p.T = (p.nbl + 3) / 4;
    p.S = 4 * (p.nss - 1) + p.T;
    return p;
}

// Byte offset of octet o (columns 8 o .. 8 o + 7) of token m.
__device__ __forceinline__ uint32_t pack_offset(const PackGeom& p, int m, int o) {
    const int b = o >> 2, ss = b >> 4, bl = b & 15;
    const int T = ss == p.nss - 1 ? p.T : 4;
    const int g = bl / T, t = bl - g * T;
    return (uint32_t)((m >> 4) * p.S + 4 * ss + t) * kStepBytes + (uint32_t)(o & 3) * kFragBytes +
           (uint32_t)(g * 16 + (m & 15)) * 16u;
}

// Activations into operand order: workgroup (tb, ss) packs 16 tokens x 512
// columns through LDS (rows in, fragments out, both in whole 1 KiB lines).
// Tokens past M and columns past K are zeros. F32: three terms, `tstride`
// bytes apart; flags[tb * nss + ss] != 0 when a second or third term is not zero.
template <bool F32>
__global__ void __launch_bounds__(256) pack_x_kernel(const void* X, int ldx, int M, int K, uint8_t* out, size_t tstride,
                                                     uint32_t* flags) {
    constexpr int NT = F32 ? 3 : 1;
    __shared__ u32x4 tile[NT][16][65];
    const PackGeom p = pack_geom(K);
    const int tb = blockIdx.x, ss = blockIdx.y, tid = threadIdx.x;
    const int T = ss == p.nss - 1 ? p.T : 4;
    bool more = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = tid + 256 * q, i = c >> 6, o = c & 63;
        const int m = tb * 16 + i, k = ss * 512 + o * 8;
        const bool in = m < M && k < K;
        if constexpr (F32) {
            float x[8] = {};
            if (in) __builtin_memcpy(x, static_cast<const float*>(X) + (size_t)m * ldx + k, sizeof(x));
            bf16x8 t[3];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const Split3 sp = split3(x[e]);
                t[0][e] = sp.p0;
                t[1][e] = sp.p1;
                t[2][e] = sp.p2;
            }
            const u32x4 low = __builtin_bit_cast(u32x4, t[1]) | __builtin_bit_cast(u32x4, t[2]);
            more |= ((low[0] | low[1] | low[2] | low[3]) & 0x7FFF7FFFu) != 0;
#pragma unroll
            for (int n = 0; n < 3; ++n) tile[n][i][o] = __builtin_bit_cast(u32x4, t[n]);
        } else {
            u32x4 v = {0, 0, 0, 0};
            if (in) v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(X) + (size_t)m * ldx + k);
            tile[0][i][o] = v;
        }
    }
    if (F32) {
        more = __syncthreads_or(more);
        if (tid == 0) flags[tb * p.nss + ss] = more ? 1u : 0u;
    } else {
        __syncthreads();
    }
    uint8_t* dst = out + (size_t)(tb * p.S + 4 * ss) * kStepBytes;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = tid + 256 * q, t = c >> 8, kk = (c >> 6) & 3, l = c & 63;
        if (t >= T) break;
        const int b = T * (l >> 4) + t;
#pragma unroll
        for (int n = 0; n < NT; ++n)
            *reinterpret_cast<u32x4*>(dst + n * tstride + (size_t)c * 16) =
                b < 16 ? tile[n][l & 15][4 * b + kk] : u32x4{0, 0, 0, 0};
    }
}

// A packed bf16 array [M][K] widened to row-major fp32 (columns K .. ldo - 1 zero).
__global__ void __launch_bounds__(256) unpack_f32_kernel(const uint8_t* in, int M, int K, float* out, int ldo) {
    const PackGeom p = pack_geom(K);
    const int no = ldo / 8;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < (int64_t)M * no; c += (int64_t)gridDim.x * 256) {
        const int m = (int)(c / no), o = (int)(c - (int64_t)m * no);
        u32x4 v = {0, 0, 0, 0};
        if (8 * o < K) v = *reinterpret_cast<const u32x4*>(in + pack_offset(p, m, o));
        float* y = out + (size_t)m * ldo + 8 * o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t w = v[e];
            y[2 * e] = bf16_bits_to_f32(w & 0xFFFFu);
            y[2 * e + 1] = bf16_bits_to_f32(w >> 16);
        }
    }
}

__device__ __forceinline__ float lo_half(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float hi_half(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }

struct PrefillArgs {
    const uint8_t* W0;
    const uint8_t* W1;
    uint32_t wbytes, rtb;
    const uint8_t* X;       // packed activations, terms tstride bytes apart
    uint32_t xbytes;        // of one term
    uint64_t tstride;
    const uint32_t* flags;  // per (16 tokens, super-step), or null: one term
    PackGeom pg;
    int M, N, act;
    int tx, ty, ks;         // token tiles, row tiles, K splits
    float* Y;               // fp32 output, or
    uint16_t* Yb;           // bf16 output, or
    uint8_t* Yp;            // packed bf16 output (the FFN's activation)
    int ldy;
    float* part;            // split K: partial tiles and arrival counters
    uint32_t* cnt;
};

// 64 lanes x 16 bytes from (rsrc, lane 16 bytes apart, soff) to LDS at byte
// `lds` + 16 lane. Written out because the compiler, which cannot tell the two
// halves of the LDS buffer apart, would wait for the load before every LDS
// read; the kernel waits for it (vmcnt) ahead of the barrier that hands the
// half over. m0 is declared as written, so that the compiler keeps no value of
// its own there across the statement (it is a reserved register, hence the
// warning: it is not preserved, as meant).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(r), "s"(soff), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// c += a b on the matrix cores. ACC: written out, with c in accumulation
// registers, so that the result stays in c's own registers: with some 100 or
// more of them the compiler, left to choose, moved accumulators between
// register files (420 moves per 256 of these) and spilled. It cannot see these writes'
// latency, so code that reads c otherwise first waits (acc_wait), and a and b
// are written two instructions or more ahead.
constexpr int kAccTiles = 24;  // f32x4 accumulators of a lane from which this holds
template <bool ACC>
__device__ __forceinline__ void mfma_acc(f32x4& c, bf16x8 a, bf16x8 b) {
    if constexpr (ACC)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else
        c = mfma16x16x32(a, b, c);
}
// The operands b are written, and two wait states have passed.
template <int RB>
__device__ __forceinline__ void settle(bf16x8 (&b)[RB]) {
#pragma unroll
    for (int q = 0; q < RB; ++q) asm volatile("" : "+v"(b[q]));
    asm volatile("s_nop 1");
}
// The accumulators hold the last products. Each is passed through a statement
// behind the wait: the compiler could otherwise read it ahead of the wait,
// which touches none of them.
template <int TB, int RB>
__device__ __forceinline__ void acc_wait(f32x4 (&acc)[TB][RB]) {
    if constexpr (TB * RB < kAccTiles) return;  // the compiler's own matrix instructions
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int q = 0; q < RB; ++q) asm volatile("" : "+a"(acc[t][q]));
}

// dequant8_mix in 17 steps of one instruction, to be spread between matrix
// instructions.
struct Dequant {
    uint32_t d, d8;
    f16x2 n[4];  // nibbles (0, 4), (1, 5), (2, 6), (3, 7)
    float w[8];
    bf16x8 r;
    __device__ __forceinline__ void step(int i, const Scale2& s) {
        if (i == 0) d8 = d >> 8;
        if (i == 1) n[0] = nib_f16x2(d, 0x000F000Fu, 0x3C083C08u);
        if (i == 2) n[1] = nib_f16x2(d, 0x00F000F0u, 0x3C803C80u);
        if (i == 3) n[2] = nib_f16x2(d8, 0x000F000Fu, 0x3C083C08u);
        if (i == 4) n[3] = nib_f16x2(d8, 0x00F000F0u, 0x3C803C80u);
        if (i >= 5 && i < 13) {
            const int e = i - 5;
            w[e] = __builtin_fmaf((float)n[e & 3][e >> 2], e & 1 ? s.s4 : s.s0, e & 1 ? s.c4 : s.c0);
        }
        if (i >= 13 && i < 17) {
            const int e = 2 * (i - 13);
            r[e] = (__bf16)w[e];
            r[e + 1] = (__bf16)w[e + 1];
        }
    }
};
constexpr int kDequantSteps = 17;

// Substeps whose activations are loaded together: enough work for the next
// ones to arrive where a CU holds one workgroup (one substep of 8 x 16 tokens
// is 2048 clocks of matrix instructions, about the latency of the L2 under this
// load), one where several workgroups cover for each other.
template <int TB>
constexpr int prefill_stage() {
    return TB == 8 ? 2 : 1;
}

// Waves per workgroup: eight, two per SIMD, where a CU's LDS and registers hold
// one such workgroup; four, several workgroups per CU, for small tiles.
template <int TB>
constexpr int prefill_wg() {
    return TB >= 8 ? 8 : 4;
}

template <int TB>
constexpr int prefill_waves() {  // waves per SIMD the register budget is set for
    return TB >= 8 ? 2 : 3;
}

// The GLU epilogue's LDS row of (gate, up) pairs, and its queue of values the
// float32 path leaves: less than one round of the nt threads kept, and all of
// two octets per thread.
constexpr int glu_stride(int rows) { return rows + 4; }
constexpr int glu_queue(int nt) { return nt + 16 * nt; }

template <int TB, int RB, bool GLU>
__global__ void __launch_bounds__((64 * prefill_wg<TB>()), (prefill_waves<TB>())) prefill_kernel(PrefillArgs a) {
    constexpr int NWV = prefill_wg<TB>(), NT = 64 * NWV;
    constexpr int RBM = GLU ? RB / 2 : RB;  // row tiles of one matrix per wave
    constexpr int PS = prefill_stage<TB>();      // substeps per stage: an LDS buffer, a barrier
    constexpr int BUF = PS * TB * kStepBytes;    // one LDS buffer
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;

    // Tile of this workgroup. Workgroups go round the 8 XCDs in turn; each XCD
    // takes a run of tiles, four token tiles by row tiles, so that its
    // workgroups share weights and activations in its L2.
    const int ntile = a.tx * a.ty;
    const int kq = blockIdx.x / ntile;
    const int id = blockIdx.x - kq * ntile;
    const int xcd = id & 7, r8 = ntile & 7;
    const int idx = xcd * (ntile >> 3) + min(xcd, r8) + (id >> 3);
    const int grp = idx / (4 * a.ty), rem = idx - grp * 4 * a.ty;
    const int gm = min(4, a.tx - 4 * grp);
    const int ty = rem / gm, tx = 4 * grp + rem - ty * gm;
    const int m0 = tx * TB * 16, rt0 = ty * NWV * RBM + wave * RBM;

    const PackGeom pg = a.pg;
    const __amdgpu_buffer_rsrc_t rw0 = make_rsrc(a.W0, a.wbytes);
    const __amdgpu_buffer_rsrc_t rw1 = make_rsrc(GLU ? a.W1 : a.W0, a.wbytes);
    const int nrt = (a.N + 15) >> 4;
    // Row tiles past the matrix load from past its end (zeros).
    const uint32_t l16 = (uint32_t)lane * 16u;
    uint32_t wbase[RBM], wlane[RBM];
#pragma unroll
    for (int q = 0; q < RBM; ++q) {
        const bool in = rt0 + q < nrt;
        wbase[q] = in ? (uint32_t)(rt0 + q) * a.rtb : 0u;
        wlane[q] = in ? l16 : a.wbytes;
    }

    int nterms = 1;
    if (a.flags) {
        const int nf = (min(m0 + TB * 16, a.M) - m0 + 15) / 16 * pg.nss;
        bool more = false;
        for (int q = tid; q < nf; q += NT) more |= a.flags[(m0 >> 4) * pg.nss + q] != 0;
        nterms = __syncthreads_or(more) ? 3 : 1;
    }
    // This split's whole super-steps [ss0, ss1), and the substeps of the last,
    // partial one (the last split's), taken once per term.
    const int nfull = pg.nbl == 16 ? pg.nss : pg.nss - 1;
    const int ss0 = kq * nfull / a.ks, ss1 = (kq + 1) * nfull / a.ks;
    const int ntail = nfull < pg.nss && kq == a.ks - 1 ? pg.T : 0;
    const int send = 4 * ss1 + ntail;  // substeps [4 ss0, send): a split's tail follows its super-steps
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    // Fragment f = 4 tb + kk of substep s, term p into its place in the LDS
    // buffers; past the last token or substep, from past the end (zeros).
    auto place = [&](int s) __attribute__((always_inline)) -> uint32_t {
        return (uint32_t)(s / PS & 1) * BUF + (uint32_t)(s % PS) * (TB * kStepBytes);
    };
    auto load_x = [&](int s, int p, int f) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.X + (size_t)p * a.tstride, a.xbytes);
        const uint32_t o = (uint32_t)(((m0 >> 4) + (f >> 2)) * pg.S + s) * kStepBytes + (f & 3) * kFragBytes;
        load_lds16(rx, l16, s >= send ? a.xbytes : min(o, a.xbytes), lds0 + place(s) + f * kFragBytes);
    };
    // The lane's 80-byte run of a whole super-step, by its 16-byte planes, of
    // every row tile: substep t multiplies dwords 5 t .. 5 t + 4.
    u32x4 u[RB][5];
    auto load_plane = [&](int ss, int pl) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < RB; ++q)
            u[q][pl] = __builtin_amdgcn_raw_buffer_load_b128(q < RBM ? rw0 : rw1, wlane[q % RBM],
                                                             wbase[q % RBM] + (uint32_t)ss * 5120u + pl * 1024u, 0);
    };
    // The 20 bytes of the lane's block of the partial super-step's substep t:
    // block T g + t, in the run of lane group (T g + t) / 4.
    auto load_tail = [&](int t, uint32_t (&w)[RB][5]) __attribute__((always_inline)) {
        const int b = pg.T * g + t;
#pragma unroll
        for (int x = 0; x < 5; ++x) {
            const int rb = 20 * (b & 3) + 4 * x;
            const uint32_t v = b < pg.nbl ? (uint32_t)(pg.nss - 1) * 5120u + (uint32_t)(rb >> 4) * 256u * (uint32_t)pg.T +
                                                (uint32_t)((b >> 2) * 16 + j) * 16u + (uint32_t)(rb & 15)
                                          : a.wbytes;
#pragma unroll
            for (int q = 0; q < RB; ++q)
                w[q][x] = __builtin_amdgcn_raw_buffer_load_b32(q < RBM ? rw0 : rw1, rt0 + q % RBM < nrt ? v : a.wbytes,
                                                               wbase[q % RBM], 0);
        }
    };

    f32x4 acc[TB][RB];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int q = 0; q < RB; ++q) acc[t][q] = f32x4{0.f, 0.f, 0.f, 0.f};

    uint32_t wt[RB][5] = {};
    bf16x8 bv[2][RB];
    Scale2 sc[RB];
    // One substep s: TT = 0 .. 3 of a whole super-step (its
    // weights in u), or 4, a partial one's (in wt). Its first octet was
    // dequantized during the substep before. The next substep's activations go
    // out first, into the other buffer. At the last octet the weights are
    // dequantized: the planes this substep used up are loaded for the next
    // super-step (two to three substeps ahead of their use, and younger than
    // the activations, so that the in-order waits for one never wait for the
    // other's latest loads), and the next substep's first octet follows. A
    // group is one row tile's dequantization between the matrix instructions
    // of G fragments.
    constexpr int G = TB / RB, R = NWV == 8 ? 6 : 8;  // R: operand reads ahead
    constexpr int XL = 4 * TB / NWV;  // fragments a wave loads per substep
    constexpr int LK = PS, LG = (PS * XL + LK * RB - 1) / (LK * RB);  // activation loads: over LK octets, per group
    static_assert(TB % RB == 0, "whole fragments per group");
    auto substep = [&](auto tt, int s, int p, int nextss) __attribute__((always_inline)) {
        constexpr int TT = decltype(tt)::value;
        auto dword = [&](int q, int i) __attribute__((always_inline)) -> uint32_t {  // of the super-step from TT's on
            if constexpr (TT == 4) return wt[q][i];
            const int d = (5 * TT + i) % 20;
            return u[q][d >> 2][d & 3];
        };
        const unsigned char* xb = smem + place(s) + l16;
        // The stage's first substep loads the next stage, its last waits for it.
        const bool first = TT < 4 ? TT % PS == 0 : s % PS == 0, last = TT < 4 ? TT % PS == PS - 1 : s % PS == PS - 1;
        auto frag = [&](int f) __attribute__((always_inline)) {  // f = kk TB + t
            return *reinterpret_cast<const bf16x8*>(xb + (4 * (f % TB) + f / TB) * kFragBytes);
        };
        bf16x8 av[R];
#pragma unroll
        for (int f = 0; f < R; ++f) av[f] = frag(f);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            if (kk == 3) {
                if constexpr (TT < 4) {
                    load_plane(nextss, TT);
                    if constexpr (TT == 3) load_plane(nextss, 4);
#pragma unroll
                    for (int q = 0; q < RB; ++q) sc[q] = make_scale2(scale_of(dword(q, 9)));
                } else {
                    load_tail(min(nextss, pg.T - 1), wt);  // nextss: the next tail substep
#pragma unroll
                    for (int q = 0; q < RB; ++q) sc[q] = make_scale2(scale_of(wt[q][4]));
                }
            }
#pragma unroll
            for (int h = 0; h < RB; ++h) {
                if (kk < LK && first)
#pragma unroll
                    for (int q = LG * (kk * RB + h); q < LG * (kk * RB + h + 1) && q < PS * XL; ++q)
                        load_x(s + PS + q / XL, p, wave * XL + q % XL);
                Dequant dq;
                dq.d = kk < 3 ? dword(h, kk + 1) : TT == 4 ? wt[h][0] : dword(h, 5);
#pragma unroll
                for (int t = G * h; t < G * h + G; ++t) {
                    const int f = kk * TB + t;
#pragma unroll
                    for (int q = 0; q < RB; ++q) {
                        mfma_acc<(TB * RB >= kAccTiles)>(acc[t][q], av[f % R], bv[kk & 1][q]);
                        const int slot = (t - G * h) * RB + q;
#pragma unroll
                        for (int i = 0; i < kDequantSteps; ++i)
                            if (i * G * RB / kDequantSteps == slot) dq.step(i, sc[h]);
                        if (q == RB - 1 && f + R < 4 * TB) av[f % R] = frag(f + R);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                bv[(kk + 1) & 1][h] = dq.r;
            }
            settle<RB>(bv[(kk + 1) & 1]);
        }
        // The activations have landed; the planes asked for since may not have.
        if (last) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TT == 4 ? 0 : TT == 3 ? (PS + 1) * RB : PS * RB) : "memory");
            lds_barrier();
        }
    };
    auto first_octet = [&](int q, uint32_t d0, uint32_t d4) __attribute__((always_inline)) {
        sc[q] = make_scale2(scale_of(d4));
        bv[0][q] = dequant8_mix(d0, sc[q]);
    };
    for (int p = 0; p < nterms; ++p) {
#pragma unroll
        for (int q = 0; q < PS * XL; ++q) load_x(4 * ss0 + q / XL, p, wave * XL + q % XL);
        if (ntail) load_tail(0, wt);
        if (ss0 < ss1) {
#pragma unroll
            for (int pl = 0; pl < 5; ++pl) load_plane(ss0, pl);
#pragma unroll
            for (int q = 0; q < RB; ++q) first_octet(q, u[q][0][0], u[q][1][0]);
            settle<RB>(bv[0]);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        for (int ss = ss0; ss < ss1; ++ss) {
            const int ns = ss + 1 < ss1 ? ss + 1 : ss0;
            substep(std::integral_constant<int, 0>{}, 4 * ss, p, ns);
            substep(std::integral_constant<int, 1>{}, 4 * ss + 1, p, ns);
            substep(std::integral_constant<int, 2>{}, 4 * ss + 2, p, ns);
            substep(std::integral_constant<int, 3>{}, 4 * ss + 3, p, ns);
        }
        if (ntail) {
#pragma unroll
            for (int q = 0; q < RB; ++q) first_octet(q, wt[q][0], wt[q][4]);
            settle<RB>(bv[0]);
            for (int t = 0; t < ntail; ++t) substep(std::integral_constant<int, 4>{}, 4 * ss1 + t, p, t + 1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    acc_wait(acc);

    // ---- split K: the last workgroup of the tile adds the partial tiles, in
    // split order (gemm_q.hip's scheme: 16-byte write-through pieces, thread
    // tid's f32x4 (t, q) at ((t RB + q) NT + tid) 16 bytes of its split).
    if (a.ks > 1) {
        const size_t tsz = (size_t)TB * RB * NT * 4;  // floats of a tile
        const __amdgpu_buffer_rsrc_t rp = make_rsrc(a.part + (size_t)idx * a.ks * tsz, (uint32_t)(a.ks * tsz * sizeof(float)));
        auto piece = [&](int k, int t, int q) -> uint32_t {
            return (uint32_t)((((size_t)k * TB + t) * RB + q) * (NT * 16) + tid * 16);
        };
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int q = 0; q < RB; ++q)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[t][q]), rp, piece(kq, t, q), 0, 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        int* last = reinterpret_cast<int*>(smem);
        __syncthreads();
        if (tid == 0)
            *last = __hip_atomic_fetch_add(&a.cnt[idx], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                    (uint32_t)(a.ks - 1);
        __syncthreads();
        const bool fin = *last;
        if (!fin) return;
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int q = 0; q < RB; ++q) acc[t][q] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < a.ks; ++k)
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int q = 0; q < RB; ++q)
                    acc[t][q] += __builtin_bit_cast(f32x4, buf_load16_sc1(rp, piece(k, t, q)));
        if (tid == 0) __hip_atomic_store(&a.cnt[idx], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();  // `last` has been read: the LDS is free
    }

    // ---- epilogue: D[4 g + r][j] of each 16 x 16 sub-tile ----------------------------
    if constexpr (GLU) {
        // bf16 (gate, up) pairs of the tile into LDS, then whole octets of the
        // activation to memory in operand order (sixteen tokens' octet is 256
        // contiguous bytes). Values the float32 path cannot settle (one in 500
        // of ordinary gates, one in 20 where gates spread over +-10) are queued
        // and evaluated together, a round of the workgroup's threads at a time:
        // one by one where they occur, nearly every octet's wave would run the
        // float64 path. (512 tokens of 3840 <-> 15360, gates 3.4 wide: 183 us,
        // as with gates 1 wide; 213 with gemm_q.hip, and 239 when more misses
        // than a queue for the tile held sent all of it to the float64 path.)
        constexpr int NR = 16 * NWV * RBM, LS = glu_stride(NR);  // rows, LDS row stride in pairs
        constexpr int OCTETS = TB * 16 * (NR / 8), BATCH = 2 * NT;  // BATCH: between two looks at the queue
        static_assert(TB * 16 * LS <= 65536, "16-bit queue entries");
        uint32_t* tile = reinterpret_cast<uint32_t*>(smem);
        uint16_t* queue = reinterpret_cast<uint16_t*>(tile + TB * 16 * LS);  // glu_queue(NT) entries
        constexpr int BATCHES = (OCTETS + BATCH - 1) / BATCH;
        __shared__ int queued[BATCHES];  // by each batch: stable once a barrier has ended it
        int waiting = 0;                 // by the batches before, not yet evaluated
        if (tid < BATCHES) queued[tid] = 0;
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int q = 0; q < RBM; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const __bf16 gb = (__bf16)acc[t][q][r], ub = (__bf16)acc[t][q + RBM][r];
                    tile[(16 * t + 4 * g + r) * LS + 16 * (wave * RBM + q) + j] =
                        (uint32_t)__builtin_bit_cast(uint16_t, gb) | (uint32_t)__builtin_bit_cast(uint16_t, ub) << 16;
                }
        __syncthreads();
        const PackGeom po = pack_geom(a.N);
        const int n0 = ty * NR;
#pragma unroll 1
        for (int b = 0; b < BATCHES; ++b) {
#pragma unroll 1
            for (int c = b * BATCH + tid; c < min(b * BATCH + BATCH, OCTETS); c += NT) {
                const int i = c & 15, o = (c >> 4) % (NR / 8), t = (c >> 4) / (NR / 8);
                const int m = m0 + 16 * t + i, n = n0 + 8 * o;
                if (m0 + 16 * t >= a.M || n >= a.N) continue;
                const u32x4* src = reinterpret_cast<const u32x4*>(tile + (16 * t + i) * LS + 8 * o);
                const u32x4 p0 = src[0], p1 = src[1];
                const uint32_t pk[8] = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
                bf16x8 y;
                uint32_t miss = 0;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float v = 0.0f;
                    if (a.act != ALV_ACT_GELU_TANH)
                        v = glu_exact(lo_half(pk[e]), hi_half(pk[e]), a.act);
                    else if (!gelu_quick(lo_half(pk[e]), hi_half(pk[e]), &v))
                        miss |= 1u << e;
                    y[e] = (__bf16)v;
                }
                if (m >= a.M) miss = 0;
                uint16_t* dst = reinterpret_cast<uint16_t*>(a.Yp + pack_offset(po, m, n >> 3));
                *reinterpret_cast<u32x4*>(dst) = m < a.M ? __builtin_bit_cast(u32x4, y) : u32x4{0, 0, 0, 0};
                while (miss) {
                    const int e = __builtin_ctz(miss);
                    miss &= miss - 1;
                    queue[waiting + atomicAdd(&queued[b], 1)] = (uint16_t)((16 * t + i) * LS + 8 * o + e);
                }
            }
            // A whole round waits (or no more will come): an entry per thread,
            // once the octets around it are in memory.
            const bool end = b == BATCHES - 1;
            if (end) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            waiting += queued[b];
            if (waiting < NT && !end) continue;
            if (!end) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
            }
#pragma unroll 1
            for (int c = tid; c < waiting; c += NT) {
                const int at = queue[c], mt = at / LS, nt = at - mt * LS;
                const uint32_t w = tile[at];
                reinterpret_cast<uint16_t*>(a.Yp + pack_offset(po, m0 + mt, (n0 + nt) >> 3))[(n0 + nt) & 7] =
                    __builtin_bit_cast(uint16_t, (__bf16)glu_exact(lo_half(w), hi_half(w), a.act));
            }
            waiting = 0;
            if (!end) __syncthreads();
        }
        // Blocks past the last, up to a whole substep, are zeros: their weights
        // are, and what the buffer held before may not be finite.
        const int npad = 4 * po.T - po.nbl;
        if (ty == a.ty - 1)
            for (int c = tid; c < TB * 64 * npad; c += NT) {
                const int i = c & 15, o = (c >> 4) % (4 * npad), t = (c >> 4) / (4 * npad);
                if (m0 + 16 * t < a.M)
                    *reinterpret_cast<u32x4*>(a.Yp + pack_offset(po, m0 + 16 * t + i, a.N / 8 + o)) = u32x4{0, 0, 0, 0};
            }
    } else {
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int q = 0; q < RB; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + 16 * t + 4 * g + r, n = 16 * (rt0 + q) + j;
                    if (m >= a.M || n >= a.N) continue;
                    if (a.Yb)
                        a.Yb[(size_t)m * a.ldy + n] = __builtin_bit_cast(uint16_t, (__bf16)acc[t][q][r]);
                    else
                        a.Y[(size_t)m * a.ldy + n] = acc[t][q][r];
                }
    }
}

struct Plan {
    int tb, rb, waves, ks;
};

// Tile and K split of a product: the least estimated time over the tiles
// built. A substep's time and a workgroup's own (prologue, epilogue) are fits,
// in us, to sweeps of every tile and split over FFNs of 3840 <-> 15360, 1152 <->
// 6912 and 1056 <-> 14400 at 70 to 3001 tokens. At 17 to 512 tokens an FFN with
// the plan's tiles takes at most 4 % more than with the fastest pair of tiles and
// splits at 3840 <-> 15360, 12 % at 1152 <-> 6912, 2048 <-> 8192 and 1056 <->
// 14400 (the fit's sizes begin at 70 tokens); 2100 one-term projections at 17 to
// 4096 tokens 2.4 % in the mean, one in twenty over 11 %. fp32 activations count
// three terms. Large tiles fill a CU alone: whole rounds of workgroups. Small ones
// share it: the longer of one workgroup's latency and the CU's throughput. A
// split adds its partial tiles' round trip.
struct TileCost {
    int tb, rb, waves;
    bool shared;            // several workgroups per CU
    float step, glu, lin;   // per substep, per workgroup with and without a GLU
    float lstep, lglu, llin;  // the same for a workgroup alone on its CU
};
constexpr TileCost kTiles[] = {
    {16, 2, 8, false, 2.93f, 20.1f, 15.f, 0, 0, 0},    {12, 2, 8, false, 1.94f, 24.6f, 14.f, 0, 0, 0},
    {8, 2, 8, false, 1.64f, 15.5f, 7.84f, 0, 0, 0},    {4, 2, 4, true, 0.72f, 2.f, 2.f, 1.17f, 5.f, 4.f},
    {2, 2, 4, true, 0.54f, 1.8f, 1.29f, 1.05f, 5.36f, 2.91f},
};

Plan prefill_plan(int M, int N, int K, int terms, bool glu) {
    const float S = (float)pack_geom(K).S * terms, cus = (float)device_cus();
    Plan best{4, 2, 4, 1};
    float least = 0.f;
    for (const TileCost& t : kTiles)
        for (int ks = 1; ks <= 16; ks *= 2) {
            const int rows = (glu ? 8 : 16) * t.waves * t.rb;
            const float tiles = (float)((M + t.tb * 16 - 1) / (t.tb * 16)) * (float)((N + rows - 1) / rows);
            const float s = S / ks, load = tiles * ks / cus;
            if (ks > 1 && (tiles > kSplitCounters || s < 8.f * terms)) break;
            float us = t.shared ? std::max(s * t.lstep + (glu ? t.lglu : t.llin), load * (s * t.step + (glu ? t.glu : t.lin)))
                                : std::ceil(load) * (s * t.step + (glu ? t.glu : t.lin));
            if (ks > 1) us += 3.8f + 0.0239f * ks * t.tb * t.rb * t.waves;
            if (least == 0.f || us < least) {
                least = us;
                best = {t.tb, t.rb, t.waves, ks};
            }
        }
    return best;
}

template <int TB, int RB, bool GLU>
hipError_t launch_tile_kernel(const PrefillArgs& a, hipStream_t s) {
    constexpr int kBufs = 2 * prefill_stage<TB>() * TB * kStepBytes;
    constexpr int kWaves = prefill_wg<TB>();
    constexpr int kPairs = GLU ? TB * 16 * glu_stride(8 * kWaves * RB) * 4 + glu_queue(64 * kWaves) * 2 : 0;
    constexpr int lds = kBufs > kPairs ? kBufs : kPairs;
    static_assert(lds + 64 <= 160 * 1024, "LDS of a CU");
    const void* k = reinterpret_cast<const void*>(&prefill_kernel<TB, RB, GLU>);
    if (lds > 64 * 1024)
        if (hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((prefill_kernel<TB, RB, GLU>), dim3(a.tx * a.ty * a.ks), dim3(64 * kWaves), lds, s, a);
    return hipGetLastError();
}

template <bool GLU>
hipError_t launch_plan(const Plan& p, const PrefillArgs& a, hipStream_t s) {
    switch (p.tb * 10 + p.rb) {
        case 162: return launch_tile_kernel<16, 2, GLU>(a, s);
        case 122: return launch_tile_kernel<12, 2, GLU>(a, s);
        case 82: return launch_tile_kernel<8, 2, GLU>(a, s);
        case 42: return launch_tile_kernel<4, 2, GLU>(a, s);
        default: return launch_tile_kernel<2, 2, GLU>(a, s);
    }
}

}  // namespace

size_t packed_bytes(int M, int K) { return (size_t)((M + 15) / 16) * pack_geom(K).S * kStepBytes; }

int launch_unpack_f32(const uint8_t* in, int M, int K, float* out, int ldo, hipStream_t s) {
    const int64_t n = (int64_t)M * (ldo / 8);
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 4096));
    hipLaunchKernelGGL(unpack_f32_kernel, dim3(grid), dim3(256), 0, s, in, M, K, out, ldo);
    return hip_check(hipGetLastError(), "unpack_f32_kernel launch");
}

int launch_prefill(const GemvLaunch& L, hipStream_t s, bool* taken) {
    *taken = false;
    const uint64_t wbytes = tile_bytes(L.N, L.K);
    const size_t xbytes = packed_bytes(L.M, L.K);
    if (!L.tiled || wbytes >= 0xF0000000ull || xbytes >= 0x7FFFF000ull) return ALV_OK;
    // (The packed output is the next product's input: blocks past N are padded
    // to a substep, so it can be the larger of the two.)
    if (L.Yp && packed_bytes(L.M, L.N) >= 0x7FFFF000ull) return ALV_OK;
    const bool f32 = L.X != nullptr && !L.Xp;
    if (!L.Xp && (f32 ? reinterpret_cast<uintptr_t>(L.X) % 4 != 0 : reinterpret_cast<uintptr_t>(L.Xb) % 16 != 0 || L.ldx % 8 != 0))
        return fail(ALV_ERR_ALIGN, "prefill activations are not aligned for 16-byte loads");
    const PackGeom pg = pack_geom(L.K);
    Plan p = prefill_plan(L.M, L.N, L.K, f32 && L.parts == 3 ? 3 : 1, L.glu);
    PrefillArgs a{};
    a.tx = (L.M + p.tb * 16 - 1) / (p.tb * 16);
    const int rows = (L.glu ? 8 : 16) * p.waves * p.rb;
    a.ty = (L.N + rows - 1) / rows;
    const int ntile = a.tx * a.ty, tbs = (L.M + 15) / 16;
    Workspace ws{};
    if (p.ks > 1 && (ntile > kSplitCounters || get_workspace(s, (size_t)ntile, &ws))) {
        clear_error();
        p.ks = 1;
    }
    // Scratch: packed activations (unless given), term flags, partial tiles.
    const size_t pack = L.Xp ? 0 : (f32 ? 3 : 1) * xbytes;
    const size_t flag_bytes = f32 ? ((size_t)tbs * pg.nss * 4 + 255) & ~(size_t)255 : 0;
    const size_t tsz = (size_t)p.tb * p.rb * p.waves * 256 * sizeof(float);
    uint8_t* sb = nullptr;
    for (;;) {
        const size_t part = p.ks > 1 ? tsz * p.ks * ntile : 0;
        if (pack + flag_bytes + part == 0) break;
        void* v = nullptr;
        if (get_scratch(s, kScratchGemm, pack + flag_bytes + part, &v) == ALV_OK) {
            sb = static_cast<uint8_t*>(v);
            break;
        }
        clear_error();  // a graph capture that would have to grow it
        if (p.ks == 1) return ALV_OK;
        p.ks = 1;
    }
    *taken = true;
    a.W0 = L.W0;
    a.W1 = L.W1;
    a.wbytes = (uint32_t)wbytes;
    a.rtb = tile_geom(L.K).rtb;
    a.X = L.Xp ? L.Xp : sb;
    a.xbytes = (uint32_t)xbytes;
    a.tstride = xbytes;
    a.pg = pg;
    a.M = L.M;
    a.N = L.N;
    a.act = L.act;
    a.ks = p.ks;
    a.Y = L.Y;
    a.Yb = L.Yb;
    a.Yp = L.Yp;
    a.ldy = L.ldy;
    a.part = reinterpret_cast<float*>(sb + pack + flag_bytes);
    a.cnt = ws.counters;
    if (!L.Xp) {
        const dim3 grid(tbs, pg.nss);
        uint32_t* flags = reinterpret_cast<uint32_t*>(sb + pack);
        if (f32) {
            hipLaunchKernelGGL((pack_x_kernel<true>), grid, dim3(256), 0, s, L.X, L.ldx, L.M, L.K, sb, xbytes, flags);
            a.flags = L.parts == 3 ? flags : nullptr;
        } else {
            hipLaunchKernelGGL((pack_x_kernel<false>), grid, dim3(256), 0, s, L.Xb, L.ldx, L.M, L.K, sb, xbytes, flags);
        }
        if (int rc = hip_check(hipGetLastError(), "pack_x_kernel launch")) return rc;
    }
    return hip_check(L.glu ? launch_plan<true>(p, a, s) : launch_plan<false>(p, a, s), "prefill_kernel launch");
}

}  // namespace alv

extern "C" int alv_prefill_plan(int M, int N, int K, int fp32, int ffn, int* tokens, int* splits) {
    using namespace alv;
    if (!tokens || !splits) return fail(ALV_ERR_ARG, "null pointer");
    if (M < 1 || N < 1 || K < 32 || K % 32) return fail(ALV_ERR_ARG, "bad shape M=%d N=%d K=%d", M, N, K);
    *tokens = 0;
    *splits = 0;
    if (ffn < 0 || ffn > 2) return fail(ALV_ERR_ARG, "ffn must be 0, 1 or 2 (got %d)", ffn);
    if (!ffn && lds_tiles_faster(M, N, K, fp32 != 0)) return ALV_OK;
    const Plan p = prefill_plan(M, N, K, fp32 && ffn < 2 ? 3 : 1, ffn == 1);
    *tokens = 16 * p.tb;
    *splits = p.ks;
    return ALV_OK;
}
