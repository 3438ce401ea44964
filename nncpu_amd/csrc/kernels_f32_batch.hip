// The bit-exact f32 matmul for several vectors (Q8_0, Q4), on the f32 matrix
// unit: the contract and the reference's order are kernels_f32.hip's.
//
// Why the matrix unit keeps the bits: v_mfma_f32_16x16x4_f32 performs, per
// output, four fused multiply-adds in k order, each rounded to nearest even
// with denormals kept (checked against fmaf over normal, denormal, overflowing,
// cancelling, signed-zero, infinite and NaN operands). So the chain
//     acc_j = fma(f32(q[32b+j]) * bf16(s[b]), x[32b+j], acc_j)
// over blocks b is a matrix product over b for each of the 32 elements j, and
// 16 rows x 16 vectors of one chain are one accumulator tile of 4 registers.
//
// Split: a wave holds 16 rows x 16 NT vectors of 8 of the 32 chains (4 w ..
// 4 w + 3 and 16 + 4 w .. + 3: one word of a Q4 block's quants, two of a Q8
// block's, two 16-byte pieces of x), four waves make a row group, R row groups
// a workgroup. Chains never split along the blocks (that would change the
// bits); at the end the four waves' chains meet in LDS in the reference's
// order. The converted weight of a lane (a conversion and a product per
// value) serves NT matrix instructions.
//
// Measured (us, before: one to four vectors per weight pass): Q8 14336 x 4096
// 16 vectors 137 -> 31.6, 64 -> 90, 301 2720 -> 350 (101 TFLOP/s), 512 573
// (105); 4096 x 4096 16 91 -> 11.3; Q4 3584 x 18944 16 244 -> 49.
//
// Bound: the f32 matrix rate (256 operations per CU and clock, 130 TFLOP/s
// measured with nothing beside it); vector instructions do not run beside f32
// matrix instructions (measured: 8 FMAs between two of them cost their full
// time), so the conversions' 72 cycles per 4 blocks come on top of NT x 256.
//
// Data moves global -> LDS directly (no registers) through a ring of NS
// stages of 8 blocks. 16-byte pieces are XOR-swizzled by row on the global
// side, so that LDS reads are spread over the banks (the LDS is active 16 to 18 %
// of the time, a quarter to a half of that in conflicts). Weights come from the
// split layout as uploaded, scales from the f32 path's padded rows (16 bytes
// are 8 blocks). In a partial last stage the missing blocks are 0 * -0 = -0,
// which leaves every accumulator as it is, -0 included.

#include "common.h"

namespace nnh {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct BatchArgs {
    const uint8_t* qs;   // quants, split layout
    const uint16_t* fs;  // scales, rows padded to nbp
    const uint16_t* bi;  // Q4 biases [rows][nb]
    const float* x;
    const float* xsum;   // Q4 block sums [n_tok][nb]
    float* y;
    size_t xs, ys;
    int rows, nb, nbp, n_tok;
    int rem;             // BF16: columns past the nb whole 32-blocks (a multiple of 8)
    int ttiles, tq, tr;  // token tiles; tile i holds tq (+ 1 for the first tr) groups of 16 vectors
    bool vec_y;          // y rows take 16-byte stores
};

// 64 lanes x 16 bytes from base (uniform) + voff into LDS at dst (uniform,
// lane l's bytes at dst + 16 l); asm because the compiler would otherwise
// drain every copy before any LDS read (the waits are explicit).
__device__ __forceinline__ void copy16(const void* base, uint32_t voff, uint32_t dst) {
    asm volatile(NNH_COPY16_ASM "%0, %1" ::"v"(voff), "s"(base), "{m0}"(dst) : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Every wave's LDS accesses so far are done, without draining the copies in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(NNH_LGKMCNT0);
    asm volatile("s_barrier" ::: "memory");
}

__device__ __forceinline__ f32x4 add4(f32x4 a, f32x4 b) {
    return f32x4{__fadd_rn(a[0], b[0]), __fadd_rn(a[1], b[1]), __fadd_rn(a[2], b[2]), __fadd_rn(a[3], b[3])};
}

// A lane's result tile column: rows row .. row + 3 of vector tok.
__device__ __forceinline__ void store4(const BatchArgs& g, f32x4 r, int row, int tok) {
    if (tok >= g.n_tok) return;
    float* yp = g.y + (size_t)tok * g.ys + row;
    if (g.vec_y && row + 4 <= g.rows) {
        *(f32x4*)yp = r;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (row + e < g.rows) yp[e] = r[e];
    }
}

template <int DT, int R, int NT, int H>
struct BatchLds {
    static constexpr int X = NT * 16384;             // [16-vector group][block][vector][8 pieces]
    static constexpr int W = R * (DT == 1 ? 4096 : 2048);
    static constexpr int S = R * 1024;               // a row's 8 scales per 16 bytes, four copies
    static constexpr int STAGE = X + W + S;
    static constexpr int PARTS = H == 1 ? 16 : 24;   // KB of chains handed over (and 4 of wave 1's v, then the bias chains)
    static constexpr int MEET_RG = (PARTS + 4 + 4 * H) * 1024;
    static constexpr int MEET = R * MEET_RG;         // the waves' meeting area at the end
};

template <int DT, int R, int NT, int H, int NS>
__device__ __forceinline__ void batch_body(const BatchArgs& g, unsigned char* lds, int row0, int tok0) {
    using L = BatchLds<DT, R, NT, H>;
    constexpr int NC = 8 / H;                           // chains per wave
    constexpr int NW = 4 * H * R, XC = 16 / NW;         // waves; x copies per wave, stage and vector group
    constexpr int CP = NT * XC + (DT == 1 && H == 1 ? 2 : 1);  // copies per wave and stage
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave / (4 * H), wl = wave % (4 * H);  // row group, wave in it
    const int w = wl & 3, half = wl >> 2;               // word of the quants; H = 2: chains 4 w .. + 3 (0) or 16 + 4 w .. + 3 (1)
    const int c16 = lane & 15, k = lane >> 4;           // row (A) or vector (B) of the tile, block of the step
    const int nb = g.nb, nst = (nb + 7) / 8;
    const uint32_t ring = (uint32_t)(uintptr_t)lds;

    // Global offsets of this lane's copies, fixed for the kernel.
    uint32_t xoff[NT];
    const float* xb = g.x + (size_t)tok0 * g.xs;
    {
        const int v8 = 8 * (wave & 1) + (lane >> 3), c = (lane & 7) ^ ((v8 >> 1) & 7);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            xoff[t] = (uint32_t)min(16 * t + v8, g.n_tok - 1 - tok0) * (uint32_t)(g.xs * 4) + 16 * c;
    }
    const int last = g.rows - 1 - row0;
    const uint8_t* wb = g.qs + (size_t)row0 * nb * (DT == 1 ? 32 : 16);
    const int wr = DT == 1 ? 16 * rg + 4 * w + (lane >> 4) : 16 * rg + 8 * (w & 1) + (lane >> 3);  // row of the copy
    const int wc = DT == 1 ? (lane & 15) ^ (wr & 15) : (lane & 7) ^ ((wr >> 1) & 7);        // its piece
    const uint32_t woff = (uint32_t)min(wr, last) * (uint32_t)(nb * (DT == 1 ? 32 : 16));
    const uint32_t wfull = woff + 16 * wc;
    const uint16_t* sb = g.fs + (size_t)row0 * g.nbp;
    const uint32_t soff = (uint32_t)min(16 * rg + c16, last) * (uint32_t)(g.nbp * 2);

    const uint32_t wlast = woff + 16 * (uint32_t)min(wc, (DT == 1 ? 2 : 1) * (nb - 8 * (nst - 1)) - 1);
    // Copy i of this wave (0 .. CP - 1) of stage st into buffer `buf`: x copies
    // are half w % 2 of the vectors of blocks w / 2 + (NW / 2) jj, then the
    // weights' and scales'. Blocks missing from a partial last stage repeat the
    // row's last one.
    const auto copy = [&](int i, int st, uint32_t buf) {
        const uint32_t d = ring + buf;
        if (i < NT * XC) {
            const int t = i / XC, jj = i % XC, blk = min(8 * st + (wave >> 1) + (NW / 2) * jj, nb - 1);
            copy16(xb + 32 * (size_t)blk, xoff[t], d + t * 16384 + (wave + NW * jj) * 1024);
        } else if (i == NT * XC && (DT == 1 ? (H == 1 || half == 0) : wl < 2)) {
            copy16(wb + (size_t)st * (DT == 1 ? 256 : 128), st == nst - 1 ? wlast : wfull,
                   d + L::X + (DT == 1 ? (4 * rg + w) * 1024 : rg * 2048 + w * 1024));
        } else {
            copy16(sb + 8 * (size_t)st, soff, d + L::X + L::W + rg * 1024);
        }
    };
    const auto issue = [&](int st, uint32_t buf) {
#pragma unroll
        for (int i = 0; i < CP; ++i) copy(i, st, buf);
    };
    constexpr int FIRST = NS >= 3 ? 2 : 1;  // stages asked for before the bias pass (its waits drain them)
#pragma unroll
    for (int p = 0; p < FIRST; ++p)
        issue(min(p, nst - 1), p * L::STAGE);

    // Q4's bias term dot_bf16(biases, xsum): 8 chains over whole groups of 8
    // blocks. This wave's: w and w + 4 (hsum8 adds those two first), with
    // H = 2 w + 4 half.
    constexpr int BC = 2 / H;
    f32x4 bsum[NT];
    if (DT == 2) {
        const int ng = nb >> 3;
        const uint16_t* br = g.bi + (size_t)(row0 + min(16 * rg + c16, last)) * nb + wl;
        const float* xr[NT];
        f32x4 b[BC][NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            xr[t] = g.xsum + (size_t)min(tok0 + 16 * t + c16, g.n_tok - 1) * nb + wl;
#pragma unroll
            for (int c = 0; c < BC; ++c) b[c][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        constexpr int U = 4;                                        // steps of 4 groups loaded together
        constexpr int V = (NT == 1 ? 24 : NT == 2 ? 16 : 8) / U;    // such batches in flight
        for (int gg = 0; gg < ng; gg += 4 * U * V) {
            uint16_t a[V][U][BC];
            float xv[V][U][BC][NT];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if (gg + 4 * U * v >= ng) break;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int e = 8 * min(gg + 4 * (U * v + u) + k, ng - 1);
#pragma unroll
                    for (int c = 0; c < BC; ++c) {
                        a[v][u][c] = br[e + 4 * c];
#pragma unroll
                        for (int t = 0; t < NT; ++t) xv[v][u][c][t] = xr[t][e + 4 * c];
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if (gg + 4 * U * v >= ng) break;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool on = gg + 4 * (U * v + u) + k < ng;
#pragma unroll
                    for (int c = 0; c < BC; ++c)
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            b[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                on ? bf16f(a[v][u][c]) : 0.0f, on ? xv[v][u][c][t] : -0.0f, b[c][t], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) bsum[t] = H == 1 ? add4(b[0][t], b[BC - 1][t]) : b[0][t];
    }
#pragma unroll
    for (int p = FIRST; p < NS - 1; ++p)
        issue(min(p, nst - 1), p * L::STAGE);

    f32x4 acc[NT][NC];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < NC; ++i) acc[t][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // LDS offsets of this lane's reads in a stage (step 0; step 1's blocks are 4 on).
    const uint32_t x0 = (uint32_t)(k * 2048 + c16 * 128 + (((w + 4 * half) ^ ((c16 >> 1) & 7)) << 4)), x1 = x0 ^ 64;
    const uint32_t s0 = (uint32_t)(L::X + L::W + rg * 1024 + c16 * 16 + 2 * k);
    const uint32_t w0 = DT == 1 ? (uint32_t)(L::X + rg * 4096 + c16 * 256 + 4 * w + 16 * ((2 * k + half) ^ c16))
                                : (uint32_t)(L::X + rg * 2048 + c16 * 128 + 4 * w + 16 * (k ^ ((c16 >> 1) & 7)));
    struct Quants {
        uint32_t q0, q1;
        uint16_t s;
    };
    const auto load_w = [&](uint32_t p, int s) {
        Quants q;
        const uint32_t o = p + (w0 ^ (s ? (DT == 1 ? 128u : 64u) : 0u));
        q.q0 = *(const uint32_t*)(lds + o);
        q.q1 = DT == 1 && H == 1 ? *(const uint32_t*)(lds + (o ^ 16u)) : 0;
        q.s = *(const uint16_t*)(lds + p + s0 + 8 * s);
        return q;
    };
    const auto load_x = [&](uint32_t p, int s, int t, f32x4(&v)[2 / H]) {
        v[0] = *(const f32x4*)(lds + p + t * 16384 + s * 8192 + x0);
        if (H == 1) v[2 / H - 1] = *(const f32x4*)(lds + p + t * 16384 + s * 8192 + x1);
    };
    const auto convert = [&](const Quants& q, float(&a)[NC]) {
        const float sc = bf16f(q.s);
        const uint32_t lo = (H == 2 && half ? q.q0 >> 4 : q.q0) & 0x0F0F0F0Fu, hi = (q.q0 >> 4) & 0x0F0F0F0Fu;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] = __fmul_rn(DT == 1 ? (float)(int8_t)(q.q0 >> (8 * i)) : (float)((lo >> (8 * i)) & 255u), sc);
            if (H == 1)
                a[NC - 4 + i] =
                    __fmul_rn(DT == 1 ? (float)(int8_t)(q.q1 >> (8 * i)) : (float)((hi >> (8 * i)) & 255u), sc);
        }
    };
    // The NC matrix instructions of a step and vector group; between(i) runs
    // after the i-th and is kept there: an LDS read or a copy issued then costs
    // the wave nothing, where a burst of them before the first matrix
    // instruction leaves the matrix unit idle until the LDS or the address unit
    // has taken them all.
    const auto mfmas = [&](const float(&a)[NC], const f32x4(&v)[2 / H], f32x4(&c)[NC], auto between) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < 2 / H; ++h) {
                c[4 * h + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[4 * h + i], v[h][i], c[4 * h + i], 0, 0, 0);
                between((2 / H) * i + h);
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    // The ring: past the last stage the copies repeat it (into buffers no longer
    // read), so that the waits count the same everywhere.
    const int full = nb >> 3;
    uint32_t cur = 0, fill = (NS - 1) * L::STAGE;  // the buffers computed from and refilled
    const auto after = [&](uint32_t p) { return p == (NS - 1) * L::STAGE ? 0 : p + L::STAGE; };
    const auto turn = [&]() {
        // This wave's copies of the stage have landed once at most those of the
        // NS - 2 later stages are outstanding; after the barrier everyone's have,
        // and everyone is done with the buffer refilled next.
        wait_vmcnt<CP*(NS - 2)>();
        lds_barrier();
    };
    constexpr int SLOTS = 2 * NT * NC;  // matrix instructions of a stage
    Quants q;
    f32x4 xv[2][2 / H];
    for (int st = 0; st < full; ++st) {
        turn();
        q = load_w(cur, 0);
        load_x(cur, 0, 0, xv[0]);
        const int sf = min(st + NS - 1, nst - 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float a[NC];
            convert(q, a);
            if (s == 0) q = load_w(cur, 1);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int v = s * NT + t;
                if (t + 1 < NT)
                    load_x(cur, s, t + 1, xv[(v + 1) & 1]);
                else if (s == 0)
                    load_x(cur, 1, 0, xv[(v + 1) & 1]);
                mfmas(a, xv[v & 1], acc[t], [&](int i) {
                    const int u = v * NC + i;
#pragma unroll
                    for (int e = u * CP / SLOTS; e < (u + 1) * CP / SLOTS; ++e) copy(e, sf, fill);
                });
            }
        }
        fill = after(fill);
        cur = after(cur);
    }
    if (full < nst) {  // the partial last stage
        wait_vmcnt<0>();
        lds_barrier();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (8 * full + 4 * s >= nb) break;
            const bool on = 8 * full + 4 * s + k < nb;
            float a[NC];
            convert(load_w(cur, s), a);
#pragma unroll
            for (int i = 0; i < NC; ++i) a[i] = on ? a[i] : 0.0f;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                f32x4 v[2 / H];
                load_x(cur, s, t, v);
#pragma unroll
                for (int h = 0; h < 2 / H; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[h][i] = on ? v[h][i] : -0.0f;
                mfmas(a, v, acc[t], [](int) {});
            }
        }
    }

    // v[l] = (a_l + a_{8+l}) + (a_{16+l} + a_{24+l}): words 2 and 3 (with H = 2
    // also the upper halves) hand their chains to waves 0 and 1; hsum8 then
    // adds wave 1's v[4..7] to wave 0's v[0..3].
    wait_vmcnt<0>();  // the repeated copies, before the ring is written over (the loop's first barrier: everyone's)
    unsigned char* m = lds + rg * L::MEET_RG + lane * 16;
    constexpr int VOFF = L::PARTS * 1024, BOFF = VOFF + 4096;
    // Where chain quad (word, half) waits: words 2, 3 of half 0, then half 1's four.
    const auto part = [&](int word, int h, int i) {
        return (f32x4*)(m + ((h == 0 ? word - 2 : H == 1 ? word : 2 + word) * 4 + i) * 1024);
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        lds_barrier();
        if (wl >= 2)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                *part(w, half, i) = acc[t][i];
                if (H == 1) *part(w, 1, i) = acc[t][NC - 4 + i];
            }
        if (DT == 2) *(f32x4*)(m + BOFF + wl * 1024) = bsum[t];
        lds_barrier();
        f32x4 v[4];
        if (wl < 2) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 up = H == 1 ? acc[t][NC - 4 + i] : *part(w, 1, i);
                v[i] = add4(add4(acc[t][i], *part(w + 2, 0, i)), add4(up, *part(w + 2, 1, i)));
                if (wl == 1) *(f32x4*)(m + VOFF + i * 1024) = v[i];
            }
        }
        lds_barrier();
        if (wl == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = add4(v[i], *(const f32x4*)(m + VOFF + i * 1024));
            f32x4 r = add4(add4(v[0], v[1]), add4(v[2], v[3]));
            const int row = row0 + 16 * rg + 4 * k, tok = tok0 + 16 * t + c16;
            if (DT == 2) {
                f32x4 p[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = *(const f32x4*)(m + BOFF + i * 1024);
                    if (H == 2) p[i] = add4(p[i], *(const f32x4*)(m + BOFF + (4 + i) * 1024));
                }
                f32x4 b = add4(add4(p[0], p[1]), add4(p[2], p[3]));
                for (int i = nb & ~7; i < nb; ++i) {
                    const float xv = g.xsum[(size_t)min(tok, g.n_tok - 1) * nb + i];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        b[e] = __fadd_rn(b[e], __fmul_rn(bf16f(g.bi[(size_t)min(row + e, g.rows - 1) * nb + i]), xv));
                }
                r = add4(r, b);
            }
            store4(g, r, row, tok);
        }
    }
}

// A workgroup's row tile, first vector and 16-vector groups. Workgroups go
// round-robin to the 8 XCDs; each XCD takes a contiguous range of logical ids,
// the token tiles of a row tile side by side, so a row tile's weights are read
// once into its L2.
__device__ __forceinline__ void batch_tile(const BatchArgs& g, int& rt, int& tok0, int& nt) {
    const int total = gridDim.x, per = total / 8, rem = total % 8, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const int id = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
    rt = id / g.ttiles;
    const int tt = id - rt * g.ttiles;
    nt = g.tq + (tt < g.tr ? 1 : 0);
    tok0 = 16 * (tt * g.tq + min(tt, g.tr));
}

// NT: 16-vector groups of the largest token tile; a launch's tiles hold NT or
// NT - 1 of them.
template <int DT, int R, int NT, int H, int NS>
__global__ __launch_bounds__(R * H * 256) void gemm_f32_kernel(BatchArgs g) {
    extern __shared__ __align__(16) unsigned char lds[];
    int rt, tok0, nt;
    batch_tile(g, rt, tok0, nt);
    if (nt == NT)
        batch_body<DT, R, NT, H, NS>(g, lds, rt * 16 * R, tok0);
    else if constexpr (NT > 1)
        batch_body<DT, R, NT - 1, H, NS>(g, lds, rt * 16 * R, tok0);
}

// BF16 weights for several vectors, the same scheme (kernels_bf16.hip names the
// reference's kernel per shape and its chains):
//   ROW32       32 chains, element j of every 32-block: a wave's chains and the
//               meeting as for Q8_0 above;
//   QUAD, ROW8  8 chains over elements 8 i + l, i in order: a matrix instruction
//               takes 4 values of i (32 columns), a wave the chain pair that is
//               added first (QUAD l = 2 w, 2 w + 1, ROW8's hsum8 l = w, w + 4),
//               so waves meet once, on (p0 + p1) + (p2 + p3).
// A stage is 256 columns: 512 bytes per row of raw weights, in 16-byte pieces
// XOR-swizzled by row. Measured (us; before: four vectors per pass of
// gemv_bf16_kernel): 6144 x 1536, 16 vectors 38.6 -> 8.4, 6143 rows 38.8 -> 8.3;
// 14336 x 4096 149 -> 34.4.
template <int R, int NT>
struct Bf16Lds {
    static constexpr int X = NT * 16384;
    static constexpr int STAGE = X + R * 8192;
};

template <int PATH, int R, int NT, int NS>
__device__ __forceinline__ void bf16_body(const BatchArgs& g, unsigned char* lds, int row0, int tok0) {
    using L = Bf16Lds<R, NT>;
    constexpr bool WIDE = PATH == BF16_PATH_ROW32, QUAD = PATH == BF16_PATH_QUAD;
    constexpr int NC = WIDE ? 8 : 2;           // chains per wave
    constexpr int STEPS = WIDE ? 2 : 8;        // matrix instructions of a chain per stage
    constexpr int NW = 4 * R, XC = 16 / NW;    // waves; x copies per wave, stage and vector group
    constexpr int CP = NT * XC + 2;            // copies per wave and stage
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave >> 2, w = wave & 3, c16 = lane & 15, k = lane >> 4;
    const int cols = 32 * g.nb + g.rem, nst = (cols + 255) / 256, full = cols / 256;
    const uint32_t ring = (uint32_t)(uintptr_t)lds;

    uint32_t xrow[NT];
    const float* xb = g.x + (size_t)tok0 * g.xs;
    const int v8 = 8 * (wave & 1) + (lane >> 3);
    const uint32_t xc = 16 * ((lane & 7) ^ ((v8 >> 1) & 7));
#pragma unroll
    for (int t = 0; t < NT; ++t) xrow[t] = (uint32_t)min(16 * t + v8, g.n_tok - 1 - tok0) * (uint32_t)(g.xs * 4);
    const int last = g.rows - 1 - row0;
    const uint8_t* wb = g.qs + (size_t)row0 * cols * 2;
    uint32_t wfull[2], wlast[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 4 * w + 2 * i + (lane >> 5), c = (lane & 31) ^ r;  // row in the group, its piece
        const uint32_t o = (uint32_t)min(16 * rg + r, last) * (uint32_t)(cols * 2);
        wfull[i] = o + 16 * c;
        wlast[i] = o + 16 * min(c, cols / 8 - 32 * (nst - 1) - 1);  // pieces past the row repeat its last one
    }
    const auto copy = [&](int i, int st, uint32_t buf) {
        const uint32_t d = ring + buf;
        if (i < NT * XC) {
            const int t = i / XC, jj = i % XC, kk = (wave >> 1) + (NW / 2) * jj;
            uint32_t o = xc + (uint32_t)(8 * st + kk) * 128;
            if (st == nst - 1) o = min(o, (uint32_t)(cols * 4 - 16));
            copy16(xb, xrow[t] + o, d + t * 16384 + (wave + NW * jj) * 1024);
        } else {
            const int j = i - NT * XC;
            copy16(wb + (size_t)st * 512, st == nst - 1 ? wlast[j] : wfull[j],
                   d + L::X + rg * 8192 + (2 * w + j) * 1024);
        }
    };
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
#pragma unroll
        for (int i = 0; i < CP; ++i) copy(i, min(p, nst - 1), p * L::STAGE);

    f32x4 acc[NT][NC];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < NC; ++i) acc[t][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
    const auto hi = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
    // The weights' operands of step s: piece 4 s + k of the row (QUAD, ROW8), or
    // the pieces of block 4 s + k.
    const auto load_w = [&](uint32_t p, int s, float(&a)[NC]) {
        const unsigned char* row = lds + p + L::X + rg * 8192 + c16 * 512;
        if (WIDE) {
            const int c = 4 * (4 * s + k) + (w >> 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint2 v = *(const uint2*)(row + 16 * ((c + 2 * h) ^ c16) + 8 * (w & 1));
                a[4 * h % NC] = lo(v.x);
                a[(4 * h + 1) % NC] = hi(v.x);
                a[(4 * h + 2) % NC] = lo(v.y);
                a[(4 * h + 3) % NC] = hi(v.y);
            }
        } else {
            const unsigned char* q = row + 16 * ((4 * s + k) ^ c16);
            if (QUAD) {
                const uint32_t v = *(const uint32_t*)(q + 4 * w);
                a[0] = lo(v);
                a[1] = hi(v);
            } else {
                a[0] = lo(*(const uint16_t*)(q + 2 * w));
                a[1] = lo(*(const uint16_t*)(q + 8 + 2 * w));
            }
        }
    };
    const int sw = (c16 >> 1) & 7;
    const auto load_x = [&](uint32_t p, int s, int t, float(&b)[NC]) {
        const unsigned char* x = lds + p + t * 16384 + (WIDE ? 4 * s + k : s) * 2048 + c16 * 128;
        if (WIDE) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 v = *(const f32x4*)(x + 16 * ((w + 4 * h) ^ sw));
#pragma unroll
                for (int i = 0; i < 4; ++i) b[(4 * h + i) % NC] = v[i];
            }
        } else if (QUAD) {
            const float2 v = *(const float2*)(x + 16 * ((2 * k + (w >> 1)) ^ sw) + 8 * (w & 1));
            b[0] = v.x;
            b[1] = v.y;
        } else {
            b[0] = *(const float*)(x + 16 * ((2 * k) ^ sw) + 4 * w);
            b[1] = *(const float*)(x + 16 * ((2 * k + 1) ^ sw) + 4 * w);
        }
    };
    uint32_t cur = 0, fill = (NS - 1) * L::STAGE;
    const auto after = [&](uint32_t p) { return p == (NS - 1) * L::STAGE ? 0 : p + L::STAGE; };
    constexpr int SLOTS = STEPS * NT * NC;
    for (int st = 0; st < full; ++st) {
        wait_vmcnt<CP*(NS - 2)>();
        lds_barrier();
        const int sf = min(st + NS - 1, nst - 1);
        float a[2][NC], b[2][NC];
        load_w(cur, 0, a[0]);
        load_x(cur, 0, 0, b[0]);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            if (s + 1 < STEPS) load_w(cur, s + 1, a[(s + 1) & 1]);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int v = s * NT + t;
                if (v + 1 < STEPS * NT) load_x(cur, (v + 1) / NT, (v + 1) % NT, b[(v + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s & 1][i], b[v & 1][i], acc[t][i], 0, 0, 0);
                    const int u = v * NC + i;
#pragma unroll
                    for (int e = u * CP / SLOTS; e < (u + 1) * CP / SLOTS; ++e) copy(e, sf, fill);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        fill = after(fill);
        cur = after(cur);
    }
    if (full < nst) {  // the partial last stage: missing steps are 0 * -0
        wait_vmcnt<0>();
        lds_barrier();
        const int left = WIDE ? (cols - 256 * full) / 32 : (cols - 256 * full) / 8;  // blocks / values of i
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            if (4 * s >= left) break;
            const bool on = 4 * s + k < left;
            float a[NC], b[NC];
            load_w(cur, s, a);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                load_x(cur, s, t, b);
#pragma unroll
                for (int i = 0; i < NC; ++i)
                    acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(on ? a[i] : 0.0f, on ? b[i] : -0.0f, acc[t][i], 0, 0,
                                                                     0);
            }
        }
    }

    wait_vmcnt<0>();  // the repeated copies, before the ring is written over
    lds_barrier();
    if constexpr (WIDE) {
        // As in batch_body: words 2 and 3 hand their chains to words 0 and 1.
        unsigned char* m = lds + rg * 20 * 1024 + lane * 16;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            lds_barrier();
            if (w >= 2)
#pragma unroll
                for (int i = 0; i < 8; ++i) *(f32x4*)(m + ((w - 2) * 8 + i) * 1024) = acc[t][i % NC];
            lds_barrier();
            f32x4 v[4];
            if (w < 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = add4(add4(acc[t][i % NC], *(const f32x4*)(m + (w * 8 + i) * 1024)),
                                add4(acc[t][(4 + i) % NC], *(const f32x4*)(m + (w * 8 + 4 + i) * 1024)));
                    if (w == 1) *(f32x4*)(m + (16 + i) * 1024) = v[i];
                }
            }
            lds_barrier();
            if (w == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = add4(v[i], *(const f32x4*)(m + (16 + i) * 1024));
                store4(g, add4(add4(v[0], v[1]), add4(v[2], v[3])), row0 + 16 * rg + 4 * k, tok0 + 16 * t + c16);
            }
        }
    } else {
        unsigned char* m = lds + rg * 4 * NT * 1024 + lane * 16;
#pragma unroll
        for (int t = 0; t < NT; ++t) *(f32x4*)(m + (4 * t + w) * 1024) = add4(acc[t][0], acc[t][1]);
        lds_barrier();
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if ((t & 3) != w) continue;
            f32x4 p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = *(const f32x4*)(m + (4 * t + i) * 1024);
            store4(g, add4(add4(p[0], p[1]), add4(p[2], p[3])), row0 + 16 * rg + 4 * k, tok0 + 16 * t + c16);
        }
    }
}

template <int PATH, int R, int NT, int NS>
__global__ __launch_bounds__(R * 256) void gemm_bf16_kernel(BatchArgs g) {
    extern __shared__ __align__(16) unsigned char lds[];
    int rt, tok0, nt;
    batch_tile(g, rt, tok0, nt);
    if (nt == NT)
        bf16_body<PATH, R, NT, NS>(g, lds, rt * 16 * R, tok0);
    else if constexpr (NT > 1)
        bf16_body<PATH, R, NT - 1, NS>(g, lds, rt * 16 * R, tok0);
}

// The launch's token tiles: n16 groups of 16 vectors spread over tiles of at most nt.
int token_tiles(BatchArgs& g, int nt) {
    const int n16 = ceil_div(g.n_tok, 16);
    g.ttiles = ceil_div(n16, nt);
    g.tq = n16 / g.ttiles;
    g.tr = n16 % g.ttiles;
    return g.ttiles;
}

template <int DT, int R, int NT, int H, int NS>
void launch_batch(BatchArgs g, hipStream_t st) {
    using L = BatchLds<DT, R, NT, H>;
    constexpr int LDS = NS * L::STAGE > L::MEET ? NS * L::STAGE : L::MEET;
    static_assert(LDS <= 160 * 1024, "the ring fits the LDS");
    static const bool once = [] {
        return hipFuncSetAttribute((const void*)gemm_f32_kernel<DT, R, NT, H, NS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
    }();
    (void)once;
    const int tiles = token_tiles(g, NT);
    gemm_f32_kernel<DT, R, NT, H, NS><<<ceil_div(g.rows, 16 * R) * tiles, R * H * 256, LDS, st>>>(g);
}

template <int PATH, int R, int NT, int NS>
void launch_bf16(BatchArgs g, hipStream_t st) {
    constexpr int LDS = NS * Bf16Lds<R, NT>::STAGE;
    static_assert(LDS <= 160 * 1024 && LDS >= R * 20 * 1024, "the ring fits the LDS and holds the meeting area");
    static const bool once = [] {
        return hipFuncSetAttribute((const void*)gemm_bf16_kernel<PATH, R, NT, NS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
    }();
    (void)once;
    const int tiles = token_tiles(g, NT);
    gemm_bf16_kernel<PATH, R, NT, NS><<<ceil_div(g.rows, 16 * R) * tiles, R * 256, LDS, st>>>(g);
}

template <int DT>
void launch_dt(const BatchArgs& g, hipStream_t st) {
    switch (batch_split(g.rows, g.n_tok, cu_count())) {
        case 1: launch_batch<DT, 1, 1, 2, 3>(g, st); break;
        case 0: launch_batch<DT, 1, 1, 1, 3>(g, st); break;
        case 2: launch_batch<DT, 2, 2, 1, 3>(g, st); break;
        default: launch_batch<DT, 2, 4, 1, 2>(g, st); break;
    }
}

template <int PATH>
void launch_path(const BatchArgs& g, hipStream_t st) {
    switch (batch_split(g.rows, g.n_tok, cu_count())) {
        case 0:
        case 1: launch_bf16<PATH, 1, 1, 3>(g, st); break;
        case 2: launch_bf16<PATH, 2, 2, 3>(g, st); break;
        default: launch_bf16<PATH, 2, 4, 2>(g, st); break;
    }
}

}  // namespace

// The split with the least time: rounds of workgroups over the CUs times a
// workgroup's time per stage of 256 columns (us, measured for Q8_0 at 14336 and
// 4096 rows; BF16's is within a tenth): 0 one row group and 16 vectors per
// workgroup, 1 the same with a workgroup or less per CU, 2 two row groups and
// 32 vectors, 3 two and 64.
int batch_split(int rows, int n_tok, int cus) {
    const int n16 = ceil_div(n_tok, 16);
    const auto cost = [&](int r, int nt, double us) {
        const long wgs = (long)ceil_div(rows, 16 * r) * ceil_div(n16, nt);
        return (double)((wgs + cus - 1) / cus) * us;
    };
    const double c11 = cost(1, 1, 0.45), c22 = cost(2, 2, 1.42), c24 = cost(2, 4, 2.6);
    if (c24 <= c11 && c24 <= c22) return 3;
    if (c22 <= c11) return 2;
    return (long)ceil_div(rows, 16) * n16 <= cus ? 1 : 0;
}

// Vectors of one launch: a grid holds less than 2^32 threads, and every split
// has at most 512 per 16 rows x 16 vectors. 0: not even 16 vectors.
int batch_slice(int rows) { return 16 * (int)(((size_t)1 << 22) / ceil_div(rows, 16)); }

// Few vectors: a group of 16 costs the same from 1 to 16, in rounds of 16 rows
// per CU, so short rows, a partial round and many rounds of two to eight vectors
// are left to the kernels of kernels_f32.hip (one vector at a time, or four at
// a time through the tall matrices' kernel). Measured, both at 2000 sizes from
// 128 x 512 to 151936 x 512 and 28672 x 4096; us, those against these: Q8_0 two
// vectors 4096 x 4096 11.7 / 10.4, 256 x 4096 9.1 / 10.1, 2048 x 12288 22.1 /
// 24.8, three 20000 x 1024 10.1 / 13.2, 28672 x 4096 58.6 / 47.4; Q4 three
// 4096 x 4096 15.7 / 15.0, 8192 x 1024 9.6 / 10.5, five 65536 x 1024 41.2 / 60.8,
// 14336 x 4096 45.4 / 36.1.
bool batch_wins(int dtype, int rows, int nb, int n_tok, bool v2) {
    if (n_tok > 12) return true;
    if (v2) {
        // The blocks per row from which these are no slower, by vectors and rows.
        constexpr short NO = 32767;
        constexpr int ROWS[5] = {12288, 16384, 24576, 32767, 49152};
        constexpr short MIN[2][6][6] = {
            {{48, 216, 216, 216, 216, 216},  // Q8_0: 2 vectors
             {48, 80, 171, 112, 171, 171},   // 3
             {48, 48, 112, 112, 144, 144},   // 4
             {0, 0, 32, 32, 0, 48},          // 5, 6
             {0, 0, 0, 0, 0, 32},            // 7, 8
             {0, 0, 0, 0, 0, 0}},            // 9 .. 12
            {{NO, NO, NO, NO, NO, NO},     // Q4
             {NO, NO, NO, NO, NO, NO},
             {NO, NO, NO, NO, NO, NO},
             {32, 48, 80, 112, 48, 112},
             {0, 32, 48, 64, 32, 80},
             {0, 0, 0, 0, 0, 32}}};
        int c = 0;
        while (c < 5 && rows > ROWS[c]) ++c;
        return nb >= MIN[dtype - 1][n_tok <= 4 ? n_tok - 2 : n_tok <= 6 ? 3 : n_tok <= 8 ? 4 : 5][c];
    }
    if (dtype == 1) {
        if (n_tok > 2) return true;
        if (rows < 2048) return nb <= 80 || nb > 256 || (rows >= 1280 && nb <= 128);
        if (rows <= 4096) return nb <= 48 || (rows >= 2560 && nb <= 96) || rows >= 3584;
        if (rows <= 8192) return nb <= 24 || rows >= 7168;
        return rows >= 11776 && nb >= 64;
    }
    if (n_tok > 4) return true;
    if (n_tok == 4) return rows <= 4096 || (rows <= 8192 ? nb >= 24 && (rows >= 6144 || nb < 384) : nb >= 48);
    if (n_tok < 3 || nb <= 32) return false;
    if (rows <= 4096) return rows < 2048 || nb <= 160 || rows >= 3584;
    return nb >= 64 && rows >= 7168;
}

// BF16: measured likewise (four vectors, us): 256 x 4096 15.8 / 12.4, 257 x 4096
// 8.2 / 10.9, 4097 x 4096 22.8 / 15.0, 14336 x 2048 13.5 / 18.3, x 4096 37.8 / 31.4;
// from five no size was slower.
bool batch_wins_bf16(int path, int rows, int cols, int n_tok) {
    if (n_tok != 4) return n_tok > 4;
    if (path == BF16_PATH_ROW32) return cols < 2048 || (rows > 2048 ? cols >= 4096 || rows > 3000 : cols > 8192);
    return rows <= 8192 || cols >= 4096 || (path == BF16_PATH_ROW8 && cols <= 520);
}

namespace {
// g's vectors by slices; xsum, if any, has a row of nb per vector.
template <class Launch>
void launch_slices(const BatchArgs& g, const Launch& launch) {
    const int step = batch_slice(g.rows);
    for (long t = 0; t < g.n_tok; t += step) {
        BatchArgs p = g;
        p.x += (size_t)t * g.xs;
        p.y += (size_t)t * g.ys;
        if (p.xsum) p.xsum += (size_t)t * g.nb;
        p.n_tok = (int)(g.n_tok - t < step ? g.n_tok - t : step);
        launch(p);
    }
}
}  // namespace

bool launch_gemm_f32(int dtype, const uint8_t* qs, const uint16_t* fs, const uint16_t* biases, const float* x,
                     size_t x_stride, float* xsum, int rows, int nb, int nbp, int n_tok, float* y, size_t y_stride,
                     bool v2, hipStream_t st) {
    if (n_tok < 2 || !batch_wins(dtype, rows, nb, n_tok, v2)) return false;
    // 16-byte pieces of x; 32-bit byte offsets within a tile's rows.
    if (((uintptr_t)x & 15) || (x_stride & 3) || x_stride >= ((size_t)1 << 23) || nb >= (1 << 21) ||
        batch_slice(rows) == 0)
        return false;
    if (dtype == 2) launch_block_sums(x, x_stride, nb, n_tok, xsum, st);
    const BatchArgs g{qs, fs,       biases, x,  xsum, y, x_stride, y_stride,
                      rows, nb, nbp, n_tok, 0, 0, 0, 0, ((uintptr_t)y & 15) == 0 && (y_stride & 3) == 0};
    launch_slices(g, [&](const BatchArgs& p) {
        if (dtype == 1)
            launch_dt<1>(p, st);
        else
            launch_dt<2>(p, st);
    });
    return true;
}

bool launch_gemm_bf16(int path, const uint16_t* raw, int rows, int cols, const float* x, size_t x_stride, int n_tok,
                      float* y, size_t y_stride, hipStream_t st) {
    if (path == BF16_PATH_F64 || !batch_wins_bf16(path, rows, cols, n_tok) || ((uintptr_t)x & 15) || (x_stride & 3) ||
        x_stride >= ((size_t)1 << 23) || cols >= (1 << 26) || batch_slice(rows) == 0)
        return false;
    const BatchArgs g{(const uint8_t*)raw, nullptr, nullptr, x, nullptr, y, x_stride, y_stride, rows, cols / 32, 0, n_tok,
                      cols % 32,           0,       0,       0, ((uintptr_t)y & 15) == 0 && (y_stride & 3) == 0};
    launch_slices(g, [&](const BatchArgs& p) {
        if (path == BF16_PATH_QUAD)
            launch_path<BF16_PATH_QUAD>(p, st);
        else if (path == BF16_PATH_ROW8)
            launch_path<BF16_PATH_ROW8>(p, st);
        else
            launch_path<BF16_PATH_ROW32>(p, st);
    });
    return true;
}

}  // namespace nnh
