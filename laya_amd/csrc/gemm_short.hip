// Short products: linear layers over a few hundred rows.
//
// At 189 rows a 768-wide projection is 12 tiles of 128 x 128, and with K split over the idle CUs a product was three
// dependent launches (operand magnitudes, the partial products, a pass that sums them), each several microseconds of
// latency whatever it computes. Here one launch does it all, on tiles of 64 x 64 down to 32 x 32 so that the grid
// covers the chip, with K dealt to the eight waves of a workgroup: each wave streams its own K range of the whole
// tile and no barrier is met until the waves' sums meet in LDS, where the epilogue adds them in wave order
// (deterministic) and reads them by rows.
//
// Operands go from memory straight into the wave's part of LDS, 32 of K at a time (16-byte direct-to-LDS loads of
// whole lines), the next stage in flight while this one is multiplied. An operand contiguous along K lies there as
// [row][32 k], the 16-byte chunks of a row XOR-ed by (row / 2) mod 8; one contiguous along its rows (dX's W, dW's dY
// and x) as [k][64 rows]: the fragment reads of both meet no bank conflict.
//
// fp32 operands are split into two fp16 pieces (split.hpp) with a power-of-two scale that each wave takes from the
// values it has just loaded and lowers as it goes (the accumulators follow, exactly), so no pass over the operands
// precedes the product.
#include <type_traits>

#include "gemm_short.hpp"
#include "elementwise.hpp"
#include "split.hpp"

namespace laya {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int UNIT = 32;  // K per stage
constexpr int CHAIN = 3;  // stages summed in one accumulator

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// Tile row (or column) r of B under the Geglu epilogue: columns 0–31 of the tile are the first half's a0 … a0 + 31,
// columns 32–63 the second half's.
__device__ __forceinline__ int geglu_row(int r, int a0, int inter) {
    return min(a0 + (r & 31), inter - 1) + (r < 32 ? 0 : inter);
}

// One wave's stage of a T-row operand contiguous along K: T x 32 floats in LDS. Rows past the edge are clamped (they
// reach only outputs that are never stored).
template <int T>
struct SideK {
    static constexpr int LDS = T * UNIT;
    __amdgpu_buffer_rsrc_t rs;
    unsigned off[T / 8];
    float* lds;
    // inter: 0, or GeGLU's width (the tile's rows taken in pairs from both halves).
    __device__ __forceinline__ SideK(const float* src, long ld, int rows, int K, int r0, int lane, float* stage, int inter)
        : rs(buffer_of(src, (unsigned)(((long)(rows - 1) * ld + K) * 4))), lds(stage) {
#pragma unroll
        for (int j = 0; j < T / 8; ++j) {
            const int r = 8 * j + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
            const int row = inter ? geglu_row(r, r0, inter) : min(r0 + r, rows - 1);
            off[j] = ((unsigned)row * (unsigned)ld + 4u * chunk) * 4u;
        }
    }
    __device__ __forceinline__ void issue(int k0) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass has no 16-byte form of the builtin
#pragma unroll
        for (int j = 0; j < T / 8; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds + j * 256), 16, off[j], k0 * 4, 0, 0);
#endif
    }
    __device__ __forceinline__ void fetch(float (&v)[T / 32][2][8], int lr, int h) const {
#pragma unroll
        for (int i = 0; i < T / 32; ++i) {
            const int r = 32 * i + lr;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int chunk = (4 * s + 2 * h + q) ^ ((r >> 1) & 7);
                    const f32x4 x = *reinterpret_cast<const f32x4*>(lds + r * UNIT + 4 * chunk);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][s][4 * q + e] = x[e];
                }
        }
    }
};

// One wave's stage of an operand contiguous along its rows (64 of them): 32 x 64 floats in LDS, [k][row]. Lane r of a
// half holds rows 2r and 2r + 1 of the half's 16 k.
struct SideMN {
    static constexpr int T = 64, LDS = T * UNIT;
    __amdgpu_buffer_rsrc_t rs;
    unsigned col, ld4;
    int row, K;
    float* lds;
    __device__ __forceinline__ SideMN(const float* src, long ld, int rows, int k, int r0, int lane, float* stage, int)
        : rs(buffer_of(src, (unsigned)(((long)(k - 1) * ld + rows) * 4))),
          col((unsigned)min(r0 + 4 * (lane & 15), rows - 4) * 4u),
          ld4((unsigned)ld * 4u),
          row(lane >> 4),
          K(k),
          lds(stage) {}
    __device__ __forceinline__ void load(int j, unsigned voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(lds + j * 256), 16, voff, soff, 0, 0);
#endif
    }
    __device__ __forceinline__ void issue(int k0) {
        if (k0 + UNIT <= K) {
            const unsigned off = (unsigned)row * ld4 + col;
#pragma unroll
            for (int j = 0; j < UNIT / 4; ++j) load(j, off, (int)((unsigned)(k0 + 4 * j) * ld4));
        } else {  // the last stage: K rows past the end repeat the last one, and are zeroed when read
#pragma unroll
            for (int j = 0; j < UNIT / 4; ++j) load(j, (unsigned)min(k0 + 4 * j + row, K - 1) * ld4 + col, 0);
        }
    }
    __device__ __forceinline__ void zero_tail(int k0) {
        for (int k = K - k0; k < UNIT; ++k) lds[k * T + (int)(threadIdx.x & 63)] = 0.0f;
    }
    __device__ __forceinline__ void fetch(float (&v)[2][2][8], int lr, int h) const {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const f32x2 x = *reinterpret_cast<const f32x2*>(lds + (16 * s + 8 * h + e) * T + 2 * lr);
                v[0][s][e] = x[0];
                v[1][s][e] = x[1];
            }
    }
};

__device__ __forceinline__ float max3_abs(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp_max(unsigned v) {
    return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true));
}

// The scale exponent of a wave's values (pair_scale_exp of the largest finite magnitude), in every lane.
template <int I>
__device__ __forceinline__ int wave_scale_exp(const float (&v)[I][2][8]) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; e += 2) m = max3_abs(m, v[i][s][e], v[i][s][e + 1]);
    auto all = [](unsigned u) {
        u = dpp_max<0x111>(u);  // row_shr 1, 2, 4, 8: the row's last lane holds its maximum
        u = dpp_max<0x112>(u);
        u = dpp_max<0x114>(u);
        u = dpp_max<0x118>(u);
        u = dpp_max<0x142>(u);  // row_bcast 15, 31: the wave's last lane holds the wave's
        u = dpp_max<0x143>(u);
        return (unsigned)__builtin_amdgcn_readlane((int)u, 63);
    };
    unsigned u = all(__builtin_bit_cast(unsigned, m));
    if (u >= 0x7f800000u) {  // an infinity or NaN among them: the largest finite one, value by value
        unsigned f = 0;
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) f = max(f, amax_bits(v[i][s][e]));
        u = all(f);
    }
    return pair_scale_exp(u);
}

// Scales of a line (a row of A, a column of B) of its own rather than of the wave's tile: each lane holds 16 of its
// line's 32 values, the lane 32 away the rest. e: the lines' exponents; lowered where a value would leave fp16's range,
// with two bits to spare (a line's later values seldom reach four times its first 32's largest; below, the low piece's
// floor is still 2^-37 of the line's largest). drop: how far; whether any line's was, in the whole wave.
constexpr int NO_SCALE = 200;  // before a line's first stage
template <int I>
__device__ __forceinline__ bool line_scale_exps(const float (&v)[I][2][8], int (&e)[I], int (&drop)[I]) {
    auto both = [](unsigned u) {
#ifdef __HIP_DEVICE_COMPILE__
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return max((unsigned)r[0], (unsigned)r[1]);
#else
        return u;
#endif
    };
    unsigned u[I], top = 0;
#pragma unroll
    for (int i = 0; i < I; ++i) {
        float m = 0.0f;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int k = 0; k < 8; k += 2) m = max3_abs(m, v[i][s][k], v[i][s][k + 1]);
        u[i] = both(__builtin_bit_cast(unsigned, m));
        top = max(top, u[i]);
    }
    if (__any(top >= 0x7f800000u)) {  // an infinity or NaN among them: the largest finite ones, value by value
#pragma unroll
        for (int i = 0; i < I; ++i) {
            unsigned f = 0;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int k = 0; k < 8; ++k) f = max(f, amax_bits(v[i][s][k]));
            u[i] = both(f);
        }
    }
#pragma unroll
    for (int i = 0; i < I; ++i) {
        const int p = pair_scale_exp(u[i]), n = e[i] > p ? p - 2 : e[i];
        drop[i] = n - e[i];
        e[i] = n;
    }
    int any = 0;
#pragma unroll
    for (int i = 0; i < I; ++i) any |= drop[i];
    return __any(any);
}

template <int NP>
struct Frag {
    f16x8 hi, lo;
    __device__ __forceinline__ void set(const float (&v)[8], float sc) {
        f16x4 h0, l0, h1, l1;
        split2h_4(f32x4{v[0], v[1], v[2], v[3]}, sc, h0, l0);
        split2h_4(f32x4{v[4], v[5], v[6], v[7]}, sc, h1, l1);
        hi = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
        lo = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    __device__ __forceinline__ void mma(const Frag& b, f32x16& c) const {
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b.hi, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b.lo, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b.hi, c, 0, 0, 0);
    }
};

template <>
struct Frag<1> {
    bf16x8 x;
    __device__ __forceinline__ void set(const float (&v)[8], float) {
        typedef float f32x8 __attribute__((ext_vector_type(8)));
        x = __builtin_convertvector((f32x8{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]}), bf16x8);
    }
    __device__ __forceinline__ void mma(const Frag& b, f32x16& c) const {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, b.x, c, 0, 0, 0);
    }
};

// LDS floats of a wave: its stage, later its sums.
template <int TM, int TN>
constexpr int wave_floats() {
    const int stage = UNIT * (TM + TN);
    return stage > TM * TN ? stage : TM * TN;
}

// One output tile by one workgroup of W waves. AK / BK: A / B contiguous along K (K a multiple of 32 then). EP: the
// epilogue; N and the leading dimensions of C and R multiples of 4, their bases 16-byte aligned. smem: W · wave_floats.
// LINES: two-piece scales by row of A and column of B instead of by wave, which keep lines far below the tile's largest.
template <bool AK, bool BK, int TM, int TN, ShortEpilogue EP, int W, int NP, bool LINES = false>
__device__ __forceinline__ void short_tile(const ShortGemm& p, int tile, float* smem) {
    constexpr int I = TM / 32, J = TN / 32, THREADS = 64 * W;
    constexpr int STAGE = UNIT * (TM + TN);
    static_assert((AK || TM == 64) && (BK || TN == 64), "operands contiguous along their rows come 64 wide");
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, h = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tn = tile / p.tiles_m, tm = tile - tn * p.tiles_m;  // rows fastest: B's tile stays on one XCD
    const int m0 = tm * TM, n0 = tn * (EP == ShortEpilogue::Geglu ? TN / 2 : TN);

    // A wave adds CHAIN stages into acc, then acc into sum: an accumulator that took every product would round 6 times
    // per stage at its full size (2.1e-7 against 1.4e-7 relative L2 at K = 2304).
    f32x16 acc[I][J], sum[I][J];
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j) f(acc[i][j], sum[i][j]);
    };
    each([](f32x16& a, f32x16& t) { a = t = f32x16{}; });
    static_assert(!LINES || NP == 2, "bf16 products have no scales");
    int ea = 126, eb = 126, la[I], lb[J];
#pragma unroll
    for (int i = 0; i < I; ++i) la[i] = NO_SCALE;
#pragma unroll
    for (int j = 0; j < J; ++j) lb[j] = NO_SCALE;
    auto rescale = [&](int i, int j, int r, int d) {
        acc[i][j][r] = __builtin_amdgcn_ldexpf(acc[i][j][r], d);
        sum[i][j][r] = __builtin_amdgcn_ldexpf(sum[i][j][r], d);
    };
    // A value of the lane that holds row 8·(r / 4) + 4h + r mod 4 of A's group, that of accumulator register r.
    auto of_row = [&](int x, int r) { return __builtin_amdgcn_ds_bpermute(4 * (8 * (r >> 2) + 4 * h + (r & 3)), x); };
    {
        float* stage = smem + w * STAGE;
        std::conditional_t<AK, SideK<TM>, SideMN> a(p.A, p.lda, p.M, p.K, m0, lane, stage, 0);
        std::conditional_t<BK, SideK<TN>, SideMN> b(p.B, p.ldb, p.N, p.K, n0, lane, stage + a.LDS,
                                                        EP == ShortEpilogue::Geglu ? p.inter : 0);
        const int units = (p.K + UNIT - 1) / UNIT;
        const int ub = units * w / W, ue = units * (w + 1) / W;
        if (ub < ue) {
            a.issue(ub * UNIT);
            b.issue(ub * UNIT);
        }
        for (int u = ub; u < ue; ++u) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if constexpr (!AK || !BK) {
                if ((u + 1) * UNIT > p.K) {
                    if constexpr (!AK) a.zero_tail(u * UNIT);
                    if constexpr (!BK) b.zero_tail(u * UNIT);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
            }
            // One operand after the other: both at once in fp32 would not fit the registers.
            Frag<NP> fa[I][2], fb[J][2];
            int na = ea, nb = eb;
            {
                float v[I][2][8];
                a.fetch(v, lr, h);
                if constexpr (LINES) {
                    int d[I];
                    if (line_scale_exps(v, la, d) && u > ub) {
#pragma unroll
                        for (int i = 0; i < I; ++i)
#pragma unroll
                            for (int r = 0; r < 16; ++r) {
                                const int dr = of_row(d[i], r);
#pragma unroll
                                for (int j = 0; j < J; ++j) rescale(i, j, r, dr);
                            }
                    }
                } else if constexpr (NP == 2) {
                    na = min(ea, wave_scale_exp(v));
                }
#pragma unroll
                for (int i = 0; i < I; ++i)
#pragma unroll
                    for (int s = 0; s < 2; ++s) fa[i][s].set(v[i][s], exp2_int(LINES ? la[i] : na));
            }
            __builtin_amdgcn_sched_barrier(0);
            {
                float v[J][2][8];
                b.fetch(v, lr, h);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this stage is read: the next may overwrite it
                if (u + 1 < ue) {
                    a.issue((u + 1) * UNIT);
                    b.issue((u + 1) * UNIT);
                }
                if constexpr (LINES) {
                    int d[J];
                    if (line_scale_exps(v, lb, d) && u > ub) {
#pragma unroll
                        for (int j = 0; j < J; ++j)
#pragma unroll
                            for (int i = 0; i < I; ++i)
#pragma unroll
                                for (int r = 0; r < 16; ++r) rescale(i, j, r, d[j]);
                    }
                } else if constexpr (NP == 2) {
                    nb = min(eb, wave_scale_exp(v));
                }
#pragma unroll
                for (int j = 0; j < J; ++j)
#pragma unroll
                    for (int s = 0; s < 2; ++s) fb[j][s].set(v[j][s], exp2_int(LINES ? lb[j] : nb));
            }
            if constexpr (NP == 2 && !LINES) {
                const int d = na + nb - ea - eb;
                if (d < 0 && u > ub)
                    each([&](f32x16& a, f32x16& t) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            a[e] = __builtin_amdgcn_ldexpf(a[e], d);
                            t[e] = __builtin_amdgcn_ldexpf(t[e], d);
                        }
                    });
                ea = na;
                eb = nb;
            }
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int j = 0; j < J; ++j)
#pragma unroll
                    for (int s = 0; s < 2; ++s) fa[i][s].mma(fb[j][s], acc[i][j]);
            if ((u - ub) % CHAIN == CHAIN - 1)
                each([](f32x16& a, f32x16& t) {
                    t += a;
                    a = f32x16{};
                });
        }
        each([](f32x16& a, f32x16& t) { a += t; });
    }

    // The waves' sums: [wave][TM][TN] in LDS (over the stages, which every wave has finished reading).
    __syncthreads();
    {
        float* red = smem + w * TM * TN;
        const int ex = -(ea + eb);
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int q = 8 * (r >> 2) + 4 * h + (r & 3), row = AK ? 32 * i + q : I * q + i;
                const int er = LINES ? of_row(la[i], r) : 0;
                float v[J];
#pragma unroll
                for (int j = 0; j < J; ++j)
                    v[j] = NP == 2 ? __builtin_amdgcn_ldexpf(acc[i][j][r], LINES ? -(er + lb[j]) : ex) : acc[i][j][r];
                if constexpr (BK) {
#pragma unroll
                    for (int j = 0; j < J; ++j) red[row * TN + 32 * j + lr] = v[j];
                } else {
#pragma unroll
                    for (int j = 0; j < J; ++j) red[row * TN + J * lr + j] = v[j];
                }
            }
    }
    __syncthreads();
    auto total = [&](int row, int col) {
        f32x4 s = *reinterpret_cast<const f32x4*>(smem + row * TN + col);
#pragma unroll
        for (int v = 1; v < W; ++v) s += *reinterpret_cast<const f32x4*>(smem + (v * TM + row) * TN + col);
        return s;
    };
    auto four = [](const float* x) { return *reinterpret_cast<const f32x4*>(x); };
    unsigned am = 0;
    if constexpr (EP == ShortEpilogue::Store || EP == ShortEpilogue::Accumulate) {
        constexpr int QUADS = TM * TN / 4;
#pragma unroll
        for (int o = 0; o < QUADS; o += THREADS) {
            const int q = o + tid, row = q / (TN / 4), col = q % (TN / 4) * 4, m = m0 + row, n = n0 + col;
            if ((QUADS % THREADS && q >= QUADS) || m >= p.M || n >= p.N) continue;
            float* c = p.C + (long)m * p.ldc + n;
            f32x4 v = total(row, col);
            if constexpr (EP == ShortEpilogue::Store) {
                if (p.bias)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += p.bias[n + e];
                if (p.R) v += four(p.R + (long)m * p.ldr + n);
            } else {
                v = four(c) + v;
            }
            *reinterpret_cast<f32x4*>(c) = v;
            am = max(am, amax_bits4(v));
        }
    } else {
        // Columns c and c + 32 of a row together: a rotation pair, or GeGLU's two halves.
        static_assert(TN == 64, "pairs lie 32 columns apart");
#pragma unroll
        for (int o = 0; o < TM * 8; o += THREADS) {
            const int q = o + tid, row = q / 8, col = q % 8 * 4, m = m0 + row;
            if ((TM * 8 % THREADS && q >= TM * 8) || m >= p.M) continue;
            f32x4 a = total(row, col), b = total(row, col + 32);
            const int na = n0 + col, nb = EP == ShortEpilogue::Geglu ? p.inter + na : na + 32;
            if (na >= (EP == ShortEpilogue::Geglu ? p.inter : p.N)) continue;
            if (p.bias) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[e] += p.bias[na + e];
                    b[e] += p.bias[nb + e];
                }
            }
            if constexpr (EP == ShortEpilogue::Rope) {
                if (n0 < p.rope_cols) {
                    const long at = (long)p.rope_pos[m] * 32 + col;
                    f32x4 v0, v1;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float cs = p.rope_cos[at + e], sn = p.rope_sin[at + e];
                        v0[e] = a[e] * cs - b[e] * sn;
                        v1[e] = b[e] * cs + a[e] * sn;
                    }
                    a = v0;
                    b = v1;
                }
                am = max(am, max(amax_bits4(a), amax_bits4(b)));
            } else {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gelu_f(a[e]) * b[e];
                *reinterpret_cast<f32x4*>(p.act + (long)m * p.inter + na) = v;
                if (p.act16)
                    *reinterpret_cast<bf16x4*>(p.act16 + (long)m * p.inter + na) = __builtin_convertvector(v, bf16x4);
                am = max(am, amax_bits4(v));
            }
            *reinterpret_cast<f32x4*>(p.C + (long)m * p.ldc + na) = a;
            *reinterpret_cast<f32x4*>(p.C + (long)m * p.ldc + nb) = b;
        }
    }
    block_amax_fold(am, p.amax);
}

// Workgroups are dealt round-robin to the 8 XCDs: of n consecutive ones, those on one XCD get a contiguous run of tiles.
__device__ __forceinline__ int xcd_tile(int block, int n) {
    const int xcd = block & 7, local = block >> 3, per = n >> 3, rem = n & 7;
    return (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + local;
}

template <bool AK, bool BK, int TM, int TN, ShortEpilogue EP, int W, int NP>
__global__ __launch_bounds__(64 * W, 2) void short_gemm_kernel(ShortGemm p) {
    __shared__ __attribute__((aligned(16))) float smem[W * wave_floats<TM, TN>()];
    short_tile<AK, BK, TM, TN, EP, W, NP>(p, xcd_tile(blockIdx.x, gridDim.x), smem);
}

// dX's tiles, then dW's, each over all XCDs: neither product reads what the other writes. LINES costs 6 to 12 % (512 x
// 768 -> 2304 27 us and 31; 256 registers and ten spilled to the rescaling) and is for pairs that would run as exact
// three-piece splits otherwise: 1618 x 2624 -> 1024 139 us there, 100 here, the worst row or column of dX and dW off by
// 1.6e-7 where rows or columns lie 2^-26 below the others, and by 4e-7 there.
template <int W, int NP, bool LINES>
__global__ __launch_bounds__(64 * W, 2) void short_pair_kernel(ShortGemm nn, ShortGemm tn, int dx_tiles) {
    __shared__ __attribute__((aligned(16))) float smem[W * 64 * 64];
    const int block = blockIdx.x;
    if (block < dx_tiles)
        short_tile<true, false, 64, 64, ShortEpilogue::Store, W, NP, LINES>(nn, xcd_tile(block, dx_tiles), smem);
    else
        short_tile<false, false, 64, 64, ShortEpilogue::Accumulate, W, NP, LINES>(
            tn, xcd_tile(block - dx_tiles, gridDim.x - dx_tiles), smem);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int layout_class(GemmLayout l) { return l == GemmLayout::NT ? 1 : l == GemmLayout::NN ? 2 : 4; }

long tiles_of(const ShortGemm& g, ShortEpilogue ep, int tm, int tn) {
    const long n = ep == ShortEpilogue::Geglu ? (g.inter + tn / 2 - 1) / (tn / 2) : (g.N + tn - 1) / tn;
    return (long)((g.M + tm - 1) / tm) * n;
}

void set_tiles(ShortGemm& g, ShortEpilogue ep, int tm, int tn) {
    g.tiles_m = (g.M + tm - 1) / tm;
    g.tiles_n = (int)(tiles_of(g, ep, tm, tn) / g.tiles_m);
}

bool short_gemm_fits(const ShortGemm& g, GemmLayout layout, ShortEpilogue ep) {
    const bool ak = layout != GemmLayout::TN, bk = layout == GemmLayout::NT;
    auto operand = [&](const float* x, long ld, int mn, bool kcontig) {
        const long lines = kcontig ? mn : g.K, width = kcontig ? g.K : mn;
        return x && aligned16(x) && ld % 4 == 0 && width % 4 == 0 && width >= 4 && ld >= width && lines >= 1 &&
               ((lines - 1 + UNIT) * ld + width) * 4 < (1L << 31);
    };
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || (ak && g.K % UNIT)) return false;
    if (!operand(g.A, g.lda, g.M, ak) || !operand(g.B, g.ldb, g.N, bk)) return false;
    if (g.N % 4 || g.ldc % 4 || !aligned16(g.C) || (g.R && (g.ldr % 4 || !aligned16(g.R)))) return false;
    if (ep == ShortEpilogue::Rope && (g.N % 64 || g.rope_cols % 64)) return false;
    if (ep == ShortEpilogue::Geglu && (g.inter % 4 || !aligned16(g.act) || (g.act16 && !aligned16(g.act16)))) return false;
    return true;
}

// Up to how many multiply-adds a product may run here: the range over which the times below were fitted.
constexpr double FORWARD_LIMIT = 4.0e9, FORWARD_LIMIT_BF16 = 2.0e9, PAIR_LIMIT = 5.0e9, PAIR_LIMIT_BF16 = 3.0e9, PAIR_LIMIT_LINES = 9.0e9;

double work_of(const ShortGemm& g) { return (double)g.M * g.N * g.K; }

bool is_bf16(const laya_ctx* ctx, GemmLayout layout) { return ctx->matmul_bf16 & layout_class(layout); }

// A product's tiles and how many waves share one.
struct Shape {
    int tm, tn, waves;
    long tiles;
};

// Smaller tiles while they would leave nearly half the CUs without one (404 x 3072 -> 768: 84 tiles of 64 x 64
// 27.6 us, 156 of 32 x 64 21.0, 312 of 32 x 32 25.9; 800 x 768 -> 768, 156 tiles: 11.6, 14.1 with 32 x 64). Past a
// tile per CU workgroups of four waves, two to a CU, hide each other's first loads and epilogues (1618 x 768 -> 2304
// 47.8 us with eight waves, 36.9 with four); under it eight waves shorten each one's K (3072 -> 768 27.6 and 34.8).
Shape shape_of(const laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, const ShortGemm& g) {
    const long few = ctx->cu_count * 9L / 16;
    Shape s{64, 64, 8, 0};
    if (layout == GemmLayout::NT) {
        if (tiles_of(g, ep, s.tm, s.tn) < few) s.tm = 32;
        if (ep == ShortEpilogue::Store && tiles_of(g, ep, s.tm, s.tn) < few) s.tn = 32;
    }
    s.tiles = tiles_of(g, ep, s.tm, s.tn);
    if (s.tm == 64 && s.tiles > ctx->cu_count) s.waves = 4;
    return s;
}

long ceil_div(long a, long b) { return (a + b - 1) / b; }

// The stages a wave goes through, one after the other.
long chain_of(const ShortGemm& g, int waves) { return ceil_div(ceil_div(g.K, UNIT), waves); }

double megabytes(double floats) { return 4e-6 * floats; }

// Memory traffic in MB: A is read by each XCD that has columns of its rows, B once (rows fastest: a tile of B stays on
// one XCD).
double traffic_of(const ShortGemm& g, long tiles_n) {
    return megabytes((double)g.M * g.K * std::min(8L, tiles_n) + (double)g.N * g.K);
}

// Microseconds a product takes here: its rounds of workgroups, each a chain of stages and an epilogue, and its traffic
// from the memory-side cache. Work alone does not say it: dW of 768 x 64 over 65,536 rows is twelve workgroups of 256
// stages a wave, 460 us here and 130 with K split over the chip; 65536 x 64 -> 768 forward is 12,288 tiles of half a
// stage a wave, 109 us here and 65 on 256-wide tiles. Fitted to 500 shapes (widths 32 … 4096, 16 … 131,072 rows, back to
// back on one stream), where it is within 10 % for four in five. Over 3,400 other products, forward, dX, dW and pairs,
// choosing by it and by the other tiles' estimate costs, against always choosing the faster, 2.4 % in sum for the forward,
// 1.4 % for dX and under 1 % for dW and pairs where the operands' magnitudes are known, and 1.9, 1.8 and about 1 % where
// they are not.
double short_time(const laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, const ShortGemm& g) {
    const bool bf16 = is_bf16(ctx, layout), accumulate = ep == ShortEpilogue::Accumulate;
    const Shape s = shape_of(ctx, layout, ep, g);
    const long chain = chain_of(g, s.waves), cu = ctx->cu_count;
    const double out = megabytes((double)g.M * g.N);
    const double moved = (bf16 ? 0.08 : 0.07) * traffic_of(g, s.tiles / ceil_div(g.M, s.tm));
    if (s.waves == 4) {  // two workgroups share a CU; the last of an odd number has it to itself
        const long each = ceil_div(s.tiles, cu);
        return 2.7 + 0.15 * out + moved + (each / 2) * ((accumulate ? 2.5 : 0.8) + (bf16 ? 1.0 : 1.83) * chain) +
               (each % 2) * ((accumulate ? 1.8 : 1.3) + (bf16 ? 0.6 : 1.05) * chain);
    }
    if (s.tn == 32) return 4.0 + moved + (bf16 ? 0.25 : 0.74) * ceil_div(s.tiles, 2 * cu) * chain;
    if (s.tm == 32) return 3.6 + moved + (bf16 ? 0.8 : 1.3) * ceil_div(s.tiles, cu) * chain;
    return 4.2 + moved + (accumulate ? 0.15 * out : 0.0) + (bf16 ? 0.95 : 1.7) * ceil_div(s.tiles, cu) * chain;
}

// As for the forward; and eight waves where dX is few tiles of a long K, which last longest (512 x 768 -> 2304, 96
// tiles: 27 us with eight waves, 32 with four; 800 rows, 156 tiles: 41 and 36). Over 340 pairs of ordinary widths and 60 to
// 3,000 rows the rule is within 0.6 % in sum of always taking the faster; it is furthest off where dX has 16 to 48 tiles
// of a K under 2048 (60 x 1536 -> 1536: 17 us with eight waves, 21 with four).
// Pairs scaled by line have at least 400 tiles: the balanced plan whose place they take needs 100 of 128 x 128 for dX.
int pair_waves(const laya_ctx* ctx, const ShortGemm& nn, long dx_tiles, long dw_tiles, bool lines) {
    return lines || (dx_tiles + dw_tiles > ctx->cu_count && (dx_tiles >= 100 || nn.K < 2048)) ? 4 : 8;
}

// The same of a pair: dX's workgroups, then dW's, of which the last begin, where they come in more than one round, as the
// others are done.
double pair_time(const laya_ctx* ctx, const ShortGemm& nn, const ShortGemm& tn, bool lines) {
    const bool bf16 = (ctx->matmul_bf16 & 6) == 6;
    const long dx = tiles_of(nn, ShortEpilogue::Store, 64, 64), dw = tiles_of(tn, ShortEpilogue::Accumulate, 64, 64);
    const int waves = pair_waves(ctx, nn, dx, dw, lines);
    const long slots = (waves == 4 ? 2L : 1L) * ctx->cu_count;
    const double a = chain_of(nn, waves) + 1.0, b = chain_of(tn, waves) + 1.0;  // an epilogue is about a stage
    double span = std::max(a, b);
    if (dx + dw > slots) span = std::max(span, (dx * a + dw * b) / slots + b);
    const long tiles_n = ceil_div(nn.N, 64);
    const double moved = traffic_of(nn, tiles_n) + traffic_of(tn, tiles_n);
    const double out = megabytes((double)nn.M * nn.N + 2.0 * tn.M * tn.N);
    if (waves == 4) return 3.1 + (bf16 ? 0.68 : lines ? 1.35 : 1.25) * span + 0.075 * moved + 0.14 * out;
    return 3.4 + (bf16 ? 0.93 : 1.7) * span + 0.06 * moved + 0.07 * out;
}

// A product runs here where the estimates' ratio is below this. bf16: only where they differ by more than they scatter
// by. fp32: also where they are even, for its sums, K dealt to a workgroup's waves and each in two accumulators, are the
// more precise (a product of 45 us here and 48 there: 1.5e-7 and 2.7e-7 of fp64). Against 0.95 that costs up to 2 % of a
// step's products at 2,200 to 4,800 tokens, whose magnitudes are known, and gives 1 % where they are not.
double margin(bool bf16) { return bf16 ? 0.87 : 1.05; }

}  // namespace

bool short_gemm_pays(const laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, const ShortGemm& g, double other) {
    const int cls = layout_class(layout);
    const bool bf16 = is_bf16(ctx, layout);
    if (!bf16 && !((ctx->matmul_pair & cls) && (ctx->matmul_split & cls))) return false;
    return work_of(g) <= (bf16 ? FORWARD_LIMIT_BF16 : FORWARD_LIMIT) && short_gemm_fits(g, layout, ep) &&
           short_time(ctx, layout, ep, g) < margin(bf16) * other;
}

bool short_pair_pays(const laya_ctx* ctx, const ShortGemm& nn, const ShortGemm& tn, bool lines, double other) {
    const bool bf16 = (ctx->matmul_bf16 & 6) == 6;
    if (!bf16 && ((ctx->matmul_bf16 & 6) || (ctx->matmul_pair & 6) != 6 || (ctx->matmul_split & 6) != 6)) return false;
    return work_of(nn) <= (bf16 ? PAIR_LIMIT_BF16 : lines ? PAIR_LIMIT_LINES : PAIR_LIMIT) &&
           short_gemm_fits(nn, GemmLayout::NN, ShortEpilogue::Store) &&
           short_gemm_fits(tn, GemmLayout::TN, ShortEpilogue::Accumulate) &&
           pair_time(ctx, nn, tn, lines) < margin(bf16) * other;
}

#define SHORT_NP(W, ...)                                                                                   \
    do {                                                                                                   \
        if (bf16)                                                                                          \
            LAYA_LAUNCH((short_gemm_kernel<__VA_ARGS__, W, 1>), grid, dim3(64 * W), 0, ctx->stream, g);    \
        else                                                                                               \
            LAYA_LAUNCH((short_gemm_kernel<__VA_ARGS__, W, 2>), grid, dim3(64 * W), 0, ctx->stream, g);    \
    } while (0)

void short_gemm(laya_ctx* ctx, GemmLayout layout, ShortEpilogue ep, ShortGemm g) {
    constexpr auto ST = ShortEpilogue::Store, AC = ShortEpilogue::Accumulate, RO = ShortEpilogue::Rope,
                   GE = ShortEpilogue::Geglu;
    LAYA_REQUIRE(layout == GemmLayout::NT ? ep != AC : ep == (layout == GemmLayout::NN ? ST : AC),
                 "short_gemm: no such product");
    const bool bf16 = is_bf16(ctx, layout);
    static const char* names[3][2] = {{"gemm_nt_h2s", "gemm_nt_bf16s"},
                                      {"gemm_nn_h2s", "gemm_nn_bf16s"},
                                      {"gemm_tn_h2s", "gemm_tn_bf16s"}};
    const Shape s = shape_of(ctx, layout, ep, g);
    const int tm = s.tm, tn = s.tn;
    set_tiles(g, ep, tm, tn);
    const dim3 grid(g.tiles_m * g.tiles_n);
    const bool w4 = s.waves == 4;
    ProfileScope scope(ctx, names[(int)layout][bf16], 2.0 * g.M * g.N * (double)g.K, 0.0);
    if (layout == GemmLayout::NT) {
        if (ep == RO && w4) SHORT_NP(4, true, true, 64, 64, RO);
        else if (ep == RO && tm == 64) SHORT_NP(8, true, true, 64, 64, RO);
        else if (ep == RO) SHORT_NP(8, true, true, 32, 64, RO);
        else if (ep == GE && w4) SHORT_NP(4, true, true, 64, 64, GE);
        else if (ep == GE && tm == 64) SHORT_NP(8, true, true, 64, 64, GE);
        else if (ep == GE) SHORT_NP(8, true, true, 32, 64, GE);
        else if (w4) SHORT_NP(4, true, true, 64, 64, ST);
        else if (tm == 64) SHORT_NP(8, true, true, 64, 64, ST);
        else if (tn == 64) SHORT_NP(8, true, true, 32, 64, ST);
        else SHORT_NP(8, true, true, 32, 32, ST);
    } else if (layout == GemmLayout::NN) {
        if (w4) SHORT_NP(4, true, false, 64, 64, ST);
        else SHORT_NP(8, true, false, 64, 64, ST);
    } else {
        if (w4) SHORT_NP(4, false, false, 64, 64, AC);
        else SHORT_NP(8, false, false, 64, 64, AC);
    }
    check_launch("short_gemm_kernel");
}
#undef SHORT_NP

void short_gemm_pair(laya_ctx* ctx, ShortGemm nn, ShortGemm tn, bool lines) {
    const bool bf16 = (ctx->matmul_bf16 & 6) == 6;
    set_tiles(nn, ShortEpilogue::Store, 64, 64);
    set_tiles(tn, ShortEpilogue::Accumulate, 64, 64);
    const int dx_tiles = nn.tiles_m * nn.tiles_n;
    const dim3 grid(dx_tiles + tn.tiles_m * tn.tiles_n);
    const bool w4 = pair_waves(ctx, nn, dx_tiles, (long)grid.x - dx_tiles, lines) == 4;
    ProfileScope scope(ctx, bf16 ? "gemm_bwd_pair_bf16s" : "gemm_bwd_pair_h2s", 4.0 * nn.M * nn.N * (double)nn.K, 0.0);
#define SHORT_PAIR(...) \
    LAYA_LAUNCH((short_pair_kernel<__VA_ARGS__>), grid, dim3(w4 ? 256 : 512), 0, ctx->stream, nn, tn, dx_tiles)
    if (bf16 && w4) SHORT_PAIR(4, 1, false);
    else if (bf16) SHORT_PAIR(8, 1, false);
    else if (lines) SHORT_PAIR(4, 2, true);
    else if (w4) SHORT_PAIR(4, 2, false);
    else SHORT_PAIR(8, 2, false);
#undef SHORT_PAIR
    check_launch("short_pair_kernel");
}

}  // namespace laya
