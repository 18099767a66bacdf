// f32 activations at more than a few rows (block size >= 32, K % 4 == 0): the matrix cores with nothing rounded below f32.
//
// An f32 value is the exact sum of three bf16 values (its 24 significant bits cut in three runs of eight) down to 2^-110, and beside values of 2^-95 and more
// what is lost below that is none of an f32 sum's bits; rows of smaller values only are scaled up first (at the second walk below). q - zp, an
// integer of at most four bits and a sign, is a bf16 value as it stands. So
//   y += scale * (sum a1*(q-zp) + sum a2*(q-zp) + sum a3*(q-zp))
// over a run of 32 weights of one block, with products that are exact and sums in f32: the reference's fp32 route
// (matmul_nbits.rs:7499-7566), three MFMAs where the f32 form of the instruction would take sixteen times the cycles of one.
//
// A wave works alone on its share of K, the next loads in flight (one run ahead on 32 x 32 tiles, three on 16 x 16), and no barrier until the waves of a
// workgroup, which split K between them, add up their sums in wave order at the end. Short grids get their parallelism from that split.
// What bounds it is a CU's vector memory path, which serves a load one cache line at a time: on 32 x 32 tiles, operand lanes that load their own rows'
// activations ask for 32 lines with each of a run's four loads. So where K is a whole number of blocks (WHOLE) eight lanes load one row's 128
// bytes of a run, eight lines a load, and the wave turns them round through LDS of its own (no bank conflicts). The weights' loads (16 bytes of 32
// columns) are left as they are.
// Measured, block 32, f32 scales, lanes loading rows of their own before: as nodes of a recorded graph, 896 -> 4864 at 200 rows 24.4 -> 21.1 us,
// 4864 -> 896 at 200 rows 33.2 -> 22.6; a 0.5B layer's nodes called in a row at 100 / 200 / 512 rows 98 -> 80, 111 -> 90, 164 -> 136. (Offsets and nibbles worked
// out in a quarter fewer instructions gave 1 % of that; a third or fourth run in flight costs registers and 8 - 12 %.) The catch-all took 1665 and 2219 us for
// the first two. Over 140 shapes of whole blocks, 5 - 512 rows, the time is 0.84 of before in the mean (0.60 - 0.99). Where K ends inside a
// block the other build has the nibbles alone: 0.99 over 90 shapes (0.97 - 1.01).
#include <type_traits>

#include "prefill_common.hiph"

namespace mnb {

// Fourteen dwords of plain arguments, which are in scalar registers when a wave starts, and what is needed behind the loads.
struct GemmF32Rest {
    const void* bias;
    void* y;
    int scale_dtype, bias_dtype, y_dtype;
};
struct GemmF32Params {
    const float* a;
    const uint8_t* b;
    const void* scales;
    const uint8_t* zp;
    int m, n, k, kb;
    int bs_log2;
    int units_per_wave;     // runs of 32 k a wave walks
};
#define MNB_GEMM_F32_ARGS const float *a, const uint8_t *b, const void *scales, const uint8_t *zp, int m, int n, int k, int kb, int bs_log2, int units_per_wave, GemmF32Rest rest

// 8 * GROUPS f32 values as three bf16 operands each: plane[p][group], in plain_nibbles' order. What a cut leaves of an infinity is NaN; with WIDE it is 0.
template <int GROUPS, bool WIDE>
__device__ __forceinline__ void cut_in_three(const uint32_t (&v)[8 * GROUPS], uint4 (&plane)[3][GROUPS])
{
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
        uint32_t out[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t lo = v[8 * g + i], hi = v[8 * g + i + 4];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                out[p][i] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);      // the upper halves: both values cut to bf16
                if (p < 2) {                                                // what the cut leaves, exactly
                    const bool lo_inf = WIDE && (lo & 0x7fffffffu) == 0x7f800000u, hi_inf = WIDE && (hi & 0x7fffffffu) == 0x7f800000u;
                    lo = lo_inf ? 0u : __float_as_uint(__uint_as_float(lo) - __uint_as_float(lo & 0xffff0000u));
                    hi = hi_inf ? 0u : __float_as_uint(__uint_as_float(hi) - __uint_as_float(hi & 0xffff0000u));
                }
            }
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) plane[p][g] = make_uint4(out[p][0], out[p][1], out[p][2], out[p][3]);
    }
}

// The matrix-core step and the shape of its operands for tiles of 32 x 32 (16 k per MFMA, a run is two of them) and of
// 16 x 16 (32 k per MFMA: a run is one). An operand lane holds 8 k of one row or column per MFMA.
typedef __attribute__((ext_vector_type(4))) float f32x4_acc_t;
template <int TILE> struct TileOps;
template <> struct TileOps<32> {
    using acc_t = float16_t;
    static constexpr int kMfmas = 2, kAcc = 16;
    static __device__ __forceinline__ acc_t mfma(const uint4& a, const uint4& b, acc_t c) { return mfma32<true>(a, b, c); }
    static __device__ __forceinline__ int row_of(int e, int lane) { return (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3); }
};
template <> struct TileOps<16> {
    using acc_t = f32x4_acc_t;
    static constexpr int kMfmas = 1, kAcc = 4;
    static __device__ __forceinline__ acc_t mfma(const uint4& a, const uint4& b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0); }
    static __device__ __forceinline__ int row_of(int e, int lane) { return (lane >> 4) * 4 + e; }
};

// TILE: 16 or 32 rows and columns per matrix-core tile. CN: tiles along N per wave. DEPTH: runs in flight. WAVES: the most
// waves a workgroup is launched with. ST: float, or uint16_t for f16 / bf16 scales.
// WHOLE: K is a whole number of blocks, so that no run is cut short: activations go through LDS, and the offsets of a wave's loads do not change from
// run to run (the run goes into the scalar offset). The other build works out per run and load whether elements lie within K.
template <int TILE, int CN, int DEPTH, int WAVES, typename ST, bool WHOLE>
__global__ __launch_bounds__(WAVES * 64) void gemm_f32_kernel(MNB_GEMM_F32_ARGS)
{
    const GemmF32Params p{a, b, scales, zp, m, n, k, kb, bs_log2, units_per_wave};
    const int64_t row_bytes = (static_cast<int64_t>(kb) << bs_log2) / 2, zp_row = (kb + 1) / 2;
    using Ops = TileOps<TILE>;
    using acc_t = typename Ops::acc_t;
    constexpr int G = Ops::kMfmas;                         // groups of 8 k a lane holds of a run
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int waves = static_cast<int>(blockDim.x >> 6);
    const int r = lane & (TILE - 1), part = lane / TILE;   // operand row (A) or column (B), and which 8 G of a run's 32 k
    const int64_t m_base = static_cast<int64_t>(blockIdx.y) * TILE;
    const int64_t n_base = static_cast<int64_t>(blockIdx.x) * (TILE * CN);
    const int64_t rows_left = p.m - m_base, cols_left = p.n - n_base;

    const __amdgpu_buffer_rsrc_t srd_a = make_srd(p.a + m_base * p.k, static_cast<uint64_t>(rows_left * p.k) * 4);
    const __amdgpu_buffer_rsrc_t srd_b = make_srd(p.b + n_base * row_bytes, static_cast<uint64_t>(cols_left * row_bytes));
    const __amdgpu_buffer_rsrc_t srd_s = make_srd(static_cast<const ST*>(p.scales) + n_base * p.kb, static_cast<uint64_t>(cols_left * p.kb) * sizeof(ST));
    const __amdgpu_buffer_rsrc_t srd_z = make_srd(p.zp ? p.zp + n_base * zp_row : nullptr, p.zp ? static_cast<uint64_t>(cols_left * zp_row) : 0);
    const uint32_t zp_mask = p.zp ? 0xfu : 0u, zp_default = p.zp ? 0u : 8u;
    const bool scale_bf16 = rest.scale_dtype == ROCM_DT_BF16;
    const uint32_t mask = __builtin_amdgcn_mov_dpp(opaque_scalar(0x000F000Fu), 0xE4, 0xf, 0xf, false), magic = opaque_scalar(0x64006400u);

    const uint32_t a_off = static_cast<uint32_t>(r) * static_cast<uint32_t>(p.k) * 4u;
    const bool row_live = r < rows_left;
    // WHOLE: eight lanes load one row's 128 bytes of a run; lane -> (row lane / 8 + 8 i, piece lane % 8). Rows beyond M lie out of range by themselves.
    // The 16-byte piece c of row x lies at c ^ (x / 2 % 8) in the wave's 128-byte rows of LDS: writes, and reads by rows, cover all banks.
    unsigned char* const a_stage = smem + wave * (TILE * 128);
    uint32_t a_piece[2 * G], a_write[2 * G];
#pragma unroll
    for (int i = 0; i < 2 * G; ++i) {
        const uint32_t x = static_cast<uint32_t>(8 * i + (lane >> 3)), c = static_cast<uint32_t>(lane & 7);
        a_piece[i] = x * static_cast<uint32_t>(p.k) * 4u + c * 16u;
        a_write[i] = x * 128u + ((c ^ ((x >> 1) & 7u)) * 16u);
    }
    const uint32_t a_read = static_cast<uint32_t>(r) * 128u + ((static_cast<uint32_t>(part * 2 * G) ^ ((static_cast<uint32_t>(r) >> 1) & 7u)) * 16u);
    uint32_t b_off[CN], s_off[CN], z_off[CN];
#pragma unroll
    for (int j = 0; j < CN; ++j) {                         // a column beyond N lies out of range by itself
        b_off[j] = static_cast<uint32_t>(j * TILE + r) * static_cast<uint32_t>(row_bytes) + static_cast<uint32_t>(part * 4 * G);
        s_off[j] = static_cast<uint32_t>(j * TILE + r) * static_cast<uint32_t>(p.kb) * static_cast<uint32_t>(sizeof(ST));
        z_off[j] = static_cast<uint32_t>(j * TILE + r) * static_cast<uint32_t>(zp_row);
    }

    struct Run {
        u32x4_t a[2 * G];
        uint32_t b[CN][G];
        typename ScaleIo<ST>::raw_t s[CN];
        uint32_t z[CN];
        uint32_t zsh;
    };
    const int u0 = wave * p.units_per_wave;
    const int u1 = min(u0 + p.units_per_wave, static_cast<int>((p.kb << p.bs_log2) >> 5));
    // No branch: a run past the wave's share, a row beyond M and elements beyond K get offsets out of range, which read zeros.
    auto request = [&](Run& x, int u) {
        const bool live = u < u1;
        if constexpr (WHOLE) {
            // (A run past the wave's share: its last one again, with scales of zero. Offsets out of range for all its loads, as below, take 2 - 5 % off 16 x 16
            // tiles (3584 -> 3584 at 16 rows 13.9 and 13.4 us) and add up to 3 % to 32 x 32 ones (4864 -> 896, block 128, 200 rows 20.3 and 20.8).)
            const int at = min(u, u1 - 1);
            const uint32_t blk = static_cast<uint32_t>(at * 32) >> p.bs_log2, oor = live ? 0u : kOutOfRange;
#pragma unroll
            for (int i = 0; i < 2 * G; ++i) x.a[i] = __builtin_amdgcn_raw_buffer_load_b128(srd_a, static_cast<int>(a_piece[i]), at * 128, 0);
#pragma unroll
            for (int j = 0; j < CN; ++j) {
                if constexpr (G == 2) {
                    const auto w = __builtin_amdgcn_raw_buffer_load_b64(srd_b, static_cast<int>(b_off[j]), at * 16, 0);
                    x.b[j][0] = w[0];
                    x.b[j][1] = w[1];
                } else {
                    x.b[j][0] = __builtin_amdgcn_raw_buffer_load_b32(srd_b, static_cast<int>(b_off[j]), at * 16, 0);
                }
                x.s[j] = ScaleIo<ST>::load_raw(srd_s, s_off[j] | oor, blk * static_cast<uint32_t>(sizeof(ST)));
                x.z[j] = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b8(srd_z, static_cast<int>(z_off[j]), static_cast<int>(blk >> 1), 0));
            }
            x.zsh = (blk & 1u) * 4u;
            return;
        }
        const int k0 = u * 32 + part * 8 * G;
#pragma unroll
        for (int i = 0; i < 2 * G; ++i) {
            const uint32_t off = live && row_live && k0 + i * 4 < p.k ? a_off + static_cast<uint32_t>(k0 + i * 4) * 4u : kOutOfRange;
            x.a[i] = __builtin_amdgcn_raw_buffer_load_b128(srd_a, static_cast<int>(off), 0, 0);
        }
        const uint32_t oor = live ? 0u : kOutOfRange;
        const uint32_t blk = static_cast<uint32_t>(u * 32) >> p.bs_log2;
#pragma unroll
        for (int j = 0; j < CN; ++j) {
            const int off = static_cast<int>((b_off[j] + static_cast<uint32_t>(u) * 16u) | oor);
            if constexpr (G == 2) {
                const auto w = __builtin_amdgcn_raw_buffer_load_b64(srd_b, off, 0, 0);
                x.b[j][0] = w[0];
                x.b[j][1] = w[1];
            } else {
                x.b[j][0] = __builtin_amdgcn_raw_buffer_load_b32(srd_b, off, 0, 0);
            }
            x.s[j] = ScaleIo<ST>::load_raw(srd_s, (s_off[j] + blk * static_cast<uint32_t>(sizeof(ST))) | oor, 0);
            x.z[j] = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b8(srd_z, static_cast<int>((z_off[j] + (blk >> 1)) | oor), 0, 0));
        }
        x.zsh = (blk & 1u) * 4u;
    };

    acc_t sum[CN], zero;
#pragma unroll
    for (int e = 0; e < Ops::kAcc; ++e) {
        zero[e] = 0.f;
#pragma unroll
        for (int j = 0; j < CN; ++j) sum[j][e] = 0.f;
    }

    uint32_t seen = 0;                                     // the bits of all this lane's activations or-ed together
    float scale_up = 1.f, scale_down[Ops::kAcc];           // of the second walk: this lane's operand row, its accumulators' rows
    auto multiply = [&](const Run& x, auto wide) {
        constexpr bool kWide = decltype(wide)::value;
        u32x4_t a[2 * G];
        if constexpr (WHOLE) {
#pragma unroll
            for (int i = 0; i < 2 * G; ++i) *reinterpret_cast<u32x4_t*>(a_stage + a_write[i]) = x.a[i];
            lds_order();
#pragma unroll
            for (int i = 0; i < 2 * G; ++i) a[i] = *reinterpret_cast<const u32x4_t*>(a_stage + (a_read ^ static_cast<uint32_t>(i * 16)));
            lds_order();
        } else {
#pragma unroll
            for (int i = 0; i < 2 * G; ++i) a[i] = x.a[i];
        }
        uint32_t v[8 * G];
#pragma unroll
        for (int i = 0; i < 2 * G; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[4 * i + e] = kWide ? __float_as_uint(__uint_as_float(a[i][e]) * scale_up) : a[i][e];
                if (!kWide) seen |= a[i][e];
            }
        uint4 plane[3][G];
        cut_in_three<G, kWide>(v, plane);
#pragma unroll
        for (int j = 0; j < CN; ++j) {
            const uint32_t zq = ((x.z[j] >> x.zsh) & zp_mask) | zp_default;
            uint4 w[G];
#pragma unroll
            for (int g = 0; g < G; ++g) w[g] = plain_nibbles<true>(x.b[j][g], zq, mask, magic);
            acc_t acc = zero;
#pragma unroll
            for (int q = 2; q >= 0; --q)                                      // smallest parts first
#pragma unroll
                for (int g = 0; g < G; ++g) acc = Ops::mfma(plane[q][g], w[g], acc);
            const float sc = ScaleIo<ST>::to_f32(x.s[j], scale_bf16);         // 0 for a column beyond N and past the end
#pragma unroll
            for (int e = 0; e < Ops::kAcc; ++e) sum[j][e] = fmaf(acc[e], kWide ? sc * scale_down[e] : sc, sum[j][e]);
        }
    };

    Run x[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) request(x[d], u0 + d);
    asm volatile("" : : "s"(rest.bias), "s"(rest.y), "s"(rest.bias_dtype), "s"(rest.y_dtype));      // there from here on, not read behind the last barrier
    for (int u = u0; u < u1; u += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            request(x[(d + DEPTH - 1) % DEPTH], u + d + DEPTH - 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(x[d], std::false_type{});
        }
    }

    // A sum that is not finite: an activation was infinite (NaN came of it above), or so large that the unscaled sum of a run overflowed,
    // or the result is what it is. Or a row whose values in the wave's share, not all of them zero, are all below 2^-95 (the or-ed exponents tell): their parts fall
    // under bf16's smallest value. The wave then walks its share once more with infinities kept whole in their first part and each row scaled
    // for itself: one with a value of 2 or more by 2^-16, so that a run's 32 products of up to 15 fit, one of tiny values by 2^64. Asked
    // once per wave, not per run; or-ing the values costs one instruction for two of them.
#pragma unroll
    for (int off = TILE; off < 64; off <<= 1) seen |= __shfl_xor(seen, off, 64);
    const bool tiny = (seen & 0x7fffffffu) != 0 && (seen & 0x70000000u) == 0;
    bool finite = true;
#pragma unroll
    for (int j = 0; j < CN; ++j)
#pragma unroll
        for (int e = 0; e < Ops::kAcc; ++e) finite = finite && __builtin_isfinite(sum[j][e]);
    if (__builtin_expect(__any(!finite || tiny), 0)) {
        scale_up = tiny ? 0x1p64f : (seen & 0x40000000u) != 0 ? 0x1p-16f : 1.f;
        const float inverse = tiny ? 0x1p-64f : (seen & 0x40000000u) != 0 ? 0x1p16f : 1.f;
#pragma unroll
        for (int e = 0; e < Ops::kAcc; ++e) scale_down[e] = __shfl(inverse, Ops::row_of(e, lane), 64);
#pragma unroll
        for (int j = 0; j < CN; ++j) sum[j] = zero;
#pragma unroll 1
        for (int u = u0; u < u1; ++u) {
            request(x[0], u);
            multiply(x[0], std::true_type{});
        }
    }

    // ---- the waves' sums through LDS, added in wave order: [wave][tile][accumulator][64] ----
    constexpr int kOuts = CN * Ops::kAcc * 64;
    float* parts = reinterpret_cast<float*>(smem);
    if constexpr (WHOLE) __syncthreads();                  // (the waves' activations lay there)
#pragma unroll
    for (int j = 0; j < CN; ++j)
#pragma unroll
        for (int e = 0; e < Ops::kAcc; ++e) parts[((wave * CN + j) * Ops::kAcc + e) * 64 + lane] = sum[j][e];
    __syncthreads();
    for (int i = t; i < kOuts; i += waves * 64) {
        float v = 0.f;
        for (int w = 0; w < waves; ++w) v += parts[w * kOuts + i];
        const int l = i & 63;
        const int64_t row = m_base + Ops::row_of((i >> 6) & (Ops::kAcc - 1), l);
        const int64_t col = n_base + (i / (Ops::kAcc * 64)) * TILE + (l & (TILE - 1));
        if (row < p.m && col < p.n) store_from_f32(rest.y, rest.y_dtype, row * p.n + col, with_bias(v, rest.bias, rest.bias_dtype, row, p.n, col, rest.y_dtype));
    }
}

template <int TILE, int CN, int DEPTH, int WAVES, typename ST, bool WHOLE>
static int launch_gemm_f32(const GemmF32Params& p, const GemmF32Rest& rest, int waves, hipStream_t stream)
{
    const dim3 grid(static_cast<unsigned>((static_cast<int64_t>(p.n) + TILE * CN - 1) / (TILE * CN)), static_cast<unsigned>((p.m + TILE - 1) / TILE));
    constexpr int kWaveLds = CN * TileOps<TILE>::kAcc * 256, kStageLds = WHOLE ? TILE * 128 : 0;
    const size_t lds = static_cast<size_t>(waves) * (kWaveLds > kStageLds ? kWaveLds : kStageLds);        // at most 64 KiB
    hipLaunchKernelGGL((gemm_f32_kernel<TILE, CN, DEPTH, WAVES, ST, WHOLE>), grid, dim3(static_cast<unsigned>(waves * 64)), lds, stream, p.a, p.b, p.scales, p.zp, p.m, p.n, p.k, p.kb, p.bs_log2, p.units_per_wave, rest);
    return static_cast<int>(hipGetLastError());
}

}  // namespace mnb

extern "C" int rocm_gemm_f32_eligible(const RocmMatMulNBitsArgs* a)
{
    if (a->a_dtype != ROCM_DT_F32 || a->m < 1 || a->n < 1 || a->k < 1 || a->block_size < 32 || a->k % 4 != 0) return 0;
    const int64_t kb = (a->k + a->block_size - 1) / a->block_size;
    if (kb * a->block_size / 2 * 64 >= 0x7ffffff0 || a->k * 4 * 32 >= 0x7ffffff0 || (a->m + 31) / 32 > 65535 || a->n > 0x7fffffff) return 0;    // 32-bit offsets inside one tile, 32-bit sizes
    return (reinterpret_cast<uintptr_t>(a->a) & 15) == 0 && (reinterpret_cast<uintptr_t>(a->b) & 7) == 0;
}

namespace {

// Tiles, and waves that share K, by the grid they make (f32 scales, block 32; us, nodes of a recorded graph):
//   * 16 x 16 tiles while they make at most one workgroup per CU: 896 -> 896 at 64 rows 6.3 against 7.0 with 32 x 32, 4864 -> 896
//     at 64 rows 17.4 against 19.3; with more of them they lose (896 -> 896 at 200 rows 12.1 against 7.3).
//   * 32 x 32 otherwise, two of them per wave once single ones make more than one workgroup per CU: the cut activations are used
//     twice (4864 -> 896 at 512 rows 39.5 against 44.3; at 200 rows, 196 workgroups, 35.3 against 23.4).
//   * eight waves share K up to one workgroup per CU, four beyond (896 -> 9728 at 512 rows 62.5 against 80.5 us), each with two runs or more.
//   * between two and three single tiles per CU (five where K is at most 1536): single tiles of eight waves, of which a CU holds two workgroups at a time, where
//     the last of the few rounds of double ones would be half empty (single / double, us: 896 -> 4864 at 100 / 200 / 256 rows, 2.4 / 4.2 / 4.8 a CU, 12.6 / 18.7 / 19.3
//     against 15.1 / 20.4 / 21.8; 3584 -> 3584 at 150, 2.2, 37.3 against 42.4; 8960 -> 1536 at 400, 2.4, 98.8 against 109.0). Beyond they lose: 3584 -> 3584 at 200 rows,
//     3.1, 48.9 against 44.5; 1536 -> 8960 at 150, 5.5, 34.2 against 31.5; 896 -> 4864 at 512, 9.5, 34.6 against 33.3.
struct F32Plan { int tile, cn, waves; };
F32Plan plan_gemm_f32(const RocmMatMulNBitsArgs* a, int units, int64_t cus)
{
    auto workgroups = [&](int rows, int cols) { return ((a->m + rows - 1) / rows) * ((a->n + cols - 1) / cols); };
    F32Plan plan{32, 1, 8};
    if (workgroups(16, 16) <= cus) plan.tile = 16;
    else if (workgroups(32, 32) > cus) plan.cn = 2;
    const int64_t single = workgroups(32, 32);
    if (single > 2 * cus && single <= (a->k <= 1536 ? 5 : 3) * cus) plan.cn = 1;
    else if (workgroups(plan.tile, plan.tile * plan.cn) > cus) plan.waves = 4;
    while (plan.waves > 1 && units < 2 * plan.waves) plan.waves >>= 1;
    return plan;
}

}  // namespace

// From five rows; up to eight rows only on grids of at most two workgroups per CU (896 -> 9728 at five rows: 9.1 against 12.9 us in two passes of the
// streaming kernel). Beyond that, five rows of a long K are the streaming kernel's (3584 -> 18944 43.6 against 45.3 us). Six to eight are not since activations go
// through LDS (eight rows 56 against 44), nor is a K of 896 (-> 151936 at five rows 95 against 53): the line is older.
extern "C" int rocm_gemm_f32_pays(const RocmMatMulNBitsArgs* a)
{
    return a->m > 8 || (a->m > 4 && (a->n + 31) / 32 <= 2 * static_cast<int64_t>(rocm_ffi_compute_units()));
}

extern "C" int rocm_launch_gemm_f32(const RocmMatMulNBitsArgs* a, rocm_stream_t stream)
{
    if (!rocm_gemm_f32_eligible(a)) return -1;
    mnb::GemmF32Params p;
    p.a = static_cast<const float*>(a->a);
    p.b = a->b;
    p.scales = a->scales;
    p.zp = a->zp;
    p.m = static_cast<int>(a->m);
    p.n = static_cast<int>(a->n);
    p.k = static_cast<int>(a->k);
    p.kb = static_cast<int>((a->k + a->block_size - 1) / a->block_size);
    p.bs_log2 = __builtin_ctz(static_cast<unsigned>(a->block_size));
    const mnb::GemmF32Rest rest{a->bias, a->y, a->scale_dtype, a->bias_dtype, a->y_dtype};
    const int64_t cus = rocm_ffi_compute_units();
    const int units = static_cast<int>(static_cast<int64_t>(p.kb) * a->block_size / 32);
    const F32Plan plan = plan_gemm_f32(a, units, cus);
    const int tile = plan.tile, cn = plan.cn, waves = plan.waves;
    p.units_per_wave = (units + waves - 1) / waves;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto st, auto whole) {
        using ST = decltype(st);
        constexpr bool W = decltype(whole)::value;
        if (tile == 16) return mnb::launch_gemm_f32<16, 1, 4, 8, ST, W>(p, rest, waves, s);
        return cn == 2 ? mnb::launch_gemm_f32<32, 2, 2, 8, ST, W>(p, rest, waves, s) : mnb::launch_gemm_f32<32, 1, 2, 8, ST, W>(p, rest, waves, s);
    };
    if (a->k % a->block_size != 0) return a->scale_dtype == ROCM_DT_F32 ? go(float{}, std::false_type{}) : go(uint16_t{}, std::false_type{});
    return a->scale_dtype == ROCM_DT_F32 ? go(float{}, std::true_type{}) : go(uint16_t{}, std::true_type{});
}
