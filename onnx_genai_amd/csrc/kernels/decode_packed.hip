// Decode path of MatMulNBits over weights repacked for streaming (f16/bf16 activations; M <= 16 at every width, up to 64 rows when N is large).
//
// When B, scales and zero points are constant initializers, the kernel object repacks them once into
// the order in which the split-K MFMA kernel consumes them, so that every vector load of a wave is
// one contiguous kilobyte and everything a group of four 128-element tiles needs lies in one chunk:
//
//   chunk(column group cg of 16 columns, tile group tg of 4 tiles) =
//       4 x [lane 0..63] 16 bytes of weights      lane (c = lane % 16, g = lane / 16) of tile u at u*1024 + lane*16
//       16 x record(column c)                     scales of the group's blocks, then one zero-point byte per block
//
// Dword j of a lane's 16 bytes holds the eight weights k = tile*128 + j*32 + g*8 + e (e = 0..7) of column c:
// one MFMA therefore covers 32 consecutive k and never mixes two blocks, whatever the block size, and no
// cross-lane transpose is needed. Inside the dword, element e sits at bit 4*(e/2) + 16*(e%2), so that
// ((w >> 4i) & 0x000F000F) | magic is the pair (e = 2i, 2i+1) as two 16-bit floats - seven VALU
// instructions per eight weights. The arithmetic is that of the unpacked decode kernel: magic-number
// operands, a second MFMA with the constant -(magic + zp), one scale per block on the f32 accumulator.
//
// The copy costs one extra byte of device memory per byte of weights plus 2 to 6 % for the records; it is
// read instead of the caller's tensors, which are not touched again.
#include <type_traits>

#include "decode_packed.hiph"
#include "decode_plain.hiph"

namespace mnb {

struct PackParams {
    const uint8_t* b;
    const void* scales;
    const uint8_t* zp;
    uint8_t* out;
    int64_t n, kb, row_bytes, zp_row;
    int bs_log2, scale_bytes;
    int groups;             // tile groups per column group
    int chunk_bytes, record;
    int bits;               // 4 or 8
};

// 8-bit weights: a tile of 128 k becomes two tiles of the stream, the first with bytes 0..3 and the second with bytes 4..7 of each lane's eight
// weights. Their zero points fill the record's bytes, and both tiles' entries are alike.

// grid (tile group, column group), 256 threads: four dwords of weights per thread, then one record per thread < 16.
__global__ __launch_bounds__(256) void pack_decode_kernel(PackParams p)
{
    const int t = threadIdx.x;
    const int64_t tg = blockIdx.x, cg = blockIdx.y;
    uint8_t* chunk = p.out + (cg * p.groups + tg) * static_cast<int64_t>(p.chunk_bytes);
    const int64_t padded_k = p.kb << p.bs_log2;
    const uint32_t* b32 = reinterpret_cast<const uint32_t*>(p.b);
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int x = it * 256 + t;              // dword of the weight part: u*256 + lane*4 + j
        const int u = x >> 8, lane = (x >> 2) & 63, j = x & 3;
        const int64_t col = cg * 16 + (lane & 15);
        const int64_t tile = tg * kGroupTiles + u;
        const int64_t k = (p.bits == 8 ? tile >> 1 : tile) * 128 + j * 32 + (lane >> 4) * 8 + (p.bits == 8 ? (tile & 1) * 4 : 0);
        uint32_t out = 0;
        if (p.bits == 8 && col < p.n && k < padded_k) {
            out = b32[(col * p.row_bytes + k) >> 2];
        } else if (col < p.n && k < padded_k) {
            const uint32_t w = b32[(col * p.row_bytes + (k >> 1)) >> 2];   // eight weights, element e at bit 4e
            uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;    // even / odd elements, one per byte
            lo = (lo | (lo >> 4)) & 0x00ff00ffu;
            lo = (lo | (lo >> 8)) & 0x0000ffffu;                            // e0 | e2 << 4 | e4 << 8 | e6 << 12
            hi = (hi | (hi >> 4)) & 0x00ff00ffu;
            hi = (hi | (hi >> 8)) & 0x0000ffffu;
            out = lo | (hi << 16);
        }
        reinterpret_cast<uint32_t*>(chunk)[x] = out;
    }
    if (t < 16) {
        const int nb = (kGroupTiles * 128) >> p.bs_log2;
        uint8_t* rec = chunk + kChunkWeights + t * p.record;
        const int64_t col = cg * 16 + t;
        for (int i = 0; i < p.record; ++i) rec[i] = 0;
        for (int bi = 0; bi < nb; ++bi) {
            const int per_tile = nb / kGroupTiles;
            const int64_t tile = tg * kGroupTiles + bi / per_tile;
            const int64_t blk = p.bits == 8 ? (tile >> 1) * per_tile + bi % per_tile : tg * nb + bi;
            const bool live = col < p.n && blk < p.kb;
            if (p.scale_bytes == 4) {
                reinterpret_cast<uint32_t*>(rec)[bi] = live ? static_cast<const uint32_t*>(p.scales)[col * p.kb + blk] : 0u;
            } else {
                reinterpret_cast<uint16_t*>(rec)[bi] = live ? static_cast<const uint16_t*>(p.scales)[col * p.kb + blk] : static_cast<uint16_t>(0);
            }
            if (p.bits == 8) {
                rec[nb * p.scale_bytes + bi] = live && p.zp ? p.zp[col * p.zp_row + blk] : 128;
            } else {
                rec[nb * p.scale_bytes + bi] = static_cast<uint8_t>(live ? zero_point_of(p.zp ? p.zp + col * p.zp_row : nullptr, blk) : 8);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// accuracy_level = 4, up to 16 rows, over the same repacked stream: v_mfma_i32_16x16x32_i8.
// ---------------------------------------------------------------------------------------------
//
// `w & 0x0f0f0f0f` and `(w >> 4) & 0x0f0f0f0f` turn a repacked dword into the eight weights as unsigned bytes in the
// order e0,e4,e1,e5 | e2,e6,e3,e7; the activation codes are stored in that same order inside every run of 8, so an
// operand costs three instructions and no byte shuffles. Arithmetic as in the unpacked int8 kernel: exact integer
// block sums, zero point through the code sums, one f32 scale-and-add per block.

typedef __attribute__((ext_vector_type(4))) int int4p_t;

// Arguments that the kernel needs only behind its first loads.
struct Acc4PackedRest {
    const void* bias;
    void* y;
    int bias_dtype, y_dtype;
    int rounding;           // FUSE: 0 = ties to even, 1 = ties away from zero
    int scales_bf16;
    int32_t* acc_probe;     // PROBE builds: int32 [M, N, kb] block accumulators, as flushed
};
// (fourteen dwords of plain arguments in front, as in PackedParams)
struct Acc4PackedParams {
    const void* rows;       // [m, padded_k] codes, packed order; FUSE: the rows themselves, f16 or bf16 [m, k], which every wave quantizes for the groups it multiplies
    const float* pairs;     // one row: [kb, 2] = scale_a, f32(sum of codes); 2 .. 16 rows: [kb, 16, 2], the same pairs block-major; FUSE: not read
    const uint8_t* packed;
    int m, n, k, kb;
    int padded_k;
    int groups, groups_per_wave, waves;
    Acc4PackedRest rest;
};
#define MNB_ACC4_ARGS const void *rows, const float *pairs, const uint8_t *packed, int m, int n, int k, int kb, int padded_k, int groups, int groups_per_wave, int waves_, Acc4PackedRest rest
#define MNB_ACC4_PARAMS Acc4PackedParams{rows, pairs, packed, m, n, k, kb, padded_k, groups, groups_per_wave, waves_, rest}

constexpr int kCodePitchP = 144;   // bytes between the rows of one tile of codes in LDS: 128 + 16

template <int NR, int NA, int NX>
struct Acc4PackedGroup {
    uint4 w[kGroupTiles];
    uint4 r[NR];
    uint4 a[NA];  // one row: 16 codes of the group (lanes 0..31). 16 rows: per tile, row lane / 8 (+ 8), piece lane % 8
    uint4 x[NX];  // one row: .x/.y = (scale_a, code sum) of block `lane` of the group. 16 rows: 16 bytes of the group's aux16 rows
};

// FUSE: 0 = codes and (scale, sum) pairs come from the workspace a quantizer kernel filled; 1 / 2 = the row arrives as
// f16 / bf16 and each wave quantizes the 512 activations of a group itself, with the arithmetic of quantize_a_kernel
// (one correctly rounded divide each for scale and inverse, one multiply and one rounding per element) - a lane holds
// 8 consecutive activations, a block is BS / 8 consecutive lanes. That is redundant across workgroups but saves the
// separate launch, which at one row costs about as much as a fifth of this kernel.
// PROBE: every flushed block accumulator (the integer acc - zp * code_sum that is about to be scaled) is also stored to
// p.acc_probe; the same code otherwise, for tests that compare the integers themselves.
// MR: rows staged, 1, 4, 8 or 16 (M <= MR). Beyond one row the codes come from the workspace (FUSE = 0): per tile a wave
// loads the rows' 128 codes, stages them in LDS at a padded pitch and reads MFMA operand j of row lane % 16 from there;
// the activation-side (scale, sum) pairs of the group's blocks are staged once per group and read when a block ends.
// With 4 (8), call row r sits in matrix row 4 r (2 r) and the rows between stay zero, so that a lane finds its rows in
// component 0 (0 and 2) of its accumulator and a block's end scales one (two) values per lane instead of four.
// ST: float, uint16_t, or Bf16Scale for the several-row builds when the 16-bit scales are bf16 - there the scale type is
// known at compile time (a run-time choice between the two conversions made the compiler prepare both for all of a
// group's blocks up front: 220 registers instead of 94 at block size 32 and 16 rows, two waves per SIMD instead of five).
struct Bf16Scale {
    uint16_t bits;
};

// (waves_per_eu: builds that the compiler, left alone, gives a few registers more than fit that many waves)
template <int BS, typename ST, int SETS, int FUSE, bool PROBE, int MR = 1>
__global__ __launch_bounds__(512)
__attribute__((amdgpu_waves_per_eu(PROBE ? 1 : MR == 8 && BS == (sizeof(ST) == 4 ? 128 : 64) ? 8 : BS == 128 && sizeof(ST) == 2 && MR == 16 ? 7 : BS == 128 && sizeof(ST) == 2 && MR == 4 && FUSE != 0 ? 6 : 1)))
void acc4_packed_kernel(MNB_ACC4_ARGS)
{
    const Acc4PackedParams p = MNB_ACC4_PARAMS;
    static_assert(MR == 1 || ((MR == 4 || MR == 8 || MR == 16) && (FUSE == 0 || MR == 4) && SETS == 1),
                  "several rows: one register set; codes from the workspace, or up to four rows quantized here");
    constexpr int U = kGroupTiles;
    constexpr int NBT = 128 / BS;
    constexpr int NB = U * NBT;
    constexpr int R = packed_record_bytes(BS, static_cast<int>(sizeof(ST)));
    constexpr int NR = R / 16;
    constexpr int NA = MR == 16 ? 2 * U : MR == 1 ? 1 : U;
    constexpr int SP = MR == 1 ? 1 : 16 / MR;                                     // matrix rows per call row
    constexpr int NX = MR == 1 ? 1 : (NB * 8 + 63) / 64;
    constexpr int kCodeStage = 16 * kCodePitchP;                                  // 16 rows: one tile of codes
    constexpr int kWaveBytes = MR == 1 ? SETS * 512 : 2 * kCodeStage + NB * 128;  // 16 rows: two tiles in turn + the group's pairs
    constexpr int kRowsKept = MR == 1 ? 1 : MR / 4;                               // call rows per lane: g * kRowsKept + r
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = p.waves;
    const int c = lane & 15;
    const int g = lane >> 4;
    const int64_t n_base = static_cast<int64_t>(blockIdx.x) * 16;
    const bool bf16_scales = std::is_same<ST, Bf16Scale>::value || (MR == 1 && p.rest.scales_bf16 != 0);

    constexpr int kChunkBytes = kChunkWeights + 16 * R;
    const uint32_t cg_stride = static_cast<uint32_t>(p.groups) * static_cast<uint32_t>(kChunkBytes);      // bytes of one column group
    const __amdgpu_buffer_rsrc_t srd_p = make_srd(p.packed + static_cast<uint64_t>(blockIdx.x) * cg_stride, cg_stride);
    const __amdgpu_buffer_rsrc_t srd_a = make_srd(p.rows, static_cast<uint64_t>(p.m) * static_cast<uint64_t>(FUSE ? 2 * static_cast<int64_t>(p.k) : p.padded_k));
    const __amdgpu_buffer_rsrc_t srd_x = make_srd(p.pairs, MR == 1 && FUSE ? 0 : static_cast<uint64_t>(p.kb) * (MR == 1 ? 8 : 128));
    constexpr int kBlockLanes = BS / 8;

    const uint32_t w_off = static_cast<uint32_t>(lane * 16);
    const uint32_t r_off = static_cast<uint32_t>(kChunkWeights + c * R);
    unsigned char* stage = smem + wave * kWaveBytes;
    unsigned char* aux_stage = stage + 2 * kCodeStage;            // 16 rows only
    // operand of MFMA j of tile u: the 8 codes of elements u*128 + j*32 + g*8 .. +8. One row: only row 0 matters, every
    // lane of a lane group reads the same 8 bytes of the group's 512. 16 rows: row lane % 16 of the staged tile.
    const uint32_t st_read = MR == 1 ? static_cast<uint32_t>(g * 8) : static_cast<uint32_t>(c * kCodePitchP + g * 8);
    // several rows: a tile's codes arrive as row lane / 8 (+ 8), piece lane % 8, and go to matrix row SP * row
    const uint32_t a_off16 = static_cast<uint32_t>(lane >> 3) * static_cast<uint32_t>(p.padded_k) + static_cast<uint32_t>((lane & 7) * 16);
    const uint32_t st_write16 = static_cast<uint32_t>((lane >> 3) * SP * kCodePitchP + (lane & 7) * 16);
    if constexpr (MR == 4 || MR == 8) {
        for (int i = lane; i < 2 * kCodeStage / 16; i += 64) *reinterpret_cast<uint4*>(stage + i * 16) = make_uint4(0, 0, 0, 0);
        lds_order();
    }

    float y[kRowsKept];
#pragma unroll
    for (int r = 0; r < kRowsKept; ++r) y[r] = 0.f;
    int4p_t acc = {0, 0, 0, 0};

    const int g_begin = wave * p.groups_per_wave;
    const int g_end = min(g_begin + p.groups_per_wave, p.groups);

    using Grp = Acc4PackedGroup<NR, NA, NX>;
    // No branch in here (a branch would make the compiler wait for every load in flight, the prefetch included): a group
    // past the wave's last one gets every offset out of range, fetches nothing and reads as zeros - it adds nothing.
    auto fetch_group = [&](Grp& grp, int gi) {
        const uint32_t oor = gi < g_end ? 0u : kOutOfRange;        // or-ed in: any offset with these bits is out of range
        const uint32_t soff = static_cast<uint32_t>(gi) * static_cast<uint32_t>(kChunkBytes);
#pragma unroll
        for (int u = 0; u < U; ++u) grp.w[u] = load16(srd_p, (w_off + static_cast<uint32_t>(u * 1024)) | oor, soff);
#pragma unroll
        for (int i = 0; i < NR; ++i) grp.r[i] = load16(srd_p, (r_off + static_cast<uint32_t>(i * 16)) | oor, soff);
        if constexpr (MR != 1 && FUSE != 0) {
            // up to four rows quantized here: a[r] = 8 activations of row r (lane * 8 of the group's 512); a row past M lies past
            // the range and reads as zeros, a piece past K would be the next row's and is kept out
            const bool beyond = static_cast<int64_t>(gi) * 512 + lane * 8 >= p.k;
#pragma unroll
            for (int r = 0; r < NA; ++r) {
                const uint32_t off = beyond ? kOutOfRange : static_cast<uint32_t>(r) * static_cast<uint32_t>(p.k) * 2u + static_cast<uint32_t>(lane * 16);
                grp.a[r] = load16(srd_a, off | oor, static_cast<uint32_t>(gi) * 1024u);
            }
        } else if constexpr (MR != 1) {
#pragma unroll
            for (int x = 0; x < NA; ++x) {
                const int u = MR == 16 ? x / 2 : x, i = MR == 16 ? x % 2 : 0;
                // a piece past the end of its row would read the next row's codes (rows past M lie past the range and read as zeros)
                const bool beyond = static_cast<int64_t>(gi * U + u) * 128 + (lane & 7) * 16 >= p.padded_k || (MR == 4 && lane >= 32);
                const uint32_t off = beyond ? kOutOfRange : a_off16 + static_cast<uint32_t>(i * 8) * static_cast<uint32_t>(p.padded_k);
                grp.a[x] = load16(srd_a, off | oor, static_cast<uint32_t>(gi * U + u) * 128u);
            }
#pragma unroll
            for (int x = 0; x < NX; ++x)
                grp.x[x] = load16(srd_x, (lane + 64 * x < NB * 8 ? static_cast<uint32_t>((lane + 64 * x) * 16) : kOutOfRange) | oor, static_cast<uint32_t>(gi * NB) * 128u);
        } else if constexpr (FUSE) {
            grp.a[0] = load16(srd_a, static_cast<uint32_t>(lane * 16) | oor, static_cast<uint32_t>(gi) * 1024u);   // 8 activations; K % 8 == 0 and the range ends the row
        } else {
            grp.a[0] = load16(srd_a, (lane < 32 ? static_cast<uint32_t>(lane * 16) : kOutOfRange) | oor, static_cast<uint32_t>(gi) * 512u);   // the range ends the row at padded_k
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(srd_x, static_cast<int>((lane < NB ? static_cast<uint32_t>(lane * 8) : kOutOfRange) | oor), static_cast<int>(gi * NB * 8), 0);
            grp.x[0].x = v[0];
            grp.x[0].y = v[1];
        }
        asm volatile("" : : "s"(p.rest.bias), "s"(p.rest.y), "s"(p.rest.bias_dtype), "s"(p.rest.y_dtype));      // there from here on, not read behind the last barrier
    };
    auto compute_group = [&](const Grp& grp, int gi, int slot) {
        unsigned char* st = stage + slot * 512;
        float sa_lane = 0.f, qs_lane = 0.f;          // FUSE: scale and f32(code sum) of the block this lane's activations lie in
        uint2 fused_codes[MR != 1 && FUSE != 0 ? MR : 1];
        // FUSE: the quantizer's arithmetic on one 16-byte piece (8 activations); the block's lanes share maximum and code sum.
        // Returns the eight codes in the byte order the repacked weights unpack to, elements 0,4,1,5 | 2,6,3,7.
        auto quantize_piece = [&](const uint4& piece) -> uint2 {
            const uint32_t d[4] = {piece.x, piece.y, piece.z, piece.w};
            float v[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (FUSE == 2) {
                    v[2 * i] = __uint_as_float(d[i] << 16);
                    v[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
                } else {
                    const half2p_t h = __builtin_bit_cast(half2p_t, d[i]);
                    v[2 * i] = static_cast<float>(h.x);
                    v[2 * i + 1] = static_cast<float>(h.y);
                }
            }
            float vmax = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) vmax = fmaxf(vmax, fabsf(v[i]));
            vmax = dpp_max<0xB1>(vmax);
            vmax = dpp_max<0x4E>(vmax);
            if constexpr (BS >= 64) vmax = dpp_max<0x141>(vmax);
            if constexpr (BS >= 128) vmax = dpp_max<0x140>(vmax);
            sa_lane = __fdiv_rn(vmax, 127.0f);
            const float inv = vmax != 0.0f ? __fdiv_rn(127.0f, vmax) : 0.0f;
            int q[8], sum = 0;
            auto round_all = [&](auto away) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float scaled = __fmul_rn(v[i], inv);
                    float r = decltype(away)::value ? roundf(scaled) : rintf(scaled);
                    r = fminf(fmaxf(r, -127.0f), 127.0f);
                    q[i] = static_cast<int>(r);
                    sum += q[i];
                }
            };
            if (p.rest.rounding == 1) round_all(std::true_type{});      // wave-uniform: one branch per group, not one select per element
            else round_all(std::false_type{});
            sum = dpp_addi<0xB1>(sum);
            sum = dpp_addi<0x4E>(sum);
            if constexpr (BS >= 64) sum = dpp_addi<0x141>(sum);
            if constexpr (BS >= 128) sum = dpp_addi<0x140>(sum);
            qs_lane = static_cast<float>(sum);                     // |sum| <= 127 * BS: exact
            const uint32_t lo = (q[0] & 0xff) | ((q[4] & 0xff) << 8) | ((q[1] & 0xff) << 16) | (static_cast<uint32_t>(q[5]) << 24);
            const uint32_t hi = (q[2] & 0xff) | ((q[6] & 0xff) << 8) | ((q[3] & 0xff) << 16) | (static_cast<uint32_t>(q[7]) << 24);
            return make_uint2(lo, hi);
        };
        if constexpr (MR != 1 && FUSE != 0) {
            // every row's piece is quantized; the first lane of a block leaves the row's (scale, code sum) where a block's end
            // reads it: pair [block][row] of the group
#pragma unroll
            for (int r = 0; r < MR; ++r) {
                fused_codes[r] = quantize_piece(grp.a[r]);
                if (lane % kBlockLanes == 0) *reinterpret_cast<float2*>(aux_stage + (lane / kBlockLanes) * 128 + r * 8) = make_float2(sa_lane, qs_lane);
            }
        } else if constexpr (MR != 1) {
#pragma unroll
            for (int x = 0; x < NX; ++x)
                if (lane + 64 * x < NB * 8) *reinterpret_cast<uint4*>(aux_stage + (lane + 64 * x) * 16) = grp.x[x];
        } else if constexpr (FUSE) {
            *reinterpret_cast<uint2*>(st + lane * 8) = quantize_piece(grp.a[0]);
        } else {
            if (lane < 32) *reinterpret_cast<uint4*>(st + lane * 16) = grp.a[0];
        }
        lds_order();
        uint32_t rr[NR * 4];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            rr[4 * i] = grp.r[i].x;
            rr[4 * i + 1] = grp.r[i].y;
            rr[4 * i + 2] = grp.r[i].z;
            rr[4 * i + 3] = grp.r[i].w;
        }
        // every dword of the record counts as used, also its padding: a load destination known to be dead is handed out
        // again at once, and writing it waits for the load in flight
#pragma unroll
        for (int i = 0; i < NR * 4; ++i) asm volatile("" : : "v"(rr[i]));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            long av[4];
            if constexpr (MR != 1) {
                unsigned char* tile = stage + (u & 1) * kCodeStage;
                if constexpr (FUSE != 0) {
                    // the lanes that hold this tile's elements (lane / 16 = u) write each row's eight codes into its matrix row
                    if ((lane >> 4) == u) {
#pragma unroll
                        for (int r = 0; r < MR; ++r) *reinterpret_cast<uint2*>(tile + r * SP * kCodePitchP + (lane & 15) * 8) = fused_codes[r];
                    }
                } else if constexpr (MR != 16) {
                    if (MR == 8 || lane < 32) *reinterpret_cast<uint4*>(tile + st_write16) = grp.a[u];
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i) *reinterpret_cast<uint4*>(tile + st_write16 + i * 8 * kCodePitchP) = grp.a[u * 2 + i];
                }
                lds_order();
#pragma unroll
                for (int j = 0; j < 4; ++j) av[j] = *reinterpret_cast<const long*>(tile + st_read + j * 32);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) av[j] = *reinterpret_cast<const long*>(st + st_read + u * 128 + j * 32);
            }
            const uint32_t wd[4] = {grp.w[u].x, grp.w[u].y, grp.w[u].z, grp.w[u].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool first = (j * 32) % BS == 0;
                const bool last = ((j + 1) * 32) % BS == 0 || j == 3;
                const uint64_t bw = static_cast<uint64_t>(wd[j] & 0x0f0f0f0fu) | (static_cast<uint64_t>((wd[j] >> 4) & 0x0f0f0f0fu) << 32);
                const int4p_t zero = {0, 0, 0, 0};
                acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[j], static_cast<long>(bw), first ? zero : acc, 0, 0, 0);
                if (last) {
                    const int bi = u * NBT + (j * 32) / BS;
                    // (a block beyond K needs no guard: its repacked scale is 0 and its codes and sums are 0)
                    const int zbyte = NB * static_cast<int>(sizeof(ST)) + bi;
                    const float zf = static_cast<float>((rr[zbyte / 4] >> ((zbyte % 4) * 8)) & 0xffu);
                    float sb;
                    if constexpr (sizeof(ST) == 4) {
                        sb = __uint_as_float(rr[bi]);
                    } else {
                        const uint32_t raw = (rr[bi / 2] >> ((bi % 2) * 16)) & 0xffffu;
                        sb = bf16_scales ? __uint_as_float(raw << 16) : f16_bits_to_f32(static_cast<uint16_t>(raw));
                    }
                    if constexpr (MR != 1) {
                        // this lane's call rows g * kRowsKept + r sit in components SP * r of its accumulator
                        const float2* pairs = reinterpret_cast<const float2*>(aux_stage + bi * 128 + g * kRowsKept * 8);
#pragma unroll
                        for (int r = 0; r < kRowsKept; ++r) {
                            const float2 pr = pairs[r];                                           // (scale, sum of codes)
                            const float f = fmaf(-zf, pr.y, static_cast<float>(acc[SP * r]));      // both terms are integers below 2^24: exact
                            y[r] = fmaf(f, __fmul_rn(pr.x, sb), y[r]);
                            if constexpr (PROBE) {
                                const int64_t blk = static_cast<int64_t>(gi) * NB + bi;
                                const int64_t row = g * kRowsKept + r;
                                if (row < p.m && n_base + c < p.n && blk < p.kb) p.rest.acc_probe[(row * p.n + n_base + c) * p.kb + blk] = static_cast<int>(f);
                            }
                        }
                    } else {
                        const int src = FUSE ? bi * kBlockLanes : bi;         // a lane of the block, or the lane that loaded its pair
                        const float sa = __int_as_float(__builtin_amdgcn_readlane(FUSE ? __float_as_int(sa_lane) : static_cast<int>(grp.x[0].x), src));
                        const float qs = __int_as_float(__builtin_amdgcn_readlane(FUSE ? __float_as_int(qs_lane) : static_cast<int>(grp.x[0].y), src));
                        const float f = fmaf(-zf, qs, static_cast<float>(acc[0]));   // both terms are integers below 2^24: exact
                        y[0] = fmaf(f, __fmul_rn(sa, sb), y[0]);
                        if constexpr (PROBE) {                                       // row 0 sits in lanes 0..15
                            const int64_t blk = static_cast<int64_t>(gi) * NB + bi;
                            if (lane < 16 && n_base + lane < p.n && blk < p.kb) p.rest.acc_probe[(n_base + lane) * p.kb + blk] = static_cast<int>(f);
                        }
                    }
                }
            }
        }
    };

    if constexpr (SETS == 2) {
        Grp ga, gb;
        fetch_group(ga, g_begin);
        int gi = g_begin;
        for (; gi + 1 < g_end; gi += 2) {                      // whole pairs, no branch inside: every wait counts loads exactly
            __builtin_amdgcn_sched_barrier(0);                 // nothing of a group moves up into the one before it
            fetch_group(gb, gi + 1);
            __builtin_amdgcn_sched_barrier(0);
            compute_group(ga, gi, 0);
            __builtin_amdgcn_sched_barrier(0);
            fetch_group(ga, gi + 2);                           // past the end this fetches nothing
            __builtin_amdgcn_sched_barrier(0);
            compute_group(gb, gi + 1, 1);
        }
        if (gi < g_end) compute_group(ga, gi, 0);              // an odd group out

    } else {
        Grp ga;
        for (int gi = g_begin; gi < g_end; ++gi) {
            fetch_group(ga, gi);
            compute_group(ga, gi, 0);
        }
    }

    // ---- split-K reduction across the waves of this workgroup, in wave order ----
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
    if constexpr (MR != 1) {                           // [waves][kRowsKept][64]: lane (c, g) holds rows g * kRowsKept + r of column c
#pragma unroll
        for (int r = 0; r < kRowsKept; ++r) red[(wave * kRowsKept + r) * 64 + lane] = y[r];
        __syncthreads();
        for (int idx = threadIdx.x; idx < kRowsKept * 64; idx += waves * 64) {
            const int r = idx >> 6;
            const int l = idx & 63;
            const int row = (l >> 4) * kRowsKept + r;
            const int64_t col = n_base + (l & 15);
            if (row < p.m && col < p.n) {
                float total = 0.f;
                for (int w = 0; w < waves; ++w) total += red[(w * kRowsKept + r) * 64 + l];
                total = with_bias(total, p.rest.bias, p.rest.bias_dtype, row, p.n, col, p.rest.y_dtype);
                store_from_f32(p.rest.y, p.rest.y_dtype, static_cast<int64_t>(row) * p.n + col, total);
            }
        }
    } else {                                           // [waves][16]: row 0 lives in lanes 0..15
        if (lane < 16) red[wave * 16 + lane] = y[0];
        __syncthreads();
        if (threadIdx.x < 16) {
            const int64_t col = n_base + threadIdx.x;
            if (col < p.n) {
                float total = 0.f;
                for (int w = 0; w < waves; ++w) total += red[w * 16 + threadIdx.x];
                total = with_bias(total, p.rest.bias, p.rest.bias_dtype, 0, p.n, col, p.rest.y_dtype);       // one row
                store_from_f32(p.rest.y, p.rest.y_dtype, col, total);
            }
        }
    }
}

template <int BS, typename ST>
static int launch_acc4_packed(Acc4PackedParams p, int waves, bool single_set, int fuse, hipStream_t stream)
{
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(p.n) + 15) / 16);
    p.waves = waves;
    if (p.m > 1) {
        if constexpr (std::is_same<ST, uint16_t>::value) {
            if (p.rest.scales_bf16) return launch_acc4_packed<BS, Bf16Scale>(p, waves, single_set, fuse, stream);
        }
        // two tiles of codes in turn + the group's pairs per wave; the reduction reuses the space (1 KiB per wave)
        const size_t lds16 = static_cast<size_t>(waves) * (2 * 16 * kCodePitchP + kGroupTiles * (128 / BS) * 128);
        if (fuse != 0) {
            // up to four f16 / bf16 rows: the kernel quantizes them itself (no codes, no pairs, no launch before this one)
            if (p.m > 4 || p.rest.acc_probe) return -1;
            if (fuse == 2) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 2, false, 4>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
            else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 1, false, 4>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
            return static_cast<int>(hipGetLastError());
        }
        if (p.m <= 4) {
            if (p.rest.acc_probe) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, true, 4>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
            else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, false, 4>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        } else if (p.m <= 8) {
            if (p.rest.acc_probe) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, true, 8>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
            else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, false, 8>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        } else if (p.rest.acc_probe) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, true, 16>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, 0, false, 16>), dim3(grid), dim3(waves * 64), lds16, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        return static_cast<int>(hipGetLastError());
    }
    if constexpr (std::is_same<ST, Bf16Scale>::value) {
        return -1;                                         // (several rows only)
    } else {
    const size_t lds = static_cast<size_t>(waves) * 1024;
    auto go = [&](auto fuse) {
        constexpr int F = decltype(fuse)::value;
        if (p.rest.acc_probe) {
            if (single_set) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, F, true>), dim3(grid), dim3(waves * 64), lds, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
            else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 2, F, true>), dim3(grid), dim3(waves * 64), lds, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        } else if (single_set) hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 1, F, false>), dim3(grid), dim3(waves * 64), lds, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
        else hipLaunchKernelGGL((acc4_packed_kernel<BS, ST, 2, F, false>), dim3(grid), dim3(waves * 64), lds, stream, p.rows, p.pairs, p.packed, p.m, p.n, p.k, p.kb, p.padded_k, p.groups, p.groups_per_wave, p.waves, p.rest);
    };
    if (fuse == 1) go(std::integral_constant<int, 1>{});
    else if (fuse == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 0>{});
    return static_cast<int>(hipGetLastError());
    }
}

static int packed_groups(const RocmMatMulNBitsArgs* a)
{
    const int64_t kb = (a->k + a->block_size - 1) / a->block_size;
    const int64_t tiles = (kb * a->block_size + 127) / 128;
    return static_cast<int>((tiles + kGroupTiles - 1) / kGroupTiles);
}

static int packed_chunk_bytes(const RocmMatMulNBitsArgs* a)
{
    return kChunkWeights + 16 * packed_record_bytes(a->block_size, a->scale_dtype == ROCM_DT_F32 ? 4 : 2);
}

}  // namespace mnb

// Rows 5..64 only run from the repacked copy in the shared-activation kernel, which wants many column groups.
// (16 rows at block size 32, 32 at 64, 64 at 128: more row blocks than that do not fit the register file)
// `pair`: the call is the fused gate/up launch or one of its two projections - both projections' columns count, since the
// paired launch streams both, and a projection launched on its own must add up the way the paired launch does.
// The shared-activation kernel's window below five rows: block 128 on 18432 .. 49151 columns, four rows of a plain call, two to
// four of a gate/up pair (whose columns count together).
static bool few_row_wide(const RocmMatMulNBitsArgs* a, bool pair)
{
    const int64_t cols = a->n * (pair ? 2 : 1);
    return a->m <= 4 && a->m >= (pair ? 2 : 4) && a->block_size == 128 && cols >= 18432 && cols < 49152;
}

static bool wide_shape(const RocmMatMulNBitsArgs* a, bool pair)
{
    const int64_t max_rows = a->block_size == 32 ? 16 : a->block_size == 64 ? 32 : 64;
    // Columns from which it beats the other kernels. 17 rows and more (against the tiled kernel and two passes of the
    // split-K kernel; bf16, 4096 -> 14336: 30.6 -> 24.4 us at 32 rows with block 128, 31.5 -> 25.7 with block 64; 33-64 rows
    // lose below 16384 columns: 32.9 -> 38.7 us). Up to 16 rows the 16-row split-K kernel over the same repacked stream is
    // the alternative, and with 4096 rows of K it stays ahead up to 16384 columns at block 128 (5 / 8 / 16 rows, 14336
    // columns: 12.0 / 12.1 / 13.8 against 13.2 / 13.3 / 14.2 us; 16384: 12.5 / 12.8 / 14.4 against 13.4 / 13.5 / 14.5; at 20480
    // it loses, 14.9-17.3 against 14.1-15.3) and up to 20480 at block 32 (14336: 13.2 / 13.2 / 14.7 against 17.1 / 17.2 / 17.7;
    // 20480: 16.9 / 17.2 / 18.6 against 17.8 / 17.9 / 18.4; at 28672 it loses, 22-25 against 20-21).
    // (block 64: 12.3 / 12.6 / 14.4 us at 14336 and 13.2 / 13.7 / 15.2 at 16384 against 15.4-16.0 in the shared-activation kernel)
    const int64_t min_cols = a->m > 32 ? 16384 : a->m > 16 ? 14336 : a->block_size == 32 ? 22528 : a->block_size == 64 ? 20480 : 18432;
    // Four rows of a plain call on 18432 .. 49151 columns at block 128 run here as well: level with the four-row split-K build
    // on a GPU that runs it well (3584 -> 37888 18.1 -> 17.6 us, 4096 -> 28672 16.0 -> 16.2, 3072 -> 32064 13.8 -> 13.5), and this kernel
    // moved far less from one GPU to the next (on two others the same three calls took 21-22.5 / 18.0-18.3 / 16.8-17.0 us there
    // against 18.8 / 16.5 / 14.9-15.4 at five rows here). More columns lose (4096 -> 128256: 56.4 -> 62.3), and so do three rows.
    // A gate/up pair counts both projections' columns, as below, and comes here from two rows: the paired four-row split-K
    // launch is further behind than the plain one (3584 -> 2 x 18944 at 2 / 3 / 4 rows: 20.2-21.2 / 20.5-21.1 / 20.9 -> 17.9 / 18.5 /
    // 18.9 us, the unfused call over 37888 columns 18.5 at four; 5120 -> 2 x 13824: 20.0 / 20.4-21.3 -> 18.6-18.9 / 19.0-19.7;
    // 4096 -> 2 x 14336 level).
    if (few_row_wide(a, pair)) return a->gamma == nullptr;
    return a->m >= 5 && a->m <= max_rows && a->n * (pair ? 2 : 1) >= min_cols;
}

extern "C" int rocm_decode_packed_eligible(const RocmMatMulNBitsArgs* a)
{
    RocmMatMulNBitsArgs base = *a;
    if (base.m > 16) base.m = 16;                         // the shared-activation kernel takes up to 64 rows
    if (!rocm_decode_mfma_eligible(&base)) return 0;
    if (a->m * a->k * 2 >= 0x7ffffff0 || a->n > 0x7fffffff) return 0;      // (sizes are 32-bit arguments)
    if (a->m > 16 && !wide_shape(a, false)) return 0;    // up to 16 rows the split-K kernel stages the rows per wave
    return static_cast<int64_t>(mnb::packed_groups(a)) * mnb::packed_chunk_bytes(a) < 0x7fffffff;
}

extern "C" uint64_t rocm_decode_packed_bytes(const RocmMatMulNBitsArgs* a)
{
    const uint64_t col_groups = static_cast<uint64_t>((a->n + 15) / 16);
    return col_groups * static_cast<uint64_t>(mnb::packed_groups(a)) * static_cast<uint64_t>(mnb::packed_chunk_bytes(a));
}

static int launch_pack_decode(const RocmMatMulNBitsArgs* a, int bits, int groups, void* packed, rocm_stream_t stream)
{
    mnb::PackParams p;
    p.bits = bits;
    p.b = a->b;
    p.scales = a->scales;
    p.zp = a->zp;
    p.out = static_cast<uint8_t*>(packed);
    p.n = a->n;
    p.kb = (a->k + a->block_size - 1) / a->block_size;
    p.row_bytes = p.kb * a->block_size * bits / 8;
    p.zp_row = (p.kb * bits + 7) / 8;
    p.bs_log2 = __builtin_ctz(static_cast<unsigned>(a->block_size));
    p.scale_bytes = a->scale_dtype == ROCM_DT_F32 ? 4 : 2;
    p.groups = groups;
    p.chunk_bytes = mnb::packed_chunk_bytes(a);
    p.record = mnb::packed_record_bytes(a->block_size, p.scale_bytes);
    const dim3 grid(static_cast<unsigned>(p.groups), static_cast<unsigned>((a->n + 15) / 16));
    hipLaunchKernelGGL(mnb::pack_decode_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return static_cast<int>(hipGetLastError());
}

extern "C" int rocm_launch_pack_decode(const RocmMatMulNBitsArgs* a, void* packed, rocm_stream_t stream)
{
    return launch_pack_decode(a, 4, mnb::packed_groups(a), packed, stream);
}

// The 4-bit call whose stream an 8-bit call's is, in everything that plans or sizes it: twice the tiles, the same activations.
static RocmMatMulNBitsArgs as_four_bits(const RocmMatMulNBitsArgs* a)
{
    RocmMatMulNBitsArgs four = *a;
    const int64_t kb = (a->k + a->block_size - 1) / a->block_size;
    four.k = (kb * a->block_size + 127) / 128 * 256;
    return four;
}

extern "C" int rocm_decode_packed8_eligible(const RocmMatMulNBitsArgs* a)
{
    const RocmMatMulNBitsArgs four = as_four_bits(a);
    return a->m <= 32 && a->k % 8 == 0 && a->scale_dtype == a->a_dtype && !a->gamma && rocm_decode_packed_eligible(&four);
}

extern "C" uint64_t rocm_decode_packed8_bytes(const RocmMatMulNBitsArgs* a)
{
    const RocmMatMulNBitsArgs four = as_four_bits(a);
    return rocm_decode_packed_bytes(&four);
}

extern "C" int rocm_launch_pack_decode8(const RocmMatMulNBitsArgs* a, void* packed, rocm_stream_t stream)
{
    const RocmMatMulNBitsArgs four = as_four_bits(a);
    return launch_pack_decode(a, 8, mnb::packed_groups(&four), packed, stream);
}

// The launch of rocm_launch_decode_packed; with `packed_up` the paired gate/up launch. `probe_only`: nothing is launched,
// the return value says whether a paired launch with this split of K fits a workgroup (1) or not (0).
// `pair_member`: the launch is one projection of a gate/up pair (or the paired launch itself): the split of K is chosen
// for the pair's column groups together, so that the separate launches and the paired one add up in the same order.
extern "C" int rocm_decode_packed_fuses_norm(const RocmMatMulNBitsArgs* a)
{
    if (!a->gamma || a->m > 4 || a->k % 128 != 0 || !rocm_decode_packed_eligible(a)) return 0;      // (with gamma, up to four rows never take the shared-activation kernel)
    // Where up to four rows take the shared-activation kernel (alone, or as one projection of a pair), the rows are normalized
    // by a launch of their own: a pair's first call runs its projections over normalized rows, and the later single launch has
    // to add up in the same order.
    if (few_row_wide(a, false) || few_row_wide(a, true)) return 0;
    if (a->gamma_dtype != ROCM_DT_F32 && a->gamma_dtype != a->a_dtype) return 0;
    return (reinterpret_cast<uintptr_t>(a->gamma) & 15) == 0;
}

// Waves per SIMD of the one-set builds, from the registers the compiler reported for them (59-76 with one row, 71-102 with
// four, 84-112 with eight, 110-134 with sixteen); a test holds the table against the build's report.
static int waves_per_simd(const RocmMatMulNBitsArgs* a, bool f32_scales)
{
    // [f16 / bf16][rows: 1, 2-4, 5-8, 9-16][block 32, 64, 128][16-bit / f32 scales]
    static const unsigned char table[2][4][3][2] = {
        {{{5, 6}, {8, 7}, {8, 8}}, {{5, 4}, {5, 6}, {6, 6}}, {{4, 4}, {5, 5}, {5, 5}}, {{4, 3}, {4, 4}, {3, 4}}},
        {{{7, 6}, {8, 7}, {8, 8}}, {{5, 4}, {6, 6}, {7, 6}}, {{4, 4}, {5, 5}, {5, 5}}, {{4, 3}, {4, 4}, {4, 4}}},
    };
    const int rows = a->m <= 1 ? 0 : a->m <= 4 ? 1 : a->m <= 8 ? 2 : 3;
    const int block = a->block_size == 32 ? 0 : a->block_size == 64 ? 1 : 2;
    return table[a->a_dtype == ROCM_DT_BF16][rows][block][f32_scales];
}

extern "C" int rocm_decode_packed_waves_per_simd(int block_size, int m, int f32_scales, int bf16)
{
    RocmMatMulNBitsArgs a{};
    a.block_size = block_size;
    a.m = m;
    a.a_dtype = bf16 ? ROCM_DT_BF16 : ROCM_DT_F16;
    return waves_per_simd(&a, f32_scales != 0);
}

// the most waves a workgroup of decode_packed_kernel may have (see the kernel's launch bounds)
static int w_max_of(const RocmMatMulNBitsArgs* a, bool f32_scales)
{
    return (a->block_size == 128 && !f32_scales && (a->m <= 8 || a->a_dtype == ROCM_DT_BF16)) ? 16 : 8;
}

// What rocm_launch_decode_packed launches for a shape, without launching it: which kernel, which build of it, how many waves
// split K and over how many register sets. Everything below is arithmetic on the shape and the chip's CU count (the
// thresholds were measured on 256 CUs and are written as multiples of that count), so a CPU test can hold the answers for
// the model shapes against a committed table: a change made for one shape cannot move another unnoticed.
struct PackedPlan {
    bool wide;          // the shared-activation kernel (plan in `w`); otherwise the split-K kernel
    mnb::WidePlan w;
    int rows_build;     // split-K kernel: rows the build stages (1, 4, 8, 16)
    int waves;          // per projection and workgroup
    int groups_per_wave;
    bool single_set;
};

static PackedPlan plan_decode_packed(const RocmMatMulNBitsArgs* a, int waves, bool pair_member, bool paired_launch, int64_t cus)
{
    PackedPlan plan{};
    const bool f32_scales = a->scale_dtype == ROCM_DT_F32;
    if (wide_shape(a, pair_member)) {
        plan.wide = true;
        plan.w = mnb::plan_wide(a->m, a->n, a->block_size, !f32_scales, paired_launch, cus);
        plan.groups_per_wave = mnb::packed_groups(a);
        plan.waves = plan.w.waves;
        return plan;
    }
    const int groups = mnb::packed_groups(a);
    // Waves per workgroup (they split K in whole tile groups). Many column groups (thousands of waves even at four per
    // group): short waves of at most two tile groups. Few column groups: enough waves per group to reach about 8k in
    // flight. Then the adjustments below: register sets, and wave counts that fit the chip.
    const int64_t wgs = (a->n + 15) / 16 * ((pair_member && a->m <= 4) ? 2 : 1);      // (a pair shares a launch up to four rows here)
    int w = waves;
    const int w_max = w_max_of(a, f32_scales);
    // One row: one tile group per wave where the workgroup can hold that many waves, no prefetch, offset and zero point
    // through the activation sums. Every byte of the call is then requested as soon as its wave starts, and what a wave
    // computes between its loads and the reduction is the least any variant here does. Measured against the few-wave
    // prefetching build it replaced on the small shapes (bf16, block 128): 3584 -> 4608 5.06 -> 4.78 us, 3584 -> 3584
    // 4.17 -> 3.97, 18944 -> 3584 9.94 -> 9.41, 3584 -> 37888 15.81 -> 15.48.
    // (a gate/up pair keeps the few-wave split: with fourteen waves a workgroup the paired launch measured 17.8 us against 15.5)
    const bool one_row = a->m <= 1 && !pair_member;
    const bool large_grid = wgs * 4 >= 24 * cus;
    if (w <= 0) {
        if (one_row) {
            w = groups;
        } else if (large_grid) {
            w = (groups + 1) / 2;
        } else {
            const int want = static_cast<int>((32 * cus + wgs - 1) / wgs);
            w = want < groups ? want : groups;               // at least one group per wave
        }
        if (w < 1) w = 1;
    }
    // One register set or two (the second holds the next group's loads while the current one is multiplied, at the price
    // of waves per SIMD). Swept over 384 .. 1024 column groups x K = 3584 .. 8192 x 1 / 2 / 4 rows x block 32 / 128: one set is
    // ahead or level nearly everywhere, by up to 30 % from K = 5120 (block 128, 4 rows, 5120 -> 16384: 12.4 against 16.5 us;
    // block 32: 15.8 against 21.7). Two sets keep:
    //  * two to four rows on small grids, where the second set's first fetch, issued before anything else, is worth 1-3 %
    //    (block 128, 3584 -> 4608: 5.56 against 5.72 us; 18944 -> 3584 at block 32: 13.3 against 13.9) - below 256 column groups at
    //    block 32, else up to 512 (two workgroups per CU: 4096 -> 8192 6.4 against 6.5 us at two rows, but 4096 -> 9216 7.7 against
    //    7.3 and 3072 -> 9216 7.75 against 6.8), or below 320 when K is more than eight groups;
    //  * one row at block size 32 with more groups than a workgroup has waves, on small grids: sixteen scale steps per group
    //    leave enough arithmetic between a wave's loads that fetching ahead pays (18944 -> 3584 12.4 -> 11.8 us; with 1024
    //    column groups it loses, 5120 -> 16384: 17.3 against 12.2; at block 128 one set stays ahead, 9.5 against 9.9 us).
    bool single_set;
    if (one_row) single_set = !(a->block_size == 32 && groups > w_max && wgs <= cus);
    else if (a->block_size == 32) single_set = wgs >= cus;
    else single_set = wgs > 2 * cus || (wgs >= cus + cus / 4 && groups > 8);
    if (w > w_max) w = w_max;
    if (w > groups) w = groups;
    // Mid-size grids: a launch whose waves do not all fit the chip at once queues workgroups behind each other, and
    // workgroups of 6, 10 or 12 waves leave slots of a CU empty on top; fewer waves of more groups each run it faster
    // (16 rows, block 128: 3072 -> 16384 13.8 -> 12.2 us, 5120 -> 13824 21.0 -> 17.6, 6144 -> 16384 24.6 -> 21.1, 5120 -> 17920
    // 24.1 -> 21.7; 8 rows: 16.2 -> 13.9 on 5120 -> 13824; one row: 7168 -> 16384 16.2 -> 14.3; 4 rows at block 32: 3584 -> 16384
    // 12.5 -> 11.4). Workgroups of eight waves of one group each fill a CU's slots exactly and stay (K = 4096, 16 rows: 14336
    // columns 13.9 against 14.9 us with four waves, 11008 11.3 against 11.6), and so do the large grids, whose waves are
    // short enough for the queue not to show (one row, 3584 -> 37888: seven waves of one group, 15.5 against 15.8 us).
    // Which of the wave counts that fit: a workgroup's waves go round the four SIMDs, so k workgroups of w waves put
    // k * ceil(w / 4) of them on the first SIMD, and with three to five waves per SIMD a workgroup of 5, 6 or 10 waves keeps
    // a CU from filling up (16 rows, 5120 -> 13824: five waves 21.4 us, four 17.5, ten 21.0; 2 rows at block 32, 8192 -> 12288:
    // six waves 18.9 us, four 16.6). Builds of up to five waves per SIMD take the count that holds the most waves per CU that way.
    if (waves <= 0 && !(w == 8 && groups == 8)) {
        const int per_simd = waves_per_simd(a, f32_scales);
        const int64_t fit = cus * 4 * per_simd / wgs;
        const int64_t least = a->m <= 1 ? 6 : a->m <= 4 ? 4 : 1;
        // A count within that bound can still be too many once the waves' places on the SIMDs are counted (576 workgroups of six
        // waves at five waves per SIMD: two workgroups a CU, 3072 slots for 3456 waves). Then the count that holds the most is
        // taken as well, if it leaves a wave two tile groups at most (block 32, two / four rows: 3072 -> 9216 8.9 / 8.9 -> 8.3 / 8.7 us,
        // 3072 -> 12288 10.0 / 10.1 -> 8.5 / 9.0; block 128, five / eight rows: 3072 -> 12288 9.2 -> 8.1; with three groups a wave it
        // lost, 5120 -> 10240 at block 32: 10.1 -> 10.8).
        const bool crowded = per_simd <= 5 && w <= fit && wgs * w > cus * static_cast<int64_t>(per_simd / ((w + 3) / 4) * w);
        if (fit >= least && (w > fit || crowded)) {
            if (w > fit) w = static_cast<int>(fit);
            const int limit = w;
            if (per_simd <= 5) {                       // (with six or more waves per SIMD the plain count is as good or better: 4 rows at block 128, 6144 -> 16384: six waves 14.2 us, four 15.4)
                int best = -1;
                for (int g = 1; g <= groups; ++g) {
                    const int cand = (groups + g - 1) / g;
                    if (cand > limit || (crowded && g > 2)) continue;
                    const int held = per_simd / ((cand + 3) / 4) * cand;
                    if (held > best) {                 // (ties: the first found, which has the most waves)
                        best = held;
                        w = cand;
                    }
                    if (cand == 1) break;
                }
            }
        }
    }
    // A projection of a gate/up pair takes at most half a workgroup's waves where that leaves a wave five tile groups or fewer,
    // so that the pair runs as one launch and not as two and the epilogue (bf16, one / two / four rows: 3072 -> 2 x 8192 at block 32
    // 14.3 -> 9.1 us at one row; 5120 -> 2 x 13824 at block 32 25.5 / 30.9 / 32.6 -> 20.6 / 25.4 / 25.7, at block 64 24.1 / 26.5 / 28.0 ->
    // 18.8 / 21.7 / 22.8; 8192 -> 2 x 8192 at block 64 22.5 / 25.3 / 26.8 -> 17.7 / 18.6 / 19.9). The projection launched alone on a
    // pair's first call takes the same count, as everything here.
    if (pair_member && a->m <= 4 && waves <= 0 && 2 * w > w_max && (groups + w_max / 2 - 1) / (w_max / 2) <= 5) w = w_max / 2;
    const int gpw = (groups + w - 1) / w;
    w = (groups + gpw - 1) / gpw;
        plan.rows_build = a->m <= 1 ? 1 : a->m <= 4 ? 4 : a->m <= 8 ? 8 : 16;
    plan.waves = w;
    plan.groups_per_wave = gpw;
    plan.single_set = a->m > 4 || single_set || (a->m > 1 && a->gamma != nullptr);
    return plan;
}

extern "C" int rocm_decode_packed_plan(const RocmMatMulNBitsArgs* a, int waves, int pair_member, int compute_units, RocmDecodePackedPlan* out)
{
    if (!a || !out || compute_units <= 0 || !rocm_decode_packed_eligible(a)) return -1;
    const PackedPlan plan = plan_decode_packed(a, waves, pair_member != 0, pair_member == 2, compute_units);
    if (plan.wide && !plan.w.ok) return -1;
    const int64_t col_groups = (a->n + 15) / 16;
    out->shared_activations = plan.wide;
    out->rows_build = plan.wide ? plan.w.rb * 16 : plan.rows_build;
    out->waves = plan.waves;
    out->groups_per_wave = plan.groups_per_wave;
    out->register_sets = plan.wide ? ((plan.w.pf ? 1 : 0) + (plan.w.deep ? 1 : 0) + 1) : (plan.single_set ? 1 : 2);
    out->activation_sums = plan.wide ? plan.w.sums : (plan.rows_build == 1 && plan.single_set);
    out->workgroups = plan.wide ? static_cast<int64_t>(plan.w.grid) : col_groups;
    return 0;
}

extern "C" int rocm_decode_packed_ahead(const RocmMatMulNBitsArgs* a, const void* packed, const void* packed_up, int waves, RocmWeightsAhead* out)
{
    if (!rocm_decode_packed_eligible(a)) return 0;
    const bool pair = packed_up != nullptr;
    const PackedPlan plan = plan_decode_packed(a, waves, pair, pair, rocm_ffi_compute_units());
    if (plan.wide && !plan.w.ok) return 0;
    const int64_t col_groups = (a->n + 15) / 16, each = plan.wide ? (pair ? plan.waves / 2 : plan.waves) : 1;
    out->first = packed;
    out->second = packed_up;
    out->bytes = static_cast<uint64_t>(each) * mnb::packed_groups(a) * mnb::packed_chunk_bytes(a);
    out->workgroups = static_cast<uint32_t>(col_groups / each);            // whole ones
    return 1;
}

// Operands and stream geometry of a launch over `a`'s stream.
static mnb::PackedParams packed_params(const RocmMatMulNBitsArgs* a, const void* packed)
{
    mnb::PackedParams p{};
    p.a = static_cast<const uint16_t*>(a->a);
    p.packed = static_cast<const uint8_t*>(packed);
    p.m = static_cast<int>(a->m);
    p.k = static_cast<int>(a->k);
    p.n = static_cast<int>(a->n);
    p.groups = mnb::packed_groups(a);
    p.rest.nodes[0] = mnb::PackedNode{a->bias, a->y, p.packed, p.n, a->bias_dtype};
    p.rest.y_dtype = a->y_dtype;
    return p;
}

static int launch_decode_packed(const RocmMatMulNBitsArgs* a, const void* packed, const void* packed_up, int decomposed, int waves, bool probe_only,
                                bool pair_member, rocm_stream_t stream, RocmStepTail* tail)
{
    if (!rocm_decode_packed_eligible(a)) return probe_only ? 0 : -1;
    const int64_t cus = rocm_ffi_compute_units();
    const PackedPlan plan = plan_decode_packed(a, waves, pair_member, packed_up != nullptr, cus);
    mnb::PackedParams p = packed_params(a, packed);
    p.packed_up = static_cast<const uint8_t*>(packed_up);
    p.rest.decomposed_silu = decomposed;
    const bool bf16 = a->a_dtype == ROCM_DT_BF16;
    if (a->gamma) {
        if (!rocm_decode_packed_fuses_norm(a)) return probe_only ? 0 : -1;
        p.gamma = a->gamma;
        p.rest.gamma_f32 = a->gamma_dtype == ROCM_DT_F32;
        p.rest.norm_epsilon = a->norm_epsilon;
    }

    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool f32_scales = a->scale_dtype == ROCM_DT_F32;
    if (plan.wide) {
        // the shared-activation kernel's paired form takes up to 16 rows (one block of rows per wave)
        if (probe_only) return a->m <= 16 ? 1 : 0;
        if (packed_up && a->m > 16) return -1;
        if (bf16) return f32_scales ? mnb::launch_wide_bs<true, float>(p, a->block_size, cus, s) : mnb::launch_wide_bs<true, uint16_t>(p, a->block_size, cus, s);
        return f32_scales ? mnb::launch_wide_bs<false, float>(p, a->block_size, cus, s) : mnb::launch_wide_bs<false, uint16_t>(p, a->block_size, cus, s);
    }
    const int w = plan.waves;
    const int w_max = w_max_of(a, f32_scales);
    const bool single_set = plan.single_set;
    p.split = static_cast<uint32_t>(plan.groups_per_wave);
    // a paired launch keeps each projection's own split of K (so that it adds up in the same order) and needs twice the waves
    if (probe_only) return a->m <= 4 && 2 * w <= w_max ? 1 : 0;
    if (packed_up && (a->m > 4 || 2 * w > w_max)) return -1;

    if (bf16) return f32_scales ? mnb::launch_packed_bs<true, float>(p, a->block_size, w, single_set, s, tail) : mnb::launch_packed_bs<true, uint16_t>(p, a->block_size, w, single_set, s, tail);
    return f32_scales ? mnb::launch_packed_bs<false, float>(p, a->block_size, w, single_set, s, tail) : mnb::launch_packed_bs<false, uint16_t>(p, a->block_size, w, single_set, s, tail);
}

extern "C" int rocm_launch_decode_packed(const RocmMatMulNBitsArgs* a, const void* packed, int waves, rocm_stream_t stream, RocmStepTail* tail)
{
    return launch_decode_packed(a, packed, nullptr, 0, waves, false, false, stream, tail);
}

extern "C" int rocm_decode_plain_eligible(const RocmMatMulNBitsArgs* a)
{
    return a->m <= 32 && !a->gamma && rocm_decode_packed_eligible(a);
}

// `a`'s call over its stream, planned as `four`'s.
static int launch_decode_plain(const RocmMatMulNBitsArgs* a, const RocmMatMulNBitsArgs* four, int bits, const void* packed, int waves, rocm_stream_t stream)
{
    const int64_t cus = rocm_ffi_compute_units();
    const PackedPlan plan = plan_decode_packed(four, waves, false, false, cus);
    mnb::PackedParams p = packed_params(four, packed);
    p.k = static_cast<int>(a->k);            // what the activations have
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool bf16 = a->a_dtype == ROCM_DT_BF16, f32_scales = a->scale_dtype == ROCM_DT_F32;
    if (plan.wide) {
        // a grid between one and one and a half workgroups of eight waves per CU: as many waves as spread it over one a CU, as in plan_wide
        // (3584 -> 37888, block 128, 16 rows: 8 bits, bf16 38.3 -> 31.6 us, act-order 4 bits, f16 26.7 -> 20.9)
        const int64_t col_groups = (a->n + 15) / 16;
        const bool in_between = a->m <= 16 && (bits == 8 || a->block_size != 32) && col_groups > cus * mnb::kWideWaves && col_groups <= cus * mnb::kWideWavesMax;
        return mnb::launch_plain_wide(p, bits, bf16, f32_scales, a->block_size, in_between ? static_cast<int>((col_groups + cus - 1) / cus) : mnb::kWideWaves, s);
    }
    p.split = static_cast<uint32_t>(plan.groups_per_wave);
    return mnb::launch_plain(p, bits, bf16, f32_scales, a->block_size, plan.waves, s);
}

extern "C" int rocm_launch_decode_plain(const RocmMatMulNBitsArgs* a, const void* packed, int waves, rocm_stream_t stream)
{
    return rocm_decode_plain_eligible(a) ? launch_decode_plain(a, a, 4, packed, waves, stream) : -1;
}

// One row in another order than the weights': gathered by the kernel where a thread has at most four pieces of it to bring to LDS and two workgroups fit a CU's.
extern "C" int rocm_decode_plain_gathers(const RocmMatMulNBitsArgs* a, int waves)
{
    if (a->m != 1 || a->k > 65536 || (reinterpret_cast<uintptr_t>(a->a) & 15) != 0 || !rocm_decode_plain_eligible(a)) return 0;
    const PackedPlan plan = plan_decode_packed(a, waves, false, false, rocm_ffi_compute_units());
    return !plan.wide && a->k <= static_cast<int64_t>(plan.waves) * 64 * 8 * mnb::kGatherPieces && mnb::plain_gather_lds(a->k, plan.waves) <= 80 * 1024;
}

extern "C" int rocm_launch_decode_plain_gathered(const RocmMatMulNBitsArgs* a, const void* packed, const uint16_t* order, int waves, rocm_stream_t stream)
{
    if (!rocm_decode_plain_gathers(a, waves)) return -1;
    const PackedPlan plan = plan_decode_packed(a, waves, false, false, rocm_ffi_compute_units());
    mnb::PackedParams p = packed_params(a, packed);
    p.gamma = order;
    p.split = static_cast<uint32_t>(plan.groups_per_wave);
    return mnb::launch_plain_gather(p, a->a_dtype == ROCM_DT_BF16, a->scale_dtype == ROCM_DT_F32, a->block_size, plan.waves, static_cast<hipStream_t>(stream));
}

extern "C" int rocm_launch_decode_packed8(const RocmMatMulNBitsArgs* a, const void* packed, int waves, rocm_stream_t stream)
{
    if (!rocm_decode_packed8_eligible(a)) return -1;
    const RocmMatMulNBitsArgs four = as_four_bits(a);
    return launch_decode_plain(a, &four, 8, packed, waves, stream);
}

extern "C" int rocm_launch_decode_packed_pair_member(const RocmMatMulNBitsArgs* a, const void* packed, int waves, rocm_stream_t stream)
{
    return launch_decode_packed(a, packed, nullptr, 0, waves, false, true, stream, nullptr);
}

extern "C" int rocm_decode_packed_pair_fits(const RocmMatMulNBitsArgs* a, int waves)
{
    return launch_decode_packed(a, nullptr, nullptr, 0, waves, true, true, nullptr, nullptr);
}

extern "C" int rocm_launch_decode_packed_pair(const RocmMatMulNBitsArgs* a, const void* packed_gate, const void* packed_up, int decomposed, int waves,
                                              rocm_stream_t stream)
{
    if (!packed_gate || !packed_up || a->y_dtype != a->a_dtype) return -1;
    return launch_decode_packed(a, packed_gate, packed_up, decomposed, waves, false, true, stream, nullptr);
}

extern "C" int rocm_acc4_packed_eligible(const RocmMatMulNBitsArgs* a)
{
    const bool bs_ok = a->block_size == 32 || a->block_size == 64 || a->block_size == 128;
    if (!(bs_ok && a->m >= 1 && a->m <= 16 && a->n >= 1)) return 0;
    if ((reinterpret_cast<uintptr_t>(a->b) & 15) != 0 || (reinterpret_cast<uintptr_t>(a->scales) & 3) != 0) return 0;
    const int64_t padded_k = (a->k + a->block_size - 1) / a->block_size * a->block_size;
    if (a->m * padded_k >= 0x7fffffff || a->n > 0x7fffffff) return 0;      // the codes are addressed with 32-bit offsets, sizes are 32-bit arguments
    return static_cast<int64_t>(mnb::packed_groups(a)) * mnb::packed_chunk_bytes(a) < 0x7fffffff;
}

extern "C" int rocm_acc4_packed_fuses_quantizer(const RocmMatMulNBitsArgs* a)
{
    if (!(rocm_acc4_packed_eligible(a) && (a->a_dtype == ROCM_DT_F16 || a->a_dtype == ROCM_DT_BF16) && a->k % 8 == 0 && (reinterpret_cast<uintptr_t>(a->a) & 15) == 0))
        return 0;
    if (a->m == 1) return 1;
    // Two to four rows: every workgroup quantizes the rows again, which more than doubles what a wave computes per tile
    // group - worth it only where the call is short enough for the quantizer's own launch (about 3 us) to weigh more:
    // 3584 -> 3584 8.2 -> 6.3 us, 3584 -> 4608 8.9 -> 8.0; 4096 -> 14336 level; 18944 -> 3584 14.5 -> 16.6 and 3584 -> 37888 19.6 -> 22.4
    // the wrong way. (The builds that probe block accumulators read the workspace's codes.)
    const int64_t work = (a->n + 15) / 16 * mnb::packed_groups(a);            // column groups x tile groups
    return a->m <= 4 && !a->acc_probe && work <= 4096;
}

// Waves per workgroup, tile groups per wave and register sets of rocm_launch_acc4_packed for a shape on a chip of `cus` CUs
// (thresholds measured on 256 CUs, written as multiples of the count). No GPU work.
static void plan_acc4_packed(const RocmMatMulNBitsArgs* a, int waves, int64_t cus, int* waves_out, int* groups_per_wave, bool* one_set)
{
    const int groups = mnb::packed_groups(a);
    const int64_t wgs = (a->n + 15) / 16;
    int w = waves;
    bool single_set = wgs * 4 >= 24 * cus;
    if (w <= 0) {
        if (single_set) {
            w = (groups + 1) / 2;
        } else {
            const int want = static_cast<int>((32 * cus + wgs - 1) / wgs);
            w = want < groups ? want : groups;
        }
        if (w < 1) w = 1;
    } else {
        single_set = wgs * w >= 24 * cus;
    }
    if (w > 8) w = 8;
    if (w > groups) w = groups;
    const int gpw = (groups + w - 1) / w;
    w = (groups + gpw - 1) / gpw;
    // One register set (one-row launches; the builds for several rows have no other): with one group per wave a second set
    // has nothing to fetch ahead (4096 -> 14336: 14.3 -> 9.8 us at block 32, 9.7 -> 8.8 at 64, 9.2 -> 8.4 at 128); at block 32 the
    // two-set build holds three waves per SIMD against eight (5120 -> 13824 21.4 -> 11.6 us, 6144 -> 16384 23.8 -> 14.4,
    // 8192 -> 8192 14.1 -> 10.5); and from a few hundred column groups on the other block sizes are level or ahead with one
    // (13824 -> 5120 at block 128: 12.3 -> 11.2; 8192 -> 10240 at 64: 12.3 -> 11.5). Small K-heavy grids keep two (18944 -> 3584 at
    // block 128: 9.3 against 10.2 us).
    if (gpw == 1 || a->block_size == 32 || wgs > cus) single_set = true;

    *waves_out = w;
    *groups_per_wave = gpw;
    *one_set = single_set;
}

extern "C" int rocm_acc4_packed_plan(const RocmMatMulNBitsArgs* a, int waves, int compute_units, int* waves_out, int* groups_per_wave, int* register_sets)
{
    if (!a || compute_units <= 0 || !rocm_acc4_packed_eligible(a)) return -1;
    int w = 0, gpw = 0;
    bool one_set = false;
    plan_acc4_packed(a, waves, compute_units, &w, &gpw, &one_set);
    if (waves_out) *waves_out = w;
    if (groups_per_wave) *groups_per_wave = gpw;
    if (register_sets) *register_sets = (one_set || a->m > 1) ? 1 : 2;
    return 0;
}

extern "C" int rocm_launch_acc4_packed(const RocmMatMulNBitsArgs* a, const void* packed, const RocmAcc4Workspace* ws, int rounding, int waves, rocm_stream_t stream)
{
    if (!rocm_acc4_packed_eligible(a)) return -1;
    const int fuse = ws ? 0 : (a->a_dtype == ROCM_DT_BF16 ? 2 : 1);
    if (!ws && !rocm_acc4_packed_fuses_quantizer(a)) return -1;
    mnb::Acc4PackedParams p{};
    p.rows = ws ? static_cast<const void*>(ws->qa) : a->a;
    p.pairs = !ws ? nullptr : a->m > 1 ? ws->aux : ws->aq;
    p.packed = static_cast<const uint8_t*>(packed);
    p.m = static_cast<int>(a->m);
    p.n = static_cast<int>(a->n);
    p.k = static_cast<int>(a->k);
    p.kb = static_cast<int>((a->k + a->block_size - 1) / a->block_size);
    p.padded_k = p.kb * a->block_size;
    p.groups = mnb::packed_groups(a);
    p.rest.bias = a->bias;
    p.rest.y = a->y;
    p.rest.bias_dtype = a->bias_dtype;
    p.rest.y_dtype = a->y_dtype;
    p.rest.rounding = rounding;
    p.rest.scales_bf16 = a->scale_dtype == ROCM_DT_BF16;
    p.rest.acc_probe = a->acc_probe;

    int w = 0, gpw = 0;
    bool single_set = false;
    plan_acc4_packed(a, waves, rocm_ffi_compute_units(), &w, &gpw, &single_set);
    p.groups_per_wave = gpw;

    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool f32_scales = a->scale_dtype == ROCM_DT_F32;
    switch (a->block_size) {
        case 32: return f32_scales ? mnb::launch_acc4_packed<32, float>(p, w, single_set, fuse, s) : mnb::launch_acc4_packed<32, uint16_t>(p, w, single_set, fuse, s);
        case 64: return f32_scales ? mnb::launch_acc4_packed<64, float>(p, w, single_set, fuse, s) : mnb::launch_acc4_packed<64, uint16_t>(p, w, single_set, fuse, s);
        default: return f32_scales ? mnb::launch_acc4_packed<128, float>(p, w, single_set, fuse, s) : mnb::launch_acc4_packed<128, uint16_t>(p, w, single_set, fuse, s);
    }
}
