// Batched prefill GEMM: Q4_0 / Q8_0 weights x Q8_0-quantized activations -> f32, on the gfx950 int8 matrix cores.
//
// Arithmetic: gemm_q4_0_q8_0_neon / gemm_q8_0_q8_0_neon
// (wick/src/backend/simd.rs:696-925, 937-1019):
//   C[i,j] = sum_b f32(isum_{i,j,b}) * (f32(f16 d_w[i,b]) * xs[j,b]),  isum exact i32
// with one scale pair per 32-element block, so i32 accumulation cannot run across
// blocks: every MFMA covers exactly one block (K = 32) and its i32 result is scaled
// into f32 accumulators on the vector ALU.
//
// Three families of block loops:
//   * gemm_tile_kernel, v_mfma_i32_32x32x32_i8: prompts, on the cheapest of six tiles for the launch (see T32 and TileL .. TileH);
//   * gemm_few_kernel, v_mfma_i32_16x16x32_i8, 32 rows x 32 or 64 tokens, several such tiles side by side past 64 tokens: where latency is what a
//     launch costs (few_applies, few_side_applies, few_tokens_per_tile);
//   * gemm_narrow_kernel, v_mfma_i32_16x16x32_i8, 128 rows x 64 tokens: the other unsplit launches of up to 48 tokens (many rows), which skip the
//     16-token columns they do not have; gemm_mfma_kernel, the same shape on 128 x 128, on request (wick_rocm_set_gemm_mfma_shape).
// The kernels are bound by the two scaling FMAs per result plus the matrix instructions, which a SIMD overlaps only in part, and by
// feeding both from LDS.  A wave issues a vector-ALU instruction only every ~4.7 cycles while a SIMD retires one every ~2.3, so two
// waves per SIMD at least, four where a wave has one result buffer.
//
// The 16x16 kernels below are described here; gemm_tile_kernel shares their data layouts and says the rest at its place.
// One stage = 4 blocks (128 elements of K).  Both operands are copied global -> LDS directly
// (global_load_lds_dwordx4: asynchronous, no registers, 1 KB per wave instruction):
//   * weights from the GEMM's own copy of the matrix, made from the raw GGUF blocks when the
//     weight is uploaded (gemm_pack_kernel, layout at StageT): int8 operand rows and
//     {scale, -bias * scale} pairs already in the order a stage of LDS holds them, so the main
//     loop neither unpacks nibbles nor converts scales nor stores to LDS;
//   * activations from the token-major Q8_0 quants; token scales through registers (they are
//     stored block-major).
// LDS holds two stages (76 KB, two workgroups per CU).  The copies of stage s+1 are issued
// before stage s is computed, so there is one barrier per stage and the load latency hides
// behind the stage's ALU work.
//
// LDS operand layout: weights [granule of 32 rows][khalf][block][row][16 bytes], activations
// [token][8 x 16 bytes, swizzled].  An MFMA lane supplies 8 consecutive K-bytes of operand row
// lane % 16, K-quarter lane / 16, so 32 consecutive lanes read 256 consecutive bytes (the two
// 8-byte halves of 16 rows): conflict-free.  For Q4_0 the low nibbles of a block ARE its first
// 16 elements and the high nibbles its last 16 (wick/src/quant.rs:82-88): the two khalf planes.
// (The K order inside an MFMA is irrelevant as long as both operands use the same one.)
//
// Roles: tokens are the MFMA "A" (M) operand, weight rows the "B" (N) operand, so in the
// 16x16 result a lane holds ONE weight row (n = lane % 16) and 4 consecutive tokens
// (m = 4*(lane/16) + r).  Its weight scale is one register pair per block and row tile;
// the token scales sit in LDS as f32, token-major, and a lane reads its four with one
// 16-byte read (a broadcast within each group of 16 lanes).
//
// Scaling is what bounds this kernel (vector ALU, not the matrix core), so it is
// cut to two FMAs per result:
//   * Q4_0 nibbles are stored as 16*(nibble-8) (the nibble moved to the top of the
//     byte, sign bit flipped: two ALU ops per four weights, no per-byte subtract);
//     the 1/16 is folded into the weight scale.
//   * The MFMA accumulates onto C = 0x4B400000 in every lane, i.e. the bit pattern
//     of 12582912.0f = 1.5 * 2^23.  Integer-adding v (|v| < 2^22) to that pattern
//     gives exactly the f32 12582912 + v, so the i32 -> f32 conversion is free.
//   * t = fma(D_as_f32, dw, -12582912*dw) = round(v * dw) exactly (single rounding;
//     12582912*dw is exact because dw has an 11-bit significand);
//     acc = fma(t, dx, acc), both plain v_fma_f32 (v_fma_mix_f32 with an f16 scale
//     operand would save registers but issues at half the rate).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "wick_rocm_device.h"
#include "wick_rocm_internal.h"

namespace wick_rocm {

namespace {

constexpr int BM = 128;       // weight rows per workgroup
constexpr int BN = 128;       // tokens per workgroup
constexpr int BN_NARROW = 64;  // ... of the narrow kernel
constexpr int KB = 4;         // blocks per stage
constexpr int THREADS = 512;  // 8 waves: 2 (rows) x 4 (tokens)
constexpr int TT = 2;          // 16-token MFMA tiles per wave
constexpr int RT = 4;          // 16-row MFMA tiles per wave
// The rules that choose tile and split count in CUs of the whole chip (the constants in them were fitted on it), two workgroups
// each.  On a partition of it they still choose launches that are right, not the fastest ones.
constexpr uint32_t kCus = 256;
constexpr uint32_t kBiasBits = 0x4B400000u;  // 12582912.0f
constexpr float kBias = 12582912.0f;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct GemmArgs {
    const uint8_t* w;
    const int8_t* xq;
    const float* xs;
    float* y;
    int32_t* dots;  // parity hook output (DUMP only)
    uint32_t m, n, k;
    uint32_t y_stride;
    uint32_t row_tiles, tok_tiles;
    int y_row_major;
    int accumulate;
    // Up to two more weights that share the activations (Q / K / V, gate / up): their row tiles follow the first
    // weight's in the launch's tile list.  tile_start[i]: first row tile of weight i + 1 (UINT32_MAX: absent).
    const uint8_t* w_more[2];
    float* y_more[2];
    uint32_t m_more[2];
    uint32_t tile_start[2];
    // Gated feed-forward launch (GATED kernels only): w = gate, w_up = up, the output is the Q8_0-quantized silu(gate) * up.
    const uint8_t* w_up;
    int8_t* q_out;   // [n][m]
    float* s_out;    // [n][m / 32]
    // K split of a narrow launch with few tiles: workgroup (tile, split) walks its share of the stages and leaves its sums
    // in partial[split][n][m]; gemm_splitk_reduce_kernel adds the shares up in a fixed order.  ksplit <= 1: off.
    uint32_t ksplit;
    float* partial;
};

// (of a launch's leading scalars) More weights than one.
constexpr uint32_t kMoreWeights = 512;

// Makes `a` describe the weight that owns row tile `row_tile` and rebases the tile index to that weight.
__device__ __forceinline__ void select_weight(GemmArgs& a, uint32_t& row_tile) {
    const bool second = row_tile >= a.tile_start[0], third = row_tile >= a.tile_start[1];
    if (second) {
        a.w = third ? a.w_more[1] : a.w_more[0];
        a.y = third ? a.y_more[1] : a.y_more[0];
        a.m = third ? a.m_more[1] : a.m_more[0];
        row_tile -= third ? a.tile_start[1] : a.tile_start[0];
    }
}

// The weights a GEMM launch reads are not the raw GGUF blocks but a copy laid out for this kernel, made once when the
// weight is uploaded (gemm_pack_kernel): rows in granules of 32, and per (granule, stage of 4 blocks) one 5120-byte slab
//   [khalf 2][block 4][row 32][16 bytes]   int8 operand rows (Q4_0: 16 * (nibble - 8)), 4096 bytes
//   [block 4][row 32] {dw, -12582912 * dw}  scale pairs (dw x 1/16 for Q4_0), 1024 bytes
// laid out [pair of granules][stage][granule of the pair]: the 64 rows x 128 K-elements a wave works on are 10 KB in one piece.  A slab is exactly what a stage of LDS holds for those 32 rows, so the weights go
// global -> LDS directly like the activations: five 1 KB copies per granule, no staging registers, no unpack and no LDS
// stores in the main loop, fully coalesced.  A tile is four granules (a gated tile: two of the gate weight and the same
// two of the up weight).  1.25 bytes per weight instead of 0.5625 (Q4_0) / 1.0625 (Q8_0).
constexpr int GR = 32;                              // rows per granule
constexpr int kSlabWt = 2 * KB * GR * 16;           // 4096
constexpr int kSlabDws = KB * GR * 8;               // 1024
constexpr int kSlab = kSlabWt + kSlabDws;           // 5120
constexpr int kSlabChunks = kSlab / 1024;           // 5 direct-to-LDS copies of 1 KB

// One stage of operands.
template <int NTOK>  // tokens per workgroup tile: BN, or BN_NARROW for the narrow kernel
struct StageT {
    uint4 wt[BM / GR][2][KB][GR];  // [granule][khalf][block][row]  int8 weights: the slabs' first 4 KB
    uint4 xt[NTOK][2 * KB];        // [token][16-byte K-chunk, swizzled] int8 activations, see dma_activations
    float2 dws[BM / GR][KB][GR];   // {dw, -12582912*dw} per granule, block and row: the slabs' last 1 KB
    float dxf[KB][NTOK];           // token scales
};
using Stage = StageT<BN>;

template <int NTOK>
struct SmemT {
    StageT<NTOK> st[2];
};
using Smem = SmemT<BN>;

// 16*(nibble-8) for the four low / four high nibbles of each byte of q.
__device__ __forceinline__ uint32_t q4_lo_x16(uint32_t q) { return ((q << 4) & 0xf0f0f0f0u) ^ 0x80808080u; }
__device__ __forceinline__ uint32_t q4_hi_x16(uint32_t q) { return (q & 0xf0f0f0f0u) ^ 0x80808080u; }

struct StageRegs {
    float4 dx;
};

// Raw blocks -> slabs.  One workgroup per (granule, stage): thread (row = t % 32, block = t / 32).  Rows past the end of
// the matrix become zero rows with zero scales.  For Q4_0 the low nibbles of a block ARE its first 16 elements and the high
// nibbles its last 16 (wick/src/quant.rs:82-88): the two khalf planes.
template <int TYPE>
__global__ __launch_bounds__(GR * KB) void gemm_pack_kernel(const uint8_t* __restrict__ raw, uint32_t m, uint32_t nb, uint8_t* __restrict__ packed) {
    constexpr int BB = TYPE == 2 ? 18 : 34;
    const uint32_t stages = nb / KB, granule = blockIdx.x / stages, stage = blockIdx.x % stages;
    const uint32_t within = threadIdx.x % GR, b = threadIdx.x / GR, row = granule * GR + within;
    uint32_t lo[4] = {0, 0, 0, 0}, hi[4] = {0, 0, 0, 0};
    float dw = 0.0f;
    if (row < m) {
        const uint16_t* blk = reinterpret_cast<const uint16_t*>(raw + ((size_t)row * nb + stage * KB + b) * BB);  // blocks are 2-byte aligned
        dw = f16_bits_to_f32(blk[0]) * (TYPE == 2 ? 0.0625f : 1.0f);
        uint32_t q[8];
#pragma unroll
        for (int i = 0; i < (BB - 2) / 4; i++) q[i] = (uint32_t)blk[1 + 2 * i] | ((uint32_t)blk[2 + 2 * i] << 16);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = TYPE == 2 ? q4_lo_x16(q[i]) : q[i];
            hi[i] = TYPE == 2 ? q4_hi_x16(q[i]) : q[4 + i];
        }
    }
    uint8_t* slab = packed + (((size_t)(granule >> 1) * stages + stage) * 2 + (granule & 1u)) * kSlab;
    reinterpret_cast<uint4*>(slab)[(0 * KB + b) * GR + within] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    reinterpret_cast<uint4*>(slab)[(1 * KB + b) * GR + within] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    reinterpret_cast<float2*>(slab + kSlabWt)[b * GR + within] = make_float2(dw, -kBias * dw);
}

// Activation tiles go global -> LDS directly (global_load_lds_dwordx4): no staging
// registers, no unpack, no ds_write, and the copy runs asynchronously under the stage's
// ALU work.  A token's 128 K-bytes of the stage are exactly one cache line, so one wave
// instruction fetches 8 tokens x 8 16-byte chunks = 8 whole lines (lane l -> token l / 8,
// position l % 8; the address unit works per line touched, and a chunk-major split would
// touch 64 lines per instruction).  Direct-to-LDS data lands lane-contiguous, i.e. as
// [token][8 positions] rows of 128 bytes, which an MFMA operand read (16 tokens, same
// chunk) would hit with an 8-way bank conflict.  So position p of token t holds K-chunk
// p ^ ((t >> 1) & 7): the lane picks its GLOBAL chunk accordingly, and 16 consecutive
// tokens reading one chunk then spread over all banks.  16 instructions per stage, four
// per loader wave (dma_stage).
__device__ __forceinline__ uint32_t xt_swizzle(uint32_t token_in_tile) { return (token_in_tile >> 1) & 7u; }
// A thread's global read positions of the stage to fetch next.  Set up once per tile; every fetch moves them one stage
// (128 K-elements) on, one 64-bit add each, instead of rebuilding row / token / block addresses per stage.
// Only the first kLoaderWaves waves of a workgroup issue the stage's global -> LDS copies (and fetch the token scales): the
// address unit takes a copy instruction every 16 cycles, so 36 of them per stage and workgroup queue up, and a wave waiting in
// that queue issues nothing else.  The later waves of a workgroup are the ones that lag in the block loop (the SIMD favours the
// older wave), so they get no copies to issue at all and the earlier ones, which would otherwise idle at the stage barrier, all.
constexpr int kLoaderWaves = 4;
template <int NTOK>
struct StagePtrs {
    const int8_t* x[NTOK / 8 / kLoaderWaves];  // this lane's 16-byte activation chunks (direct-to-LDS copies)
    const uint8_t* wc;                          // this lane's 16 bytes of the first kilobyte of granule `wave`'s slab
    const uint8_t* dx;                          // threads 0 .. NTOK - 1: a token's four scales
};
// Where chunk c (0 .. 19) of a tile's stage lands: granule c / 5, its weights' kilobyte c % 5 or (the fifth) its scale pairs.
template <int NTOK>
__device__ __forceinline__ void* chunk_dst(StageT<NTOK>& s, uint32_t c) {
    const uint32_t g = c / kSlabChunks, part = c % kSlabChunks;
    return part < 4 ? static_cast<void*>(reinterpret_cast<uint8_t*>(&s.wt[g][0][0][0]) + 1024u * part) : static_cast<void*>(&s.dws[g][0][0]);
}
template <int NTOK>
__device__ __forceinline__ void dma_stage(StagePtrs<NTOK>& p, StageT<NTOK>& s) {
    constexpr int PER_WAVE = NTOK / 8 / kLoaderWaves;  // activation instructions per loader wave and stage
    static_assert(BM / GR == kLoaderWaves, "one granule's slab per loader wave");
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (wave >= (uint32_t)kLoaderWaves) return;  // uniform per wave
#pragma unroll
    for (int j = 0; j < PER_WAVE; j++) {
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)p.x[j],
                                         (void __attribute__((address_space(3)))*)&s.xt[8u * (PER_WAVE * wave + j)][0], 16, 0, 0);
        p.x[j] += KB * 32;
    }
#pragma unroll
    for (int part = 0; part < kSlabChunks; part++)
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(p.wc + 1024 * part),
                                         (void __attribute__((address_space(3)))*)chunk_dst(s, kSlabChunks * wave + part), 16, 0, 0);
    p.wc += 2 * kSlab;
}

template <int NTOK>
__device__ __forceinline__ void init_stage_ptrs(const GemmArgs& a, uint32_t row_tile, uint32_t tok0, uint32_t kb0, StagePtrs<NTOK>& p) {
    constexpr int PER_WAVE = NTOK / 8 / kLoaderWaves;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wave = min((uint32_t)__builtin_amdgcn_readfirstlane((int)(t >> 6)), (uint32_t)kLoaderWaves - 1u);  // (later waves: unused values)
    const uint32_t nb = a.k >> 5, stages = nb / KB;
#pragma unroll
    for (int j = 0; j < PER_WAVE; j++) {
        const uint32_t tt = 8u * (PER_WAVE * wave + j) + (lane >> 3);  // token within the tile
        const uint32_t chunk = (lane & 7u) ^ xt_swizzle(tt);
        const uint32_t tok = min(tok0 + tt, a.n - 1);
        p.x[j] = a.xq + (size_t)tok * a.k + (size_t)kb0 * 32 + 16u * chunk;
    }
    const uint32_t granules = (a.m + GR - 1) / GR;
    {
        const uint32_t g = wave;
        const uint32_t granule = min((BM / GR) * row_tile + g, granules - 1u);  // past the end of the matrix: any rows, their results are not stored
        p.wc = a.w + (((size_t)(granule >> 1) * stages + kb0 / KB) * 2 + (granule & 1u)) * kSlab + 16u * lane;
    }
    p.dx = nullptr;
    if (t < NTOK && a.xs) {  // xs is null only for the parity hook, which never scales
        const uint32_t tok = min(tok0 + t, a.n - 1);
        p.dx = reinterpret_cast<const uint8_t*>(a.xs + (size_t)tok * nb + kb0);
    }
}

// Thread -> rest of a stage: one float4 (4 blocks) of token scales per token, threads 0 .. NTOK - 1 (loader waves), through registers
// (they are stored block-major).
template <int NTOK>
__device__ __forceinline__ void load_stage(StagePtrs<NTOK>& p, StageRegs& r) {
    if (p.dx) {
        r.dx = *reinterpret_cast<const float4*>(p.dx);
        p.dx += KB * sizeof(float);
    } else {
        r.dx = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

template <int NTOK>
__device__ __forceinline__ void store_stage(StageT<NTOK>& s, const StageRegs& r) {
    const uint32_t t = threadIdx.x;
    if (t < NTOK) {
        const uint32_t u = t;
        s.dxf[0][u] = r.dx.x;
        s.dxf[1][u] = r.dx.y;
        s.dxf[2][u] = r.dx.z;
        s.dxf[3][u] = r.dx.w;
    }
}

// Per-block operands of a wave's TT x RT MFMA tiles: 8 K-bytes of this lane's operand row.
struct Mats {
    long av[TT], bv[RT];
};
struct Scales {
    float2 dw[RT];  // {dw, -12582912*dw} of this lane's weight row, per row tile
    v4f dx[TT];     // scales of this lane's four tokens, per token tile
};

// All LDS reads of the main loop are inline assembly on purpose.  While direct-to-LDS
// copies (of the NEXT stage, into the other buffer) are in flight, the compiler makes
// every LDS read it can see wait for all of them, which would put the whole global-memory
// latency at the start of each stage.  These reads touch only the current buffer; the
// copies are waited for explicitly before the barrier that ends the stage.  Data arrives
// in issue order; lds_wait<N> is the matching wait (at most N later LDS reads still
// outstanding) and ties the registers, so nothing can use them earlier.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const void __attribute__((address_space(3)))*)p;
}
// A lane's four LDS read addresses (its rows of xt / wt / dws and its tokens of dxf for the
// block being fetched).  Tile indices are immediate offsets; moving to the next block costs
// three additions and, for the swizzled activation tile, one xor + shift-add:
// xt = xbase + ((block ^ xsh) << 5).
struct LaneAddr {
    uint32_t xt, wt, dws, dxf;
    uint32_t xbase, xsh;
};
constexpr int kOffWt = sizeof(uint4) * GR;            // one block of wt (within a granule's khalf plane)
constexpr int kOffDws = sizeof(float2) * GR;          // one block of dws (within a granule)
constexpr int kOffDxf = sizeof(float) * BN;           // one block of dxf
__device__ __forceinline__ void next_block(LaneAddr& la, uint32_t block, bool advance) {
    la.xt = la.xbase + (((advance ? block + 1 : block) ^ la.xsh) << 5);
    la.wt += advance ? kOffWt : 0;
    la.dws += advance ? kOffDws : 0;
    la.dxf += advance ? kOffDxf : 0;
}
template <int OFF>
__device__ __forceinline__ void lds_read16(uint32_t addr, v4f& dst) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read8(uint32_t addr, long& dst) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read8(uint32_t addr, float2& dst) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
__device__ __forceinline__ void load_mats(const LaneAddr& la, Mats& m) {  // TT + RT = 6 reads
    lds_read8<0 * 16 * 128>(la.xt, m.av[0]);  // 16 tokens further: same swizzle
    lds_read8<1 * 16 * 128>(la.xt, m.av[1]);
    lds_read8<0>(la.wt, m.bv[0]);  // row tiles 0, 1: the two halves of the wave's first granule; 2, 3: of its second
    lds_read8<256>(la.wt, m.bv[1]);
    lds_read8<kSlabWt>(la.wt, m.bv[2]);
    lds_read8<kSlabWt + 256>(la.wt, m.bv[3]);
}
__device__ __forceinline__ void load_row_scales(const LaneAddr& la, Scales& s) {  // RT = 4 reads
    lds_read8<0>(la.dws, s.dw[0]);
    lds_read8<128>(la.dws, s.dw[1]);
    lds_read8<kSlabDws>(la.dws, s.dw[2]);
    lds_read8<kSlabDws + 128>(la.dws, s.dw[3]);
}
template <int T>
__device__ __forceinline__ void load_tok_scales(const LaneAddr& la, Scales& s) {  // 1 read
    lds_read16<T * 64>(la.dxf, s.dx[T]);
}
template <int N>
__device__ __forceinline__ void lds_wait(Mats& m) {
    asm volatile("s_waitcnt lgkmcnt(%6)"
                 : "+v"(m.av[0]), "+v"(m.av[1]), "+v"(m.bv[0]), "+v"(m.bv[1]), "+v"(m.bv[2]), "+v"(m.bv[3])
                 : "n"(N)
                 : "memory");
}
template <int N>
__device__ __forceinline__ void lds_wait(Scales& s) {
    asm volatile("s_waitcnt lgkmcnt(%6)"
                 : "+v"(s.dw[0]), "+v"(s.dw[1]), "+v"(s.dw[2]), "+v"(s.dw[3]), "+v"(s.dx[0]), "+v"(s.dx[1])
                 : "n"(N)
                 : "memory");
}

// Scales one 16 x 16 MFMA result (4 values per lane) into the f32 accumulators: two
// full-rate v_fma_f32 per value.
__device__ __forceinline__ void scale_tile(const v4i& d, const float2 dw, const v4f& dx, float (&acc)[4]) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float v = __builtin_fmaf(__int_as_float(d[r]), dw.x, dw.y);
        acc[r] = __builtin_fmaf(v, dx[r], acc[r]);
    }
}

// Parity hook: the raw i32 block dots of one MFMA result.  row = this lane's weight row,
// tok = the first of its four tokens.
template <int TYPE>
__device__ __forceinline__ void dump_tile(const GemmArgs& a, const v4i& d, uint32_t row, uint32_t tok, uint32_t nb, uint32_t block) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (row < a.m && tok + r < a.n) {
            int v = d[r] - (int)kBiasBits;
            if (TYPE == 2) v >>= 4;  // weights were stored x16; exact
            a.dots[((size_t)(tok + r) * a.m + row) * nb + block] = v;
        }
    }
}

// Workgroup -> tile, XCD- and L2-aware.  Hardware hands consecutive workgroup ids to
// the 8 XCDs round-robin, so ids with equal (id % 8) share an L2 (4 MB).  Each XCD
// takes a contiguous run of a tile list that walks the output in 8 x 8 "supertiles"
// (8 row tiles x 8 token tiles, row-major inside): the ~64 workgroups resident on an
// XCD at one time then touch 8 weight panels + 8 activation panels (~3.3 MB at
// k = 2048), which fit its L2, instead of a 4 x 16 strip whose activation panels
// alone overflow it.
__device__ __forceinline__ void tile_of_block(uint32_t bid, uint32_t row_tiles, uint32_t tok_tiles, uint32_t& row_tile,
                                              uint32_t& tok_tile, bool& valid) {
    constexpr uint32_t S = 8;
    const uint32_t tiles = row_tiles * tok_tiles;
    const uint32_t per_xcd = (tiles + 7u) / 8u;
    const uint32_t t = (bid & 7u) * per_xcd + (bid >> 3);
    valid = (bid >> 3) < per_xcd && t < tiles;
    const uint32_t tt = valid ? t : 0;
    const uint32_t sr_count = (row_tiles + S - 1) / S, sc_count = (tok_tiles + S - 1) / S;
    const uint32_t sr = min(tt / (S * tok_tiles), sr_count - 1);  // supertile row (all but the last hold S*tok_tiles tiles)
    const uint32_t t1 = tt - sr * S * tok_tiles;
    const uint32_t h = min(S, row_tiles - sr * S);
    const uint32_t sc = min(t1 / (h * S), sc_count - 1);
    const uint32_t t2 = t1 - sc * h * S;
    const uint32_t w = min(S, tok_tiles - sc * S);
    row_tile = sr * S + t2 / w;
    tok_tile = sc * S + t2 % w;
}

// Results of a wave's MFMA tiles into the output (or into a K share's partial sums): element (tt, rt, r) of the wave tile is
// (row + RSTEP rt, tok + TSTEP tt + r), `row` / `tok` being this lane's first row and token (16 / 16 for the 16x16 MFMA
// layout: a lane holds 4 consecutive tokens of one row per tile; 8 / 32 for the 32x32 layout: 4 groups of 4 tokens, 8 apart).  One instantiation per output layout
// so that the inner index is an immediate offset of the store; CHECK = false for wave tiles that lie inside the matrix (no
// predicates at all), ACC adds onto what is there.  The mode is uniform per launch, the bounds are uniform per wave: the
// callers branch once, not per element.
template <int NTT, int NRT, int TSTEP, int RSTEP, bool ROW_MAJOR, bool CHECK, bool ACC, typename F>
__device__ __forceinline__ void store_results(float* __restrict__ base, size_t stride, uint32_t row, uint32_t tok, uint32_t m, uint32_t n,
                                              F&& value) {
    // accumulating inside the matrix: all old values on their way before the first is used, not one round trip per value
    constexpr bool AHEAD = ACC && !CHECK;
    float old[AHEAD ? NTT * NRT * 4 : 1];
    if constexpr (AHEAD) {
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int rt = 0; rt < NRT; rt++)
                    old[(tt * 4 + r) * NRT + rt] = ROW_MAJOR ? base[(size_t)(row + RSTEP * rt) * stride + tok + TSTEP * tt + r]
                                                             : base[(size_t)(tok + TSTEP * tt + r) * stride + row + RSTEP * rt];
    }
    if constexpr (ROW_MAJOR) {
#pragma unroll
        for (int rt = 0; rt < NRT; rt++) {
            float* q = base + (size_t)(row + RSTEP * rt) * stride + tok;
#pragma unroll
            for (int tt = 0; tt < NTT; tt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (CHECK && !(row + RSTEP * rt < m && tok + TSTEP * tt + r < n)) continue;
                    const float v = value(tt, rt, r);
                    q[TSTEP * tt + r] = AHEAD ? old[(tt * 4 + r) * NRT + rt] + v : (ACC ? q[TSTEP * tt + r] + v : v);
                }
        }
    } else {
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float* q = base + (size_t)(tok + TSTEP * tt + r) * stride + row;
#pragma unroll
                for (int rt = 0; rt < NRT; rt++) {
                    if (CHECK && !(row + RSTEP * rt < m && tok + TSTEP * tt + r < n)) continue;
                    const float v = value(tt, rt, r);
                    q[RSTEP * rt] = AHEAD ? old[(tt * 4 + r) * NRT + rt] + v : (ACC ? q[RSTEP * rt] + v : v);
                }
            }
    }
}
// The launch's output mode picked once per wave: a K share's partial sums [share][n][m], or y in either layout, plain or accumulating.
template <int NTT, int NRT, int TSTEP = 16, int RSTEP = 16, typename F>
__device__ __forceinline__ void store_wave_tile(const GemmArgs& a, uint32_t ksplit, uint32_t split, uint32_t row, uint32_t tok, F&& value) {
    // the wave tile's corner is the same for every lane: keep the test (and the branches on it) scalar
    const uint32_t row_end = (uint32_t)__builtin_amdgcn_readfirstlane((int)(row - (row & (uint32_t)(RSTEP - 1)))) + (uint32_t)(RSTEP * NRT);
    const uint32_t tok_end = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tok - (tok & (uint32_t)(TSTEP - 1)))) + (uint32_t)(TSTEP * NTT);
    const bool inside = row_end <= a.m && tok_end <= a.n;
    if (ksplit > 1) {  // this share's sums; the reduce launch (or the caller's next kernel) adds the shares up
        float* base = a.partial + (size_t)split * a.n * a.m;
        if (inside) store_results<NTT, NRT, TSTEP, RSTEP, false, false, false>(base, a.m, row, tok, a.m, a.n, value);
        else store_results<NTT, NRT, TSTEP, RSTEP, false, true, false>(base, a.m, row, tok, a.m, a.n, value);
    } else if (a.y_row_major) {
        if (a.accumulate && inside) store_results<NTT, NRT, TSTEP, RSTEP, true, false, true>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else if (a.accumulate) store_results<NTT, NRT, TSTEP, RSTEP, true, true, true>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else if (inside) store_results<NTT, NRT, TSTEP, RSTEP, true, false, false>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else store_results<NTT, NRT, TSTEP, RSTEP, true, true, false>(a.y, a.y_stride, row, tok, a.m, a.n, value);
    } else {
        if (a.accumulate && inside) store_results<NTT, NRT, TSTEP, RSTEP, false, false, true>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else if (a.accumulate) store_results<NTT, NRT, TSTEP, RSTEP, false, true, true>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else if (inside) store_results<NTT, NRT, TSTEP, RSTEP, false, false, false>(a.y, a.y_stride, row, tok, a.m, a.n, value);
        else store_results<NTT, NRT, TSTEP, RSTEP, false, true, false>(a.y, a.y_stride, row, tok, a.m, a.n, value);
    }
}

template <int TYPE, bool DUMP>
__global__ __launch_bounds__(THREADS, 4) void gemm_mfma_kernel(GemmArgs a) {
    __shared__ Smem sm;
    uint32_t row_tile, tok_tile;
    bool valid_tile;
    // K split (plain single-weight launches only): workgroup (tile, share) walks the stages [first, first + stages) of its tile
    const uint32_t ksplit = DUMP || a.ksplit < 2 ? 1u : a.ksplit;
    const uint32_t split = ksplit > 1 ? blockIdx.x % ksplit : 0u;
    tile_of_block(ksplit > 1 ? blockIdx.x / ksplit : blockIdx.x, a.row_tiles, a.tok_tiles, row_tile, tok_tile, valid_tile);
    if (!valid_tile) return;  // whole workgroup leaves together
    select_weight(a, row_tile);
    const uint32_t row0 = row_tile * BM;
    const uint32_t tok0 = tok_tile * BN;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t l16 = lane & 15u;
    const uint32_t kq = lane >> 4;            // which 8-byte quarter of the block this lane feeds
    const uint32_t wrow0 = (wave >> 2) * 64;  // wave's rows within the tile
    const uint32_t wtok0 = (wave & 3u) * 32;  // wave's tokens within the tile
    const uint32_t nb = a.k >> 5;
    const uint32_t all_stages = nb / KB;
    const uint32_t first = split * all_stages / ksplit;  // shares differ by at most one stage, none is empty
    const uint32_t stages = (split + 1u) * all_stages / ksplit - first;

    float acc[TT][RT][4];
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[tt][rt][r] = 0.0f;

    v4i cbias = {(int)kBiasBits, (int)kBiasBits, (int)kBiasBits, (int)kBiasBits};
    asm volatile("" : "+v"(cbias));  // keep it in registers (left alone, the compiler rebuilds it before every MFMA)

    StageRegs regs;
    StagePtrs<BN> ptrs;
    init_stage_ptrs<BN>(a, row_tile, tok0, first * KB, ptrs);
    dma_stage(ptrs, sm.st[0]);
    load_stage(ptrs, regs);
    store_stage(sm.st[0], regs);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's direct-to-LDS copies have landed
    __syncthreads();

    // This lane's LDS read addresses: block 0 of buffer 0 here, moved from block to block by next_block and from one buffer to
    // the other at the end of every stage (four additions instead of rebuilding them).
    LaneAddr la;
    {
        const Stage& s = sm.st[0];
        // this lane's token row; K-chunk 2*block + (kq >> 1) sits at position chunk ^ swizzle
        la.xsh = xt_swizzle(wtok0 + l16) >> 1;
        la.xbase = lds_addr(&s.xt[wtok0 + l16][0]) + ((((kq >> 1) ^ xt_swizzle(wtok0 + l16)) & 1u) << 4) + 8 * (kq & 1u);
        la.xt = la.xbase + (la.xsh << 5);
        la.wt = lds_addr(&s.wt[wrow0 / GR][kq >> 1][0][l16]) + 8 * (kq & 1u);  // the wave's 64 rows are two granules
        la.dws = lds_addr(&s.dws[wrow0 / GR][0][l16]);
        la.dxf = lds_addr(&s.dxf[0][wtok0 + 4 * kq]);
    }

    for (uint32_t st = 0; st < stages; st++) {
        if (st + 1 < stages) {
            // the other LDS stage was last read in stage st-1 and every wave has passed the
            // barrier that ended it, so it can be refilled from here on
            dma_stage(ptrs, sm.st[(st + 1) & 1u]);
            load_stage(ptrs, regs);
        }

        // 8 MFMA tiles per block, software-pipelined by hand: four result buffers, the matrix
        // core runs up to four tiles ahead of the vector ALU, and every operand register is
        // refilled from LDS (for block b+1) as soon as its last use in block b has been
        // issued, so LDS latency stays out of the wave's dependency chain.  The scheduling
        // barriers pin that order; the block loop stays rolled.
        // Tile order: t = 4 * token tile + row tile.
        Mats mt;
        Scales sc;
        load_mats(la, mt);              // 6 reads
        load_tok_scales<0>(la, sc);     // 1
        load_tok_scales<1>(la, sc);     // 1
        load_row_scales(la, sc);        // 4
#pragma unroll 1
        for (int b = 0; b < KB; b++) {
            next_block(la, (uint32_t)b, b + 1 < KB);  // last iteration: harmless re-read of its own block
            const uint32_t row = row0 + wrow0 + l16, tok = tok0 + wtok0 + 4 * kq, blk = (first + st) * KB + b;
            v4i d[4];
            lds_wait<6>(mt);  // the six reads issued after the matrices may still be in flight
#pragma unroll
            for (int t = 0; t < 4; t++) d[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(mt.av[0], mt.bv[t], cbias, 0, 0, 0);
            lds_wait<0>(sc);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int tt = t >> 2, rt = t & 3;
                if constexpr (DUMP) dump_tile<TYPE>(a, d[t & 3], row + 16 * rt, tok + 16 * tt, nb, blk);
                else scale_tile(d[t & 3], sc.dw[rt], sc.dx[tt], acc[tt][rt]);
                __builtin_amdgcn_sched_barrier(0);
                if (t < 4) {
                    d[t & 3] = __builtin_amdgcn_mfma_i32_16x16x32_i8(mt.av[1], mt.bv[t], cbias, 0, 0, 0);
                    if (t == 3) {
                        load_mats(la, mt);           // all eight MFMAs of this block have been issued
                        load_tok_scales<0>(la, sc);  // token tile 0 is done
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            load_tok_scales<1>(la, sc);
            load_row_scales(la, sc);
        }
        lds_wait<0>(sc);  // nothing of this stage's buffer is read past this point
        {   // block 0 of the other buffer (the block loop left wt / dws / dxf at block KB - 1)
            const uint32_t other = (st & 1u) ? 0u - (uint32_t)sizeof(Stage) : (uint32_t)sizeof(Stage);
            la.xbase += other;
            la.xt = la.xbase + (la.xsh << 5);
            la.wt += other - (KB - 1) * kOffWt;
            la.dws += other - (KB - 1) * kOffDws;
            la.dxf += other - (KB - 1) * kOffDxf;
        }

        // The other buffer was last read in stage st-1; every wave has passed the barrier
        // that ended that stage, so it is free to be refilled now.
        if (st + 1 < stages) store_stage(sm.st[(st + 1) & 1u], regs);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // direct-to-LDS copies of the next stage have landed
        __syncthreads();
    }

    if constexpr (!DUMP) {
        store_wave_tile<TT, RT>(a, ksplit, split, row0 + wrow0 + l16, tok0 + wtok0 + 4 * kq,
                                [&](int tt, int rt, int r) { return acc[tt][rt][r]; });
    }
}

// ---------------------------------------------------------------------------------------
// The tiles of a prompt: T32<RT, TT, WR, WT, SB, ..> = WR x WT waves, each RT granules of 32 weight rows x TT groups of 32 tokens, on
// v_mfma_i32_32x32x32_i8, SB blocks of K per stage.  Layout of a 32x32 result: lane l holds weight row n = l % 32 of its granule and
// the 16 tokens m = 8 g + 4 (l / 32) + r, g = 0..3, r = 0..3 -- one row-scale pair per granule and 16 token scales per token group.
//
// What bounds it: a SIMD runs its matrix instructions and its scaling FMAs one after the other (32 FMAs + one MFMA per 32 x 32 block
// result, ~124 cycles together), and every operand comes through the CU's one LDS.  A wave of 64 rows x 32 tokens reads 128 bytes per
// lane for 64 FMAs, which with four such waves per SIMD keeps the LDS as busy as the SIMDs; 128 rows x 64 tokens reads 256 bytes for
// 256 FMAs, half as much per FMA, and needs 2 waves per SIMD instead of 4.  The block loop alone, fed from LDS: 1217 TOP/s for 64 x 32
// with four waves per SIMD, 1250 for 64 x 64 and 1346 for 128 x 64 with two.
//
// TWO result buffers: the MFMA of tile t + 1 is issued before the FMAs of tile t, so that one wave alone keeps its SIMD busy (the other
// wave may be waiting at its stage's barrier).  Every operand register is refilled from LDS for the next block as soon as its last use
// has been issued; all LDS addresses are immediates on four lane bases (the stage loop is written out for both buffers), so the block
// loop holds FMAs, MFMAs, LDS reads and waits only.
typedef int v16i __attribute__((ext_vector_type(16)));

// WAVES: per SIMD, what the registers have to leave room for.  SCALE_FIRST: a result's 16 FMAs with the row scale go out ahead of its 16
// with the token scales, in the result's registers, so that no FMA waits for the one before it: with two waves per SIMD the register-only
// block loop runs at 1.52 instead of 1.32 POP/s (1.60 either way with four); smaller tiles have not the registers for it.  COPIED_SCALES: how a
// slab's token scales get into LDS, see load_dx.
template <int RT_, int TT_, int WR_, int WT_, int SB_, int WAVES, bool SCALE_FIRST = false, bool COPIED_SCALES = false>
struct T32 {
    static constexpr int RT = RT_, TT = TT_, WR = WR_, WT = WT_, SB = SB_, kOcc = WAVES;
    static constexpr bool kScaleFirst = SCALE_FIRST, kCopiedScales = COPIED_SCALES;
    static constexpr int kWaves = WR * WT, kThreads = 64 * kWaves;
    static constexpr int kGranules = WR * RT, kRows = GR * kGranules, kTokens = 32 * WT * TT;
    static constexpr int kTiles = RT * TT;  // 32 x 32 results per wave and block
    static_assert(kGranules % 2 == 0 && (SB == 2 || SB == 4) && (kTiles == 1 || (RT >= 2 && kTiles % 2 == 0)), "pairs of granules, half a slab or a slab per stage, alternating result buffers");
    // One stage in LDS.  xt: [token][2 SB chunks of 16 bytes], swizzled so that consecutive tokens reading one chunk spread over all
    // banks: position p of token t holds chunk p ^ swizzle(t).
    struct Stage {
        uint4 wt[kGranules][2][SB][GR];  // [granule][khalf][block][row]
        float2 dws[kGranules][SB][GR];
        uint4 xt[kTokens][2 * SB];
    };
    struct Smem {
        Stage st[2];
        float dxf[2][KB][kTokens];  // token scales of a slab (4 blocks), two slabs
    };
    static __device__ __forceinline__ uint32_t swizzle(uint32_t t) { return SB == 4 ? (t >> 1) & 7u : (t >> 2) & 3u; }
};

template <int I>
struct Idx {
    static constexpr int value = I;
};
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(Idx<I>{});
        static_for<N, I + 1>(f);
    }
}

template <int OFF>
__device__ __forceinline__ void lds_read16(uint32_t addr, v4i& dst) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read4(uint32_t addr, float& dst) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
// At most N LDS reads outstanding; ties what becomes valid with it.
template <int N, typename V>
__device__ __forceinline__ void lds_arrived(V& v) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(N) : "memory");
}
template <typename V>
__device__ __forceinline__ void tie(V& v) {
    asm volatile("" : "+v"(v));
}

// (DUMP, the parity hook: all registers that there are, which it would otherwise take from scratch, up to 840 bytes a lane.)
// The leading scalars repeat fields of `a` (preloaded into scalar registers at wave launch, see gemm_few_kernel): what the first copies need.
template <int TYPE, bool DUMP, bool GATED, typename C>
__global__ __launch_bounds__(C::kThreads, DUMP ? 1 : C::kOcc) void gemm_tile_kernel(Address p_w, Address p_xq, Address p_xs, Address p_w_up, uint32_t p_m,
                                                                                   uint32_t p_n, uint32_t p_k, uint32_t p_row_tiles, uint32_t p_tok_tiles, uint32_t p_flags, GemmArgs a) {
    a.w = in_global<const uint8_t>(p_w), a.xq = in_global<const int8_t>(p_xq), a.xs = in_global<const float>(p_xs), a.w_up = in_global<const uint8_t>(p_w_up);
    a.m = p_m, a.n = p_n, a.k = p_k, a.row_tiles = p_row_tiles, a.tok_tiles = p_tok_tiles;
    constexpr int RT = C::RT, TT = C::TT, SB = C::SB, T = C::kTiles;
    __shared__ __align__(16) typename C::Smem sm;
    uint32_t row_tile, tok_tile;
    bool valid_tile;
    // K split (plain single-weight launches only): workgroup (tile, share) walks the slabs [first, first + slabs) of its tile
    const uint32_t shift = DUMP || GATED ? 0u : p_flags & 31u, ksplit = 1u << shift, split = blockIdx.x & (ksplit - 1u);
    tile_of_block(blockIdx.x >> shift, a.row_tiles, a.tok_tiles, row_tile, tok_tile, valid_tile);
    if (!valid_tile) return;  // whole workgroup leaves together
    if (!GATED && (p_flags & kMoreWeights)) select_weight(a, row_tile);
    const uint32_t row0 = row_tile * (GATED ? C::kRows / 2 : C::kRows);
    const uint32_t tok0 = tok_tile * C::kTokens;
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, kh = lane >> 5;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t wr = wave / C::WT, wt = wave % C::WT;
    const uint32_t nb = a.k >> 5, all_slabs = nb / KB;
    const uint32_t first = split * all_slabs >> shift;  // shares differ by at most one slab, none is empty
    const uint32_t slabs = ((split + 1u) * all_slabs >> shift) - first;

    // ---- the stage's copies: global -> LDS directly, 1 KB per wave instruction, uniform bases that move one stage on per copy round ----
    constexpr int kPairs = C::kGranules / 2, kXChunks = C::kTokens * 2 * SB / 64;
    constexpr int kPairWaves = kPairs < C::kWaves ? kPairs : C::kWaves;  // waves that copy weights (the others: activations only)
    constexpr int kPairsPer = kPairs / kPairWaves;
    constexpr int kXPer = kXChunks / C::kWaves;
    static_assert(kXChunks % C::kWaves == 0 && kPairs % kPairWaves == 0, "copies deal out evenly");
    const uint32_t pairs_total = (a.m + 2 * GR - 1) / (2 * GR);
    const uint8_t* wsrc[kPairsPer];
#pragma unroll
    for (int i = 0; i < kPairsPer; i++) {
        const uint32_t lp = min(wave, (uint32_t)kPairWaves - 1u) * kPairsPer + i;
        // the tile's pair lp: rows 64 lp ..; a gated tile: its pairs of gate, then the same ones of up
        const bool up = GATED && lp >= kPairs / 2;
        const uint32_t p = GATED ? row_tile * (kPairs / 2) + lp - (up ? kPairs / 2 : 0) : row_tile * kPairs + lp;
        const uint8_t* w = up ? a.w_up : a.w;
        wsrc[i] = w + ((size_t)min(p, pairs_total - 1u) * all_slabs + first) * (2 * kSlab);  // past the end: any rows, never stored
    }
    uint32_t woff = 16u * lane;                                               // this lane's 16 bytes of a kilobyte of operand rows
    uint32_t soff = SB == 4 ? 16u * lane : 16u * l32 + (uint32_t)kSlab * kh;  // ... of a kilobyte of scale pairs (SB = 2: 512 B of either granule)
    uint32_t xoff[kXPer];
#pragma unroll
    for (int j = 0; j < kXPer; j++) {
        const uint32_t tt = (64u / (2 * SB)) * (kXPer * wave + j) + lane / (2 * SB);  // token within the tile
        const uint32_t chunk = (lane % (2 * SB)) ^ C::swizzle(tt);
        xoff[j] = min(tt, a.n - 1u - tok0) * a.k + 16u * chunk;
    }
    const int8_t* xsrc = a.xq + (size_t)tok0 * a.k + (size_t)first * (KB * 32);
    auto copy_lds = [](const void* g, void* l) {
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)g, (void __attribute__((address_space(3)))*)l, 16, 0, 0);
    };
    // stage h (SB = 2: half a slab, SB = 4: a slab) into its buffer; then the bases move on
    auto copy_stage = [&](uint32_t h_) {
        typename C::Stage& s = sm.st[h_ & 1u];
        const uint32_t half = SB == 2 ? h_ & 1u : 0u;
        tie(woff), tie(soff);  // (opaque, or the compiler keeps a 64-bit address per copy in registers)
        if (wave < (uint32_t)kPairWaves) {
#pragma unroll
            for (int i = 0; i < kPairsPer; i++) {
                const uint32_t lp = wave * kPairsPer + i;
#pragma unroll
                for (int g = 0; g < 2; g++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int c = 0; c < SB / 2; c++)
                            copy_lds(wsrc[i] + (g * kSlab + h * 2048 + (SB == 2 ? half * 1024 : c * 1024)) + woff,
                                     reinterpret_cast<uint8_t*>(&s.wt[2 * lp + g][h][0][0]) + 1024 * c);
                if constexpr (SB == 2) copy_lds(wsrc[i] + (kSlabWt + half * 512) + soff, &s.dws[2 * lp][0][0]);
                else {
                    copy_lds(wsrc[i] + kSlabWt + soff, &s.dws[2 * lp][0][0]);
                    copy_lds(wsrc[i] + kSlab + kSlabWt + soff, &s.dws[2 * lp + 1][0][0]);
                }
                wsrc[i] += SB == 4 || half == 1 ? 2 * kSlab : 0;
            }
        }
#pragma unroll
        for (int j = 0; j < kXPer; j++) tie(xoff[j]), copy_lds(xsrc + xoff[j], reinterpret_cast<uint8_t*>(&s.xt[0][0]) + 1024u * (kXPer * wave + j));
        xsrc += SB * 32;
    };
    // Token scales of a slab (token-major in memory), into block-major LDS with neighbours swapped (see the FMA that reads them).  Through registers, one
    // float4 per token, threads 0 .. kTokens - 1, stored when the stage before the slab is done; or (copied) global -> LDS like the operands, a
    // block's 64 tokens per wave: no registers, but a cache line per lane and block instead of per lane and slab.  TileQ, whose registers do
    // not hold the float4 (the compiler parked it in scratch, and its waves waited for memory ahead of the next stage's copies), gains by the
    // copies what the others lose: gated 4608 x 1024 over 555 tokens 26.0 -> 23.9 us, 3072 x 1024 over 2048 25.7 -> 23.7; TileX 62.7 -> 63.6
    // (gated 4608 x 1024 over 2048), TileN 24.6 -> 26.0 and TileH 25.9 -> 26.6 (3072 x 1024 over 2048).
    constexpr bool kCopied = C::kCopiedScales;
    static_assert(kCopied ? KB * C::kTokens == C::kThreads && T > 1 : C::kTokens <= C::kThreads, "a block of 64 tokens per wave, or a thread per token");
    const bool has_dx = (kCopied || threadIdx.x < (uint32_t)C::kTokens) && a.xs;  // xs is null only for the parity hook, which never scales
    const uint8_t* dxsrc = reinterpret_cast<const uint8_t*>(a.xs + (size_t)tok0 * nb + (size_t)first * KB);
    uint32_t dxoff = (min(kCopied ? lane ^ 1u : threadIdx.x, a.n - 1u - tok0) * nb + (kCopied ? wave : 0u)) * (uint32_t)sizeof(float);
    [[maybe_unused]] float4 dxr = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load_dx = [&]([[maybe_unused]] uint32_t buf) {
        tie(dxoff);
        if (has_dx) {
            if constexpr (kCopied)
                __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(dxsrc + dxoff),
                                                 (void __attribute__((address_space(3)))*)&sm.dxf[buf][wave][0], 4, 0, 0);
            else dxr = *reinterpret_cast<const float4*>(dxsrc + dxoff);
        }
        dxsrc += KB * sizeof(float);
    };
    auto store_dx = [&]([[maybe_unused]] uint32_t buf) {
        if constexpr (!kCopied) {
            if (threadIdx.x < (uint32_t)C::kTokens) {
                const uint32_t at = T == 1 ? threadIdx.x : threadIdx.x ^ 1u;
                sm.dxf[buf][0][at] = dxr.x;
                sm.dxf[buf][1][at] = dxr.y;
                sm.dxf[buf][2][at] = dxr.z;
                sm.dxf[buf][3][at] = dxr.w;
            }
        }
    };

    v16f acc[RT][TT];  // [granule][token group]: elements 4 g + r
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < TT; j++) acc[i][j] = v16f{};
    v16i cbias;
#pragma unroll
    for (int i = 0; i < 16; i++) cbias[i] = (int)kBiasBits;
    asm volatile("" : "+v"(cbias));  // keep it in registers (left alone, the compiler rebuilds it before every MFMA)

    // This lane's LDS bases; everything else of an address is an immediate.
    // (granule rt of a wave: its RT consecutive ones of the tile, or its RT / 2 of gate and the same RT / 2 of up; RT == 1: one of either)
    constexpr int kOwn = GATED && RT > 1 ? RT / 2 : RT;
    uint32_t a_wt = lds_addr(&sm.st[0].wt[kOwn * wr][kh][0][l32]);
    uint32_t a_dws = lds_addr(&sm.st[0].dws[kOwn * wr][0][l32]);
    // token scales: the first of the lane's four groups of four, or (T == 1) the lane of every 16 that holds the scale of their result e reads
    // that one, 8 (e / 4) + 4 kh + e % 4
    uint32_t a_dxf = lds_addr(&sm.dxf[0][0][32 * TT * wt + 4 * kh + (T == 1 ? 8 * ((lane & 15u) >> 2) + (lane & 3u) : 0u)]);
    uint32_t a_xt[SB];  // chunk 2 b + kh of this lane's token sits at position chunk ^ swizzle
#pragma unroll
    for (int b = 0; b < SB; b++) a_xt[b] = lds_addr(&sm.st[0].xt[32 * TT * wt + l32][(2u * b + kh) ^ C::swizzle(l32)]);
    constexpr uint32_t kBuf = sizeof(typename C::Stage);

    constexpr auto granule = [](int rt) { return rt < kOwn ? rt : C::kGranules / 2 + rt - kOwn; };
    // LDS reads of block b of the stage
    auto read_ab = [&](auto b, v4i (&A)[TT], v4i (&B)[RT]) {  // TT + RT reads
        static_for<TT>([&](auto t) { lds_read16<32 * decltype(t)::value * 32 * SB>(a_xt[decltype(b)::value], A[decltype(t)::value]); });
        static_for<RT>([&](auto r) { lds_read16<1024 * SB * granule(decltype(r)::value) + 512 * decltype(b)::value>(a_wt, B[decltype(r)::value]); });
    };
    auto read_dw = [&](auto b, auto r, float2& dw) { lds_read8<256 * SB * granule(decltype(r)::value) + 256 * decltype(b)::value>(a_dws, dw); };
    [[maybe_unused]] auto read_dx = [&](auto b, auto t, auto g, v4f& dx) {
        lds_read16<decltype(b)::value * 4 * C::kTokens + 128 * decltype(t)::value + 32 * decltype(g)::value>(a_dxf, dx);
    };
    // (parity checks) dot of element e of one result
    [[maybe_unused]] auto dump = [&](int d, uint32_t rt, uint32_t tt, uint32_t e, uint32_t blk) {
        const uint32_t row = row0 + GR * (RT * wr + rt) + l32, tok = tok0 + 32 * (TT * wt + tt) + 4 * kh + 8 * (e >> 2) + (e & 3u);
        if (row < a.m && tok < a.n) {
            const int v = d - (int)kBiasBits;
            a.dots[((size_t)tok * a.m + row) * nb + blk] = TYPE == 2 ? v >> 4 : v;  // (type 2: weights were stored x16; exact)
        }
    };

    // One stage: SB blocks, the first of them block blk0 of the row.
    auto compute_stage = [&](uint32_t blk0) {
        v16i D[2];
        if constexpr (T == 1) {
            // One result per wave and block: the operands are read two blocks ahead, the next block's MFMA goes out before this one's FMAs. A
            // small tile is bound by what it reads from the LDS, 104 bytes per lane and block, 64 of them token scales, which every lane reads
            // alike: here each lane reads the scale of one of its row's sixteen tokens, 4 bytes, and the FMAs take it from there.
            v4i A[2][1], B[2][1];
            float2 dw[2];
            float xs[2];
            const auto read_scales = [&](auto b) {
                constexpr int at = decltype(b)::value;
                read_dw(b, Idx<0>{}, dw[at & 1]);
                lds_read4<at * 4 * C::kTokens>(a_dxf, xs[at & 1]);
            };
            read_ab(Idx<0>{}, A[0], B[0]), read_scales(Idx<0>{});
            read_ab(Idx<1>{}, A[1], B[1]), read_scales(Idx<1>{});
            lds_arrived<6>(A[0][0]), tie(B[0][0]);
            D[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[0][0], B[0][0], cbias, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            static_for<SB>([&](auto b_) {
                constexpr int b = decltype(b_)::value, at = b & 1, ahead = b + 2 < SB ? b + 2 : 0;
                // requested and not waited for yet, in order: scales of b (b == 0), operands of b + 1, scales of b + 1; (b > 0) scales of b first
                if constexpr (b + 1 < SB) {
                    lds_arrived<2>(A[at ^ 1][0]), tie(B[at ^ 1][0]), tie(dw[at]), tie(xs[at]);
                    D[at ^ 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[at ^ 1][0], B[at ^ 1][0], cbias, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    lds_arrived<0>(dw[at]), tie(xs[at]);
                }
                if constexpr (b + 2 < SB) read_ab(Idx<ahead>{}, A[at], B[at]);
                v16i& d = D[at];
                if constexpr (DUMP) {
#pragma unroll
                    for (int e = 0; e < 16; e++) dump(d[e], 0, 0, e, blk0 + b);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; e++) d[e] = __float_as_int(__builtin_fmaf(__int_as_float(d[e]), dw[at].x, dw[at].y));
                    __builtin_amdgcn_sched_barrier(0);
                    fmac_row_lanes(acc[0][0], xs[at], __builtin_bit_cast(v16f, d));
                    tie(acc[0][0]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (b + 2 < SB) read_scales(Idx<ahead>{});
            });
        } else {
            v4i A[TT], B[RT];
            float2 dw[RT];
            v4f dx[4];
            read_ab(Idx<0>{}, A, B);
            static_for<RT - 1>([&](auto r) { read_dw(Idx<0>{}, r, dw[decltype(r)::value]); });
            static_for<4>([&](auto g) { read_dx(Idx<0>{}, Idx<0>{}, g, dx[decltype(g)::value]); });
            read_dw(Idx<0>{}, Idx<RT - 1>{}, dw[RT - 1]);
            // (the reads behind the operands' may still be in flight)
            lds_arrived<RT + 4>(A[0]);
            static_for<TT>([&](auto t) { tie(A[decltype(t)::value]); });
            static_for<RT>([&](auto r) { tie(B[decltype(r)::value]); });
            D[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[0], B[0], cbias, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            static_for<SB>([&](auto b_) {
                constexpr int b = decltype(b_)::value;
                constexpr bool next = b + 1 < SB;
                static_for<T>([&](auto t_) {
                    constexpr int t = decltype(t_)::value, tt = t / RT, rt = t % RT;
                    if constexpr (t + 1 < T) {
                        constexpr int tt1 = (t + 1) / RT, rt1 = (t + 1) % RT;
                        D[(t + 1) & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[tt1], B[rt1], cbias, 0, 0, 0);
                    } else if constexpr (next) {
                        lds_arrived<1>(A[0]);  // all operands of the next block; its scale pair of granule RT - 2 may still be on its way
                        static_for<TT>([&](auto i) { tie(A[decltype(i)::value]); });
                        static_for<RT>([&](auto i) { tie(B[decltype(i)::value]); });
                        D[(t + 1) & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[0], B[0], cbias, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    constexpr bool fetch = next && t == T - 2;  // all MFMAs of this block have been issued
                    if constexpr (fetch) read_ab(Idx<next ? b + 1 : 0>{}, A, B);
                    constexpr int kFetched = fetch ? TT + RT : 0;  // reads that a wait below may leave outstanding on top
                    if constexpr (rt == RT - 1 && tt == 0) lds_arrived<kFetched + (TT == 1 && next ? 1 : 0)>(dw[rt]);
                    if constexpr (!DUMP && C::kScaleFirst) {
                        if constexpr (rt == 0 && tt == 0) {
                            lds_arrived<5 + kFetched>(dw[0]);  // (behind them: the token scales and the last granule's pair)
                            static_for<RT - 1>([&](auto i) { tie(dw[decltype(i)::value]); });
                        }
#pragma unroll
                        for (int e = 0; e < 16; e++) D[t & 1][e] = __float_as_int(__builtin_fmaf(__int_as_float(D[t & 1][e]), dw[rt].x, dw[rt].y));
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    static_for<4>([&](auto g_) {
                        constexpr int g = decltype(g_)::value;
                        if constexpr (rt == 0) {
                            lds_arrived<(tt == 0 ? 4 : 3) - g + kFetched>(dx[g]);
                            if constexpr (!(!DUMP && C::kScaleFirst) && g == 0 && tt == 0) static_for<RT - 1>([&](auto i) { tie(dw[decltype(i)::value]); });
                        }
                        if constexpr (DUMP) {
#pragma unroll
                            for (int r = 0; r < 4; r++) dump(D[t & 1][4 * g + r], rt, tt, 4 * g + r, blk0 + b);
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                float v = __int_as_float(D[t & 1][4 * g + r]);
                                if constexpr (!C::kScaleFirst) v = __builtin_fmaf(v, dw[rt].x, dw[rt].y);
                                acc[rt][tt][4 * g + r] = __builtin_fmaf(v, dx[g][r ^ 1], acc[rt][tt][4 * g + r]);
                            }
                            // (without this the compiler lets the MFMAs of all tiles run ahead of their FMAs, and spills)
                            if constexpr (!C::kScaleFirst || g == 3) tie(acc[rt][tt]);
                        }
                        // this group's token scales are done with: the next token group's, or the next block's first
                        if constexpr (rt == RT - 1) {
                            if constexpr (tt + 1 < TT) read_dx(Idx<b>{}, Idx<tt + 1 < TT ? tt + 1 : 0>{}, g_, dx[g]);
                            else if constexpr (next) read_dx(Idx<next ? b + 1 : b>{}, Idx<0>{}, g_, dx[g]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    if constexpr (tt == TT - 1 && next) read_dw(Idx<next ? b + 1 : 0>{}, Idx<rt>{}, dw[rt]);
                });
            });
        }
    };
    // The stage's reads are all done (nothing is outstanding past its last wait) and the next stage's copies have landed.
    auto end_stage = [] {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    constexpr uint32_t HS = KB / SB;  // stages per slab
    const uint32_t stages = slabs * HS;
    load_dx(0);
    copy_stage(0);
    store_dx(0);
    end_stage();
    for (uint32_t h = 0; h < stages; h++) {
        const uint32_t h1 = h + 1;
        const bool more = h1 < stages, new_slab = more && h1 % HS == 0;
        if (new_slab) load_dx((h1 / HS) & 1u);
        if (more) copy_stage(h1);
        compute_stage((first * HS + h) * SB);
        const uint32_t other = h & 1u ? 0u - kBuf : kBuf;  // to the other buffer
        a_wt += other, a_dws += other;
#pragma unroll
        for (int b = 0; b < SB; b++) a_xt[b] += other;
        // token scales: blocks 0 .. 7 of the two slabs of dxf, then from the start
        a_dxf += (h1 % (2 * HS) == 0 ? 0u - (2 * HS - 1) * SB : (uint32_t)SB) * (uint32_t)(sizeof(float) * C::kTokens);
        if (new_slab) store_dx((h1 / HS) & 1u);
        end_stage();
    }

    if constexpr (GATED && RT == 1) {
        // The same as below where a wave has a granule of gate or of up: it takes sixteen tokens of both, hands the other wave the other sixteen and
        // quantizes its own.
        constexpr int kRow = 36;
        static_assert(C::WR == 4 && TT == 1 && sizeof(sm) >= sizeof(float) * (8 * 64 + 16 * kRow) * C::kWaves, "gate waves, then up waves");
        float* const ex = reinterpret_cast<float*>(&sm);  // [wave][8][lane]
        float* const h = ex + 8 * 64 * C::kWaves + 16 * kRow * wave;
        const bool up = wr >= 2u;
#pragma unroll
        for (int e = 0; e < 8; e++) ex[64 * (8 * wave + e) + lane] = up ? acc[0][0][e] : acc[0][0][8 + e];
        __syncthreads();
        float g[8], u[8], v[8], far = 0.0f, small = 1.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float its = ex[64 * (8 * (wave ^ (2u * C::WT)) + e) + lane];
            g[e] = up ? its : acc[0][0][e], u[e] = up ? acc[0][0][8 + e] : its;
            v[e] = silu_mul_near(g[e], u[e], far, small);
        }
        if (__builtin_amdgcn_ballot_w64(!silu_mul_was_near(far, small)) != 0) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = silu_mul(g[e], u[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) h[kRow * (4 * kh + 8 * (e >> 2) + (e & 3)) + l32] = v[e];
        const uint32_t rbase = row0 + 32u * (wr & 1u), tok = tok0 + 32 * wt + (up ? 16u : 0u) + (lane >> 3), mine = lane & 1u;
        if (rbase < a.m) {
            float4 x[2];
            float amax[2], id;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                x[i] = *reinterpret_cast<const float4*>(&h[kRow * (8u * i + (lane >> 3)) + 4u * (lane & 7u)]);
                amax[i] = group_max8(fmaxf(fmaxf(fabsf(x[i].x), fabsf(x[i].y)), fmaxf(fabsf(x[i].z), fabsf(x[i].w))));
            }
            const float scale = q8_scale_and_inverse(mine ? amax[1] : amax[0], id);
            if ((lane & 7u) < 2u && tok + 8u * mine < a.n) a.s_out[(size_t)(tok + 8u * mine) * (a.m >> 5) + (rbase >> 5)] = scale;
            static_for<2>([&](auto i_) {
                constexpr int i = decltype(i_)::value;
                const float idi = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(id), 0x55 * i, 0xf, 0xf, false));
                const uint32_t packed = q8_pack4(x[i].x, x[i].y, x[i].z, x[i].w, idi);
                if (tok + 8u * i < a.n) *reinterpret_cast<uint32_t*>(a.q_out + (size_t)(tok + 8u * i) * a.m + rbase + 4u * (lane & 7u)) = packed;
            });
        }
    } else if constexpr (GATED) {
        // silu(gate) * up and the Q8_0 quantizer, element for element what silu_mul_quantize_kernel computes from the two float
        // results: granules 0 .. RT / 2 - 1 of the wave are gate rows, the others the same rows of up, 32 rows = one Q8_0 block of a
        // token.  The gated values go through a wave-private piece of LDS (the stages are done with), so that eight lanes own a block
        // with four rows each: one scale per block and eight lanes instead of 32, and 4-byte stores.  It is bound by its instructions: with
        // the shorter silu (silu_mul_near) and a quarter of the scales' divisions per lane, 4608 x 1024 over 555 tokens 24.8 -> 23.0 us,
        // 6912 x 2048 over 2002 155 -> 152.5.
        constexpr int kRow = 36;  // floats per token row: 16-byte aligned, neighbouring tokens on other banks
        static_assert(sizeof(sm) >= sizeof(float) * kRow * 32 * C::kWaves, "a 32 x 32 block of floats per wave");
        float* const h = reinterpret_cast<float*>(&sm) + kRow * 32 * wave;
#pragma unroll
        for (int j = 0; j < kOwn; j++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                float v[16], far = 0.0f, small = 1.0f;
#pragma unroll
                for (int e = 0; e < 16; e++) v[e] = silu_mul_near(acc[j][tt][e], acc[kOwn + j][tt][e], far, small);
                if (__builtin_amdgcn_ballot_w64(!silu_mul_was_near(far, small)) != 0) {  // some lane outside what that takes
#pragma unroll
                    for (int e = 0; e < 16; e++) v[e] = silu_mul(acc[j][tt][e], acc[kOwn + j][tt][e]);
                }
#pragma unroll
                for (int e = 0; e < 16; e++) h[kRow * (4 * kh + 8 * (e >> 2) + (e & 3)) + l32] = v[e];
                const uint32_t rbase = row0 + 32u * (kOwn * wr + j);
                if (rbase < a.m) {  // m % 32 == 0: a block is inside the matrix or not at all
                    // Eight lanes have four tokens' blocks: each lane works out the scale of one of the four and hands its inverse round.
                    float4 x[4];
                    float amax[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        x[i] = *reinterpret_cast<const float4*>(&h[kRow * (8u * i + (lane >> 3)) + 4u * (lane & 7u)]);
                        amax[i] = group_max8(fmaxf(fmaxf(fabsf(x[i].x), fabsf(x[i].y)), fmaxf(fabsf(x[i].z), fabsf(x[i].w))));
                    }
                    const uint32_t mine = lane & 3u, tok = tok0 + 32 * (TT * wt + tt) + (lane >> 3);
                    float id;
                    const float scale = q8_scale_and_inverse(mine < 2u ? (mine == 0u ? amax[0] : amax[1]) : (mine == 2u ? amax[2] : amax[3]), id);
                    if ((lane & 7u) < 4u && tok + 8u * mine < a.n) a.s_out[(size_t)(tok + 8u * mine) * (a.m >> 5) + (rbase >> 5)] = scale;
                    static_for<4>([&](auto i_) {
                        constexpr int i = decltype(i_)::value;
                        const float idi = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(id), 0x55 * i, 0xf, 0xf, false));  // of lane i of the four
                        const uint32_t packed = q8_pack4(x[i].x, x[i].y, x[i].z, x[i].w, idi);
                        if (tok + 8u * i < a.n) *reinterpret_cast<uint32_t*>(a.q_out + (size_t)(tok + 8u * i) * a.m + rbase + 4u * (lane & 7u)) = packed;
                    });
                }
            }
    } else if constexpr (!DUMP) {
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
            store_wave_tile<4, RT, 8, 32>(a, ksplit, split, row0 + GR * RT * wr + l32, tok0 + 32 * (TT * wt + tt) + 4 * kh,
                                          [&](int g, int rt, int r) { return acc[rt][tt][4 * g + r]; });
    }
}

// ---------------------------------------------------------------------------------------
// Narrow variant for launches of up to 48 tokens that gemm_few_kernel does not take (an LM head, or a long K, over a short
// prompt; up to 64 tokens, and few tiles of more, where the 16x16x32 loop is asked for): tile = 128 weight rows x 64 tokens,
// every one of the 8 waves owns 16 rows x all 64 tokens (one row tile x four token tiles), so no matrix or scaling work is
// spent on token columns that do not exist beyond the 64, and the weights -- the only large operand -- are streamed exactly
// once per 64 tokens.  Same staging, LDS layouts and arithmetic as the wide kernel; 60 KB of LDS, two workgroups per CU.  TTN (1 .. 4): how many of the four token tiles the launch has tokens
// for -- a launch of n <= 16 / 32 / 48 tokens reads and multiplies only those (these launches
// are bound by their block loop, so the unused tiles were a third to three quarters of their time).
struct NarrowMats {
    long av[4], bv;
};
struct NarrowScales {
    float2 dw;
    v4f dx[4];
};
constexpr int kOffDxfNarrow = sizeof(float) * BN_NARROW;
// TTN: the token tiles (of 16) the launch has tokens for; the others are neither read nor multiplied.
template <int TTN>
__device__ __forceinline__ void load_mats(const LaneAddr& la, NarrowMats& m) {  // TTN + 1 reads
    lds_read8<0 * 16 * 128>(la.xt, m.av[0]);
    if constexpr (TTN > 1) lds_read8<1 * 16 * 128>(la.xt, m.av[1]);
    if constexpr (TTN > 2) lds_read8<2 * 16 * 128>(la.xt, m.av[2]);
    if constexpr (TTN > 3) lds_read8<3 * 16 * 128>(la.xt, m.av[3]);
    lds_read8<0>(la.wt, m.bv);
}
template <int TTN>
__device__ __forceinline__ void load_scales(const LaneAddr& la, NarrowScales& s) {  // TTN + 1 reads
    lds_read8<0>(la.dws, s.dw);
    lds_read16<0 * 64>(la.dxf, s.dx[0]);
    if constexpr (TTN > 1) lds_read16<1 * 64>(la.dxf, s.dx[1]);
    if constexpr (TTN > 2) lds_read16<2 * 64>(la.dxf, s.dx[2]);
    if constexpr (TTN > 3) lds_read16<3 * 64>(la.dxf, s.dx[3]);
}
template <int N>
__device__ __forceinline__ void lds_wait(NarrowMats& m) {
    asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(m.av[0]), "+v"(m.av[1]), "+v"(m.av[2]), "+v"(m.av[3]), "+v"(m.bv) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void lds_wait(NarrowScales& s) {
    asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(s.dw), "+v"(s.dx[0]), "+v"(s.dx[1]), "+v"(s.dx[2]), "+v"(s.dx[3]) : "n"(N) : "memory");
}

template <int TYPE, bool DUMP, int TTN = 4>
__global__ __launch_bounds__(THREADS, 4) void gemm_narrow_kernel(GemmArgs a) {
    __shared__ SmemT<BN_NARROW> sm;
    uint32_t row_tile, tok_tile;
    bool valid_tile;
    const uint32_t ksplit = DUMP || a.ksplit < 2 ? 1u : a.ksplit;
    const uint32_t split = ksplit > 1 ? blockIdx.x % ksplit : 0u;  // the splits of a tile are neighbours: different XCDs, same time
    tile_of_block(ksplit > 1 ? blockIdx.x / ksplit : blockIdx.x, a.row_tiles, a.tok_tiles, row_tile, tok_tile, valid_tile);
    if (!valid_tile) return;  // whole workgroup leaves together
    select_weight(a, row_tile);
    const uint32_t row0 = row_tile * BM;
    const uint32_t tok0 = tok_tile * BN_NARROW;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t l16 = lane & 15u;
    const uint32_t kq = lane >> 4;      // which 8-byte quarter of the block this lane feeds
    const uint32_t wrow0 = wave * 16;   // wave's rows within the tile
    const uint32_t nb = a.k >> 5;
    // this workgroup's stages: [first, first + stages)
    const uint32_t all_stages = nb / KB;
    // shares differ by at most one stage and none is empty (the host splits only where all_stages >= 2 * ksplit)
    const uint32_t first = split * all_stages / ksplit;
    const uint32_t stages = (split + 1u) * all_stages / ksplit - first;

    float acc[4][4];
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[tt][r] = 0.0f;

    v4i cbias = {(int)kBiasBits, (int)kBiasBits, (int)kBiasBits, (int)kBiasBits};
    asm volatile("" : "+v"(cbias));

    StageRegs regs;
    StagePtrs<BN_NARROW> ptrs;
    init_stage_ptrs<BN_NARROW>(a, row_tile, tok0, first * KB, ptrs);
    dma_stage(ptrs, sm.st[0]);
    load_stage(ptrs, regs);
    store_stage(sm.st[0], regs);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's direct-to-LDS copies have landed
    __syncthreads();

    LaneAddr la;  // block 0 of buffer 0; moved on as in the wide kernel
    {
        const StageT<BN_NARROW>& s = sm.st[0];
        la.xsh = xt_swizzle(l16) >> 1;
        la.xbase = lds_addr(&s.xt[l16][0]) + ((((kq >> 1) ^ xt_swizzle(l16)) & 1u) << 4) + 8 * (kq & 1u);
        la.xt = la.xbase + (la.xsh << 5);
        la.wt = lds_addr(&s.wt[wrow0 / GR][kq >> 1][0][(wrow0 % GR) + l16]) + 8 * (kq & 1u);  // the wave's 16 rows: half a granule
        la.dws = lds_addr(&s.dws[wrow0 / GR][0][(wrow0 % GR) + l16]);
        la.dxf = lds_addr(&s.dxf[0][4 * kq]);
    }

    for (uint32_t st = 0; st < stages; st++) {
        if (st + 1 < stages) {
            dma_stage(ptrs, sm.st[(st + 1) & 1u]);
            load_stage(ptrs, regs);
        }

        NarrowMats mt{};
        NarrowScales sc{};
        load_mats<TTN>(la, mt);    // TTN + 1 reads
        load_scales<TTN>(la, sc);  // TTN + 1 reads
#pragma unroll 1
        for (int b = 0; b < KB; b++) {
            // addresses of block b+1 (last iteration: harmless re-read of its own block)
            const bool adv = b + 1 < KB;
            la.xt = la.xbase + ((((uint32_t)(adv ? b + 1 : b)) ^ la.xsh) << 5);
            la.wt += adv ? kOffWt : 0;
            la.dws += adv ? kOffDws : 0;
            la.dxf += adv ? kOffDxfNarrow : 0;
            const uint32_t row = row0 + wrow0 + l16, tok = tok0 + 4 * kq, blk = (first + st) * KB + b;
            v4i d[TTN];
            lds_wait<TTN + 1>(mt);  // the scale reads issued after the matrices may still be in flight
#pragma unroll
            for (int tt = 0; tt < TTN; tt++) d[tt] = __builtin_amdgcn_mfma_i32_16x16x32_i8(mt.av[tt], mt.bv, cbias, 0, 0, 0);
            load_mats<TTN>(la, mt);  // in place: the MFMAs that read block b's operands have been issued
            lds_wait<TTN + 1>(sc);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int tt = 0; tt < TTN; tt++) {
                if constexpr (DUMP) dump_tile<TYPE>(a, d[tt], row, tok + 16 * tt, nb, blk);
                else scale_tile(d[tt], sc.dw, sc.dx[tt], acc[tt]);
            }
            __builtin_amdgcn_sched_barrier(0);
            load_scales<TTN>(la, sc);
        }
        lds_wait<0>(sc);  // nothing of this stage's buffer is read past this point
        {
            const uint32_t other = (st & 1u) ? 0u - (uint32_t)sizeof(StageT<BN_NARROW>) : (uint32_t)sizeof(StageT<BN_NARROW>);
            la.xbase += other;
            la.xt = la.xbase + (la.xsh << 5);
            la.wt += other - (KB - 1) * kOffWt;
            la.dws += other - (KB - 1) * kOffDws;
            la.dxf += other - (KB - 1) * kOffDxfNarrow;
        }

        if (st + 1 < stages) store_stage(sm.st[(st + 1) & 1u], regs);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // direct-to-LDS copies of the next stage have landed
        __syncthreads();
    }

    if constexpr (!DUMP) {
        store_wave_tile<TTN, 1>(a, ksplit, split, row0 + wrow0 + l16, tok0 + 4 * kq, [&](int tt, int, int r) { return acc[tt][r]; });
    }
}

// ---------------------------------------------------------------------------------------
// Few tokens (a chat turn, the tail of a prompt; up to a few hundred where the rows are few).  Such a launch is one latency after the other.  A workgroup
// takes ONE granule of 32 rows x 32 TG tokens (blockIdx.y: which) of one share of K; a wave multiplies 16 rows x 16 tokens (or two such) with all of K in order, on
// v_mfma_i32_16x16x32_i8, so that nothing is handed from wave to wave and the bits are those of the tiles.  The operands go global -> LDS
// directly, R slabs deep: everything that fits is requested in one go when the launch starts, and a wave waits for a slab, not for memory.
// Where a workgroup has more waves than tiles (32 tokens, eight waves) the other half of them sends the copies.
//
// What bounds it: a launch, a memory round trip, then each tile's chain of a slab (operands out of LDS, MFMA, four multiply-adds by the row
// scale, four by the token scale: ~0.26 us with one wave per SIMD), and how fast the slabs come, 1.25 bytes a weight.  A 16 x 16 tile has four
// results a lane: its token scales are read from LDS once per SLAB, 4 bytes a lane -- lane i of a row of 16 has that of block i / 4 and of
// its row's token i % 4 -- and taken from there by the multiply-adds.  (Before, a wave multiplied slabs of its own on 32 x 32 tiles, left
// isum * dw of every block in LDS, and all threads walked the blocks in order: half a megabyte through the LDS of a CU for gate | up of 1024
// elements.)  Back to back, weights cold, us: 23 tokens 1024 x 1024 in 4 shares 4.0 -> 3.3, 1024 x 4608 in 8 5.4 -> 4.6, 2048 x 6912 in 8 8.0 -> 6.5,
// 9216 x 1024 7.9 -> 6.1; 48 tokens 1024 x 1024 in 4 4.8 -> 3.5, 1024 x 4608 in 8 7.3 -> 5.1; gated 4608 x 1024 over 23 8.7 -> 6.5, 6912 x 2048 14.9 -> 10.4.
// Tried and left: the ring deeper than R (8 slabs: 7.4 -> 8.9, the first slab waits behind the burst), shallower (3: 1 - 3 % faster up to
// 8 slabs of K, 8 % slower at 16); a slab's operands in registers ahead of its turn, or a slab scaled under the next one's reads
// (both 5 - 8 % slower: more code, and code that runs once has to be fetched).
//
// Shares of K (split_k_factor): side by side, a workgroup each, or walked one after the other and added up in the same order as elsewhere, in
// the same workgroup: no scratch and no second launch.
//
// GATED: gate | up over few tokens with the SiLU gate and the down projection's quantizer behind it.  A workgroup takes a granule of gate
// rows and the same one of up, half of the waves each; a granule is one Q8_0 block of every token, so the gated values are exchanged
// through LDS and leave as blocks, element for element what the two projections and silu_mul_quantize_kernel compute.

// sums[e] += x of lane 4 B + e of this lane's row of 16, times v[e].  One piece with its wait: see fmac_row_lanes.
template <int B>
__device__ __forceinline__ void fmac_row_lanes4(v4f& sums, float x, const v4f& v) {
    float s0 = sums[0], s1 = sums[1], s2 = sums[2], s3 = sums[3];
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
        : "+&v"(s0), "+&v"(s1), "+&v"(s2), "+&v"(s3)
        : "v"(x), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "n"(4 * B), "n"(4 * B + 1), "n"(4 * B + 2), "n"(4 * B + 3));
    sums[0] = s0, sums[1] = s1, sums[2] = s2, sums[3] = s3;
}

// The leading scalars repeat fields of `a` (p_more: w_up of a gated launch, else partial), so that the hardware preloads them into scalar registers at wave
// launch (the build asks for that, -amdgpu-kernarg-preload-count): everything that the first copies need is there at the first instruction, and a
// launch of 4 us does not begin with four scalar loads one after the other.  p_flags: log2 of the shares of K; kFewSide: they are side by
// side; kMoreWeights: more weights than one.
// (1024 x 1024 in 4 3.8 -> 3.5 us.)
constexpr uint32_t kFewSide = 256;
template <int TYPE, bool DUMP, bool GATED, int TG, int WV>
__global__ __launch_bounds__(64 * WV, 2) void gemm_few_kernel(Address p_w, Address p_xq, Address p_xs, Address p_more, uint32_t p_n, uint32_t p_k, uint32_t p_row_tiles,
                                                              uint32_t p_flags, GemmArgs a) {
    static_assert(!(GATED && DUMP), "the parity hook runs the plain launch");
    constexpr int MS = GATED ? 2 : 1;                                                   // weights
    constexpr int TILES = MS * 4 * TG, MW = WV < TILES ? WV : TILES, TPW = TILES / MW;  // 16 x 16 tiles, waves that multiply, tiles of each
    constexpr int CW = WV > TILES ? WV - TILES : WV;                                    // waves that copy: the others, or all
    constexpr int kW = MS * kSlabChunks, kX = 4 * TG, kUnits = kW + kX + (DUMP ? 0 : 1), kPer = (kUnits + CW - 1) / CW;
    // A slab's operands in LDS, a kilobyte per copy: the slab of each weight as it is in memory ([khalf][block][row] 16 bytes, [block][row] scale pairs),
    // [token][16-byte chunk, swizzled], [token] {scales of the four blocks}.
    constexpr uint32_t kStage = 1024 * (kW + kX + 1), kAtX = 1024 * kW, kAtDx = kAtX + 1024 * kX;
    constexpr int R = 4;      // of them: more requested at once delay the first
    constexpr int kRow = 36;  // (GATED) floats of a token's 32 gated values: 16-byte aligned, tokens spread over the banks
    static_assert(kStage * R <= 80 * 1024, "two workgroups on a CU");
    static_assert(!GATED || (WV * 8 >= 32 * TG && kStage * R >= sizeof(float) * 2 * 32 * TG * kRow), "eight threads and two rows of LDS per token");
    __shared__ __align__(16) uint8_t sm[R * kStage];
    // shares of K: side by side, a workgroup each, into a.partial; or (no partial) one after the other in this one
    const uint32_t shift = DUMP || GATED ? 0u : p_flags & 31u;
    const bool side = !DUMP && !GATED && (p_flags & kFewSide);
    const uint32_t my_share = side ? blockIdx.x & ((1u << shift) - 1u) : 0u;
    uint32_t granule = side ? blockIdx.x >> shift : blockIdx.x;  // within the launch's weights
    if (granule >= p_row_tiles) return;                          // (grids are rounded up)
    a.w = in_global<const uint8_t>(p_w);
    if (!GATED && (p_flags & kMoreWeights)) select_weight(a, granule);
    const uint32_t lane = threadIdx.x & 63u, l16 = lane & 15u, kq = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nb = p_k >> 5, all_slabs = nb / KB;
    const uint32_t first = side ? my_share * all_slabs >> shift : 0u;  // this workgroup's slabs; shares differ by at most one
    const uint32_t slabs = side ? ((my_share + 1u) * all_slabs >> shift) - first : all_slabs;
    const uint32_t lds = lds_addr(sm);
    const uint32_t tok0 = 32u * TG * blockIdx.y, n_here = p_n - tok0;  // this workgroup's tokens

    // ---- copies: the kilobytes of a stage dealt out over the copying waves, the same number to each (the last one more than once where they do not
    // come out even), so that waiting for a stage is a count of those behind it ----
    const bool copies = CW == WV || wave >= (uint32_t)MW;
    const uint8_t* src[kPer];
    uint32_t off[kPer], step[kPer], dst[kPer];
    if (copies) {
        const uint32_t cw = CW == WV ? wave : wave - MW;
        const uint8_t* const slab0 = a.w + (((size_t)(granule >> 1) * all_slabs + first) * 2 + (granule & 1u)) * kSlab;
        const size_t to_up = GATED ? p_more - p_w - kSlab : 0;
        const uint32_t t = lane >> 3, x0 = 16u * ((lane & 7u) ^ xt_swizzle(t));  // (eight tokens on: four on in the swizzle)
        static_for<kPer>([&](auto j_) {
            constexpr int j = decltype(j_)::value, lo = CW * j, hi = lo + CW - 1;  // the units that this one can be
            const uint32_t u = min(cw + (uint32_t)lo, (uint32_t)kUnits - 1u);
            dst[j] = lds + 1024u * u;
            src[j] = slab0 + 1024u * u + (GATED && u >= (uint32_t)kSlabChunks ? to_up : 0), step[j] = 2 * kSlab, off[j] = 16u * lane;
            if (hi >= kW && (lo >= kW || u >= (uint32_t)kW)) {
                const uint32_t c = u - kW;
                src[j] = in_global<const uint8_t>(p_xq) + (size_t)tok0 * p_k + first * (32u * KB), step[j] = 32 * KB;
                off[j] = min(8u * c + t, n_here - 1u) * p_k + (x0 ^ (64u * (c & 1u)));
            }
            if (!DUMP && hi >= kW + kX && u >= (uint32_t)(kW + kX)) {
                src[j] = in_global<const uint8_t>(p_xs) + ((size_t)tok0 * nb + first * KB) * sizeof(float), step[j] = KB * sizeof(float);
                off[j] = min(lane, n_here - 1u) * nb * (uint32_t)sizeof(float);
            }
            const uint64_t p = reinterpret_cast<uint64_t>(src[j]);  // (said again that it is the same for the wave: the compiler puts it in vector registers otherwise)
            src[j] = reinterpret_cast<const uint8_t*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)p) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32);
            step[j] = (uint32_t)__builtin_amdgcn_readfirstlane((int)step[j]);
        });
    }
    uint32_t at = 0;  // of the stage that is written
    const auto copy_stage = [&] {
#pragma unroll
        for (int j = 0; j < kPer; j++) {
            tie(off[j]);
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(src[j] + off[j]),
                                             (void __attribute__((address_space(3)))*)(dst[j] + at), 16, 0, 0);
            src[j] += step[j];
        }
        at = at == (R - 1) * kStage ? 0u : at + kStage;
    };
    if (copies)
        for (uint32_t s = 0; s < R - 1u && s < slabs; s++) copy_stage();

    // ---- this wave's tiles: 16 rows, TPW groups of 16 tokens ----
    const uint32_t half = wave & 1u, mat = GATED ? (wave >> 1) & 1u : 0u, tg0 = (GATED ? wave >> 2 : wave >> 1) * TPW;
    const bool multiplies = wave < (uint32_t)MW && 16u * tg0 < n_here;
    uint32_t a_wt = lds + kSlab * mat + 2048u * (kq >> 1) + 16u * (16 * half + l16) + 8u * (kq & 1u);
    uint32_t a_dx = lds + kAtDx + 16u * (16 * tg0 + 4 * kq + (l16 & 3u)) + 4u * (l16 >> 2);
    uint32_t a_dws = lds + kSlab * mat + kSlabWt + 8u * (16 * half + l16);
    uint32_t a_xt[KB];  // chunk 2 b + kq / 2 of this lane's token (the second tile's is 16 tokens on: the same swizzle)
#pragma unroll
    for (uint32_t b = 0; b < (uint32_t)KB; b++) a_xt[b] = lds + kAtX + 128u * (16 * tg0 + l16) + 16u * ((2 * b + (kq >> 1)) ^ xt_swizzle(l16)) + 8u * (kq & 1u);

    v4i cbias;
#pragma unroll
    for (int i = 0; i < 4; i++) cbias[i] = (int)kBiasBits;
    asm volatile("" : "+v"(cbias));
    v4f acc[TPW], total[TPW];
#pragma unroll
    for (int i = 0; i < TPW; i++) acc[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f}, total[i] = acc[i];
    const bool walks = !DUMP && !GATED && shift != 0 && !side;
    uint32_t share = 1, share_end = walks ? all_slabs >> shift : UINT32_MAX, stage = 0;
    for (uint32_t s = 0; s < slabs; s++) {
        if (copies) {  // slab s is there once no more copies are under way than those of the R - 2 slabs behind it
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 2) * kPer) : "memory");
            if (s + (R - 2u) >= slabs) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (copies && s + (R - 1u) < slabs) copy_stage();  // where slab s - 1 was, which every wave has left
        if (multiplies) {
            if (__builtin_expect(s == share_end, 0)) {  // the next share of K starts
#pragma unroll
                for (int i = 0; i < TPW; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) total[i][r] = share == 1 ? acc[i][r] : total[i][r] + acc[i][r], acc[i][r] = 0.0f;
                share++;
                share_end = share * all_slabs >> shift;
            }
            long w[KB], x[TPW][KB];
            float2 dw[KB];
            float dx[TPW];
            v4i D[TPW][KB];
            static_for<KB>([&](auto b_) {
                constexpr int b = decltype(b_)::value;
                lds_read8<512 * b>(a_wt, w[b]);
                static_for<TPW>([&](auto i) { lds_read8<16 * 128 * decltype(i)::value>(a_xt[b], x[decltype(i)::value][b]); });
            });
            if constexpr (!DUMP) {
                static_for<TPW>([&](auto i) { lds_read4<16 * 16 * decltype(i)::value>(a_dx, dx[decltype(i)::value]); });
                static_for<KB>([&](auto b) { lds_read8<256 * decltype(b)::value>(a_dws, dw[decltype(b)::value]); });
            }
            constexpr int kScales = DUMP ? 0 : TPW + KB;
            static_for<KB>([&](auto b_) {
                constexpr int b = decltype(b_)::value, behind = (KB - 1 - b) * (1 + TPW) + kScales;
                lds_arrived<(behind < 15 ? behind : 15)>(w[b]);
                static_for<TPW>([&](auto i_) {
                    constexpr int i = decltype(i_)::value;
                    tie(x[i][b]);
                    D[i][b] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[i][b], w[b], cbias, 0, 0, 0);
                });
            });
            if constexpr (!DUMP) {
                static_for<KB>([&](auto b_) {
                    constexpr int b = decltype(b_)::value;
                    lds_arrived<KB - 1 - b>(dw[b]);
                    static_for<TPW>([&](auto i_) {
                        constexpr int i = decltype(i_)::value;
                        if constexpr (b == 0) tie(dx[i]);
                        v4f t;
#pragma unroll
                        for (int r = 0; r < 4; r++) t[r] = __builtin_fmaf(__int_as_float(D[i][b][r]), dw[b].x, dw[b].y);
                        fmac_row_lanes4<b>(acc[i], dx[i], t);
                    });
                });
            } else {
#pragma unroll
                for (int i = 0; i < TPW; i++)
#pragma unroll
                    for (int b = 0; b < KB; b++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const uint32_t rw = GR * granule + 16 * half + l16, t = 16 * (tg0 + i) + 4 * kq + r;
                            if (rw < a.m && t < n_here) {
                                int v = D[i][b][r] - (int)kBiasBits;
                                if (TYPE == 2) v >>= 4;  // weights were stored x16; exact
                                a.dots[((size_t)(tok0 + t) * a.m + rw) * nb + s * KB + b] = v;
                            }
                        }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this slab's reads are done
            stage++;
            const uint32_t next = (stage & (R - 1u)) == 0 ? 0u - (R - 1u) * kStage : kStage;
            a_wt += next, a_dws += next, a_dx += next;
#pragma unroll
            for (int b = 0; b < KB; b++) a_xt[b] += next;
        }
    }
    static_assert((R & (R - 1)) == 0, "stages are counted in a mask");
    if constexpr (GATED) {
        // The waves of gate and of up have the same elements: each hands half of its own to the other and gates the rest.
        __syncthreads();
        float* const h = reinterpret_cast<float*>(sm);  // [token][row] of gate * up
        float* const other = h + 32 * TG * kRow;        // [token][row] of what is handed over
        const uint32_t el = kRow * (16 * tg0 + 4 * kq) + 16 * half + l16, mine = mat ? 2u : 0u;
#pragma unroll
        for (int i = 0; i < TPW; i++)
#pragma unroll
            for (uint32_t r = 0; r < 2; r++) other[el + kRow * (16 * i + 2 - mine + r)] = mat ? acc[i][r] : acc[i][2 + r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TPW; i++)
#pragma unroll
            for (uint32_t r = 0; r < 2; r++) {
                const float own = mat ? acc[i][2 + r] : acc[i][r], its = other[el + kRow * (16 * i + mine + r)];
                h[el + kRow * (16 * i + mine + r)] = silu_mul(mat ? its : own, mat ? own : its);
            }
        __syncthreads();
        const uint32_t tok = threadIdx.x >> 3, quad = threadIdx.x & 7u;
        if (tok < 32u * TG) {
            const float4 x = *reinterpret_cast<const float4*>(&h[kRow * tok + 4u * quad]);
            float id;
            const float scale = q8_scale_and_inverse(group_max8(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)))), id);
            const uint32_t packed = q8_pack4(x.x, x.y, x.z, x.w, id);
            if (tok < n_here) {
                *reinterpret_cast<uint32_t*>(a.q_out + (size_t)(tok0 + tok) * a.m + GR * granule + 4u * quad) = packed;
                if (quad == 0) a.s_out[(size_t)(tok0 + tok) * (a.m >> 5) + granule] = scale;
            }
        }
    } else if constexpr (!DUMP) {
        const uint32_t row = GR * granule + 16 * half + l16;
        if (!multiplies || row >= a.m) return;
        const size_t tok_step = side ? a.m : (a.y_row_major ? 1u : a.y_stride), row_step = side || !a.y_row_major ? 1u : a.y_stride;
        const bool add = !side && a.accumulate;
        float* y = (side ? in_global<float>(p_more) + (size_t)my_share * p_n * a.m : a.y) + row * row_step + tok0 * tok_step;
#pragma unroll
        for (int i = 0; i < TPW; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t t = 16 * (tg0 + i) + 4 * kq + r;
                if (t >= n_here) continue;
                const float v = walks ? total[i][r] + acc[i][r] : acc[i][r];
                y[t * tok_step] = add ? y[t * tok_step] + v : v;
            }
    }
}

// y (+)= partial[0] + partial[1] + ... in that order, element by element (token-major partials [split][n][m]).
// (S a template parameter: all of an element's loads are in flight together instead of one round trip per share.)
template <int S>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ partial, uint32_t n, uint32_t m,
                                                                 float* __restrict__ y, uint32_t y_stride, int y_row_major, int accumulate) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, total = (size_t)n * m;
    if (i >= total) return;
    const uint32_t tok = (uint32_t)(i / m), row = (uint32_t)(i % m);
    float* dst = y_row_major ? y + (size_t)row * y_stride + tok : y + (size_t)tok * y_stride + row;
    float p[S];
#pragma unroll
    for (int s_ = 0; s_ < S; s_++) p[s_] = partial[(size_t)s_ * total + i];
    const float old = accumulate ? *dst : 0.0f;
    float sum = p[0];
#pragma unroll
    for (int s_ = 1; s_ < S; s_++) sum += p[s_];
    *dst = accumulate ? old + sum : sum;
}

// How many ways a single-weight launch is split over K: only narrow launches that leave at least half of the CUs without
// a tile, with K long enough (>= 8 stages) that the shorter walk pays for the second launch, every share >= 2 stages (a stage
// of a launch with few tiles costs a whole memory round trip, 1.2 - 1.4 us: nothing else is there to hide it).
// Also a long-K launch of 64 .. 256 tiles of 128 x 128 (the down projection of a long prompt: 1024 x 2002 x 4608 is 128 of them), up to two
// (tile, share) pairs per CU: the large tiles' block loops are the faster ones, and without shares they would leave half of the chip
// idle.  Shares of >= 8 stages.  (The shares fix the order of a row's sum, so they follow from the shape alone, whichever tile then runs.)
uint32_t wide_split_factor(uint32_t m, uint32_t n, uint32_t k, uint32_t max_splits) {
    const uint32_t tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN), stages = (k >> 5) / KB;
    if (n <= BN_NARROW || tiles < kCus / 4 || tiles > kCus || stages < 32) return 1;
    uint32_t s_ = 1;
    while (2 * s_ <= max_splits && tiles * 2 * s_ <= 2 * kCus && stages / (2 * s_) >= 8) s_ *= 2;
    return s_;
}

// Launches of few 128 x 128 tiles (at most one per CU): the ones that may be split over K.
bool narrow_tiles(uint64_t row_tiles, uint32_t n) { return n <= BN_NARROW || row_tiles * ((n + BN - 1) / BN) <= kCus; }

// Launches of gemm_few_kernel: up to 64 tokens and few enough granules that latency and not the chip's throughput is what they cost (every workgroup
// fetches all tokens' activations for its 32 rows; beyond, the 128-row tiles are the cheaper readers).  Above 32 tokens up to the two workgroups a CU
// that it holds at once, up to 32 to three, or four over shorter rows.  Tiles / here, us, weights cold, in a graph:
//   up to 32:  1024 x 4608 over 23 29 / 12.5; 16384 x 1024 10.9 / 6.6, x 3072 24.7 / 13.2, x 4096 over 32 32.9 / 19.3; 8192 x 8192 59.2 / 21.6; 24576 x 1024 11.6 / 8.6, x 4096 over
//              32 34.5 / 28.1; 32768 x 1024 12.8 / 10.5, x 2048 20.8 / 18.3, x 4096 over 32 36.5 / 37.2; 40960 x 2048 over 32 24.1 / 24.2; 65536 x 1024 17.7 / 18.2, x 2048 over 16 29.3 / 31.9
//   above:     8192 x 1024 over 40 10.8 / 6.1, x 8192 over 64 52.6 / 29.5; 9216 x 1024 over 48 10.6 / 7.4; 16384 x 1024 over 33 11.3 / 7.7, x 2048 over 64 16.9 / 15.3, x 4096 29.9 / 27.2;
//              18432 x 1024 over 64 11.3 / 12.0, 20480 x 2048 18.8 / 19.8, 24576 x 1024 over 48 12.0 / 12.5
bool few_applies(uint64_t rows, uint32_t n, uint32_t k) {
    const uint64_t units = (rows + GR - 1) / GR;
    if (n > 32) return n <= 64 && units <= 2 * kCus;
    return units <= (k <= 16 * KB * 32 ? 4 : 3) * kCus;
}

// Shares of K side by side on the same kernel, a workgroup each.  Above 32 tokens while the chip holds them all at once, two workgroups a CU; up to 32
// always (there are four a CU at most).  128-row or 64-row tiles / here with the addition, us: 1024 x 4608 in 8 over 23 tokens 6.7 / 4.6; 2048 x 6912 over 37
// 10.0 / 8.9, over 64 12.6 / 12.2; 2048 x 4096 over 48 10.5 / 10.2; past two a CU, over 23 2560 x 4096 9.7 / 9.2, 4096 x 4096 11.4 / 10.5, 8192 x 2048 11.1 / 10.2, 16384 x 2048
// 14.6 / 12.9, over 32 4096 x 2048 9.4 / 9.2, 16384 x 3072 18.4 / 17.6; over 48 2560 x 4096 10.9 / 11.8, 4096 x 4096 12.8 / 14.1, 6144 x 2048 11.7 / 12.3.
bool few_side_applies(uint64_t rows, uint32_t n, uint32_t shares) {
    return n <= 32 || (n <= 64 && (rows + GR - 1) / GR * shares <= 2 * kCus);
}

// More tokens on that kernel, side by side in tiles of 32 or 64 (0: not): while the chip holds all of the workgroups at once, each slab is a
// quarter of a 32 x 32 tile's chain and three slabs of cold weights are under way, not one.  In tiles of 32 while they are 7/4 a CU at most (beyond,
// the 64-token tile's half as many weight copies count for more), else of 64 up to two a CU (their LDS); past that the larger tiles do more per byte read
// from LDS.  64-row or 128-row tiles / 32 / 64 tokens here, us:
//   one share:  1024 x 1024 over 100 7.7 / 4.7 / 5.4, 300 7.8 / 5.5 / 5.6, 555 8.0 / 7.6 / 7.0, 1300 10.1 / 11.9 / 11.1; 2048 x 2048 over 160 15.3 / 8.2 / 8.9,
//               256 15.3 / 11.0 / 9.7, 400 15.5 / 16.0 / 12.6, 555 15.9 / 19.5 / 17.9; 4608 x 1024 over 130 9.6 / 8.6 / 7.9, 256 11.0 / 12.3 / 11.5; 3072 x 2048 over 300 15.8 / 17.6 / 13.9
//   in shares:  1024 x 1024 in 4 over 130 4.5 / 3.9 / 3.8, 300 5.5 / 5.6 / 6.0; 1024 x 4608 in 8 over 72 7.3 / 6.5 / 6.0, 130 8.4 / 8.4 / 8.7; 2048 x 6912 in 8 over 72 11.2 / 12.9 / 12.4
// Up to 2048 tokens, where the few granules that are left re-read activations that an XCD's L2 no longer holds: 1024 x 1024 over 1000 8.1 / 7.5, 256 x 512 over
// 1220 5.5 / 3.8, over 2211 5.6 / 4.7, 704 x 3072 over 1459 19.3 / 18.0, 512 x 2048 over 2048 12.7 / 12.6; 256 x 2048 over 3000 12.4 / 13.3, over 4000 12.7 / 14.7.
// Small weights gain the same: in a graph 512 x 512 over 65 5.0 / 3.2, over 832 5.5 / 3.9; 1024 x 256 over 400 4.1 / 3.2; 32 x 128 over 66 3.1 / 2.1; and
// back to back, in shares and with their addition or walked, 512 x 512 over 400 5.2 / 3.9, 64 x 4096 over 200 7.4 / 6.5, 128 x 2048 over 100 6.4 / 6.5.
uint32_t few_tokens_per_tile(uint64_t rows, uint32_t n, uint32_t shares) {
    const uint64_t units = (rows + GR - 1) / GR * shares;
    if (n <= 64 || n > 2048) return 0;
    if (4 * units * ((n + 31) / 32) <= 7 * kCus) return 32;
    return units * ((n + 63) / 64) <= 2 * kCus ? 64 : 0;
}

// Workgroups of such a launch per token tile (blockIdx.y).  Rounded up to whole rounds over the XCDs, a granule's token tiles are all on one, which
// reads its weights once; but with a last round that is not full the first XCDs have more of them, and where that is another workgroup for their
// 32 CUs, the launch waits for those: there the token tiles go round the XCDs one after the other.  Tiles of other kernels / rounded / not, us:
// 1312 x 1024 over 768 8.2 / 10.3 / 7.8, 1056 x 1024 over 832 8.0 / 9.9 / 7.6, 5408 x 2688 over 130 19.5 / 18.0 / 14.9, 1568 x 2048 over 300 13.8 / 10.2 / 8.9;
// as many either way: 2208 x 1024 over 200 8.4 / 6.2 / 6.5, 7712 x 1024 over 128 9.8 / 9.0 / 9.3, 544 x 1024 over 300 7.7 / 4.7 / 4.8.
// Shares are rounded up together, not eight granules of each: a workgroup without work still takes its turn on a CU.  Tiles of other kernels / eight granules /
// here, with the addition: 1344 x 7040 in 4 over 163 16.5 / 18.0 / 14.2, 192 x 3968 in 8 over 635 9.4 / 10.7 / 9.2, 544 x 7040 in 4 over 405 16.8 / 18.0 / 14.3.
uint32_t few_grid(uint32_t granules, uint32_t shares, uint32_t tok_tiles) {
    const auto per_cu = [](uint32_t on_an_xcd) { return (on_an_xcd + kCus / 8 - 1) / (kCus / 8); };
    const uint32_t n = granules * shares;
    const bool uneven = per_cu((n + 7) / 8 * tok_tiles) > per_cu((n * tok_tiles + 7) / 8);
    return uneven ? n : (n + 7) / 8 * 8;
}

// Shares of K one after the other in one launch of that kernel: ~0.3 us a slab up to 32 tokens, twice that above, against shares side by side and
// the launch that adds them up, or, with `deferrable`, the additions in the norm's kernel behind the projection.  With the norm, side by
// side is the faster way up to two workgroups a CU (1024 x 1024 in 4 over 23 tokens 3.5 and 0.4 more in the norm, here 4.7); beyond, and plain:
//   plain, 9 tokens:        1024 x 1024 6.3 / 4.5, x 1792 7.5 / 6.5, x 2048 (8 shares, not 4) 6.7 / 7.1; 4096 x 2048 7.0 / 7.3
//   plain, 24:              1024 x 1024 6.6 / 4.9, x 1792 8.0 / 6.8, x 2048 7.0 / 7.4; 3072 x 2048 7.6 / 7.5, 4096 x 2048 8.5 / 7.5
//   plain, 40:              1024 x 1024 7.2 / 7.0, 4096 x 1024 8.2 / 7.1, 9216 x 1024 over 48 10.8 / 7.6, 16384 x 1024 over 33 12.5 / 7.6, over 64 14.8 / 9.2; 2048 x 2048 8.2 / 11.5
//   with the norm, 24:      4096 x 2048 13.3 / 12.5; over 40 tokens 3072 x 1024 11.3 / 11.6, 4096 x 1024 12.9 / 12.3
// Without room for shares side by side: all that needs none, the faster way or not.
// Above 64 tokens, against shares on the 64-row or 128-row tiles: the walk costs 0.3 us a slab and the other way the sums' round trip through memory:
//   plain:                  3072 x 1024 over 66 8.7 / 5.4, 130 10.0 / 6.2, 320 13.3 / 8.0; 1024 x 1024 over 512 11.3 / 6.1; 2048 x 2048 over 66 9.4 / 7.7, 256 13.6 / 9.5;
//                           1024 x 3072 over 96 8.5 / 9.7, 160 10.3 / 9.8; 1024 x 4608 over 200 12.1 / 13.7, 256 13.8 / 13.7; 512 x 4096 over 400 11.7 / 12.2, 512 12.9 / 12.3
//   plain, longer rows, weights cold; warm and with the quantizer: 640 x 7296 over 761 25.4 / 35.8 (warm); 512 x 6144 over 832 18.3 / 23.8 (cold); 4128 x 4352 over 82
//                           19.3 / 16.5; 20.9 / 15.5.  In tiles of 32 tokens 512 x 3072 over 832 13.2 / 10.9; 18.5 / 19.0, 1024 x 4608 over 400 16.0 / 15.0; 19.3 / 20.9, 768 x
//                           4352 over 566 15.0 / 13.7; 19.2 / 21.6.  Of 64 1216 x 5248 over 519 24.2 / 22.0; 28.0 / 27.4, 1024 x 6144 over 800 27.9 / 28.2; 31.1 / 34.1.
//                           Over more tokens, cold; warm: 1024 x 3584 over 887 21.1 / 17.4; 25.3 / 23.5, 512 x 5120 over 1144 22.1 / 26.0; 28.3 / 33.1, 256 x 2560 over 1651
//                           12.6 / 12.2; 18.1 / 19.1, 544 x 2176 over 1100 14.0 / 10.8; 19.3 / 17.2.
//                           (A walk is a chain of slabs, behind which cold weights hide; warm ones shorten what it is compared with.  The lines are where neither
//                           loses what the other gains: 190 launches of 16 to 64 slabs.)
//   with the norm, a prompt of the 350M shape, all of it: 220 tokens 839 / 840, 300 963 / 947, 420 1039 / 1016, 680 1388 / 1394; of the 1.2B shape's first six layers
//                           (2048 x 2048): 200 550 / 559, 300 689 / 685, 400 742 / 734
bool few_applies_split(uint64_t rows, uint32_t n, uint32_t k, uint32_t shares, bool deferrable, bool room) {
    const uint64_t units = (rows + GR - 1) / GR, slabs = k / (KB * 32), cost = n <= 32 ? 1u : 2u;
    if (n > 64) {
        const uint32_t tokens = few_tokens_per_tile(rows, n, 1);
        if (!tokens) return false;
        if (deferrable) return slabs <= 16 && n <= 512 && rows * n >= 32768 * slabs && !few_tokens_per_tile(rows, n, shares);
        if (!room) return slabs <= 9 + rows * n / 9500;  // (all that walks with room, at least)
        return slabs <= 9 + rows * n / 11000 && slabs <= (n > 1024 ? 17u : (n <= 768 && tokens == 64) || n <= 96 ? 42u : 26u);
    }
    if (units > 2 * kCus || slabs * cost > (cost == 1 && units < 96 ? 15u : 16u)) return false;
    if (deferrable && 12 * slabs * cost > 72 + units) return false;
    return !room || !(deferrable && units * shares <= 2 * kCus);
}

uint32_t split_k_factor(uint32_t m, uint32_t n, uint32_t k, uint32_t max_splits) {
    const uint32_t ws = wide_split_factor(m, n, k, max_splits);
    if (ws > 1) return ws;
    const uint32_t row_tiles = (m + BM - 1) / BM;
    if (!narrow_tiles(row_tiles, n)) return 1;
    const uint32_t tiles = row_tiles * ((n + BN_NARROW - 1) / BN_NARROW), stages = (k >> 5) / KB;
    if (stages < 8) return 1;
    uint32_t s_ = 1;
    while (2 * s_ <= max_splits && tiles * 2 * s_ <= kCus && stages / (2 * s_) >= 2) s_ *= 2;
    return s_;
}

// The second launch of a split GEMM: y (+)= the shares in ascending order.
hipError_t launch_reduce(const GemmArgs& a, const Launch& L) {
    const size_t total = (size_t)a.n * a.m;
    const auto reduce = [&](auto kernel) {
        return launch_kernel(L, kFamGemm, kernel, dim3((uint32_t)((total + 255) / 256)), dim3(256), static_cast<const float*>(a.partial), a.n, a.m, a.y,
                             a.y_stride, a.y_row_major, a.accumulate);
    };
    if (a.ksplit == 2) return reduce(gemm_splitk_reduce_kernel<2>);
    if (a.ksplit == 4) return reduce(gemm_splitk_reduce_kernel<4>);
    if (a.ksplit == 8) return reduce(gemm_splitk_reduce_kernel<8>);
    return hipErrorInvalidValue;  // split_k_factor makes 2, 4 or 8 shares
}

// The tiles of a launch over a prompt, and what each costs: us per slab (128 elements of K) of a share with 1 .. kPerCu workgroups on a CU, and us
// per workgroup for filling, draining and storing it (and 3 us a launch, the same for all) -- plain launches first, those with the gate
// in the epilogue second (0: not built).  Fitted to 130 launches (3072, 2048, 1024 x 1024, 1024 x 4608, 6144, 3072, 2048 x 2048, 2048 x 6912 and gate | up 4608 x 1024,
// 6912 x 2048, each over 80 .. 2048 tokens, weights and activations of random bits: a launch that keeps the chip busy runs at the
// power limit), which they meet to 5 % rms; the tile they choose is 0.3 % behind the best of the six.  Below the fit, over 115 launches of
// 33 .. 96 tokens (14 shapes of 512 .. 16384 rows and 512 .. 8192 of K, split as the library does it): 5.4 % rms, 1.2 % behind the best, at worst
// 8.5 % (8192 x 4096 over 56 in four shares: N where H is best, which cost 17 and 7 % more than they are given).  TileQ's constants are what they were
// times what copied token scales (load_dx) made of its launches: 0.85 .. 0.93 over 300 launches of 35 .. 4000 tokens, of which the tile chosen is now
// 0.6 % (plain, 219) and 0.3 % (gated, 79) behind the best, 0.9 and 1.6 % before.  A launch is workgroups on 256
// CUs, kPerCu at a time, and what the last round leaves idle is what separates the tiles: large ones do more per operand byte, small ones leave
// less over, and a CU with a single workgroup on it wants that one's waves to be many.
struct TileCost {
    float slab[4], fixed;
};
struct TileL : T32<4, 2, 2, 2, 2, 2, true> {  // 256 x 128, 4 waves of 128 x 64
    static constexpr int kPerCu = 2;
    static constexpr TileCost kCost[2] = {{{3.10f, 4.36f}, 2.10f}, {{3.06f, 4.00f}, 6.15f}};
};
struct TileX : T32<2, 2, 2, 2, 2, 3> {  // 128 x 128, 4 waves of 64 x 64
    static constexpr int kPerCu = 3;
    static constexpr TileCost kCost[2] = {{{1.79f, 2.38f, 3.42f}, 1.43f}, {{1.79f, 2.23f, 3.27f}, 2.24f}};
};
struct TileS : T32<2, 1, 2, 2, 4, 2> {  // 128 x 64, 4 waves of 64 x 32
    static constexpr int kPerCu = 2;
    static constexpr TileCost kCost[2] = {{{0.94f, 1.32f}, 1.25f}, {{0.99f, 1.37f}, 0.92f}};
};
struct TileQ : T32<2, 1, 2, 2, 2, 4, false, true> {  // the same with half a slab per stage: four of them on a CU
    static constexpr int kPerCu = 4;
    static constexpr TileCost kCost[2] = {{{1.12f, 1.40f, 1.87f, 2.36f}, 1.25f}, {{1.20f, 1.45f, 1.78f, 2.39f}, 0.97f}};
};
struct TileN : T32<1, 1, 4, 2, 4, 4> {  // 128 x 64, 8 waves of 32 x 32
    static constexpr int kPerCu = 2;
    static constexpr TileCost kCost[2] = {{{0.70f, 1.25f}, 1.53f}, {{0.94f}, 0.9f}};  // (with the gate: one on a CU, see gated_tile_n)
};
struct TileH : T32<1, 1, 2, 2, 4, 4> {  // 64 x 64, 4 waves of 32 x 32
    static constexpr int kPerCu = 4;
    static constexpr TileCost kCost[2] = {{{0.53f, 0.76f, 1.06f, 1.32f}, 0.73f}, {}};
};
template <typename C>
float tile_cost(uint64_t row_tiles, uint32_t n, uint32_t k, uint32_t shares, bool gated = false) {
    const uint64_t tiles = row_tiles * ((n + C::kTokens - 1) / C::kTokens) * shares, per_cu = (tiles + kCus - 1) / kCus;
    const TileCost& c = C::kCost[gated];
    const uint32_t rest = (uint32_t)(per_cu % C::kPerCu);
    float per_slab = (float)(per_cu / C::kPerCu) * c.slab[C::kPerCu - 1] + (rest ? c.slab[rest - 1] : 0.0f);
    // Shares of K whose second workgroup only some CUs have: the small tile gives way by what the others leave it of the caches (128-row / 64-row tile, us,
    // and workgroups a CU: 1024 x 4608 in 2 over 555 19.0 / 17.8 and 1.13, 700 19.4 / 18.6 and 1.38, 900 in 4 18.3 / 20.0; in 4 over 300 11.8 / 11.2 and 1.25,
    // 420 12.2 / 12.0 and 1.63, 480 12.4 / 12.4 and 1.88; 2048 x 6912 in 2 over 300 27.2 / 25.3 and 1.25, 360 27.9 / 28.6 and 1.5).
    if (shares > 1 && C::kRows == 64 && per_cu == 2) per_slab *= 1.0f - 0.14f * (2.0f - (float)tiles / (float)kCus);
    // Past the four that are on a CU at a time its many stores of shares count (TileQ / 64-row tile, us: 2048 x 6912 in 4 over 555 32.3 / 35.0, 620
    // 35.2 / 37.2; in 2 over 1200 56.6 / 57.2).
    if (shares > 1 && C::kRows == 64 && per_cu > 4) per_slab *= 1.06f;
    return per_slab * (float)k / (float)(KB * 32 * shares) + (float)per_cu * c.fixed;
}
// go(tile) for the one of them that cost(tile) is lowest for.
template <typename... Tiles, typename Cost, typename Go>
hipError_t cheapest_tile(Cost&& cost, Go&& go) {
    const float costs[] = {cost(Tiles{})...};
    uint32_t best = 0;
    for (uint32_t i = 1; i < sizeof...(Tiles); i++)
        if (costs[i] < costs[best]) best = i;
    hipError_t e = hipErrorInvalidValue;
    uint32_t i = 0;
    (void)((i++ == best ? (e = go(Tiles{}), true) : false) || ...);
    return e;
}

// A launch with the leading scalars of its kernel: none (the 16x16x32 kernels), a tile's, the few-token kernel's.
using TileKernel = void (*)(Address, Address, Address, Address, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, GemmArgs);
template <typename Kernel>
hipError_t enqueue(Kernel kernel, uint32_t grid, uint32_t threads, const GemmArgs& a, uint32_t shares, bool more, const Launch& L) {
    const uint32_t flag = more ? kMoreWeights : 0u;
    const uint32_t shift = shares >= 8 ? 3u : (shares >= 4 ? 2u : shares >= 2 ? 1u : 0u);  // (split_k_factor makes 2, 4 or 8 shares)
    if constexpr (std::is_same<Kernel, void (*)(GemmArgs)>::value) {
        return launch_kernel(L, kFamGemm, kernel, dim3(grid), dim3(threads), a);
    } else if constexpr (std::is_same<Kernel, TileKernel>::value) {
        return launch_kernel(L, kFamGemm, kernel, dim3(grid), dim3(threads), address(a.w), address(a.xq), address(a.xs), address(a.w_up), a.m, a.n, a.k,
                             a.row_tiles, a.tok_tiles, shift | flag, a);
    } else {
        const Address p_more = a.w_up ? address(a.w_up) : address(a.partial);
        return launch_kernel(L, kFamGemm, kernel, dim3(grid, a.tok_tiles), dim3(threads), address(a.w), address(a.xq), address(a.xs), p_more, a.n, a.k, a.row_tiles,
                             shift | (shift && a.partial ? kFewSide : 0u) | flag, a);
    }
}

// in_launch: the launch walks its shares of K itself (gemm_split_in_launch).  The parity hook comes with the product launch's share
// count and in_launch, runs its kernel, and walks K whole.
template <bool DUMP>
hipError_t launch(int type, GemmArgs& a, const Launch& L, bool in_launch, uint32_t more = 0, bool defer_reduce = false) {
    if (a.m == 0 || a.n == 0) return hipSuccess;
    const auto tile_rows = [&](uint32_t rows) {  // row tiles of `rows` rows over the launch's weights
        uint64_t t = (a.m + (uint64_t)rows - 1) / rows;
        for (uint32_t i = 0; i < more; i++) t += (a.m_more[i] + (uint64_t)rows - 1) / rows;
        return t;
    };
    uint32_t ksplit = a.ksplit > 1 ? a.ksplit : 1u;
    const bool wide_split = more == 0 && ksplit > 1 && wide_split_factor(a.m, a.n, a.k, ksplit) == ksplit;
    if (!wide_split && !narrow_tiles(tile_rows(BM), a.n)) ksplit = 1;  // only few-tile launches carry a split
    a.ksplit = DUMP ? 1u : ksplit;
    const auto go = [&](auto kernel, uint32_t rows, uint32_t tokens, uint32_t threads, bool whole = false) {
        a.row_tiles = (a.m + rows - 1) / rows;
        a.tile_start[0] = a.tile_start[1] = UINT32_MAX;
        for (uint32_t i = 0; i < more; i++) {
            a.tile_start[i] = a.row_tiles;
            a.row_tiles += (a.m_more[i] + rows - 1) / rows;
        }
        a.tok_tiles = (a.n + tokens - 1) / tokens;
        const uint32_t shares = a.ksplit;
        if ((uint64_t)a.row_tiles * a.tok_tiles * shares > 0x7fffff00ull) return hipErrorInvalidValue;  // beyond a launch's grid
        // every XCD gets the same number of slots of the tile map; tile id = blockIdx.x / shares runs over all of them
        const uint32_t side = whole ? 1u : shares;  // whole: a workgroup takes all shares of its rows
        const uint32_t grid = rows == GR ? few_grid(a.row_tiles, side, a.tok_tiles) : (a.row_tiles * a.tok_tiles + 7u) / 8u * 8u * side;
        const hipError_t e = enqueue(kernel, grid, threads, a, shares, more != 0, L);
        if (e != hipSuccess || shares == 1 || defer_reduce || whole) return e;  // deferred: the caller's next kernel adds the shares up itself
        return launch_reduce(a, L);
    };
    // (The product kernels do not depend on the weight type: the copy they read is the same for both.  The parity hook's do.)
    const bool q8 = DUMP && type != kTypeQ4_0;
    const auto tile = [&](auto cfg) {
        using C = decltype(cfg);
        if constexpr (DUMP)
            if (q8) return go(gemm_tile_kernel<8, true, false, C>, C::kRows, C::kTokens, C::kThreads);
        return go(gemm_tile_kernel<2, DUMP, false, C>, C::kRows, C::kTokens, C::kThreads);
    };
    const uint32_t few_tiled = L.gemm_mfma16 ? 0 : few_tokens_per_tile(GR * tile_rows(GR), a.n, in_launch ? 1u : ksplit);
    const bool few = !L.gemm_mfma16 && (few_tiled || (ksplit > 1 ? in_launch || few_side_applies(a.m, a.n, ksplit) : few_applies(GR * tile_rows(GR), a.n, a.k)));
    const bool narrow = !wide_split && narrow_tiles(tile_rows(BM), a.n);
    if (few) {
        // 32 tokens, 40 KB of LDS: four waves, a 16 x 16 tile each, that also copy, or, while every CU gets one workgroup at most, four more that copy for
        // them: as fast in a graph (8192 x 1024 over 23 5.3 / 5.4 us, x 3072 10.0 / 9.9), past it 1 - 5 % slower (16384 x 1024 6.6 / 6.9).  64 tokens, 56 KB: eight
        // tiles, a wave each (four waves with two tiles each / eight: 8192 x 1024 over 48 6.4 / 6.2, 16384 x 1024 over 40 8.5 / 8.0, 2048 x 6912 in 8 over 48 11.2 / 10.8).
        const bool whole = DUMP || ksplit == 1 || in_launch;
        const auto waves = [&](auto tg, auto wv) {
            constexpr int TG = decltype(tg)::value, WV = decltype(wv)::value;
            if constexpr (DUMP)
                if (q8) return go(gemm_few_kernel<8, true, false, TG, WV>, GR, 32 * TG, 64 * WV, whole);
            return go(gemm_few_kernel<2, DUMP, false, TG, WV>, GR, 32 * TG, 64 * WV, whole);
        };
        if (few_tiled) return few_tiled == 32 ? waves(Idx<1>{}, Idx<4>{}) : waves(Idx<2>{}, Idx<8>{});
        if (a.n > 32) return waves(Idx<2>{}, Idx<8>{});
        return tile_rows(GR) * (whole ? 1u : ksplit) <= kCus ? waves(Idx<1>{}, Idx<8>{}) : waves(Idx<1>{}, Idx<4>{});
    }
    if (narrow && ((ksplit == 1 && a.n <= 48) || L.gemm_mfma16)) {
        // a launch of at most 16 / 32 / 48 tokens computes one / two / three of the tile's four 16-token MFMA tiles (the parity
        // hook: all four).  These launches are bound by their block loop, not by memory: 65536 x 16 x 2048 40 -> 34 us.
        // (Shares of K over as many: gemm_few_kernel above, or the tiles.)
        if constexpr (!DUMP) {
            if (a.n <= 16) return go(gemm_narrow_kernel<2, false, 1>, BM, BN_NARROW, THREADS);
            if (a.n <= 32) return go(gemm_narrow_kernel<2, false, 2>, BM, BN_NARROW, THREADS);
            if (a.n <= 48) return go(gemm_narrow_kernel<2, false, 3>, BM, BN_NARROW, THREADS);
        }
        if constexpr (DUMP)
            if (q8) return go(gemm_narrow_kernel<8, true>, BM, BN_NARROW, THREADS);
        return go(gemm_narrow_kernel<2, DUMP>, BM, BN_NARROW, THREADS);
    }
    if (L.gemm_mfma16) {
        if constexpr (DUMP)
            if (q8) return go(gemm_mfma_kernel<8, true>, BM, BN, THREADS);
        return go(gemm_mfma_kernel<2, DUMP>, BM, BN, THREADS);
    }
    const auto cost = [&](auto cfg) { return tile_cost<decltype(cfg)>(tile_rows(decltype(cfg)::kRows), a.n, a.k, ksplit); };
    return cheapest_tile<TileL, TileX, TileS, TileQ, TileN, TileH>(cost, tile);
}

}  // namespace

uint32_t gemm_split_k(uint32_t m, uint32_t n, uint32_t k, uint32_t max_splits) { return split_k_factor(m, n, k, max_splits); }
bool gemm_split_in_launch(uint32_t m, uint32_t n, uint32_t k, uint32_t max_splits, const Launch& L, bool deferrable, bool room) {
    return !L.gemm_mfma16 && few_applies_split(m, n, k, split_k_factor(m, n, k, max_splits), deferrable, room);
}

// The GEMM's own copy of a weight (slabs, see StageT): its size, and the kernel that makes it from the raw blocks.
size_t gemm_packed_bytes(uint32_t m, uint32_t k) { return (size_t)((m + 2 * GR - 1) / (2 * GR)) * 2 * ((k >> 5) / KB) * kSlab; }

hipError_t launch_gemm_pack(int type, const uint8_t* d_raw, uint32_t m, uint32_t k, uint8_t* d_packed, const Launch& L) {
    const uint32_t nb = k >> 5;
    if (m == 0 || nb == 0 || nb % KB != 0) return hipErrorInvalidValue;
    const uint64_t blocks = (uint64_t)((m + 2 * GR - 1) / (2 * GR)) * 2 * (nb / KB);  // whole pairs: a last odd granule gets a zero partner
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    if (type == kTypeQ4_0) return launch_kernel(L, kFamOther, gemm_pack_kernel<2>, dim3((uint32_t)blocks), dim3(GR * KB), d_raw, m, nb, d_packed);
    if (type == kTypeQ8_0) return launch_kernel(L, kFamOther, gemm_pack_kernel<8>, dim3((uint32_t)blocks), dim3(GR * KB), d_raw, m, nb, d_packed);
    return hipErrorInvalidValue;
}

// splits > 1 (= gemm_split_k(m, n, k, ...)): d_partial holds splits * n * m floats, or is null and the launch walks the shares itself
// (only where gemm_split_in_launch says so).
hipError_t launch_gemm_mfma(int type, const uint8_t* d_w, uint32_t m, uint32_t k, const int8_t* d_q,
                            const float* d_scales, uint32_t n, float* d_y, uint32_t y_stride, int y_layout,
                            int accumulate, const Launch& L, uint32_t splits, float* d_partial, bool defer_reduce) {
    GemmArgs a{};
    a.w = d_w, a.xq = d_q, a.xs = d_scales, a.y = d_y, a.dots = nullptr;
    a.m = m, a.n = n, a.k = k, a.y_stride = y_stride;
    a.y_row_major = (y_layout == 1);
    a.accumulate = accumulate;
    const bool in_launch = splits > 1 && !d_partial;
    if (splits > 1) {
        if (splits != split_k_factor(m, n, k, splits) || (in_launch && !gemm_split_in_launch(m, n, k, splits, L, false, false)))
            return hipErrorInvalidValue;  // the shape does not carry that split
        a.ksplit = splits, a.partial = d_partial;
    }
    if (defer_reduce && (splits <= 1 || in_launch)) return hipErrorInvalidValue;  // nothing to defer
    return launch<false>(type, a, L, in_launch, 0, defer_reduce);
}

// One token of a launch over more.  A row's sum is fixed by the shares of K and by nothing else of the launch.
hipError_t launch_gemm_mfma_row(const uint8_t* d_w, uint32_t m, uint32_t k, const int8_t* d_q, const float* d_scales, float* d_y, const Launch& L,
                                uint32_t splits, float* d_partial) {
    if (L.gemm_mfma16 || (splits > 1 && !d_partial)) return hipErrorInvalidValue;
    GemmArgs a{};
    a.w = d_w, a.xq = d_q, a.xs = d_scales, a.y = d_y;
    a.m = m, a.n = 1, a.k = k, a.y_stride = m;
    a.accumulate = 1;
    if (splits > 1) a.ksplit = splits, a.partial = d_partial;
    return launch<false>(kTypeQ4_0, a, L, false);
}

// The same launch over up to three weights of one type and k that share the activations: outputs y[i] (same stride,
// layout and accumulate flag), tiles of all weights in one tile list.
hipError_t launch_gemm_mfma_multi(int type, const uint8_t* const* d_w, const uint32_t* m, uint32_t count, uint32_t k, const int8_t* d_q,
                                  const float* d_scales, uint32_t n, float* const* d_y, uint32_t y_stride, int y_layout, int accumulate,
                                  const Launch& L) {
    if (count == 0 || count > 3) return hipErrorInvalidValue;
    GemmArgs a{};
    a.w = d_w[0], a.xq = d_q, a.xs = d_scales, a.y = d_y[0], a.dots = nullptr;
    a.m = m[0], a.n = n, a.k = k, a.y_stride = y_stride;
    a.y_row_major = (y_layout == 1);
    a.accumulate = accumulate;
    for (uint32_t i = 1; i < count; i++) a.w_more[i - 1] = d_w[i], a.y_more[i - 1] = d_y[i], a.m_more[i - 1] = m[i];
    return launch<false>(type, a, L, false, count - 1);
}

// Gate and up projection of a feed-forward block over n tokens in one launch whose epilogue applies the SiLU gate and
// quantizes: out = Q8_0(silu(W_gate x) * (W_up x)), [n][m] quants + [n][m / 32] scales, bit-identical to the two
// projections + silu_mul_quantize_kernel.  The float projections (2 * n * m * 4 bytes) are never written.
bool gemm_gated_applies(uint32_t m, uint32_t n, uint32_t k) {
    // wide tiles only (the narrow kernel's waves own 16 rows: no block in one wave), and enough of them to fill the chip
    return m % 32u == 0 && k % 128u == 0 && n > BN_NARROW && (uint64_t)((m + 63u) / 64u) * ((n + BN - 1) / BN) > kCus;
}

namespace {
// The few-token form of the launch: one workgroup per granule and CU, and 32 or 64 tokens (0: not).  Above 64 tokens, workgroups side by
// side in tiles of 32 up to 7/4 a CU, else of 64 while every workgroup of more than 24 tokens has a CU, or from 16 slabs on up to five quarters of a CU's worth, tiles of 16
// tokens that have any counted.  TileQ's kind / 32 / 64 tokens here, us: 4608 x 1024 over 72 13.1 / 8.7 / 10.2, 2816 x 1024 over 130 13.0 / 8.6 / 10.2;
// 2048 x 1024 over 256 13.0 / 9.0 / 9.2; over 280 13.0 / - / 10.7 and TileN below 11.3; 6912 x 2048 over 72 23.0 / 20.5 / 20.4; 1024 x 2048 over 400 20.3 / 12.9 / 13.2; 4096 x 4096 over 160 39.1 / 40.8 / 31.7.
uint32_t gated_few_tokens(uint32_t m, uint32_t n, uint32_t k) {
    const uint64_t units = m / GR;
    if (n <= 64) return units > kCus ? 0 : (n <= 32 ? 32 : 64);
    if (4 * units * ((n + 31) / 32) <= 7 * kCus) return 32;
    if (units * ((n + 39) / 64) <= kCus) return 64;
    return k >= 16 * KB * 32 && units * ((n + 15) / 16) <= 5 * kCus ? 64 : 0;
}

// TileN with the gate: past those, while every workgroup has a CU, whose eight waves make shorter slabs of it than four do (its cost is that of one a
// CU, and lower there than the other tiles').  The cheapest of the other tiles or 64 tokens above / here, us: 4608 x 1024 over 128 12.5 / 11.7, 160 13.4 / 11.8, 200 (288 workgroups) 15.9 / 16.4; 6912 x 2048 over 100 22.7 / 20.8, 160
// (324) 28.6 / 28.6; 2816 x 1024 over 300 13.3 / 11.6; 2048 x 1024 over 400 13.3 / 11.4; 4096 x 4096 over 200 41.3 / 36.6, 300 (320) 48.8 / 49.5.
bool gated_tile_n(uint32_t m, uint32_t n) { return n > 64 && (uint64_t)((m + 63) / 64) * ((n + 63) / 64) <= kCus; }

// Where that form is the faster way: it saves a launch and the floats (2.7 us together), once, and each weight has half of a workgroup's waves, so that
// it loses time with every slab against the projections alone, which run on gemm_few_kernel too.  us a layer that a prompt gains (+) or loses by it,
// hidden x feed-forward size:
//   up to 32 tokens, a CU for every granule of both: 1024 x 1024 over 9 3.3, over 24 2.5, 1280 x 2048 1.5, 2048 x 1024 1.2, x 2048 1.0, x 4096 1.1, 2560 x 2048 0.8, 2816 x 2048 0.6;
//                     3072 x 1024 0.2, x 2048 -0.2, x 3584 0.8, 4096 x 1024 -0.3, x 2048 -0.9, x 3072 0.3, x 4096 0.7; 6144 x 2048 -1.6, x 4096 -0.4, 8192 x 4096 -1.5
//   more granules:    1024 x 4608 over 24 1.9, 2048 x 6912 2.5, 4096 x 4608 3.7, over 32 5.1, 6144 x 6912 over 24 6.6, 8192 x 8192 5.7
//   above 32:         1280 x 4096 over 40 0.1, 1536 x 4096 -0.2, x 2048 -0.5, 2048 x 1024 -1.4, x 3584 -0.8, over 64 -0.9
//   more granules:    1024 x 4608 over 40 2.3, 2048 x 4608 1.9, over 64 4.1, x 8192 over 48 3.5, 4096 x 4608 over 64 6.7, 8192 x 8192 over 64 12.7
bool gated_few_faster(uint32_t m, uint32_t n, uint32_t k) {
    const uint32_t slabs = k / (KB * 32);
    if (2 * m / GR > kCus) return true;
    if (n > 32) return slabs <= 11;
    return slabs <= 22 || (m >= 3072 && slabs <= 32);
}

template <typename C>
float gated_tile_cost(uint32_t m, uint32_t n, uint32_t k) {
    if (std::is_same<C, TileN>::value && !gated_tile_n(m, n)) return INFINITY;
    return tile_cost<C>((m + C::kRows / 2 - 1) / (C::kRows / 2), n, k, 1, true);
}
}  // namespace

// Where the launch is expected to be faster than the two projections in one launch and the gate kernel behind it (2.7 us and the floats'
// round trip).  In one launch / two, us: 4608 x 1024 over 128 tokens 12.2 / 13.1, 300 14.8 / 17.9; 6912 x 2048 over 200 25.0 / 28.4.
bool gemm_gated_faster(uint32_t m, uint32_t n, uint32_t k, const Launch& L) {
    if (gemm_gated_applies(m, n, k)) return true;
    if (L.gemm_mfma16 || m % GR != 0 || k % (KB * 32) != 0 || m == 0 || n == 0) return false;
    if (gated_few_tokens(m, n, k)) return n > 64 || gated_few_faster(m, n, k);
    if (n <= 48 && (uint64_t)2 * m / GR > 2 * kCus) return false;  // the few-token kernel's or the narrow one's
    const auto plain = [&](auto cfg) {
        using C = decltype(cfg);
        return tile_cost<C>(2 * (uint64_t)((m + C::kRows - 1) / C::kRows), n, k, 1);
    };
    const float separate = std::min({plain(TileL{}), plain(TileX{}), plain(TileS{}), plain(TileQ{}), plain(TileN{}), plain(TileH{})});
    const float gated = std::min({gated_tile_cost<TileL>(m, n, k), gated_tile_cost<TileX>(m, n, k), gated_tile_cost<TileS>(m, n, k), gated_tile_cost<TileQ>(m, n, k),
                                  gated_tile_cost<TileN>(m, n, k)});
    return !few_applies(2 * (uint64_t)m, n, k) && gated < separate + 2.7f + (float)n * (float)m * 3e-6f;
}

// Any n; d_out_* as for gemm_gated_applies.
hipError_t launch_gemm_mfma_gated(int /*type: the copies are the same for both*/, const uint8_t* d_w_gate, const uint8_t* d_w_up, uint32_t m, uint32_t k, const int8_t* d_q,
                                  const float* d_scales, uint32_t n, int8_t* d_out_q, float* d_out_scales, const Launch& L) {
    if (m == 0 || n == 0) return hipSuccess;
    if (m % GR != 0 || k % (KB * 32) != 0) return hipErrorInvalidValue;
    GemmArgs a{};
    a.w = d_w_gate, a.w_up = d_w_up, a.xq = d_q, a.xs = d_scales, a.q_out = d_out_q, a.s_out = d_out_scales;
    a.m = m, a.n = n, a.k = k;
    a.tile_start[0] = a.tile_start[1] = UINT32_MAX;
    if (const uint32_t tokens = gated_few_tokens(m, n, k)) {
        a.row_tiles = m / GR, a.tok_tiles = (n + tokens - 1) / tokens;
        if (tokens == 64) return enqueue(gemm_few_kernel<2, false, true, 2, 8>, a.row_tiles, 512, a, 1, false, L);
        return enqueue(gemm_few_kernel<2, false, true, 1, 8>, a.row_tiles, 512, a, 1, false, L);
    }
    const auto tile = [&](auto cfg) {
        using C = decltype(cfg);
        a.row_tiles = (m + C::kRows / 2 - 1) / (C::kRows / 2), a.tok_tiles = (n + C::kTokens - 1) / C::kTokens;
        if ((uint64_t)a.row_tiles * a.tok_tiles > 0x7fffff00ull) return hipErrorInvalidValue;
        return enqueue(gemm_tile_kernel<2, false, true, C>, (a.row_tiles * a.tok_tiles + 7u) / 8u * 8u, C::kThreads, a, 1, false, L);
    };
    return cheapest_tile<TileL, TileX, TileS, TileQ, TileN>([&](auto cfg) { return gated_tile_cost<decltype(cfg)>(m, n, k); }, tile);
}

// Parity hook through the matrix-core path: the same loads, unpack, LDS layout and
// MFMA as the GEMM, writing the raw i32 block dots instead of scaling them.
hipError_t launch_block_dots_mfma(int type, const uint8_t* d_w, uint32_t m, uint32_t k, const int8_t* d_q, uint32_t n,
                                  int32_t* d_out, uint32_t max_splits, const Launch& L) {
    GemmArgs a{};
    a.w = d_w, a.xq = d_q, a.xs = nullptr, a.y = nullptr, a.dots = d_out;
    a.m = m, a.n = n, a.k = k, a.y_stride = 0;
    a.ksplit = split_k_factor(m, n, k, max_splits);
    return launch<true>(type, a, L, gemm_split_in_launch(m, n, k, max_splits, L, false, true));
}

}  // namespace wick_rocm
