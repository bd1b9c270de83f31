// Grouped expert GEMM on CDNA4 MFMA for prefill-sized token groups (the fast-order path).
//
// Each 32-element block's integer dot is computed exactly by the matrix cores:
//   - MXFP4 weights: v_cvt_scalef32_pk_f16_fp4 (scale 2) gives the doubled-e2m1 integers as f16,
//     activations are the int8 Q8_0 codes as f16, and v_mfma_f32_16x16x32_f16 sums the 32
//     products of one block; every partial sum is an integer below 2^24, so the block dot is
//     exact in fp32 whatever the order inside the matrix core.
//   - Q8_0 weights: v_mfma_i32_16x16x32_i8 on the int8 codes (exact int32).
// The block dot is then scaled (MXFP4: ldexp(d_act, e - 128); Q8_0: fp16(d_w) * d_act, the
// CPU's own products) and accumulated in fp32 block after block. That accumulation order is not
// the CPU's 8-lane chains, so outputs agree with the reference within fp32 rounding (the
// tolerance-checked order), while every integer block dot is bit-exact. The x86 VPSIGNB corner
// (activation code -128 against a negative weight) is applied as an exact correction on rows
// flagged by their quantizer.
//
// MFMA 16x16x32 lane layouts (checked on the device): A: lane l holds row l%16, k = 8(l/16)..+7;
// B: k = 8(l/16)..+7 of column l%16; D: rows 4(l/16)..+3 of column l%16. The bank's slice layout
// puts slices 2q and 2q+1 of a block (elements 8q..8q+7) in two 16-byte group entries, which is
// exactly lane group q's k range, so a lane's A operand is two dwords of the bank as stored.
//
// A workgroup (4 waves) computes 256 bank rows x one job tile (up to 64 jobs) of one expert; a wave owns
// 64 of the rows as a 4 x (up to 4) grid of 16 x 16 fragments. What bounds it is the vector ALU: one FMA
// per output and block is as long as the block's MFMA, and the weight conversions (MXFP4) or the
// int-to-float conversions (Q8_0) come on top, so the layout keeps everything else off it: weights
// in registers (no address or LDS work per operand), 64-row waves (four MFMAs per activation read) and
// sums placed under the MFMAs.
#include <algorithm>
#include <type_traits>

#include "vbm_device.hpp"
#include "vbm_internal.hpp"

namespace vbm {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_g __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4g __attribute__((ext_vector_type(4)));
typedef unsigned u32x2g __attribute__((ext_vector_type(2)));
typedef _Float16 half4_g __attribute__((ext_vector_type(4)));

constexpr int kGemmThreads = 256;
constexpr int kMxJobTile = 64;                             // the MXFP8 experiment's job tile

template <class T>
__device__ __forceinline__ const __attribute__((address_space(4))) T * cst(const void * p) {
    return (const __attribute__((address_space(4))) T *)(p);
}

// A wave-uniform pointer the compiler holds in vector registers, back in scalar ones.
template <class T>
__device__ __forceinline__ T * uniform_ptr(T * p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<T *>((static_cast<uint64_t>(hi) << 32) | lo);
}

struct GemmShape {
    int nb, rows, interleave;
    size_t slot_bytes;
    int64_t codes_bytes, n_slots;
};

struct GemmArgs {
    const uint8_t * bank;
    GemmShape shape;
    const int32_t * expert_to_slot;
    const uint8_t * rows_in;   // activation rows (GemmRowLayout lay)
    GemmRowLayout lay;
    int64_t n_ids, b_ne1;
    const int32_t * counts;
    const int32_t * offsets;
    const int32_t * jobs;      // grouped job list (token * n_ids + rank)
    const int32_t * tile_expert;
    const int32_t * tile_start;
    const int32_t * n_tiles;
    const float * bias;        // [n_expert][rows] in ggml row order, or null
    const float * row_scale;   // epilogue 0: per-job factor applied after the bias (routing weights), or null
    float * dst;               // epilogue 0: [job][rows]
    int row_units;             // 256-row units of the bank
    int split;                 // log2 of the most parts a job tile may run in (rows_item)
    uint8_t * rows_out;        // epilogue 1: GLU output rows for the down projection (out_lay)
    GemmRowLayout out_lay;
    int activation;
    float alpha, limit;
    int dst_vec4;              // epilogue 0: dst is 16-byte aligned (rows are multiples of 32)
};

__device__ __forceinline__ half2_g fp4x2(unsigned dw, int sel, float scale = 2.0f) {
    // sel is a compile-time constant at every call site after unrolling
    switch (sel) {
        case 0: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(dw, scale, 0);
        case 1: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(dw, scale, 1);
        case 2: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(dw, scale, 2);
        default: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(dw, scale, 3);
    }
}

// Weight operand of one block from the dwords w0, w1 of slices 2q, 2q+1 that hold it: MXFP4
// bytes 2b, 2b+1 of a 16-byte slice entry carry the slice's 4 nibbles of block b, so block b is
// half (b & 1) of dword b / 2. The e2m1 values come out multiplied by `scale` (a power of two):
// 2 gives the doubled-table integers; 2^(e+1) folds the block exponent e in as well.
__device__ __forceinline__ half8_t mx_a_operand(unsigned w0, unsigned w1, int odd, float scale = 2.0f) {
    half2_g p0, p1, p2, p3;
    if (odd) {
        p0 = fp4x2(w0, 2, scale), p1 = fp4x2(w0, 3, scale), p2 = fp4x2(w1, 2, scale), p3 = fp4x2(w1, 3, scale);
    } else {
        p0 = fp4x2(w0, 0, scale), p1 = fp4x2(w0, 1, scale), p2 = fp4x2(w1, 0, scale), p3 = fp4x2(w1, 1, scale);
    }
    return half8_t{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

// Exact VPSIGNB correction of one fragment column: contract minus true product is 256 * w for
// every element whose activation code is -128 and whose weight is negative. Computed by a second
// f16 MFMA on (min(w, 0), 256 [a == -128]) operands accumulating into the block dot (all partial
// sums stay integers below 2^24); only for waves holding flagged rows. Q8_0 takes the same route
// with its int8 codes widened to f16.
__device__ __forceinline__ half8_t neg_part(half8_t w) {
    half8_t r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = w[i] < static_cast<_Float16>(0.0f) ? w[i] : static_cast<_Float16>(0.0f);
    return r;
}
__device__ __forceinline__ half8_t is_neg128_x256(half8_t a) {
    half8_t r;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        r[i] = a[i] == static_cast<_Float16>(-128.0f) ? static_cast<_Float16>(256.0f) : static_cast<_Float16>(0.0f);
    return r;
}
__device__ __forceinline__ half8_t i8_to_f16(long v) {
    half8_t r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = static_cast<_Float16>(static_cast<signed char>(v >> (8 * i)));
    return r;
}
// Global-to-LDS DMA (global_load_lds_*): lane l's bytes land at LDS address m0 + l * size. The
// loads are issued through inline assembly so that the compiler's wait-count pass, which would
// wait for every such load before any LDS read it cannot prove disjoint, leaves the multi-stage
// ring alone; the kernel waits for them explicitly (lds_dma_wait) before each barrier. The
// compiler's own waits stay correct: loads it does not know of only make its counts stricter.
// M0 is a register the compiler reserves; the kernels of this file use it for nothing else (no
// v_movrel, s_sendmsg or LDS-DMA builtin: their assembly holds no other M0 access), so the
// clobber it is told of costs nothing and -Winline-asm's caution about reserved registers does
// not apply. A load to LDS reads M0 one wait state after a scalar write of it at the earliest: the
// compiler puts that s_nop between its own instructions, and it is written out here.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_dma_x4(const void * src, uint32_t m0) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m0) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void lds_dma_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The GLU of the fast accumulation order's epilogue: the formulas of glu() (SwiGLU-OAI with its
// clamps, or SiLU), with the device library's fast exp (__expf) and a fast divide (__fdividef)
// instead of the correctly rounded exp and the IEEE division the exact order needs. The fast
// order is held to the tolerance of the fp32 layer outputs, not to bits.
__device__ __forceinline__ float glu_fast(int activation, float g0, float u0, float alpha, float limit) {
    if (activation == VBM_ACT_SWIGLU_OAI) {
        const float g = limit < g0 ? limit : g0;
        const float u = u0 < -limit ? -limit : (limit < u0 ? limit : u0);
        return __fdividef(g, 1.0f + __expf(alpha * (-g))) * (u + 1.0f);
    }
    return __fdividef(g0, 1.0f + __expf(-g0)) * u0;
}

// ------------------------------------------------------------------------ MXFP4 grouped GEMM
// A wave owns 64 bank rows (a tile pair, so a whole 32-element GLU block of an interleaved bank) and
// up to 64 jobs: a 4 x 4 grid of 16 x 16 fragments. Its weights go from the bank straight into
// registers, one 8-block group ahead (no other wave of the workgroup needs them; as A operand, lane
// (q, r) of a fragment takes the 16-byte entries of slices 2q and 2q + 1 of its row as stored), and
// only the activation rows, which the workgroup's four waves all read, are staged in LDS: a stage is a
// bank group (eight blocks) of the codes and block scales of up to 64 jobs, two of them in turn, so
// one wait and one barrier per group. A workgroup takes 256 rows x one job tile.
// Each wave's block products are summed with one FMA per output and block in block order: the split
// over waves changes no bit of the result. One layer of 2048 tokens top-4 over 128 experts, hidden = inter =
// 2880: gate_up 976 -> 470..530 us, down 502 -> 255..290 us by box (512 to 578 and 468 to 533 TFLOP/s, from 278 and
// 271) against 32 x 32 waves with dword-staged weights; two-wave workgroups of 128 rows, a stage of half a group
// or 128-job tiles split over wave pairs measured 7 to 9 % slower.
// Registers are full (two workgroups per CU leave 256): 31 or 32 values are spilled, around the K loop, but for
// the kernel for caller-quantized rows, which holds both paths' code and reads four back in each group of four columns.
//
// The block exponents ride in the A operand when every exponent e of the wave's rows lies in
// [-14, 12] (2^(e+1) times the e2m1 values is then an exact normal f16), which the wave checks
// first; otherwise, and for waves holding -128 codes (FLAGGED), the wave takes the general path:
// doubled-integer operands, ldexp(d_act, e) per output, and the exact -128 correction.
struct MxStageLayout {
    static constexpr int kJobs = 64;
    static constexpr int ROW = 8 * 64;                         // f16 codes of a job and stage
    static constexpr int DA = kJobs * 8 * 4;                   // [job][8 blocks] fp32 block scales, both stages first
    static constexpr int OFF_ACT = 2 * DA, ACT = kJobs * ROW;  // (every fragment read then has a 16-bit offset)
    static constexpr int OFF_EXP = OFF_ACT + 2 * ACT;          // [stage][wave][64 rows] x 8 exponent bytes
    static constexpr int OFF_ROW = OFF_EXP + 2 * 4 * 512;      // [job] address of the row
    static constexpr int BYTES = OFF_ROW + kJobs * 8;
};
// Weights of a wave and group: entry [i][s] is slice 2q + s of row 16i + lr (dword d holds blocks
// 2d, 2d + 1). Their exponents are staged in LDS: as registers too they would spill.
struct MxGroupRegs {
    u32x4g c[4][2];
};

// Every stored exponent byte (signed e) of the dword in [-14, 12]: e + 14 and e + 19 both in [0, 32).
__device__ __forceinline__ unsigned mx_unfoldable(unsigned w) {
    const unsigned lo = w & 0x7F7F7F7Fu, sg = w & 0x80808080u;
    return (((lo + 0x0E0E0E0Eu) ^ sg) | ((lo + 0x13131313u) ^ sg)) & 0xE0E0E0E0u;
}

// A workgroup's work in the grouped GEMMs below: 256 rows (four tile pairs from pair0) of one expert x the
// live jobs of one job tile.
struct RowsItem {
    int expert, j0, joff, live, slot, pair0;
};

// Workgroups that the card holds at once (two per CU by LDS). A launch of few items splits every job tile into
// quarters or halves of 16 or 32 jobs (at most as the launch allows): a workgroup's K loop
// is then as long as its one or two fragment columns, not four, on CUs that would otherwise be idle, and the parts
// read the same weights, from L2. One expert of 4096 x 4096 and 64 tokens (16 items): Q8_0 66.8 -> 35 us, MXFP4 60.5 ->
// 38; 128 items, 32 jobs an expert: 59 -> 51 and 54 -> 49. Halves pay while CUs are left over: 64 rows for each of 8
// experts of 2880 x 2880 (142 items) Q8_0 57 -> 51 us; with one workgroup per CU already (256 items, 48 jobs) they
// took 93 against 78.
constexpr int kGemmSlots = 512;
__device__ __forceinline__ int tile_split(int n_items, int most) {   // log2 of a tile's parts
    const int fits = n_items * 4 <= kGemmSlots ? 2 : (n_items * 2 <= kGemmSlots - kGemmSlots / 8 ? 1 : 0);
    return fits < most ? fits : most;
}

// XCD-aware order: workgroup i runs on XCD i % 8, so each XCD takes a contiguous range of (tile, row unit) items;
// the units of one job tile share its activation rows in one L2. An XCD's first parts come before its second ones:
// the parts without jobs are then the last, not every other one, which left the live ones on every other CU (85
// tokens top-4 over 15 experts of 2880 x 2880: 110 against 80 us). False: no item, or one whose expert is not
// resident in this bank. The latter writes NaN outputs, as the decode kernels do (a tile filter removes the experts a
// pass skips on purpose, so this is a bad map).
template <int EPI>
__device__ __forceinline__ bool rows_item(const GemmArgs & A, int job_tile, RowsItem & it) {
    const int n_items = *cst<int32_t>(A.n_tiles) * A.row_units, split = tile_split(n_items, A.split);
    const int per_xcd = (n_items + 7) >> 3;
    const int slot8 = static_cast<int>(blockIdx.x >> 3);
    if (slot8 >= per_xcd << split) return false;
    const int part = slot8 >= 2 * per_xcd ? (slot8 >= 3 * per_xcd ? 3 : 2) : (slot8 >= per_xcd ? 1 : 0);
    const int item = static_cast<int>(blockIdx.x & 7) * per_xcd + slot8 - part * per_xcd;
    if (item >= n_items) return false;
    const int ti = item / A.row_units;
    it.pair0 = (item - ti * A.row_units) * 4;
    it.expert = cst<int32_t>(A.tile_expert)[ti];
    const int count = cst<int32_t>(A.counts)[it.expert];
    int t0 = cst<int32_t>(A.tile_start)[ti], share = job_tile;
    if (count > job_tile && n_items <= kGemmSlots) {
        // all items run at once: an expert's tiles share its jobs evenly, in fragment columns of 16, so that
        // 80 jobs run as 48 + 32, not 64 + 16 (80 jobs each of 24 experts, 1536 x 4096: Q8_0 107 -> 92 us)
        const int tiles = (count + job_tile - 1) / job_tile;
        share = ((count + tiles - 1) / tiles + 15) & ~15;
        t0 = t0 / job_tile * share;
    }
    const int p0 = part * (job_tile >> split);
    it.j0 = t0 + p0;
    it.joff = cst<int32_t>(A.offsets)[it.expert];
    it.slot = A.expert_to_slot ? cst<int32_t>(A.expert_to_slot)[it.expert] : it.expert;
    it.live = std::min(std::min(count - t0, share) - p0, job_tile >> split);
    if (it.live <= 0) return false;                          // a part past the tile's last job
    const GemmShape & S = A.shape;
    if (it.slot >= 0 && it.slot < S.n_slots) return true;
    const float nan = __builtin_nanf("");
    if (EPI == 0) {
        for (int i = threadIdx.x; i < it.live * 256; i += kGemmThreads) {
            const int64_t brow = static_cast<int64_t>(it.pair0) * 64 + i % 256;
            if (brow < S.rows)
                A.dst[static_cast<size_t>(A.jobs[it.joff + it.j0 + i / 256]) * S.rows + ggml_row(brow, S.rows, S.interleave)] = nan;
        }
    } else {
        for (int i = threadIdx.x; i < it.live * 4; i += kGemmThreads)
            if ((it.pair0 + i % 4) * 64 < S.rows)
                reinterpret_cast<float *>(A.rows_out + static_cast<int64_t>(A.jobs[it.joff + it.j0 + i / 4]) * A.out_lay.stride() +
                                          A.out_lay.da_offset())[it.pair0 + i % 4] = nan;
    }
    return false;
}

// Activation row of live local job jl.
__device__ __forceinline__ const uint8_t * job_row(const GemmArgs & A, const RowsItem & it, int jl) {
    const uint32_t jb = static_cast<uint32_t>(A.jobs[it.joff + it.j0 + jl]);
    return A.rows_in + A.lay.row_offset(A.b_ne1 == 1 ? jb / static_cast<uint32_t>(A.n_ids) : jb);
}

// Epilogue, from registers: lane (q, lr) holds rows 16i + 4q .. + 3 of tile pair `pair` for job 16jh + lr, jh < nf.
// Biases (ggml row order), then fp32 rows (times the routing weight when given) as one 16-byte store per
// fragment, or GLU + Q8_0 requantization: fragments 0 / 1 and 2 / 3 are the gate / up rows of the block's
// elements 4q .. + 3 and 16 + 4q .. + 3.
template <int TYPE, int EPI>
__device__ __forceinline__ void rows_epilogue(const GemmArgs & A, const RowsItem & it, int pair, int nf, const f32x4 (&acc)[4][4]) {
    const GemmShape & S = A.shape;
    const int lane = threadIdx.x & 63, lr = lane & 15, q = lane >> 4;
    const bool two_tiles = pair * 64 + 32 < S.rows;          // the last pair may be one tile
    // ggml rows of the lane's fragments: aligned runs of 4 device rows are 4 consecutive ggml rows, also in
    // interleaved banks (tile 2 pair + i / 2; its rows 16.. are the up rows there)
    uint32_t grow[4];
    float bias[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        grow[i] = S.interleave ? static_cast<uint32_t>((i & 1) * (S.rows / 2) + (2 * pair + (i >> 1)) * 16 + 4 * q)
                               : static_cast<uint32_t>(64 * pair + 16 * i + 4 * q);
        const bool row_live = i < 2 || two_tiles;
#pragma unroll
        for (int j = 0; j < 4; ++j) bias[i][j] = A.bias && row_live ? A.bias[static_cast<size_t>(it.expert) * S.rows + grow[i] + j] : 0.0f;
    }
    int jobs[4];
    float scales[4];
#pragma unroll
    for (int jh = 0; jh < 4; ++jh) jobs[jh] = A.jobs[it.joff + it.j0 + (16 * jh + lr < it.live ? 16 * jh + lr : 0)];
#pragma unroll
    for (int jh = 0; jh < 4; ++jh) scales[jh] = EPI == 0 && A.row_scale ? A.row_scale[jobs[jh]] : 1.0f;
#pragma unroll
    for (int jh = 0; jh < 4; ++jh) {
        if (jh >= nf) break;
        const bool jlive = 16 * jh + lr < it.live;
        const int job = jobs[jh];
        if constexpr (EPI == 0) {
            const float rs = scales[jh];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!jlive || (i >= 2 && !two_tiles)) continue;
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = acc[i][jh][j];
                    if (A.bias) v[j] = v[j] + bias[i][j];
                    if (A.row_scale) v[j] = v[j] * rs;
                }
                float * out = A.dst + static_cast<size_t>(job) * S.rows + grow[i];
                if (A.dst_vec4) {
                    f32x4 vv = {v[0], v[1], v[2], v[3]};
                    asm volatile("" : "+v"(vv));             // (merged with the scalar form it becomes dword stores)
                    *reinterpret_cast<f32x4 *>(out) = vv;
                } else {
                    asm volatile("" : "+v"(out));
#pragma unroll
                    for (int j = 0; j < 4; ++j) out[j] = v[j];
                }
            }
        } else {
            float x[2][4], amax = 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float gv = acc[2 * t][jh][j], uv = acc[2 * t + 1][jh][j];
                    if (A.bias) gv = gv + bias[2 * t][j], uv = uv + bias[2 * t + 1][j];
                    x[t][j] = glu_fast(A.activation, gv, uv, A.alpha, A.limit);
                    amax = fmaxf(amax, fabsf(x[t][j]));
                }
            amax = fmaxf(amax, __shfl_xor(amax, 16));        // the block's other lanes of this job
            amax = fmaxf(amax, __shfl_xor(amax, 32));
            const float d = amax / 127.0f;
            const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
            if (!jlive) continue;
            uint8_t * out = A.rows_out + static_cast<int64_t>(job) * A.out_lay.stride();
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                half4_g c;
                unsigned c8 = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float v = rintf(x[t][j] * id);
                    v = v > 127.0f ? 127.0f : (v < -128.0f ? -128.0f : v);
                    if (TYPE == 39) c[j] = static_cast<_Float16>(v);
                    else c8 |= static_cast<unsigned>(static_cast<uint8_t>(static_cast<signed char>(v))) << (8 * j);
                }
                const int64_t e0 = static_cast<int64_t>(pair) * 32 + 16 * t + 4 * q;
                if (TYPE == 39) *reinterpret_cast<half4_g *>(out + e0 * 2) = c;
                else *reinterpret_cast<unsigned *>(out + e0) = c8;
            }
            if (q == 0) {
                reinterpret_cast<float *>(out + A.out_lay.da_offset())[pair] = static_cast<float>(static_cast<_Float16>(d));
                if (pair == 0) *reinterpret_cast<int *>(out + A.out_lay.flag_offset()) = 0;   // never -128
            }
        }
    }
}

template <int EPI, bool FLAGGED>
__global__ __launch_bounds__(kGemmThreads, 2) void mx_rows_gemm_kernel(GemmArgs A) {
    using L = MxStageLayout;
    __shared__ __attribute__((aligned(256))) uint8_t lds[L::BYTES];
    RowsItem it;
    if (!rows_item<EPI>(A, L::kJobs, it)) return;
    const GemmShape S = A.shape;
    const int live = it.live;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int lr = lane & 15, q = lane >> 4;
    const int nb = S.nb, groups = nb / 8, tail = nb % 8;
    const int n_groups = groups + (tail ? 1 : 0);
    const int pair = it.pair0 + wave;
    const bool pair_live = pair * 64 < S.rows;
    const int nf = pair_live ? (live + 15) / 16 : 0;         // live fragment columns, 0..4
    const uint8_t * slot_base = A.bank + static_cast<size_t>(it.slot) * S.slot_bytes;

    // weight stream: a buffer descriptor over the pair's codes (a dead pair reads the unit's first pair
    // and drops it; a missing second tile reads the first)
    const int src_pair = pair_live ? pair : it.pair0;
    const int tile1 = __builtin_amdgcn_readfirstlane(src_pair * 64 + 32 < S.rows ? 1 : 0);   // index of fragments 2, 3's tile
    const int code_tile = 32 * nb * 16, meta_tile = 32 * nb;
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(const_cast<uint8_t *>(slot_base + static_cast<size_t>(src_pair) * 2 * code_tile)), static_cast<short>(0),
        __builtin_amdgcn_readfirstlane((1 + tile1) * code_tile), 0x00020000);
    const uint8_t * exp_base = slot_base + S.codes_bytes + static_cast<size_t>(src_pair) * 2 * meta_tile;
    // A full group holds 16 bytes of codes per (slice, row) and 8 exponent bytes per row, the tail's 2, 4
    // or 6 blocks 2 tail and tail bytes. The tail takes the same code loads with its own lane stride:
    // what they read past a row's entry is not used (past the descriptor: zeros).
    auto load_group = [&](int g, MxGroupRegs & w) __attribute__((always_inline)) {
        const int cs = g < groups ? 16 : 2 * tail;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int so = (i >> 1) * tile1 * code_tile + g * 4096;
            w.c[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rc, (2 * q * 32 + 16 * (i & 1) + lr) * cs, so, 0);
            w.c[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rc, ((2 * q + 1) * 32 + 16 * (i & 1) + lr) * cs, so, 0);
        }
    };
    // The loads of `w` are complete (an lds_dma_wait<0> came before): a use that takes the compiler's
    // own wait for them here, where it costs nothing. At their first real use, behind the next
    // stage's DMA, that wait would be for the DMA too.
    auto landed = [&](MxGroupRegs & w) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(w.c[i][0]), "+v"(w.c[i][1]));
    };
    // Fold check over every exponent of the wave's rows (k <= 4096: 8 KiB at most; all loads in flight
    // together).
    unsigned unfold = 0;
    {
        u32x4g m[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int o = lane * 16 + i * 1024;
            m[i] = *reinterpret_cast<const u32x4g *>(exp_base + (o < (1 + tile1) * meta_tile ? o : 0));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) unfold |= mx_unfoldable(m[i][0]) | mx_unfoldable(m[i][1]) | mx_unfoldable(m[i][2]) | mx_unfoldable(m[i][3]);
    }

    // activation stages: DMA k = wave + 4i (1 KiB) holds jobs 2k, 2k + 1; the 16-byte part p = 4b + q of a
    // job's 512 bytes sits at part p ^ (job & 15), so that a fragment read (16 jobs, one part) covers
    // all banks. A load whose jobs are all past the tile's live ones is skipped; a dead job in a load
    // with a live one reads the tile's first job.
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const int part = (lane & 31) ^ (2 * wave + (lane >> 5)); // of the loads with even i; odd i flip bit 3 (2k mod 16)
    const int djob = 32 * (wave & 1) + (lane >> 1);          // block scales: waves 0 and 1, 32 jobs x 32 bytes
    const uint32_t da_off = static_cast<uint32_t>(A.lay.da_offset());
    const uint8_t ** row_tab = reinterpret_cast<const uint8_t **>(lds + L::OFF_ROW);
    if (threadIdx.x < L::kJobs) row_tab[threadIdx.x] = job_row(A, it, static_cast<int>(threadIdx.x) < live ? static_cast<int>(threadIdx.x) : 0);
    __syncthreads();
    // (the rows' addresses are read back from LDS by every group: kept in registers they would spill, and
    // the spills' reloads wait for the DMA in flight)
    auto dma_stage = [&](int g) __attribute__((always_inline)) {
        const uint32_t sb = lds0 + L::OFF_ACT + (g & 1) * L::ACT;
        const uint8_t * row[8], * drow = row_tab[djob];
#pragma unroll
        for (int i = 0; i < 8; ++i) row[i] = row_tab[2 * (wave + 4 * i) + (lane >> 5)];
        // the tail's stage: parts past its blocks read one of the first two blocks' again
        const int parts = g < groups ? 32 : 4 * tail;
        const uint32_t pe = g * L::ROW + 16 * (part < parts ? part : part & 7);
        const uint32_t po = g * L::ROW + 16 * ((part ^ 8) < parts ? part ^ 8 : part & 7);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = wave + 4 * i;
            if (2 * k < live) lds_dma_x4(row[i] + (i & 1 ? po : pe), sb + k * 1024);
        }
        if (wave < 2 && 32 * wave < live)                    // (a tail of at most four blocks has no second 16 bytes)
            lds_dma_x4(drow + (da_off + 16 * (2 * g + (parts > 16 ? lane & 1 : 0))),
                       lds0 + (g & 1) * L::DA + wave * 1024);
    };
    // the wave's exponents of group g: lanes 0..15 / 16..31 bring the 256 bytes of its two tiles (the
    // tail's 32 tail bytes)
    auto dma_exps = [&](int g) __attribute__((always_inline)) {
        if (lane < 32 && (lane & 15) * 16 < 32 * (g < groups ? 8 : tail))
            lds_dma_x4(exp_base + (lane >> 4) * tile1 * meta_tile + g * 256 + (lane & 15) * 16,
                       lds0 + L::OFF_EXP + ((g & 1) * 4 + wave) * 512);
    };

    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jh = 0; jh < 4; ++jh) acc[i][jh] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bool flagged = false;                                    // wave-uniform: a live job holds -128 codes
    if constexpr (FLAGGED) {
        int f = 0;
        if (lane < live)
            f = *reinterpret_cast<const int *>(job_row(A, it, lane) + A.lay.flag_offset());
        flagged = __any(f != 0);
    }

    // K loop over NF live fragment columns; GENERAL: the general path (see above).
    auto k_loop = [&](auto nf_c, auto general_c) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf_c)::value;
        constexpr bool GENERAL = decltype(general_c)::value;
        // this lane's part of block 0 of fragment column 0; block b's is at the address with bits 6..8
        // flipped by b (recomputed from an opaque copy at each use, a register less per block)
        const uint32_t act0 = static_cast<uint32_t>(lr * L::ROW + ((q ^ lr) << 4));
        // Blocks 4H .. of group g (stage ST), its weights in w (nblk: 4, or 2 at the end of a row); TAIL:
        // exponents packed by tail bytes per row. `issue` starts the next group's DMA and loads: the
        // half's first LDS reads go out before it, so that they land while it issues.
        auto half_group = [&](int ST, auto h_c, auto tail_c, const MxGroupRegs & w, int nblk, auto && issue) __attribute__((always_inline)) {
            constexpr int H = decltype(h_c)::value;
            constexpr bool TAIL = decltype(tail_c)::value;
            const uint8_t * exps = lds + L::OFF_EXP + (ST * 4 + wave) * 512;
            auto exp_dword = [&](int i, int r) __attribute__((always_inline)) -> unsigned {   // row r of fragment i
                if constexpr (!TAIL) return *reinterpret_cast<const unsigned *>(exps + i * 128 + r * 8 + 4 * H);
                const uint16_t * p = reinterpret_cast<const uint16_t *>(exps + (i >> 1) * 256 + (16 * (i & 1) + r) * tail + 4 * H);
                return static_cast<unsigned>(p[0]) | (static_cast<unsigned>(p[1]) << 16);
            };
            f32x4 da[NF];
#pragma unroll
            for (int jh = 0; jh < NF; ++jh)
                da[jh] = *reinterpret_cast<const f32x4 *>(lds + ST * L::DA + (16 * jh + lr) * 32 + 16 * H);
            uint32_t ablk = act0;
            auto act = [&](int jh, int bb) __attribute__((always_inline)) {
                return *reinterpret_cast<const half8_t *>(lds + L::OFF_ACT + ST * L::ACT + jh * 16 * L::ROW + (ablk ^ ((4 * H + bb) << 6)));
            };
            if constexpr (!GENERAL) {
                constexpr int PB = 2;                        // activation operands read this many steps ahead
                half8_t a_op[4], bv[PB + 1];
                unsigned ew[4];                              // raw e8m0 bytes of the half's four blocks
#pragma unroll
                for (int i = 0; i < 4; ++i) ew[i] = exp_dword(i, lr);
#pragma unroll
                for (int t = 0; t < PB; ++t) bv[t] = act(t % NF, t / NF);
                issue();
#pragma unroll
                for (int i = 0; i < 4; ++i) ew[i] ^= 0x80808080u;
                auto weights = [&](int i, int bb) __attribute__((always_inline)) {
                    const float sc = bb == 0 ? exp2_byte<0>(ew[i]) : (bb == 1 ? exp2_byte<1>(ew[i]) : (bb == 2 ? exp2_byte<2>(ew[i]) : exp2_byte<3>(ew[i])));   // 2^(e+1)
                    return mx_a_operand(w.c[i][0][2 * H + (bb >> 1)], w.c[i][1][2 * H + (bb >> 1)], bb & 1, sc);
                };
                // Software pipeline over the (block, column) steps: fragment i's product of the previous
                // step is summed right before its register takes this step's MFMA (a matrix result is
                // some 16 cycles away; left to itself the compiler waits for each). A step also reads the
                // next step's activation operand and, at a block's last column, converts the next
                // block's weights.
                f32x4 d[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) a_op[i] = weights(i, 0);
                auto sum = [&](int t, int i) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][t % NF][j] = __builtin_fmaf(da[t % NF][t / NF], d[i][j], acc[i][t % NF][j]);
                };
#pragma unroll
                for (int t = 0; t < 4 * NF; ++t) {
                    if (t == 2 * NF && nblk <= 2) break;
                    if ((t + PB) % NF == 0) asm volatile("" : "+v"(ablk));
                    if (t + PB < 4 * NF) bv[(t + PB) % (PB + 1)] = act((t + PB) % NF, (t + PB) / NF);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (t > 0) sum(t - 1, i);
                        d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_op[i], bv[t % (PB + 1)], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                        if (t % NF == NF - 1 && t / NF < 3) a_op[i] = weights(i, t / NF + 1);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);          // the activation read
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (t > 0) __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);             // the sums,
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                        // one MFMA,
                        if (t % NF == NF - 1) __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);  // the conversion
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (nblk <= 2) sum(2 * NF - 1, i);
                    else sum(4 * NF - 1, i);
                }
                // keeps the sums in this place: moved past the branches that follow the half group, they
                // would hold every block's products in registers
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int jh = 0; jh < NF; ++jh) asm volatile("" : "+v"(acc[i][jh]));
            } else {
                issue();
#pragma clang loop unroll(disable)
                for (int bb = 0; bb < nblk; ++bb) {
                    half8_t bv[NF];
                    float dv[NF];
#pragma unroll
                    for (int jh = 0; jh < NF; ++jh) {
                        bv[jh] = act(jh, bb);
                        dv[jh] = bb == 0 ? da[jh][0] : (bb == 1 ? da[jh][1] : (bb == 2 ? da[jh][2] : da[jh][3]));
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const unsigned w0 = bb < 2 ? w.c[i][0][2 * H] : w.c[i][0][2 * H + 1];
                        const unsigned w1 = bb < 2 ? w.c[i][1][2 * H] : w.c[i][1][2 * H + 1];
                        const half8_t a_op = mx_a_operand(w0 >> (16 * (bb & 1)), w1 >> (16 * (bb & 1)), 0);
                        int e[4];                            // exponents of output rows 16i + 4q + j
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            e[j] = static_cast<signed char>(exp_dword(i, 4 * q + j) >> (8 * bb));
#pragma unroll
                        for (int jh = 0; jh < NF; ++jh) {
                            f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_op, bv[jh], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                            if constexpr (FLAGGED)
                                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(neg_part(a_op), is_neg128_x256(bv[jh]), d, 0, 0, 0);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                acc[i][jh][j] = __builtin_fmaf(__builtin_amdgcn_ldexpf(dv[jh], e[j]), d[j], acc[i][jh][j]);
                        }
                    }
                }
            }
        };
        constexpr std::integral_constant<int, 0> h0{};
        constexpr std::integral_constant<int, 1> h1{};
        // One full group: its weights are in `cur`; the next group's loads go into `nxt` (past the last
        // group: the last one's again, so that the loads have no branch around them and the
        // compiler's wait counts stay exact).
        auto group_step = [&](int st, int g, const MxGroupRegs & cur, MxGroupRegs & nxt) __attribute__((always_inline)) {
            const bool next = g + 1 < n_groups;
            half_group(st, h0, std::false_type{}, cur, 4, [&] {
                if (next) {
                    dma_stage(g + 1);
                    dma_exps(g + 1);
                }
                load_group(__builtin_amdgcn_readfirstlane(next ? g + 1 : g), nxt);
            });
            half_group(st, h1, std::false_type{}, cur, 4, [] {});
            lds_dma_wait<0>();
            landed(nxt);
            __syncthreads();
        };
        MxGroupRegs wa, wb;
        load_group(0, wa);
        lds_dma_wait<0>();
        landed(wa);
        __syncthreads();
#pragma clang loop unroll(disable)
        for (int g = 0; g < groups; g += 2) {
            group_step(0, g, wa, wb);
            if (g + 1 < groups) group_step(1, g + 1, wb, wa);
            else wa = wb;
        }
        if (tail) {   // 2, 4 or 6 blocks
            half_group(groups & 1, h0, std::true_type{}, wa, tail < 4 ? tail : 4, [] {});
            if (tail == 6) half_group(groups & 1, h1, std::true_type{}, wa, 2, [] {});
        }
    };
    dma_stage(0);
    dma_exps(0);
    // Waves may take different instantiations: each issues the same stage loads and reaches the same
    // number of barriers.
    const bool general = __any(unfold != 0) || flagged;
    if (nf == 0) {
        lds_dma_wait<0>();
        __syncthreads();
        for (int g = 1; g < n_groups; ++g) {
            dma_stage(g);
            lds_dma_wait<0>();
            __syncthreads();
        }
        if (!tail) __syncthreads();
        return;
    }
    constexpr std::false_type fold{};
    if (general) k_loop(std::integral_constant<int, 4>{}, std::true_type{});
    else if (nf == 4) k_loop(std::integral_constant<int, 4>{}, fold);
    else if (nf == 3) k_loop(std::integral_constant<int, 3>{}, fold);
    else if (nf == 2) k_loop(std::integral_constant<int, 2>{}, fold);
    else k_loop(std::integral_constant<int, 1>{}, fold);
    rows_epilogue<39, EPI>(A, it, pair, nf, acc);
}

// ------------------------------------------------------------------------- Q8_0 grouped GEMM
// The same work split as the MXFP4 kernel above (64 rows x up to 64 jobs per wave, weights in registers,
// activation stages of eight blocks in LDS) for int8 codes: a bank group is four blocks, so a stage is two
// of them, each prefetched half a stage ahead. Block dots come from v_mfma_i32_16x16x32_i8, and the scale
// products fp16(d_w) * d_act of four blocks of a 16 x 16 fragment from one v_mfma_f32_16x16x4_4b_f16, whose
// four K = 4 blocks each hold one quantization block's scales at k = 0 and zeros: exact fp32 products of
// two fp16 values, a quarter of a matrix instruction per block and nothing on the vector ALU, which is
// left the int-to-float conversion and the FMA of every output and block. One layer of 2048 tokens top-8 over 128
// experts, hidden 2048, inter 768: gate_up 260 -> 200..212 us, down 180 -> 122..133 us by box against the former 32-row
// waves. 14 to 16 values are spilled, around the K loop. The kernel for caller-quantized rows spills 172: it reads ten back
// per block of the -128 path, and in its full stages one for four columns and five for two; rows without such codes take
// 45 to 51 us where the former kernel, which spilled none, took 94 (517 tokens x 6 ids over 64 experts, 2048 x 1408).
struct Q8StageLayout {
    static constexpr int kJobs = 64;
    static constexpr int ROW = 8 * 32;                         // int8 codes of a job and stage
    static constexpr int DA = kJobs * 8 * 4;                   // [job][8 blocks] fp32 block scales, both stages first
    static constexpr int OFF_ACT = 2 * DA, ACT = kJobs * ROW;
    static constexpr int OFF_SC = OFF_ACT + 2 * ACT;           // [stage][wave][tile][group][32 rows] x 4 fp16
    static constexpr int OFF_ROW = OFF_SC + 2 * 4 * 1024;      // [job] address of the row
    static constexpr int BYTES = OFF_ROW + kJobs * 8;
};
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int EPI, bool FLAGGED>
__global__ __launch_bounds__(kGemmThreads, 2) void q8_rows_gemm_kernel(GemmArgs A) {
    using L = Q8StageLayout;
    __shared__ __attribute__((aligned(256))) uint8_t lds[L::BYTES];
    RowsItem it;
    if (!rows_item<EPI>(A, L::kJobs, it)) return;
    const GemmShape S = A.shape;
    const int live = it.live;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int lr = lane & 15, q = lane >> 4;
    const int nb = S.nb, stages = nb / 8, tail = nb % 8;      // full stages; blocks of a last partial one
    const int n_stages = stages + (tail ? 1 : 0);
    const int groups = nb / 4, n_groups = groups + (nb % 4 ? 1 : 0);   // a bank tail holds two blocks
    const int pair = it.pair0 + wave;
    const bool pair_live = pair * 64 < S.rows;
    const int nf = pair_live ? (live + 15) / 16 : 0;         // live fragment columns, 0..4
    const uint8_t * slot_base = A.bank + static_cast<size_t>(it.slot) * S.slot_bytes;

    // weight stream, as in the MXFP4 kernel
    const int src_pair = pair_live ? pair : it.pair0;
    const int tile1 = __builtin_amdgcn_readfirstlane(src_pair * 64 + 32 < S.rows ? 1 : 0);   // index of fragments 2, 3's tile
    const int code_tile = 32 * nb * 32, scale_tile = 32 * nb * 2;
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(const_cast<uint8_t *>(slot_base + static_cast<size_t>(src_pair) * 2 * code_tile)), static_cast<short>(0),
        __builtin_amdgcn_readfirstlane((1 + tile1) * code_tile), 0x00020000);
    const uint8_t * scale_base = slot_base + S.codes_bytes + static_cast<size_t>(src_pair) * 2 * scale_tile;
    auto load_group = [&](int g, MxGroupRegs & w) __attribute__((always_inline)) {
        const int cs = g < groups ? 16 : 8;                  // bytes per (slice, row)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int so = (i >> 1) * tile1 * code_tile + g * 4096;
            w.c[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rc, (2 * q * 32 + 16 * (i & 1) + lr) * cs, so, 0);
            w.c[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rc, ((2 * q + 1) * 32 + 16 * (i & 1) + lr) * cs, so, 0);
        }
    };
    auto landed = [&](MxGroupRegs & w) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(w.c[i][0]), "+v"(w.c[i][1]));
    };

    // activation stages: DMA k = wave + 4i (1 KiB) holds jobs 4k..4k + 3; the 16-byte part p = 2b + q / 2 of a
    // job's 256 bytes sits at part p ^ (job & 15)
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const int part = (lane & 15) ^ (4 * wave + (lane >> 4)); // 4k = 4 wave (mod 16): one part for every load
    const int djob = 32 * (wave & 1) + (lane >> 1);          // block scales: waves 0 and 1, 32 jobs x 32 bytes
    const uint32_t da_off = static_cast<uint32_t>(A.lay.da_offset());
    const uint8_t ** row_tab = reinterpret_cast<const uint8_t **>(lds + L::OFF_ROW);
    if (threadIdx.x < L::kJobs) row_tab[threadIdx.x] = job_row(A, it, static_cast<int>(threadIdx.x) < live ? static_cast<int>(threadIdx.x) : 0);
    __syncthreads();
    auto dma_stage = [&](int s) __attribute__((always_inline)) {
        const uint32_t sb = lds0 + L::OFF_ACT + (s & 1) * L::ACT;
        const uint8_t * row[4], * drow = row_tab[djob];
#pragma unroll
        for (int i = 0; i < 4; ++i) row[i] = row_tab[4 * (wave + 4 * i) + (lane >> 4)];
        // the last stage: parts past its blocks read one of the first two blocks' again
        const int parts = s < stages ? 16 : 2 * tail;
        const uint32_t p = s * L::ROW + 16 * (part < parts ? part : part & 3);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = wave + 4 * i;
            if (4 * k < live) lds_dma_x4(row[i] + p, sb + k * 1024);
        }
        if (wave < 2 && 32 * wave < live)                    // (a tail of at most four blocks has no second 16 bytes)
            lds_dma_x4(drow + (da_off + 16 * (2 * s + (parts > 8 ? lane & 1 : 0))), lds0 + (s & 1) * L::DA + wave * 1024);
    };
    // the wave's weight scales of stage s: each half-wave brings the 512 bytes of one tile (the last
    // stage's: 64 bytes per block)
    auto dma_scales = [&](int s) __attribute__((always_inline)) {
        if ((lane & 31) * 16 < 64 * (s < stages ? 8 : tail))
            lds_dma_x4(scale_base + (lane >> 5) * tile1 * scale_tile + s * 512 + (lane & 31) * 16,
                       lds0 + L::OFF_SC + ((s & 1) * 4 + wave) * 1024);
    };

    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jh = 0; jh < 4; ++jh) acc[i][jh] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bool flagged = false;                                    // wave-uniform: a live job holds -128 codes
    if constexpr (FLAGGED) {
        int f = 0;
        if (lane < live)
            f = *reinterpret_cast<const int *>(job_row(A, it, lane) + A.lay.flag_offset());
        flagged = __any(f != 0);
    }

    // K loop over NF live fragment columns; GENERAL: with the exact -128 correction.
    auto k_loop = [&](auto nf_c, auto general_c) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf_c)::value;
        constexpr bool GENERAL = decltype(general_c)::value;
        // this lane's 8 bytes of block 0 of fragment column 0; block b's are at the address with bits 5..7
        // flipped by b
        const uint32_t act0 = static_cast<uint32_t>(lr * L::ROW + (((q >> 1) ^ lr) << 4) + 8 * (q & 1));
        // Bank group H of stage buffer st, its weights in w (nblk: 4, or the bank tail's 2, whose scales are
        // packed by two per row).
        auto half_stage = [&](int st, int H, const MxGroupRegs & w, int nblk, auto && issue) __attribute__((always_inline)) {
            const uint8_t * sc_lds = lds + L::OFF_SC + (st * 4 + wave) * 1024 + H * 256;
            const int srow = 2 * nblk;                       // scale bytes per row
            const uint8_t * da_lds = lds + st * L::DA + 16 * H;
            const uint8_t * act_lds = lds + L::OFF_ACT + st * L::ACT;
            const uint32_t ah = act0 ^ (H << 7);
            auto act = [&](int jh, int bb) __attribute__((always_inline)) {
                return *reinterpret_cast<const long *>(act_lds + jh * 16 * L::ROW + (ah ^ (bb << 5)));
            };
            if constexpr (!GENERAL) {
                half4_g as[4], bs[NF];                       // scales of block q of the group, at k = 0
                unsigned dw[4];
                float da[NF];
                long bv[2][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) dw[i] = *reinterpret_cast<const uint16_t *>(sc_lds + (i >> 1) * 512 + (16 * (i & 1) + lr) * srow + 2 * q);
#pragma unroll
                for (int jh = 0; jh < NF; ++jh) da[jh] = *reinterpret_cast<const float *>(da_lds + (16 * jh + lr) * 32 + 4 * q);
#pragma unroll
                for (int bb = 0; bb < 4; ++bb) bv[0][bb] = act(0, bb);
                issue();
#pragma unroll
                for (int i = 0; i < 4; ++i) as[i] = __builtin_bit_cast(half4_g, u32x2g{dw[i], 0u});
#pragma unroll
                for (int jh = 0; jh < NF; ++jh)              // d_act holds fp16 values: exact
                    bs[jh] = __builtin_bit_cast(half4_g, u32x2g{__builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(da[jh], 0.0f)), 0u});
                // Software pipeline over the (column, fragment) steps: block bb's product of the previous step is
                // scaled and summed right before its register takes this step's MFMA.
                i32x4 d[4];
                f32x16 sc[2];
                auto sum = [&](int t, int bb) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[t % 4][t / 4][j] = __builtin_fmaf(sc[t & 1][4 * bb + j], static_cast<float>(d[bb][j]), acc[t % 4][t / 4][j]);
                };
#pragma unroll
                for (int t = 0; t < 4 * NF; ++t) {
                    const int i = t % 4, jh = t / 4;
                    sc[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f16(as[i], bs[jh], f32x16{}, 0, 0, 0);
                    if (i == 0 && jh + 1 < NF) {
#pragma unroll
                        for (int bb = 0; bb < 4; ++bb) bv[(jh + 1) & 1][bb] = act(jh + 1, bb);
                    }
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        if (bb >= 2 && nblk <= 2) break;
                        if (t > 0) sum(t - 1, bb);
                        const long a = static_cast<long>(static_cast<uint64_t>(w.c[i][0][bb]) | (static_cast<uint64_t>(w.c[i][1][bb]) << 32));
                        d[bb] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, bv[jh & 1][bb], i32x4{0, 0, 0, 0}, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    if (i == 0 && jh + 1 < NF) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
                    for (int bb = 0; bb < 4; ++bb) {
                        if (t > 0) __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int bb = 0; bb < 4; ++bb)
                    if (bb < 2 || nblk > 2) sum(4 * NF - 1, bb);
                // keeps the sums in this place (see the MXFP4 kernel)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int jh = 0; jh < NF; ++jh) asm volatile("" : "+v"(acc[i][jh]));
            } else {
                issue();
#pragma clang loop unroll(disable)
                for (int bb = 0; bb < nblk; ++bb) {
                    half8_t b16[NF];
                    float da[NF];
#pragma unroll
                    for (int jh = 0; jh < NF; ++jh) {
                        b16[jh] = i8_to_f16(act(jh, bb));
                        da[jh] = *reinterpret_cast<const float *>(da_lds + (16 * jh + lr) * 32 + 4 * bb);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        auto pick = [&](const u32x4g & c) __attribute__((always_inline)) { return bb == 0 ? c[0] : (bb == 1 ? c[1] : (bb == 2 ? c[2] : c[3])); };
                        const half8_t a16 = i8_to_f16(static_cast<long>(static_cast<uint64_t>(pick(w.c[i][0])) | (static_cast<uint64_t>(pick(w.c[i][1])) << 32)));
                        float dw[4];                         // scales of output rows 16i + 4q + j
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            dw[j] = half_bits_to_float(*reinterpret_cast<const uint16_t *>(sc_lds + (i >> 1) * 512 + (16 * (i & 1) + 4 * q + j) * srow + 2 * bb));
#pragma unroll
                        for (int jh = 0; jh < NF; ++jh) {
                            f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a16, b16[jh], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(neg_part(a16), is_neg128_x256(b16[jh]), d, 0, 0, 0);
#pragma unroll
                            for (int j = 0; j < 4; ++j) acc[i][jh][j] = __builtin_fmaf(dw[j] * da[jh], d[j], acc[i][jh][j]);
                        }
                    }
                }
            }
        };
        MxGroupRegs wa, wb;
        load_group(0, wa);
        lds_dma_wait<0>();
        landed(wa);
        __syncthreads();
#pragma clang loop unroll(disable)
        for (int s = 0; s < stages; ++s) {
            const int st = s & 1;
            half_stage(st, 0, wa, 4, [&]() __attribute__((always_inline)) {
                if (s + 1 < n_stages) {
                    dma_stage(s + 1);
                    dma_scales(s + 1);
                }
                load_group(2 * s + 1, wb);
            });
            half_stage(st, 1, wb, 4, [&]() __attribute__((always_inline)) {
                load_group(__builtin_amdgcn_readfirstlane(2 * s + 2 < n_groups ? 2 * s + 2 : n_groups - 1), wa);
            });
            lds_dma_wait<0>();
            landed(wa);
            __syncthreads();
        }
        if (tail) {   // 2, 4 or 6 blocks: a bank tail, a group, or both
            const int st = stages & 1;
            if (tail == 2) {
                half_stage(st, 0, wa, 2, [] {});
            } else {
                half_stage(st, 0, wa, 4, [&]() __attribute__((always_inline)) { load_group(n_groups - 1, wb); });
                if (tail == 6) half_stage(st, 1, wb, 2, [] {});
            }
        }
    };
    dma_stage(0);
    dma_scales(0);
    // Waves may take different instantiations: each issues the same stage loads and reaches the same
    // number of barriers.
    if (nf == 0) {
        lds_dma_wait<0>();
        __syncthreads();
        for (int s = 1; s < n_stages; ++s) {
            dma_stage(s);
            lds_dma_wait<0>();
            __syncthreads();
        }
        if (!tail) __syncthreads();
        return;
    }
    constexpr std::false_type fast{};
    if constexpr (FLAGGED) {
        if (flagged) {
            k_loop(std::integral_constant<int, 4>{}, std::true_type{});
            rows_epilogue<8, EPI>(A, it, pair, nf, acc);
            return;
        }
    }
    if (nf == 4) k_loop(std::integral_constant<int, 4>{}, fast);
    else if (nf == 3) k_loop(std::integral_constant<int, 3>{}, fast);
    else if (nf == 2) k_loop(std::integral_constant<int, 2>{}, fast);
    else k_loop(std::integral_constant<int, 1>{}, fast);
    rows_epilogue<8, EPI>(A, it, pair, nf, acc);
}

// Tiles of job_tile jobs per active expert, in active order: one workgroup, wave scans plus a
// scan of the 16 wave totals.
__global__ __launch_bounds__(1024) void gemm_tiles_kernel(const int32_t * counts, const int32_t * active,
                                                          const int32_t * n_active, const int32_t * filter, int job_tile,
                                                          int max_tiles,
                                                          int32_t * tile_expert, int32_t * tile_start, int32_t * n_tiles,
                                                          int32_t * error) {
    __shared__ int s_wave[16];
    const int na = *n_active;
    const int a = threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = a < na ? active[a] : 0;
    const bool kept = a < na && (filter == nullptr || filter[e] >= 0);   // filtered experts get no tiles
    const int nt = kept ? (counts[e] + job_tile - 1) / job_tile : 0;
    int incl = nt;
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    int before = 0;
    for (int w = 0; w < wave; ++w) before += s_wave[w];
    const int base = before + incl - nt;
    for (int t = 0; t < nt; ++t) {
        if (base + t < max_tiles) {
            tile_expert[base + t] = e;
            tile_start[base + t] = t * job_tile;
        } else {
            *error = 1;
        }
    }
    if (threadIdx.x == 1023) {
        const int total = before + incl;
        *n_tiles = total < max_tiles ? total : max_tiles;
    }
}

// x86 quantize_row_q8_0 of fp32 rows into GEMM activation rows (row-major codes as f16 or int8,
// fp16-rounded fp32 block scales, and a 0 flag: this quantizer never produces -128).
// Workgroup (row, 64-block segment seg) of it; four threads per block, eight elements each.
__device__ __forceinline__ void gemm_rows_segment(const float * __restrict__ x, int vec4, int nb, int64_t x_stride,
                                                  const GemmRowLayout & L, uint8_t * __restrict__ out, int64_t row,
                                                  int seg) {
    const int bq = seg * 64 + static_cast<int>(threadIdx.x >> 2);
    const bool live = bq < nb;
    const int b = live ? bq : 0;
    const int part = static_cast<int>(threadIdx.x & 3);
    float v[8];
    const float * src = x + row * x_stride + b * 32 + part * 8;
    if (vec4) {   // 16-byte aligned rows: two 16-byte loads per thread
        const float4 lo = live ? *reinterpret_cast<const float4 *>(src) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        const float4 hi = live ? *reinterpret_cast<const float4 *>(src + 4) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = live ? src[i] : 0.0f;
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = quad_max(amax);
    if (!live) return;
    const float d = amax / 127.0f;
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    uint8_t * o = out + row * L.stride();
    const int64_t e0 = b * 32 + part * 8;
    if (L.weight_type == 39) {
        half8_t c;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float q = rintf(v[i] * id);
            q = q > 127.0f ? 127.0f : (q < -128.0f ? -128.0f : q);
            c[i] = static_cast<_Float16>(q);
        }
        *reinterpret_cast<half8_t *>(o + e0 * 2) = c;
    } else {
        uint64_t c = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float q = rintf(v[i] * id);
            q = q > 127.0f ? 127.0f : (q < -128.0f ? -128.0f : q);
            c |= static_cast<uint64_t>(static_cast<uint8_t>(static_cast<signed char>(q))) << (8 * i);
        }
        *reinterpret_cast<uint64_t *>(o + e0) = c;
    }
    if (part == 0) {
        reinterpret_cast<float *>(o + L.da_offset())[b] = static_cast<float>(static_cast<_Float16>(d));
        if (b == 0) *reinterpret_cast<int *>(o + L.flag_offset()) = 0;
    }
}

__global__ __launch_bounds__(256) void gemm_rows_from_f32_kernel(const float * __restrict__ x, int vec4, int nb,
                                                                 int64_t x_stride, GemmRowLayout L, uint8_t * __restrict__ out) {
    gemm_rows_segment(x, vec4, nb, x_stride, L, out, blockIdx.x, static_cast<int>(blockIdx.y));
}

// The prefill's top-k + softmax (given logits; workgroups 0 .. ceil(T / 4) - 1, one wave per
// token) and its GEMM activation rows (the other workgroups, one per (row, 64-block segment)) in
// one launch: the two only share the launch.
template <int NPL>
__global__ __launch_bounds__(256) void topk_gemm_rows_kernel(const float * __restrict__ logits, int n_expert, int top_k,
                                                             int32_t * __restrict__ ids, float * __restrict__ weights,
                                                             int64_t n_tokens, int64_t topk_wgs, const float * __restrict__ x,
                                                             int vec4, int nb, int64_t x_stride, GemmRowLayout L,
                                                             int segments, uint8_t * __restrict__ out) {
    const int64_t b = blockIdx.x;
    if (b < topk_wgs) {
        const int64_t t = b * 4 + (threadIdx.x >> 6);
        if (t < n_tokens) wave_topk_softmax<NPL>(logits + t * n_expert, n_expert, top_k, ids + t * top_k, weights + t * top_k);
        return;
    }
    const int64_t r = b - topk_wgs;
    gemm_rows_segment(x, vec4, nb, x_stride, L, out, r / segments, static_cast<int>(r % segments));
}

// ggml Q8_0 block rows -> GEMM activation rows, with each row's -128 flag.
__global__ __launch_bounds__(256) void gemm_rows_from_q8_kernel(const uint8_t * __restrict__ q8, int nb, int64_t row_bytes,
                                                                GemmRowLayout L, uint8_t * __restrict__ out) {
    __shared__ int s_flag;
    const int64_t row = blockIdx.x;
    const uint8_t * src = q8 + row * row_bytes;
    uint8_t * o = out + row * L.stride();
    if (threadIdx.x == 0) s_flag = 0;
    __syncthreads();
    int neg = 0;
    for (int idx = threadIdx.x; idx < nb * 32; idx += 256) {
        const int b = idx >> 5, e = idx & 31;
        const signed char q = static_cast<signed char>(src[b * 34 + 2 + e]);
        neg |= q == -128;
        if (L.weight_type == 39) reinterpret_cast<_Float16 *>(o)[idx] = static_cast<_Float16>(q);
        else o[idx] = static_cast<uint8_t>(q);
    }
    for (int b = threadIdx.x; b < nb; b += 256)
        reinterpret_cast<float *>(o + L.da_offset())[b] =
            half_bits_to_float(static_cast<uint16_t>(src[b * 34] | (src[b * 34 + 1] << 8)));
    if (neg) atomicOr(&s_flag, 1);
    __syncthreads();
    if (threadIdx.x == 0) *reinterpret_cast<int *>(o + L.flag_offset()) = s_flag;
}

// `experts` with jobs at most, `entries` jobs in all. Parts of 16 or 32 jobs are launched where the experts hold
// more on average and the tiles are likely few enough (a grid of 512 for 140 workgroups with jobs cost a layer's two
// launches 2 us of 50).
template <int TYPE, int EPI, bool FLAGGED>
void launch_rows_gemm(const GemmArgs & a, int64_t rows, int max_tiles, int64_t experts, int64_t entries, hipStream_t stream) {
    GemmArgs b = a;
    b.row_units = static_cast<int>((rows + 255) / 256);
    const int64_t mean = entries / experts, whole = static_cast<int64_t>(b.row_units) * max_tiles;
    const int64_t likely = std::min(whole, b.row_units * experts * ((mean + 63) / 64));
    b.split = mean > 16 && likely * 4 <= kGemmSlots ? 2 : (mean > 32 && likely * 2 <= kGemmSlots ? 1 : 0);
    // every tile that there can be, or the parts of so few of them that they are split
    const int64_t tiles = (whole + 7) / 8 * 8;
    const dim3 grid(static_cast<unsigned>(std::max(tiles, std::min<int64_t>(tiles << b.split, b.split ? kGemmSlots : 0))));
    if constexpr (TYPE == 39) hipLaunchKernelGGL((mx_rows_gemm_kernel<EPI, FLAGGED>), grid, dim3(kGemmThreads), 0, stream, b);
    else hipLaunchKernelGGL((q8_rows_gemm_kernel<EPI, FLAGGED>), grid, dim3(kGemmThreads), 0, stream, b);
    check_hip(hipGetLastError(), "grouped GEMM launch");
}

// ------------------------------------------------------------------ MXFP4 x MXFP8 experiment
// The CDNA4 block-scaled matrix core (v_mfma_scale_f32_16x16x128_f8f6f4) takes MXFP4 weights as
// they are stored (e2m1 codes, e8m0 exponents) and 8-bit activations with their own e8m0 block
// scales, applies both scales and accumulates four 32-element blocks per instruction: no
// per-block scale-accumulate work is left on the vector ALUs. Its activations must be an MX
// format, so this path quantizes them to MXFP8 (OCP MX e4m3, one e8m0 scale per 32 values)
// instead of the reference's Q8_0: a measured experiment beside the f16 MFMA path, outside the
// parity contract.
//
// Operand layout of one 128-element K step (blocks blk = 0..3), checked on the device:
//   A: lane row + 16 blk holds block blk of its row, element i at nibble i (low nibble first);
//      scale_a of that lane is the block's e8m0 exponent;
//   B: lane col + 16 g, byte j holds block g / 2 + 2 (j / 16), element 16 (g % 2) + j % 16;
//      scale_b of lane col + 16 blk is the block's e8m0 scale;
//   D: lane l holds column l % 16, rows 4 (l / 16) .. + 3.
// Products and block sums inside the instruction are not rounded as an fp32 chain would be (a
// random-data check puts the difference near 6e-5 of the sum of |products|).
typedef int mx_v8i __attribute__((ext_vector_type(8)));

// MXFP8 (e4m3) quantization of fp32 rows, one e8m0 scale X per 32 values: the smallest power of two
// with amax / X <= 448 (the e4m3 maximum), i.e. the OCP MX choice 2^(floor(log2 amax) - 8) raised
// by one when amax / 2^floor(log2 amax) > 1.75, so no value saturates; code = e4m3 of v / X
// rounded to nearest even; scale byte = 127 + log2 X. One thread per 4 values; the 8 threads of a
// block are adjacent lanes.
__device__ __forceinline__ uint32_t e4m3_rne(float v) {
    const uint32_t sign = __builtin_bit_cast(uint32_t, v) >> 31 << 7;
    float a = fabsf(v);
    a = a > 448.0f ? 448.0f : a;
    if (!(a >= 0.015625f)) {                                   // below 2^-6: subnormal steps of 2^-9
        const float m = rintf(a * 512.0f);                     // 0..8 (8 rounds up to the smallest normal)
        return sign | static_cast<uint32_t>(m);
    }
    const int e = static_cast<int>((__builtin_bit_cast(uint32_t, a) >> 23) & 0xFF) - 127;   // -6..8
    float m = rintf(__builtin_amdgcn_ldexpf(a, 3 - e));         // 8..16
    int ee = e;
    if (m >= 16.0f) { m = 8.0f; ++ee; }                        // carry into the next binade (<= 448 by the clamp)
    return sign | static_cast<uint32_t>((ee + 7) << 3) | (static_cast<uint32_t>(m) - 8u);
}

__global__ __launch_bounds__(256) void quantize_mxfp8_kernel(const float * __restrict__ x, int64_t n_rows, int nb,
                                                             int64_t x_stride, uint8_t * __restrict__ codes,
                                                             uint8_t * __restrict__ scales) {
    const int64_t t = blockIdx.x * 256ll + threadIdx.x;
    const bool live = t < n_rows * nb * 8;
    const int64_t blk = live ? t / 8 : 0;
    const int part = static_cast<int>(t & 7);
    const int64_t row = blk / nb, b = blk % nb;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = live ? x[row * x_stride + b * 32 + part * 4 + i] : 0.0f;
    float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    const uint32_t ab = __builtin_bit_cast(uint32_t, amax);
    const int ea = ab >= 0x00800000u ? static_cast<int>(ab >> 23) - 127 : -127;   // subnormal or zero: X = 2^-127
    int sx = ea - 8 + (ab >= 0x00800000u && (ab & 0x7FFFFFu) > 0x600000u ? 1 : 0);
    sx = sx < -127 ? -127 : (sx > 127 ? 127 : sx);
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) packed |= e4m3_rne(__builtin_amdgcn_ldexpf(v[i], -sx)) << (8 * i);
    if (live) {
        reinterpret_cast<uint32_t *>(codes + row * nb * 32 + b * 32)[part] = packed;
        if (part == 0) scales[row * nb + b] = static_cast<uint8_t>(sx + 127);
    }
}

struct MxArgs {
    const uint8_t * bank;
    GemmShape shape;
    const int32_t * expert_to_slot;
    const uint8_t * codes;     // MXFP8 rows [n_rows][nb * 32]
    const uint8_t * scales;    // [n_rows][nb]
    int64_t n_ids, b_ne1;
    const int32_t * counts;
    const int32_t * offsets;
    const int32_t * jobs;
    const int32_t * tile_expert;
    const int32_t * tile_start;
    const int32_t * n_tiles;
    int row_pairs;
    float * dst;               // [job][rows]
};

// A workgroup (4 waves) computes 64 bank rows (a tile pair) x 64 jobs of one expert, like the f16
// path; wave w owns rows 32 (w & 1) .. + 31 and jobs 32 (w >> 1) .. + 31 as 2 x 2 fragments. Per
// bank group (8 blocks = two 128-element K steps) the tile pair's codes are restaged in LDS as
// [block][row][16 B], the operand order of the matrix core, and its exponents as [block][row]; the
// activation operands go from the MXFP8 rows straight into registers. The next group's loads
// (codes, exponents, activation operands) are in flight while the current group computes.
struct MxStage {
    uint32_t w[2][4];          // two (tile, slice, row) code entries: 8 blocks x 2 bytes each
    uint32_t m[2];             // threads 0..63: the row's 8 exponent bytes (stored as e - 128)
    u32x4g b[2][2][2];         // [K step][job half][low / high 16 bytes] activation operand
    int sb[2][2];              // [K step][job half] activation block scale
};

__global__ __launch_bounds__(256) void mx_gemm_kernel(MxArgs A) {
    __shared__ __attribute__((aligned(16))) uint8_t wl[8 * 64 * 16];
    __shared__ uint8_t el[8 * 64];
    const int n_items = *cst<int32_t>(A.n_tiles) * A.row_pairs;
    const int per_xcd = (n_items + 7) >> 3;
    const int slot8 = static_cast<int>(blockIdx.x >> 3);
    const int item = static_cast<int>(blockIdx.x & 7) * per_xcd + slot8;
    if (slot8 >= per_xcd || item >= n_items) return;
    const int ti = item / A.row_pairs;
    const int pair = item - ti * A.row_pairs;
    const int expert = cst<int32_t>(A.tile_expert)[ti];
    const int j0 = cst<int32_t>(A.tile_start)[ti];
    const int count = cst<int32_t>(A.counts)[expert];
    const int joff = cst<int32_t>(A.offsets)[expert];
    const int slot = A.expert_to_slot ? cst<int32_t>(A.expert_to_slot)[expert] : expert;
    const GemmShape S = A.shape;
    const int nb = S.nb, groups = nb / 8, tail = nb % 8;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, q = lane >> 4;
    const bool slot_ok = slot >= 0 && slot < S.n_slots;
    const uint8_t * slot_base = A.bank + static_cast<size_t>(slot_ok ? slot : 0) * S.slot_bytes;

    // this lane's two job columns
    const uint8_t * bcode[2];
    const uint8_t * bscale[2];
    int job[2];
    bool jlive[2];
#pragma unroll
    for (int jh = 0; jh < 2; ++jh) {
        const int jl = 32 * (wave >> 1) + 16 * jh + lr;
        jlive[jh] = j0 + jl < count;
        job[jh] = jlive[jh] ? A.jobs[joff + j0 + jl] : 0;
        const int64_t row_index = A.b_ne1 == 1 ? job[jh] / A.n_ids : job[jh];
        bcode[jh] = A.codes + row_index * nb * 32;
        bscale[jh] = A.scales + row_index * nb;
    }
    // this thread's two staging entries: e = t + 256 h -> tile tt, slice k, row r
    auto load = [&](int g, MxStage & R) {
        const bool is_tail = g == groups;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = threadIdx.x + 256 * h;
            const int tile = pair * 2 + (e >> 8), k = (e >> 5) & 7, r = e & 31;
#pragma unroll
            for (int d = 0; d < 4; ++d) R.w[h][d] = 0u;
            if (tile * 32 < S.rows) {
                const uint8_t * ct = slot_base + static_cast<size_t>(tile) * 32 * nb * 16;
                if (!is_tail) {
                    const u32x4g v = *reinterpret_cast<const u32x4g *>(ct + static_cast<size_t>(g) * 4096 + (k * 32 + r) * 16);
                    R.w[h][0] = v[0], R.w[h][1] = v[1], R.w[h][2] = v[2], R.w[h][3] = v[3];
                } else {
                    const uint8_t * tp = ct + static_cast<size_t>(groups) * 4096 + (k * 32 + r) * (tail * 2);
#pragma unroll
                    for (int b = 0; b < 8; ++b)       // constant indices keep the stage in registers
                        if (b < tail)
                            R.w[h][b >> 1] |= static_cast<uint32_t>(*reinterpret_cast<const uint16_t *>(tp + 2 * b)) << (16 * (b & 1));
                }
            }
        }
        R.m[0] = R.m[1] = 0x80808080u;                         // blocks past the tail: 2^0
        if (threadIdx.x < 64) {
            const int row = threadIdx.x, tile = pair * 2 + (row >> 5), r = row & 31;
            if (tile * 32 < S.rows) {
                const uint8_t * mt = slot_base + S.codes_bytes + static_cast<size_t>(tile) * 32 * nb;
                if (!is_tail) {
                    const u32x2g v = *reinterpret_cast<const u32x2g *>(mt + static_cast<size_t>(g) * 256 + r * 8);
                    R.m[0] = v[0], R.m[1] = v[1];
                } else {
#pragma unroll
                    for (int b = 0; b < 8; ++b) {
                        if (b < tail) {
                            const uint32_t byte = mt[groups * 256 + r * tail + b];
                            R.m[b >> 2] = (R.m[b >> 2] & ~(0xFFu << (8 * (b & 3)))) | (byte << (8 * (b & 3)));
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const int b0 = 8 * g + 4 * st, blo = b0 + (q >> 1), bhi = b0 + 2 + (q >> 1);
#pragma unroll
            for (int jh = 0; jh < 2; ++jh) {
                R.b[st][jh][0] = R.b[st][jh][1] = u32x4g{0u, 0u, 0u, 0u};
                if (jlive[jh] && blo < nb) R.b[st][jh][0] = *reinterpret_cast<const u32x4g *>(bcode[jh] + blo * 32 + 16 * (q & 1));
                if (jlive[jh] && bhi < nb) R.b[st][jh][1] = *reinterpret_cast<const u32x4g *>(bcode[jh] + bhi * 32 + 16 * (q & 1));
                R.sb[st][jh] = jlive[jh] && b0 + q < nb ? bscale[jh][b0 + q] : 127;
            }
        }
    };
    auto stage = [&](const MxStage & R) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = threadIdx.x + 256 * h;
            const int row = 32 * (e >> 8) + (e & 31), k = (e >> 5) & 7;
#pragma unroll
            for (int b = 0; b < 8; ++b)
                *reinterpret_cast<uint16_t *>(wl + (b * 64 + row) * 16 + 2 * k) = static_cast<uint16_t>(R.w[h][b >> 1] >> (16 * (b & 1)));
        }
        if (threadIdx.x < 64) {
#pragma unroll
            for (int b = 0; b < 8; ++b) el[b * 64 + threadIdx.x] = static_cast<uint8_t>((R.m[b >> 2] >> (8 * (b & 3))) ^ 0x80u);
        }
    };
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int jh = 0; jh < 2; ++jh) acc[i][jh] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int n_groups = groups + (tail > 0 ? 1 : 0);
    MxStage cur, nxt;
    load(0, cur);
    stage(cur);
    __syncthreads();
    for (int g = 0; g < n_groups; ++g) {
        if (g + 1 < n_groups) load(g + 1, nxt);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            if (8 * g + 4 * st >= nb) break;
            mx_v8i bop[2];
#pragma unroll
            for (int jh = 0; jh < 2; ++jh) {
                const u32x4g lo = cur.b[st][jh][0], hi = cur.b[st][jh][1];
                bop[jh] = mx_v8i{static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(lo[2]), static_cast<int>(lo[3]),
                                 static_cast<int>(hi[0]), static_cast<int>(hi[1]), static_cast<int>(hi[2]), static_cast<int>(hi[3])};
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = 32 * (wave & 1) + 16 * i + lr;
                const u32x4g a = *reinterpret_cast<const u32x4g *>(wl + ((4 * st + q) * 64 + row) * 16);
                const mx_v8i aop = mx_v8i{static_cast<int>(a[0]), static_cast<int>(a[1]), static_cast<int>(a[2]), static_cast<int>(a[3]), 0, 0, 0, 0};
                const int sa = el[(4 * st + q) * 64 + row];
#pragma unroll
                for (int jh = 0; jh < 2; ++jh)
                    acc[i][jh] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(aop, bop[jh], acc[i][jh], 4, 0, 0, sa, 0, cur.sb[st][jh]);
            }
        }
        __syncthreads();
        if (g + 1 < n_groups) {
            stage(nxt);
            cur = nxt;
        }
        __syncthreads();
    }
    const float nan = __builtin_nanf("");
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int jh = 0; jh < 2; ++jh) {
            if (!jlive[jh]) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t brow = static_cast<int64_t>(pair) * 64 + 32 * (wave & 1) + 16 * i + 4 * q + j;
                if (brow < S.rows)
                    A.dst[static_cast<size_t>(job[jh]) * S.rows + ggml_row(brow, S.rows, S.interleave)] = slot_ok ? acc[i][jh][j] : nan;
            }
        }
}

}  // namespace

void launch_job_tiles(const GroupBuffers & g, const int32_t * filter, int job_tile, int64_t max_tiles,
                      int32_t * tile_expert, int32_t * tile_start, int32_t * n_tiles, hipStream_t stream) {
    require(job_tile >= 1 && max_tiles >= 1 && max_tiles < (1ll << 31), "job tile list shape out of range");
    hipLaunchKernelGGL(gemm_tiles_kernel, dim3(1), dim3(1024), 0, stream, g.counts, g.active, g.n_active, filter, job_tile,
                       static_cast<int>(max_tiles), tile_expert, tile_start, n_tiles, g.error);
    check_hip(hipGetLastError(), "job tile list launch");
}

int64_t gemm_max_tiles(int64_t n_as, int64_t n_entries, int job_tile) {
    return (n_entries + job_tile - 1) / job_tile + (n_as < n_entries ? n_as : n_entries);
}

// sized for the smaller job tile of the two kernels that share it
size_t gemm_tiles_bytes(int64_t n_as, int64_t n_entries) {
    return static_cast<size_t>((2 * gemm_max_tiles(n_as, n_entries, kMxJobTile) + 8) * sizeof(int32_t));
}

void launch_gemm_rows_from_f32(const float * x, int64_t n_rows, int64_t k, int64_t x_stride, const GemmRowLayout & lay,
                               uint8_t * rows, hipStream_t stream) {
    require(k > 0 && k % 32 == 0 && n_rows > 0 && x_stride >= k && lay.nb == k / 32, "GEMM quantize shape mismatch");
    require(n_rows < (1ll << 31), "too many GEMM activation rows for one launch");
    const unsigned segments = static_cast<unsigned>((k / 32 + 63) / 64);
    const int vec4 = reinterpret_cast<uintptr_t>(x) % 16 == 0 && x_stride % 4 == 0;
    hipLaunchKernelGGL(gemm_rows_from_f32_kernel, dim3(static_cast<unsigned>(n_rows), segments), dim3(256), 0, stream,
                       x, vec4, static_cast<int>(k / 32), x_stride, lay, rows);
    check_hip(hipGetLastError(), "GEMM quantize launch");
}

void launch_topk_gemm_rows(const float * logits, int64_t n_expert, int64_t top_k, int32_t * ids, float * weights,
                           const float * x, int64_t n_rows, int64_t k, const GemmRowLayout & lay, uint8_t * rows,
                           hipStream_t stream) {
    require(k > 0 && k % 32 == 0 && n_rows > 0 && lay.nb == k / 32, "GEMM quantize shape mismatch");
    require(n_expert > 0 && n_expert <= 1024 && top_k > 0 && top_k <= n_expert && top_k <= 64,
            "router supports 1..1024 experts and top_k <= 64");
    const int segments = static_cast<int>((k / 32 + 63) / 64);
    const int64_t topk_wgs = (n_rows + 3) / 4, total = topk_wgs + n_rows * segments;
    require(total < (1ll << 31), "too many GEMM activation rows for one launch");
    const int vec4 = reinterpret_cast<uintptr_t>(x) % 16 == 0 && k % 4 == 0;
    const int ne = static_cast<int>(n_expert), tk = static_cast<int>(top_k), nb = static_cast<int>(k / 32);
    const dim3 grid(static_cast<unsigned>(total));
    if (n_expert <= 128)
        hipLaunchKernelGGL(topk_gemm_rows_kernel<2>, grid, dim3(256), 0, stream, logits, ne, tk, ids, weights, n_rows, topk_wgs,
                           x, vec4, nb, k, lay, segments, rows);
    else if (n_expert <= 256)
        hipLaunchKernelGGL(topk_gemm_rows_kernel<4>, grid, dim3(256), 0, stream, logits, ne, tk, ids, weights, n_rows, topk_wgs,
                           x, vec4, nb, k, lay, segments, rows);
    else
        hipLaunchKernelGGL(topk_gemm_rows_kernel<16>, grid, dim3(256), 0, stream, logits, ne, tk, ids, weights, n_rows,
                           topk_wgs, x, vec4, nb, k, lay, segments, rows);
    check_hip(hipGetLastError(), "top-k + GEMM rows launch");
}

void launch_gemm_rows_from_q8(const uint8_t * q8, int64_t n_rows, int64_t row_bytes, const GemmRowLayout & lay,
                              uint8_t * rows, hipStream_t stream) {
    require(n_rows > 0 && n_rows < (1ll << 31) && row_bytes == lay.nb * 34, "GEMM expand shape mismatch");
    hipLaunchKernelGGL(gemm_rows_from_q8_kernel, dim3(static_cast<unsigned>(n_rows)), dim3(256), 0, stream, q8,
                       static_cast<int>(lay.nb), row_bytes, lay, rows);
    check_hip(hipGetLastError(), "GEMM expand launch");
}

void launch_grouped_gemm(const GemmParams & p, hipStream_t stream) {
    const vbm_bank & bank = *p.bank;
    require(bank.nb <= 4096 / 32 && p.lay.nb == bank.nb && p.lay.weight_type == bank.type,
            "GEMM activation layout does not match the bank");
    require(p.epilogue == 0 || (bank.interleave && bank.rows % 64 == 0 && p.rows_out && p.out_layout.nb == bank.rows / 64),
            "GLU epilogue needs an interleaved gate|up bank with rows % 64 == 0 and a matching output layout");
    require(p.epilogue == 1 || p.dst != nullptr, "missing GEMM output");
    require(p.n_as >= 1 && p.n_as <= 1024 && p.n_entries >= 1, "GEMM group shape out of range");
    const int job_tile_n = kGemmJobTile;
    const int64_t max_tiles = gemm_max_tiles(p.n_as, p.n_entries, job_tile_n);
    // calls of up to some 8.4 (MXFP4) or 12.6 (Q8_0) million entries: the limit on tiles of 128 and 192 jobs that the
    // entry points have always had, beyond which nothing was measured
    require(gemm_max_tiles(p.n_as, p.n_entries, bank.type == VBM_TYPE_MXFP4 ? 128 : 192) <= 65535, "too many GEMM tiles for one launch");
    int32_t * tile_expert = static_cast<int32_t *>(p.tiles);
    int32_t * tile_start = tile_expert + max_tiles;
    int32_t * n_tiles = tile_start + max_tiles;
    if (!p.tiles_ready) {
        hipLaunchKernelGGL(gemm_tiles_kernel, dim3(1), dim3(1024), 0, stream, p.group.counts, p.group.active,
                           p.group.n_active, p.tile_filter, job_tile_n, static_cast<int>(max_tiles), tile_expert, tile_start,
                           n_tiles, p.group.error);
        check_hip(hipGetLastError(), "GEMM tile list launch");
    }
    GemmArgs a{};
    a.bank = bank.base;
    a.shape = GemmShape{static_cast<int>(bank.nb), static_cast<int>(bank.rows), bank.interleave, bank.slot_bytes,
                        bank.geometry().codes_bytes(), bank.n_slots};
    a.expert_to_slot = p.expert_to_slot;
    a.rows_in = p.rows_in;
    a.lay = p.lay;
    a.n_ids = p.n_ids;
    a.b_ne1 = p.b_ne1;
    a.counts = p.group.counts;
    a.offsets = p.group.offsets;
    a.jobs = p.group.rows;
    a.tile_expert = tile_expert;
    a.tile_start = tile_start;
    a.n_tiles = n_tiles;
    a.bias = p.bias;
    a.row_scale = p.row_scale;
    a.dst = p.dst;
    a.dst_vec4 = p.dst != nullptr && reinterpret_cast<uintptr_t>(p.dst) % 16 == 0 && bank.rows % 4 == 0;
    a.rows_out = p.rows_out;
    a.out_lay = p.out_layout;
    a.activation = p.activation;
    a.alpha = p.alpha;
    a.limit = p.limit;
    require(!p.flagged_rows || p.epilogue == 0, "flagged activation rows only with the plain epilogue");
    // the launch covers max_tiles tiles, or the caller's bound on this call's tiles (its tile filter
    // leaves only the experts whose tiles it counted)
    require(p.grid_tiles >= 0 && (p.grid_tiles == 0 || p.tile_filter != nullptr), "grid tile bound needs a tile filter");
    const int mt = static_cast<int>(p.grid_tiles > 0 ? std::min<int64_t>(p.grid_tiles, max_tiles) : max_tiles);
    if (bank.type == VBM_TYPE_MXFP4) {
        if (p.flagged_rows) launch_rows_gemm<39, 0, true>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
        else if (p.epilogue == 0) launch_rows_gemm<39, 0, false>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
        else launch_rows_gemm<39, 1, false>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
    } else {
        if (p.flagged_rows) launch_rows_gemm<8, 0, true>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
        else if (p.epilogue == 0) launch_rows_gemm<8, 0, false>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
        else launch_rows_gemm<8, 1, false>(a, bank.rows, mt, std::min(p.n_as, p.n_entries), p.n_entries, stream);
    }
}

void launch_quantize_mxfp8(const float * x, int64_t n_rows, int64_t k, int64_t x_stride, uint8_t * codes, uint8_t * scales,
                           hipStream_t stream) {
    require(k > 0 && k % 32 == 0 && n_rows > 0 && x_stride >= k, "MXFP8 quantize shape mismatch");
    const int64_t threads = n_rows * (k / 32) * 8;
    hipLaunchKernelGGL(quantize_mxfp8_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, stream, x,
                       n_rows, static_cast<int>(k / 32), x_stride, codes, scales);
    check_hip(hipGetLastError(), "MXFP8 quantize launch");
}

void launch_mx_gemm(const vbm_bank & bank, const int32_t * expert_to_slot, const uint8_t * codes, const uint8_t * scales,
                    int64_t n_ids, int64_t b_ne1, int64_t n_as, int64_t n_entries, const GroupBuffers & group, void * tiles,
                    float * dst, hipStream_t stream) {
    require(bank.type == VBM_TYPE_MXFP4, "the MXFP8 experiment runs on MXFP4 banks");
    require(n_as >= 1 && n_as <= 1024 && n_entries >= 1, "GEMM group shape out of range");
    const int64_t max_tiles = gemm_max_tiles(n_as, n_entries, kMxJobTile);
    require(max_tiles <= 65535, "too many GEMM tiles for one launch");
    int32_t * tile_expert = static_cast<int32_t *>(tiles);
    int32_t * tile_start = tile_expert + max_tiles;
    int32_t * n_tiles = tile_start + max_tiles;
    hipLaunchKernelGGL(gemm_tiles_kernel, dim3(1), dim3(1024), 0, stream, group.counts, group.active, group.n_active,
                       nullptr, kMxJobTile, static_cast<int>(max_tiles), tile_expert, tile_start, n_tiles, group.error);
    check_hip(hipGetLastError(), "GEMM tile list launch");
    MxArgs a{};
    a.bank = bank.base;
    a.shape = GemmShape{static_cast<int>(bank.nb), static_cast<int>(bank.rows), bank.interleave, bank.slot_bytes,
                        bank.geometry().codes_bytes(), bank.n_slots};
    a.expert_to_slot = expert_to_slot;
    a.codes = codes;
    a.scales = scales;
    a.n_ids = n_ids;
    a.b_ne1 = b_ne1;
    a.counts = group.counts;
    a.offsets = group.offsets;
    a.jobs = group.rows;
    a.tile_expert = tile_expert;
    a.tile_start = tile_start;
    a.n_tiles = n_tiles;
    a.row_pairs = static_cast<int>((bank.rows + 63) / 64);
    a.dst = dst;
    const int64_t items = static_cast<int64_t>(a.row_pairs) * max_tiles;
    hipLaunchKernelGGL(mx_gemm_kernel, dim3(static_cast<unsigned>((items + 7) / 8 * 8)), dim3(256), 0, stream, a);
    check_hip(hipGetLastError(), "MXFP8 GEMM launch");
}

}  // namespace vbm
