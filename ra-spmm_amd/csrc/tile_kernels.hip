// tile_kernels.hip — TC_DIRECT / COMMUNITY_TC / SEGMENT_HYBRID on gfx950.
//
// Work item = one window (TC_DIRECT, COMMUNITY_TC) or one segment
// (SEGMENT_HYBRID): 8 output rows and a run of blocks [b0, b1).
//
// FP16/BF16 route (tile_mfma_kernel): one wavefront per (item, 16*CPL-column
// slice), or a workgroup where the item is long or the launch small
// (shared_items), v_mfma_f32_16x16x32_{f16,bf16}.  A step consumes 4 blocks (32
// vectors = the MFMA K).  Lane (j = lane & 15, q = lane >> 4):
//   - gathers B rows atox[(b+q)*8 + v], v < 8, CPL contiguous elements each at
//     columns col0 + j*CPL (one 16-byte load per vector for CPL = 8), then
//     transposes in registers so MFMA number cc sees K = vectors, N = column
//     col0 + j*CPL + cc;
//   - feeds block b+q as the A fragment in block-diagonal form: rows 0-7 of the
//     16-row MFMA carry blocks b, b+1 and rows 8-15 carry b+2, b+3, so an 8-row
//     window fills the 16x16x32 shape; the two halves are summed at the end.
// FP32 route (the `_tf32` entry points): replaces the reference's TF32 path
// (gfx950 has no xf32 MFMA) with exact fp32 FMA of the stored fp16/bf16 values
// and fp32 B, run as a CSR SpMM over the plan's stored values
// (tile_f32_route.hip).
//
// Reference: fs_tile_spmm[_staged]_kernel tc/ra_tc_direct.cu:109-179, 270-328;
//            ct_fs_tile_spmm_perm_kernel tc/ra_community_tc.cu:106-190;
//            sh_fs_tile_spmm_seg_kernel / sh_merge_split_kernel
//            tc/ra_segment_hybrid.cu:90-221; convert_b_to_half_kernel
//            tc/ra_tc_direct.cu:85-104.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>

#include "ra_internal.hpp"
#include "tile_format.hpp"

namespace {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWave * kWavesPerBlock;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <int CPL> struct HalfRun;  // CPL contiguous 16-bit elements
template <> struct HalfRun<1> { typedef unsigned short T; };
template <> struct HalfRun<2> { typedef unsigned short T __attribute__((ext_vector_type(2))); };
template <> struct HalfRun<4> { typedef unsigned short T __attribute__((ext_vector_type(4))); };
template <> struct HalfRun<8> { typedef u16x8 T; };

template <int CPL>
__device__ __forceinline__ unsigned short run_elem(const typename HalfRun<CPL>::T& r, int i) {
    if constexpr (CPL == 1) return r;
    else return r[i];
}

template <bool BF16>
__device__ __forceinline__ f32x4 mfma32(u16x8 a, u16x8 b, f32x4 c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Where the gathered rows of the 16-bit B are.  A column index becomes a key
// before the lanes hand it to each other; -1 (padding of a window's last block)
// gathers zeros.
//
// HalfBuffer: key = byte offset of the row, gathered through a buffer
// descriptor of K rows: the offset of row -1 lies past its end, where the
// bounds check returns 0.  A step's eight gathers then leave back to back; with
// a branch around each the compiler waits for earlier loads in between: 512,000
// community rows at N = 512 1,215 -> 1,157 us, 64,000 at N = 128 48.3 -> 43.4,
// 150,000 social rows of 200 at N = 128 769 -> 690, 50,000 of 80 109 -> 91.
// HalfPointer: 64-bit addresses and a branch per gather, for a B of 4 GiB and more
// and for windows that should stay in step (swept_in_step).
template <int CPL>
struct HalfBuffer {
    typedef typename HalfRun<CPL>::T Run;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t row_bytes, col_bytes;
    __device__ __forceinline__ HalfBuffer(const uint16_t* Bh, int K, int ldb, int col)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(Bh), 0,
                                                 static_cast<int>(static_cast<uint32_t>(K) * (ldb * 2u)), 0x00027000)),
          row_bytes(ldb * 2u), col_bytes(col * 2u) {}
    __device__ __forceinline__ int key(int col) const { return static_cast<int>(static_cast<uint32_t>(col) * row_bytes); }
    __device__ __forceinline__ Run load(int key) const {
        const uint32_t off = static_cast<uint32_t>(key) + col_bytes;
        if constexpr (CPL == 8)
            return __builtin_bit_cast(Run, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
        else if constexpr (CPL == 4)
            return __builtin_bit_cast(Run, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0));
        else if constexpr (CPL == 2)
            return __builtin_bit_cast(Run, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
        else
            return __builtin_amdgcn_raw_buffer_load_b16(rsrc, off, 0, 0);
    }
};

template <int CPL>
struct HalfPointer {
    typedef typename HalfRun<CPL>::T Run;
    const uint16_t* base;
    int64_t ldb;
    __device__ __forceinline__ HalfPointer(const uint16_t* Bh, int, int ld, int col) : base(Bh + col), ldb(ld) {}
    __device__ __forceinline__ int key(int col) const { return col; }
    __device__ __forceinline__ Run load(int key) const {
        return key >= 0 ? *reinterpret_cast<const Run*>(base + key * ldb) : Run{};
    }
};

// Index chunk of a lane: four consecutive column indices, -1 past the item.
// They become keys when their steps begin, not when they are loaded (a chunk
// ahead): the loop does not wait for the load.
__device__ __forceinline__ int4 load_chunk4(const int32_t* __restrict__ atox, int64_t at, bool inside) {
    int4 v = make_int4(-1, -1, -1, -1);
    if (inside) v = *reinterpret_cast<const int4*>(atox + at);
    return v;
}
template <typename BRows>
__device__ __forceinline__ int4 chunk_keys(const BRows& rows, const int4& v) {
    return make_int4(rows.key(v.x), rows.key(v.y), rows.key(v.z), rows.key(v.w));
}

// The eight keys held by lanes l0 and l0 + 1.
__device__ __forceinline__ void share_keys(const int4& chunk, int l0, int (&keys)[8]) {
    keys[0] = __shfl(chunk.x, l0, kWave);
    keys[1] = __shfl(chunk.y, l0, kWave);
    keys[2] = __shfl(chunk.z, l0, kWave);
    keys[3] = __shfl(chunk.w, l0, kWave);
    keys[4] = __shfl(chunk.x, l0 + 1, kWave);
    keys[5] = __shfl(chunk.y, l0 + 1, kWave);
    keys[6] = __shfl(chunk.z, l0 + 1, kWave);
    keys[7] = __shfl(chunk.w, l0 + 1, kWave);
}

// The lane's eight gathers of a step.
template <typename BRows, typename Run>
__device__ __forceinline__ void gather8(const BRows& rows, const int (&keys)[8], Run (&raw)[8]) {
#pragma unroll
    for (int v = 0; v < 8; ++v) raw[v] = rows.load(keys[v]);
}

struct Items {
    const int32_t* block_offsets;
    const int32_t* seg_window;
    const int32_t* seg_bbegin;
    const int32_t* seg_bend;
    const int32_t* seg_slot;
    const int32_t* win_rows;       // COMMUNITY_TC's row order, NULL for rows in order
    const int32_t* order;          // items of this launch, the long ones first (NULL: in order)
    int item_base;                 // first segment of this launch
    int num_long;                  // items that a whole workgroup shares
    int cell_base;                 // partition * windows (column partitions)
    int accumulate;                // add into C (partitions after the first)
};

// Write (or, for later column partitions, add) one output value / 16-byte run.
__device__ __forceinline__ void put1(float* dst, float v, bool add) {
    if (add) v += *dst;
    *dst = v;
}
template <typename V4>
__device__ __forceinline__ void put4(float* dst, V4 v, bool add) {
    if (add) v += *reinterpret_cast<const V4*>(dst);
    __builtin_nontemporal_store(v, reinterpret_cast<V4*>(dst));
}

// Work item i = segment i (a whole window unless the window was split).
__device__ __forceinline__ void item_range(const Items& it, int i, int& w, int& b0, int& b1,
                                           int& slot) {
    i += it.item_base;
    if (it.order) i = it.order[i];
    w = static_cast<int>(static_cast<uint32_t>(it.seg_window[i]) & 0x7FFFFFFFu) - it.cell_base;
    b0 = it.seg_bbegin[i];
    b1 = it.seg_bend[i];
    slot = it.seg_slot[i];
}

// Destination of window slot m (0..H-1): a C row, or a partial-slot row.
template <int H = ra::kTileWindow>
__device__ __forceinline__ float* item_row(const Items& it, float* C, float* scratch, int w,
                                           int slot, int m, int M, int N) {
    if (slot >= 0) return scratch + ((int64_t)slot * H + m) * N;
    const int row = it.win_rows ? it.win_rows[(int64_t)w * H + m] : w * H + m;
    if (row < 0 || row >= M) return nullptr;
    return C + (int64_t)row * N;
}

// What a wave runs: blocks [b0, b1) of one item, in one column slice.
struct WaveWork {
    int slice, w, b0, b1, slot;
    bool shared;  // a quarter of the item; the workgroup's waves sum up
};

// 1-D grid of workgroups: num_long * nslices that share one item each, then
// groups of 4 items, one a wave.  The slice runs fastest, so all slices of a
// window run back to back and share its atox/vals in L2.
// order bit 0: each XCD (workgroups are dealt round-robin over 8) takes one
// contiguous range of the groups of 4, keeping neighbouring windows in one L2;
// shared items stay dealt.  Bit 1: slice slowest (all windows of slice 0, then
// slice 1, ...), which shrinks the gathered working set to one slice of each
// B row when B is far larger than the L2.
// A shared item is cut into quarters of whole steps of `step` blocks.  False:
// nothing to do (for the whole workgroup, where it is shared).
__device__ __forceinline__ bool wave_work(const Items& it, int num_items, int nslices, int order, int step,
                                          WaveWork& k) {
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const uint32_t ns = static_cast<uint32_t>(nslices), head = it.num_long * ns;
    uint32_t bid = blockIdx.x;
    k.shared = bid < head;
    int item;
    if (k.shared) {
        item = static_cast<int>(bid / ns);
        k.slice = static_cast<int>(bid - item * ns);
    } else {
        bid -= head;
        const uint32_t nb = gridDim.x - head;
        if (order & 1) {
            const uint32_t q = nb / 8, r = nb % 8, x = bid % 8, i = bid / 8;
            bid = x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
        }
        const uint32_t n = (order & 2) ? nb / ns : ns;
        const uint32_t hi = bid / n, lo = bid - hi * n;
        k.slice = static_cast<int>((order & 2) ? hi : lo);
        item = it.num_long + static_cast<int>((order & 2) ? lo : hi) * kWavesPerBlock + wave;
    }
    if (item >= num_items) return false;
    item_range(it, item, k.w, k.b0, k.b1, k.slot);
    if (k.shared) {
        const int steps = (k.b1 - k.b0 + step - 1) / step;
        const int per = (steps + kWavesPerBlock - 1) / kWavesPerBlock * step;
        k.b0 += wave * per;
        k.b1 = min(k.b0 + per, k.b1);
    }
    return true;
}

// Write one window row's CPL columns from col on (16-byte streaming stores where
// the rows allow it: C is written once and never read back here).
template <int CPL>
__device__ __forceinline__ void put_run(float* dst, int col, int N, const float (&out)[CPL], bool vec, bool add) {
    if constexpr (CPL % 4 == 0) {
        if (vec && col + CPL <= N) {
#pragma unroll
            for (int cc = 0; cc < CPL; cc += 4)
                put4(dst + col + cc, f32x4{out[cc], out[cc + 1], out[cc + 2], out[cc + 3]}, add);
            return;
        }
    }
#pragma unroll
    for (int cc = 0; cc < CPL; ++cc)
        if (col + cc < N) put1(dst + col + cc, out[cc], add);
}

// Sum of the four waves' accumulators, in wave order, for row r = wave of every
// group of four rows: out[c] = sum over waves of acc[c][r].  Four accumulators
// at a time, so the LDS (16 KB) bounds no kernel's occupancy.
template <int COUNT>
__device__ __forceinline__ void sum_waves(const f32x4 (&acc)[COUNT], float (&out)[COUNT]) {
    constexpr int kStage = COUNT < 4 ? COUNT : 4;
    __shared__ float part[kWavesPerBlock][kStage * 4][kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
#pragma unroll
    for (int c0 = 0; c0 < COUNT; c0 += kStage) {
        if (c0) __syncthreads();
#pragma unroll
        for (int c = 0; c < kStage; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][c * 4 + r][lane] = acc[c0 + c][r];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < kStage; ++c) {
            float v = part[0][c * 4 + wave][lane];
#pragma unroll
            for (int k = 1; k < kWavesPerBlock; ++k) v += part[k][c * 4 + wave][lane];
            out[c0 + c] = v;
        }
    }
}

// ------------------------------------------------------------ MFMA route
template <int CPL, bool BF16, typename BRows>
__global__ __launch_bounds__(kBlock) void tile_mfma_kernel(
    Items it, const int32_t* __restrict__ atox, const uint16_t* __restrict__ vals,
    const uint16_t* __restrict__ Bh, int K, int ldb, float* __restrict__ C, float* __restrict__ scratch,
    int M, int N, int num_items, int nslices, int order, float unscale, int vec_store) {
    const int lane = threadIdx.x & (kWave - 1);
    WaveWork wk;
    if (!wave_work(it, num_items, nslices, order, 4, wk)) return;
    const int b0 = wk.b0, b1 = wk.b1;
    const int j = lane & 15;
    const int q = lane >> 4;
    const int col = wk.slice * (16 * CPL) + j * CPL;
    const bool in_row = col < ldb;  // ldb % 8 == 0 and CPL | 8: whole runs
    const BRows rows(Bh, K, ldb, col);
    const bool a_half = (j < 8) == (q < 2);

    f32x4 acc[CPL];
#pragma unroll
    for (int cc = 0; cc < CPL; ++cc) acc[cc] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Column keys come 32 blocks (8 steps) at a time: one 16-byte load per
    // lane (lane L: indices 4L..4L+3, half L&1 of block c0 + L/2), handed to
    // step s's lane group q (block c0 + 4s + q) from lanes 8s + 2q and
    // 8s + 2q + 1 by lane permutes, which use the LDS unit, not the address
    // unit.  A fragments come two steps per load: lane j needs block b+q's
    // row j&7 on even steps when a_half, and its partner lane j^8 (same q and
    // row, !a_half) loads the same row of block b+4+q, handed over on the odd
    // step by a lane exchange.  The pair is loaded one step ahead.
    auto load_chunk = [&](int c0) {
        return load_chunk4(atox, (int64_t)c0 * 8 + lane * 4, c0 + (lane >> 1) < b1);
    };
    auto load_pair = [&](int b) {  // b = first block of an even step
        const int blk = b + q + (a_half ? 0 : 4);
        u16x8 a = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (blk < b1) a = *reinterpret_cast<const u16x8*>(vals + (int64_t)blk * 64 + (j & 7) * 8);
        return a;
    };
    int4 chunk, chunk_next = make_int4(-1, -1, -1, -1);
    u16x8 apair = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (b0 < b1) {
        chunk = chunk_keys(rows, load_chunk(b0));
        apair = load_pair(b0);
    }
    for (int b = b0; b < b1; b += 4) {
        const int t = (b - b0) >> 2;
        const int s = t & 7;
        if (s == 0 && b + 32 < b1) chunk_next = load_chunk(b + 32);  // one chunk ahead
        int keys[8];
        share_keys(chunk, 8 * s + 2 * q, keys);
        u16x8 a;
        if ((t & 1) == 0) {
            a = a_half ? apair : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        } else {
            // The partner's register holds this step's row of block b+q.
            const u32x4 mine = __builtin_bit_cast(u32x4, apair);
            u32x4 o;
            o[0] = __shfl_xor(mine[0], 8, kWave);
            o[1] = __shfl_xor(mine[1], 8, kWave);
            o[2] = __shfl_xor(mine[2], 8, kWave);
            o[3] = __shfl_xor(mine[3], 8, kWave);
            a = a_half ? __builtin_bit_cast(u16x8, o) : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        }
        typename BRows::Run raw[8];
        // Lanes past the row's end or the item's last block load nothing.
        if (in_row && b + q < b1) {
            gather8(rows, keys, raw);
        } else {
#pragma unroll
            for (int v = 0; v < 8; ++v) raw[v] = typename BRows::Run{};
        }
        if ((t & 1) == 1 && b + 4 < b1) apair = load_pair(b + 4);
        if (s == 7) chunk = chunk_keys(rows, chunk_next);
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) {
            u16x8 bop;
#pragma unroll
            for (int v = 0; v < 8; ++v) bop[v] = run_elem<CPL>(raw[v], cc);
            acc[cc] = mfma32<BF16>(a, bop, acc[cc]);
        }
    }

    // D[m][n]: lane holds rows 4*(lane>>4)+r, column n = lane & 15.  Rows m and
    // m+8 are partial sums of the same window row (block-diagonal A): lanes L
    // and L^32 exchange them.
    const bool add = it.accumulate && wk.slot < 0;
    float out[CPL];
    if (wk.shared) {
        sum_waves(acc, out);
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) out[cc] = (out[cc] + __shfl_xor(out[cc], 32, kWave)) * unscale;
        if (lane >= 32) return;
        float* dst = item_row(it, C, scratch, wk.w, wk.slot, 4 * (lane >> 4) + static_cast<int>(threadIdx.x >> 6), M, N);
        if (dst) put_run<CPL>(dst, col, N, out, vec_store, add);
    } else {
        // Both halves then hold the window's sums and each half stores two of
        // its four rows (every lane stores).
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[cc][r] += __shfl_xor(acc[cc][r], 32, kWave);
        const bool upper = lane >= 32;  // rows 2, 3 of the lane's group of four
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int m = 4 * ((lane >> 4) & 1) + (upper ? 2 : 0) + k;
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) out[cc] = (upper ? acc[cc][2 + k] : acc[cc][k]) * unscale;  // exact
            float* dst = item_row(it, C, scratch, wk.w, wk.slot, m, M, N);
            if (dst) put_run<CPL>(dst, col, N, out, vec_store, add);
        }
    }
}

// ------------------------------------------------- MFMA route, tall windows
// Windows of H = 16*RG rows; a block is 32 vectors (one MFMA K) with values
// [RG][4][16][8]: lane (j, q) of row group g loads the 16-byte run of row
// 16g + j over vectors 8q..8q+7.  Every gathered B row feeds RG MFMAs (one per
// row group), so a B row shared by several of the H rows is gathered once.
// Per step: one index load (lane pairs exchange halves), 8 B-row gathers,
// RG A loads; no block-diagonal padding.
template <int CPL, bool BF16, int RG, typename BRows>
__global__ __launch_bounds__(kBlock) void tile_mfma_tall_kernel(
    Items it, const int32_t* __restrict__ atox, const uint16_t* __restrict__ vals,
    const uint16_t* __restrict__ Bh, int K, int ldb, float* __restrict__ C, float* __restrict__ scratch,
    int M, int N, int num_items, int nslices, int order, float unscale, int vec_store) {
    constexpr int H = 16 * RG;
    constexpr int BV = H * 32;  // values per block
    const int lane = threadIdx.x & (kWave - 1);
    WaveWork wk;
    if (!wave_work(it, num_items, nslices, order, 1, wk)) return;
    const int b0 = wk.b0, b1 = wk.b1;
    const int j = lane & 15;
    const int q = lane >> 4;
    const int col = wk.slice * (16 * CPL) + j * CPL;
    // Lanes past the row's end gather its last run again and store nothing.
    const BRows rows(Bh, K, ldb, min(col, ldb - CPL));

    f32x4 acc[RG * CPL];
#pragma unroll
    for (int i = 0; i < RG * CPL; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Column keys come 8 blocks at a time: one 16-byte load per lane
    // covers the 256 indices of blocks [c0, c0 + 8) (lane L: indices 4L..4L+3),
    // and step b takes its 8 from lanes 8s + 2q and 8s + 2q + 1 (s = b - c0)
    // by lane permutes, which use the LDS unit, not the address unit.
    auto load_chunk = [&](int c0) {
        return load_chunk4(atox, (int64_t)c0 * 32 + lane * 4, c0 + (lane >> 3) < b1);
    };
    auto load_a = [&](int b, u16x8 (&a)[RG]) {
#pragma unroll
        for (int g = 0; g < RG; ++g)
            a[g] = *reinterpret_cast<const u16x8*>(vals + (int64_t)b * BV + ((g * 4 + q) * 16 + j) * 8);
    };
    int4 chunk, chunk_next = make_int4(-1, -1, -1, -1);
    u16x8 a_next[RG];
    if (b0 < b1) {
        chunk = chunk_keys(rows, load_chunk(b0));
        load_a(b0, a_next);
    }
    for (int b = b0; b < b1; ++b) {
        const int s = (b - b0) & 7;
        if (s == 0 && b + 8 < b1) chunk_next = load_chunk(b + 8);  // one chunk ahead
        int keys[8];
        share_keys(chunk, 8 * s + 2 * q, keys);
        u16x8 a[RG];
#pragma unroll
        for (int g = 0; g < RG; ++g) a[g] = a_next[g];
        typename BRows::Run raw[8];
        gather8(rows, keys, raw);
        if (b + 1 < b1) load_a(b + 1, a_next);
        if (s == 7) chunk = chunk_keys(rows, chunk_next);
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) {
            u16x8 bop;
#pragma unroll
            for (int v = 0; v < 8; ++v) bop[v] = run_elem<CPL>(raw[v], cc);
#pragma unroll
            for (int g = 0; g < RG; ++g) acc[g * CPL + cc] = mfma32<BF16>(a[g], bop, acc[g * CPL + cc]);
        }
    }

    // D of row group g: lane holds rows 16g + 4q + r, column j's CPL outputs.
    const bool add = it.accumulate && wk.slot < 0;
    auto put = [&](int g, int r, const float (&out)[CPL]) {
        float* dst = item_row<H>(it, C, scratch, wk.w, wk.slot, 16 * g + 4 * q + r, M, N);
        if (dst) put_run<CPL>(dst, col, N, out, vec_store, add);
    };
    float out[CPL];
    if (wk.shared) {
        float sums[RG * CPL];
        sum_waves(acc, sums);
#pragma unroll
        for (int g = 0; g < RG; ++g) {
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) out[cc] = sums[g * CPL + cc] * unscale;
            put(g, threadIdx.x >> 6, out);
        }
    } else {
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc) out[cc] = acc[g * CPL + cc][r] * unscale;  // exact: power of two
                put(g, r, out);
            }
    }
}

// ------------------------------ MFMA route, 32-row windows on 32x32x16 MFMA
// The 32-row tall layout run with v_mfma_f32_32x32x16_{f16,bf16}: lane
// (j = lane & 31, q = lane >> 5) feeds row j over k = 8q..8q+7 of a half block
// (16 vectors) as the A operand and gathers B columns col0 + 8j .. +7 of those
// 8 vectors (one 16-byte load each, register transpose) as the B operand.  A
// wave covers 256 columns: each 64-lane gather reads 2 B rows of 512 bytes
// instead of 4 rows of 256 bytes, and a block's A values are read once per
// 256 columns instead of once per 128.  D of MFMA cc: lane holds rows
// 8(i/4) + 4q + i%4 (i < 16) of column col0 + 8j + cc.
template <bool BF16>
__device__ __forceinline__ f32x16 mfma3232(u16x8 a, u16x8 b, f32x16 c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool BF16, typename BRows>
__global__ __launch_bounds__(kBlock, 2) void tile_mfma_tall32_kernel(
    Items it, const int32_t* __restrict__ atox, const uint16_t* __restrict__ vals,
    const uint16_t* __restrict__ Bh, int K, int ldb, float* __restrict__ C, float* __restrict__ scratch,
    int M, int N, int num_items, int nslices, int order, float unscale, int vec_store) {
    constexpr int H = 32;
    constexpr int BV = H * 32;  // values per block
    const int lane = threadIdx.x & (kWave - 1);
    WaveWork wk;
    if (!wave_work(it, num_items, nslices, order, 1, wk)) return;
    const int b0 = wk.b0, b1 = wk.b1;
    const int j = lane & 31;
    const int q = lane >> 5;
    const int col = wk.slice * 256 + j * 8;
    const BRows rows(Bh, K, ldb, min(col, ldb - 8));
    // A operand of row j, k-group q4: offset in the [2][4][16][8] block layout.
    const int a_row = ((j >> 4) * 4) * 16 + (j & 15);

    f32x16 acc[8];
#pragma unroll
    for (int cc = 0; cc < 8; ++cc)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[cc][i] = 0.f;

    // Column indices: one 16-byte load per lane covers blocks [c0, c0 + 8);
    // block s, k-group q4 sits in lanes 8s + 2q4 and 8s + 2q4 + 1.
    auto load_chunk = [&](int c0) {
        return load_chunk4(atox, (int64_t)c0 * 32 + lane * 4, c0 + (lane >> 3) < b1);
    };
    int4 chunk = chunk_keys(rows, load_chunk(b0)), chunk_next = make_int4(-1, -1, -1, -1);
    for (int b = b0; b < b1; ++b) {
        const int s = (b - b0) & 7;
        if (s == 0 && b + 8 < b1) chunk_next = load_chunk(b + 8);
#pragma unroll 1
        for (int h = 0; h < 2; ++h) {
            const int q4 = 2 * h + q;
            int keys[8];
            share_keys(chunk, 8 * s + 2 * q4, keys);
            const u16x8 a = *reinterpret_cast<const u16x8*>(vals + (int64_t)b * BV + (a_row + q4 * 16) * 8);
            u16x8 raw[8];
            gather8(rows, keys, raw);
#pragma unroll
            for (int cc = 0; cc < 8; ++cc) {
                u16x8 bop;
#pragma unroll
                for (int v = 0; v < 8; ++v) bop[v] = raw[v][cc];
                acc[cc] = mfma3232<BF16>(a, bop, acc[cc]);
            }
        }
        if (s == 7) chunk = chunk_keys(rows, chunk_next);
    }

    const bool add = it.accumulate && wk.slot < 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 8 * (i >> 2) + 4 * q + (i & 3);
        float* dst = item_row<H>(it, C, scratch, wk.w, wk.slot, m, M, N);
        float out[8];
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) out[cc] = acc[cc][i] * unscale;  // exact: power of two
        if (dst) put_run<8>(dst, col, N, out, vec_store, add);
    }
}

// ------------------------------------------------ SEGMENT_HYBRID merge
// C[w*8+m][n] = ((slot0 + slot1) + ...) in ascending slot order
// (tc/ra_segment_hybrid.cu:198-221).  A thread owns one column of one window
// row and loads kDeep slots at a time, so a long window's chain is its additions
// and not a memory latency per slot.  Index: 32 bits where the window's H * N
// elements and the last step of the grid fit them.
template <typename Index>
__global__ __launch_bounds__(kBlock) void tile_merge_kernel(
    const int32_t* __restrict__ split_windows, const int32_t* __restrict__ split_offsets,
    const int32_t* __restrict__ win_rows, const float* __restrict__ scratch, float* __restrict__ C,
    int M, int N, int H, int cell_base, int accumulate) {
    constexpr int kDeep = 8;
    const int sw = blockIdx.x;
    const int o0 = split_offsets[sw], o1 = split_offsets[sw + 1];
    const int64_t window = split_windows[sw] - cell_base;
    const Index count = static_cast<Index>(H) * N;
    // grid.y is capped by the launch; stride over the window's H*N elements.
    for (Index e = blockIdx.y * kBlock + threadIdx.x; e < count; e += gridDim.y * kBlock) {
        const uint32_t m = static_cast<uint32_t>(e / static_cast<Index>(N));
        const int64_t slot_row = window * H + m;
        const int row = win_rows ? win_rows[slot_row] : static_cast<int>(slot_row);
        if (row < 0 || row >= M) continue;
        const float* part = scratch + e;
        float acc = part[(int64_t)o0 * count];
        int o = o0 + 1;
        for (; o + kDeep <= o1; o += kDeep) {
            float x[kDeep];
#pragma unroll
            for (int k = 0; k < kDeep; ++k) x[k] = part[(int64_t)(o + k) * count];
#pragma unroll
            for (int k = 0; k < kDeep; ++k) acc += x[k];
        }
        for (; o < o1; ++o) acc += part[(int64_t)o * count];
        float* dst = C + (int64_t)row * N + (e - static_cast<Index>(m) * N);
        *dst = accumulate ? *dst + acc : acc;
    }
}

// --------------------------------------------------------------- convert
// fp32 [rows, cols] -> 16-bit [rows, ldo], RNE, columns cols..ldo-1 zeroed.
// One thread writes 8 consecutive outputs (one 16-byte store) from two 16-byte
// loads, which need 4-byte alignment only; scalar loads are left to the run that
// crosses the row's end.  FLAT (ldo == cols): runs are consecutive in both.
// Bound by its bytes: 150,000 x 100 took 31 us with scalar loads and a 64-bit
// division per run, 18.5 us so (91 MB); 512,000 x 256 119 us either way
// (786 MB, 6.6 TB/s).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

template <bool BF16>
__device__ __forceinline__ u16x8 convert8(const float (&x)[8]) {
    u16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if constexpr (BF16) o[i] = __builtin_bit_cast(unsigned short, static_cast<__bf16>(x[i]));
        else o[i] = __builtin_bit_cast(unsigned short, static_cast<_Float16>(x[i]));
    }
    return o;
}

template <bool BF16, bool FLAT, typename Index>
__global__ __launch_bounds__(kBlock) void convert_kernel(const float* __restrict__ in,
                                                         uint16_t* __restrict__ out, Index total,
                                                         int cols, int groups) {
    for (Index g = (Index)blockIdx.x * kBlock + threadIdx.x; g < total; g += (Index)gridDim.x * kBlock) {
        const float* src = in + (int64_t)g * 8;
        int left = 8;
        if constexpr (!FLAT) {
            const Index r = g / static_cast<Index>(groups);
            const int c0 = static_cast<int>(g - r * static_cast<Index>(groups)) * 8;
            src = in + (int64_t)r * cols + c0;
            left = cols - c0;
        }
        float x[8];
        if (left >= 8) {
            const f32x4u lo = __builtin_nontemporal_load(reinterpret_cast<const f32x4u*>(src));
            const f32x4u hi = __builtin_nontemporal_load(reinterpret_cast<const f32x4u*>(src + 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = lo[i];
                x[4 + i] = hi[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = i < left ? src[i] : 0.f;
        }
        *reinterpret_cast<u16x8*>(out + (int64_t)g * 8) = convert8<BF16>(x);
    }
}

ra_status launch_convert(const float* in, void* out, int64_t rows, int32_t cols, int32_t ldo,
                         bool bf16, hipStream_t st) {
    if (rows <= 0 || ldo <= 0) return RA_OK;
    const int groups = ldo / 8;
    const int64_t total = rows * groups;
    const int blocks = static_cast<int>(std::min<int64_t>((total + kBlock - 1) / kBlock, 1 << 16));
    uint16_t* o = static_cast<uint16_t*>(out);
    auto run = [&](auto kernel, auto n) { kernel<<<blocks, kBlock, 0, st>>>(in, o, n, cols, groups); };
    // 32-bit run numbers, with room for the last step of the grid.
    const bool small = total < (int64_t{1} << 31);
    const uint32_t n32 = static_cast<uint32_t>(total);
    if (ldo == cols && small) run(bf16 ? convert_kernel<true, true, uint32_t> : convert_kernel<false, true, uint32_t>, n32);
    else if (ldo == cols) run(bf16 ? convert_kernel<true, true, int64_t> : convert_kernel<false, true, int64_t>, total);
    else if (small) run(bf16 ? convert_kernel<true, false, uint32_t> : convert_kernel<false, false, uint32_t>, n32);
    else run(bf16 ? convert_kernel<true, false, int64_t> : convert_kernel<false, false, int64_t>, total);
    RA_LAUNCH_CHECK("convert_kernel");
    return RA_OK;
}

}  // namespace

namespace {

// RA_TILE_XCD_REMAP=0 turns the XCD-contiguous window order off.  It is never
// used for COMMUNITY_TC: the leading-column order clusters the heavy rows at
// the front, and contiguous ranges would hand all of them to one XCD.
int tile_remap() {
    static const int r = [] {
        const char* e = std::getenv("RA_TILE_XCD_REMAP");
        return e ? (std::atoi(e) != 0) : 1;
    }();
    return r;
}

// RA_TILE_CPL caps the columns per lane of the MFMA kernel (1, 2, 4 or 8):
// fewer columns per lane = fewer registers = more resident waves.
int tile_max_cpl() {
    static const int c = [] {
        const char* e = std::getenv("RA_TILE_CPL");
        const int v = e ? std::atoi(e) : 8;
        return v >= 8 ? 8 : v >= 4 ? 4 : v >= 2 ? 2 : 1;
    }();
    return c;
}

// RA_TILE_SLICE_MAJOR: 1 = always, 0 = never; unset = with the XCD window
// remap on and the row split into 4 or more slices (N > 384), where the
// whole-row working set is 4x the slice's.  Measured on C4 N=512 with 8 column
// partitions: TC_DIRECT (remapped) 14.4 -> 9.5 ms with slice-major order;
// COMMUNITY_TC (never remapped) 9.85 -> 8.94 ms without it.  At 2 slices the
// re-read A stream cancels the gain.
int tile_slice_major(int nslices, bool remapped) {
    static const int r = [] {
        const char* e = std::getenv("RA_TILE_SLICE_MAJOR");
        return e ? (std::atoi(e) != 0 ? 1 : 0) : -1;
    }();
    return r >= 0 ? r : (nslices >= 4 && remapped ? 1 : 0);
}

// One launch's share of a plan: all of it, or one column partition.
struct Part {
    int item_base, num_items, cell_base, accumulate, split_base, num_splits, num_long;
};

Part whole_plan(const ra_tile_plan* p) {
    return Part{0, p->num_items, 0, 0, 0, p->info.num_split_windows, p->part_long[0]};
}

Items plan_items(const ra_tile_plan* p, const Part& part) {
    Items it{};
    it.item_base = part.item_base;
    it.cell_base = part.cell_base;
    it.accumulate = part.accumulate;
    it.order = p->has_long ? p->item_order.get<int32_t>() : nullptr;
    it.block_offsets = p->block_offsets.get<int32_t>();
    it.seg_window = p->seg_window.get<int32_t>();
    it.seg_bbegin = p->seg_bbegin.get<int32_t>();
    it.seg_bend = p->seg_bend.get<int32_t>();
    it.seg_slot = p->seg_slot.get<int32_t>();
    it.win_rows = p->info.kind == RA_TILE_COMMUNITY_TC ? p->win_rows.get<int32_t>() : nullptr;
    return it;
}

// How one launch runs: columns per lane, the grid and the scheduling order.
struct TileLaunch {
    Items items;
    int cpl, nslices, order;
    dim3 grid;
    int vec_store;
    float unscale;
};

// Bytes of B that a launch gathers (an even share of the plan's blocks).
double gathered_bytes(const ra_tile_plan* p, int N) {
    const int vb = p->info.rows_per_window == ra::kTileWindow ? ra::kTileVec : 32;
    return 2.0 * N * vb * p->info.num_blocks / std::max(p->info.col_parts, 1);
}
constexpr double kGatherBound = 1.75 * (1u << 30);

// Blocks of the plan's longest item over those of its mean one.
double item_skew(const ra_tile_plan* p) {
    const int vb = p->info.rows_per_window == ra::kTileWindow ? ra::kTileVec : 32;
    const int limit =
        (p->info.kind == RA_TILE_SEGMENT_HYBRID ? ra::kTileSegBlocks : ra::kTileDirectSplitBlocks) * ra::kTileVec / vb;
    return static_cast<double>(std::min(p->info.max_window_blocks, limit)) * std::max(p->num_items, 1) /
           std::max(p->info.num_blocks, 1);
}

// Waves of the kernel that the chip holds at once (VGPRs and AGPRs at 1, 2, 4 and 8
// columns a lane: 8 rows 51, 55, 71, 110; 16 rows 45, 50, 70, 102; 32 rows 56, 72, 96,
// 140).
int64_t resident_waves(const ra_tile_plan* p, int cpl) {
    constexpr int kCus = 256;
    if (p->info.rows_per_window == 32) return kCus * (cpl == 1 ? 32 : cpl == 2 ? 28 : cpl == 4 ? 20 : 12);
    return kCus * (cpl <= 2 ? 32 : cpl == 4 ? 28 : 16);
}

// Items of one launch that a whole workgroup shares.
// All of them while the four times as many waves still find room: a wave then has
// a quarter of the steps, but all of an item's prologue (its tables, the first
// indices and keys) and the sum over LDS.  8-row windows of equal length gain up
// to twice the resident waves (N = 128: 1,000 windows of 15 steps 12.4 -> 9.6 us, 2,000
// of 15 18.6 -> 18.5) and lose beyond (2,600 of 7.5 15 -> 18, 4,000 of 25 44 -> 68);
// 16-row ones up to 0.8 times, 32-row ones 0.6, where they are long 0.9 (N = 128: 500
// of 16 steps 12.2 -> 11.8, 500 of 8 8.7 -> 10.6, 750 of 28 23.3 -> 20.4; N = 64: 1,000
// of 4 6.2 -> 5.3).  The longer the longest item against the mean one, the later that
// is: its chain would outlast the rest (3,000 8-row windows of 15 steps at N = 64, the
// longest 3.3 times the mean, 30 -> 20 us, 23 with the long ones shared), until the
// shared long ones alone do as well (5,000 of 15 at N = 128 71 against 81 for all).
// Items of fewer than 6 steps (4 tall) do not pay for it (2,000 of 5 at N = 256 17 ->
// 20).
// Otherwise the long ones, where they are exceptional (the longest twice the mean,
// or at most a quarter of the items), whose chains of gathers (128 steps of ~0.6 us
// in a window of 512 blocks) outlast the rest of a small launch: 50,000 rows of 80
// at N = 128 91 -> 84 us, 20,000 of 60 at N = 64 42 -> 21; of 6,000 windows of 200
// blocks each all would be long (N = 64 84 -> 102).  Where the gathered bytes take longer than any chain (1.75 GiB, ~200 us)
// it only spreads the columns that are gathered at a time: 100,000 rows of 60 at N
// = 256 33 -> 31 % L2 hits, 371 -> 387 us.
int shared_items(const ra_tile_plan* p, const Part& part, int N, int nslices, int cpl) {
    const bool tall = p->info.rows_per_window != ra::kTileWindow;
    const int64_t waves = (int64_t)part.num_items * nslices;
    const double steps = static_cast<double>(p->info.num_blocks) / std::max(p->num_items, 1) / (tall ? 1 : 4);
    const double skew = item_skew(p), more = std::min(skew, 4.0) - 1.0;
    const double room = tall ? (steps < 6 || p->info.rows_per_window == 16 ? 0.8 : 0.6 + 0.015 * std::max(steps - 8, 0.0)) + more
                             : std::min(2.0 + 1.4 * more, 4.0);
    if (kWavesPerBlock * waves <= room * resident_waves(p, cpl) && steps >= (tall ? 4 : 6)) return part.num_items;
    const bool exceptional = skew >= 2 || 4 * static_cast<int64_t>(part.num_long) <= part.num_items;
    return exceptional && gathered_bytes(p, N) < kGatherBound ? part.num_long : 0;
}

TileLaunch tile_launch(const ra_tile_plan* p, const Part& part, const float* C, const float* scratch, int N,
                       bool wide) {
    TileLaunch l{};
    l.cpl = std::min(N <= 16 ? 1 : N <= 32 ? 2 : N <= 64 ? 4 : 8, tile_max_cpl());
    const int slice_cols = wide ? 256 : 16 * l.cpl;
    l.nslices = (N + slice_cols - 1) / slice_cols;
    const bool remap = p->info.kind != RA_TILE_COMMUNITY_TC && tile_remap();
    l.order = (remap ? 1 : 0) | (tile_slice_major(l.nslices, remap) ? 2 : 0);
    l.items = plan_items(p, part);
    l.items.num_long = wide ? 0 : shared_items(p, part, N, l.nslices, l.cpl);
    l.items.order = l.items.num_long == part.num_long ? l.items.order : nullptr;
    const int64_t groups =
        l.items.num_long + ((int64_t)part.num_items - l.items.num_long + kWavesPerBlock - 1) / kWavesPerBlock;
    l.grid = dim3(static_cast<unsigned>(groups * l.nslices));
    l.vec_store = (N % 4 == 0) && ra::aligned16(C) && (!scratch || ra::aligned16(scratch));
    l.unscale = std::ldexp(1.0f, -p->info.value_scale_log2);
    return l;
}

// B of K rows fits HalfBuffer: the offset of row -1 lies past its end.
bool half_buffer_fits(int64_t K, int64_t ldb) { return (K + 1) * ldb * 2 <= int64_t{0xFFFFFFFF}; }

// Launches of 8-row windows that keep the branches (HalfPointer): windows in
// flight together sweep the columns side by side, and the faster their gathers
// leave the further they drift apart.
// Windows of about equal length sweep in step by themselves, which shows as soon
// as the rows of B they sweep (one slice of them where the slices are outermost)
// pass the 4 MB of an L2 by some; us, buffer / pointers at N = 256: 28,000 rows of
// 60 75 / 66, 32,000 of 100 135 / 125; at N = 128: 48,000 of 40 46 / 43; but 32,000 of 60
// at N = 64 (4 MB) 22 / 23; at N = 32, where short windows and less even ones lose:
// 128,000 of 60 91 / 73, 144,000 of 12 29 / 34, 96,000 of 60 (6 MB) 57 / 66.  Shared
// items have no step to keep.
// Unequal ones only where the gathers bound the launch: 100,000 rows of 60 at N =
// 256 32.5 and 34.8 % L2 hits, 357 and 352 us; 250,000 of 500 at N = 512 8,880 and 8,800;
// 150,000 of 100 at N = 256 880 and 871.  With fewer bytes (50,000 of 80 at N = 128: 91 and
// 104) or a slice of B that an L2 nearly holds (25,000 of 200 at N = 256: 128 and
// 140) it is the other way round.
bool swept_in_step(const ra_tile_plan* p, const Part& part, const TileLaunch& l, int N) {
    const int64_t slice = static_cast<int64_t>(p->info.K) * std::min(N, 16 * l.cpl) * 2;
    if (gathered_bytes(p, N) >= kGatherBound && slice > (int64_t{8} << 20)) return true;
    const int64_t swept = (l.order & 2) ? slice : static_cast<int64_t>(p->info.K) * N * 2;
    if (l.items.num_long >= part.num_items) return false;
    if (l.cpl == 2) return item_skew(p) < 1.5 && p->info.num_blocks >= 28LL * p->num_items && swept >= 7000000;
    return item_skew(p) < 2 && swept >= 8000000;
}

#define RA_TILE_ARGS                                                                                       \
    l.items, p->atox.get<int32_t>(), p->vals.get<uint16_t>(), Bh, p->info.K, ldb, C, scratch, \
        p->info.M, N, part.num_items, l.nslices, l.order, l.unscale, l.vec_store

template <int CPL, bool BF16, template <int> class BRows>
void launch_tile(const ra_tile_plan* p, const Part& part, const TileLaunch& l, const uint16_t* Bh, int ldb, float* C,
                 float* scratch, int N, hipStream_t st) {
    const int h = p->info.rows_per_window;
    if (h == 32) tile_mfma_tall_kernel<CPL, BF16, 2, BRows<CPL>><<<l.grid, kBlock, 0, st>>>(RA_TILE_ARGS);
    else if (h == 16) tile_mfma_tall_kernel<CPL, BF16, 1, BRows<CPL>><<<l.grid, kBlock, 0, st>>>(RA_TILE_ARGS);
    else tile_mfma_kernel<CPL, BF16, BRows<CPL>><<<l.grid, kBlock, 0, st>>>(RA_TILE_ARGS);
}

template <bool BF16, template <int> class BRows>
void launch_cpl(const ra_tile_plan* p, const Part& part, const TileLaunch& l, const uint16_t* Bh, int ldb, float* C,
                float* scratch, int N, hipStream_t st) {
    auto f = l.cpl == 1   ? launch_tile<1, BF16, BRows>
             : l.cpl == 2 ? launch_tile<2, BF16, BRows>
             : l.cpl == 4 ? launch_tile<4, BF16, BRows>
                          : launch_tile<8, BF16, BRows>;
    f(p, part, l, Bh, ldb, C, scratch, N, st);
}

// 32-row windows run on the 32x32x16 MFMA kernel at N >= 512 (C3 N=512:
// 1.048 -> 0.968 ms; at N=256 its two waves per SIMD, one per window, lose:
// 0.498 -> 0.533 ms).  RA_TILE_MFMA32=1 forces it at N > 128, 0 turns it off.
bool tile_use_mfma32(int N) {
    static const int v = [] {
        const char* e = std::getenv("RA_TILE_MFMA32");
        return e ? std::atoi(e) : -1;
    }();
    if (v == 0) return false;
    if (v == 1) return N > 128;
    return N >= 512;
}

template <bool BF16>
ra_status launch_part(const ra_tile_plan* p, const Part& part, const uint16_t* Bh, int ldb, float* C, float* scratch,
                      int N, hipStream_t st) {
    if (part.num_items == 0) return RA_OK;
    const bool wide = p->info.rows_per_window == 32 && tile_use_mfma32(N);
    const TileLaunch l = tile_launch(p, part, C, scratch, N, wide);
    const bool buf = half_buffer_fits(p->info.K, ldb) && !(p->info.rows_per_window == ra::kTileWindow && swept_in_step(p, part, l, N));
    if (!wide) (buf ? launch_cpl<BF16, HalfBuffer> : launch_cpl<BF16, HalfPointer>)(p, part, l, Bh, ldb, C, scratch, N, st);
    else if (buf) tile_mfma_tall32_kernel<BF16, HalfBuffer<8>><<<l.grid, kBlock, 0, st>>>(RA_TILE_ARGS);
    else tile_mfma_tall32_kernel<BF16, HalfPointer<8>><<<l.grid, kBlock, 0, st>>>(RA_TILE_ARGS);
    RA_LAUNCH_CHECK("tile_mfma_kernel");
    return RA_OK;
}
#undef RA_TILE_ARGS

ra_status launch_merge(const ra_tile_plan* p, const Part& part, float* C, int N, hipStream_t st) {
    if (part.num_splits == 0) return RA_OK;
    const int H = p->info.rows_per_window;
    dim3 grid(part.num_splits,
              static_cast<unsigned>(std::min<int64_t>(((int64_t)H * N + kBlock - 1) / kBlock, 65535)));
    const int32_t* wr = p->info.kind == RA_TILE_COMMUNITY_TC ? p->win_rows.get<int32_t>() : nullptr;
    const bool small = static_cast<int64_t>(H) * N + 65535LL * kBlock <= int64_t{0xFFFFFFFF};
    (small ? tile_merge_kernel<uint32_t> : tile_merge_kernel<int64_t>)<<<grid, kBlock, 0, st>>>(
        p->split_windows.get<int32_t>() + part.split_base, p->split_offsets.get<int32_t>() + part.split_base, wr,
        p->scratch.get<float>(), C, p->info.M, N, H, part.cell_base, part.accumulate);
    RA_LAUNCH_CHECK("tile_merge_kernel");
    return RA_OK;
}

// FP16/BF16 MFMA route over 16-bit B (converted, or passed in by the caller).
ra_status run_common(ra_tile_plan* p, const uint16_t* Bh, int ldb, bool bf16, float* C, int N, hipStream_t st) {
    float* scratch = nullptr;
    if (p->info.num_split_segs > 0) {
        RA_TRY(p->scratch.ensure((size_t)p->info.num_split_segs * p->info.rows_per_window * N * sizeof(float), st));
        scratch = p->scratch.get<float>();
    }
    // Column partitions run one after another on the stream, each adding into
    // C what the earlier ones wrote: the per-element sum order is fixed.
    const int P = std::max(p->info.col_parts, 1);
    for (int q = 0; q < P; ++q) {
        const Part part = P == 1 ? whole_plan(p)
                                 : Part{p->part_items[q], p->part_items[q + 1] - p->part_items[q],
                                        q * p->info.num_windows, q > 0 ? 1 : 0, p->part_splits[q],
                                        p->part_splits[q + 1] - p->part_splits[q], p->part_long[q]};
        RA_TRY(bf16 ? launch_part<true>(p, part, Bh, ldb, C, scratch, N, st)
                    : launch_part<false>(p, part, Bh, ldb, C, scratch, N, st));
        RA_TRY(launch_merge(p, part, C, N, st));
    }
    return RA_OK;
}

}  // namespace

extern "C" {

ra_status ra_convert_f32(const float* d_in, void* d_out, int64_t rows, int32_t cols, int32_t ldo,
                         int32_t out_dtype, ra_stream_t stream) {
    if (rows < 0 || cols < 0 || ldo < cols || (ldo % 8) != 0)
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "convert: need ldo >= cols and ldo % 8 == 0");
    if (out_dtype != RA_DTYPE_F16 && out_dtype != RA_DTYPE_BF16)
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "convert: out_dtype must be F16 or BF16");
    if (rows > 0 && (!d_in || !d_out)) return ra::fail(RA_ERR_INVALID_ARGUMENT, "convert: NULL buffer");
    if (!ra::aligned16(d_out)) return ra::fail(RA_ERR_INVALID_ARGUMENT, "convert: output not 16-byte aligned");
    return launch_convert(d_in, d_out, rows, cols, ldo, out_dtype == RA_DTYPE_BF16,
                          reinterpret_cast<hipStream_t>(stream));
}

ra_status ra_tile_plan_create(int32_t kind, const int32_t* h_rowptr, const int32_t* h_colind,
                              const float* h_vals, int32_t M, int32_t K, int32_t N,
                              int32_t value_dtype, ra_tile_plan** out) {
    if (!out) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: out is NULL");
    *out = nullptr;
    const auto t0 = std::chrono::steady_clock::now();
    ra_tile_host host;
    try {
        RA_TRY(ra::tile_host_build(kind, h_rowptr, h_colind, h_vals, M, K, N, value_dtype, host));
    } catch (const std::bad_alloc&) {
        return ra::fail(RA_ERR_OUT_OF_MEMORY, "tile: host build out of memory");
    }
    auto p = new (std::nothrow) ra_tile_plan();
    if (!p) return ra::fail(RA_ERR_OUT_OF_MEMORY, "tile: plan allocation");
    ra_status s = ra_tile_host_get_info(&host, &p->info);
    if (s == RA_OK && host.active) {
        if ((s = p->block_offsets.upload(host.block_offsets)) == RA_OK &&
            (s = p->atox.upload(host.atox)) == RA_OK && (s = p->vals.upload(host.vals)) == RA_OK &&
            (s = p->win_rows.upload(host.win_rows)) == RA_OK &&
            (s = p->seg_window.upload(host.seg_window)) == RA_OK &&
            (s = p->seg_bbegin.upload(host.seg_bbegin)) == RA_OK &&
            (s = p->seg_bend.upload(host.seg_bend)) == RA_OK &&
            (s = p->seg_slot.upload(host.seg_slot)) == RA_OK &&
            (s = p->split_windows.upload(host.split_windows)) == RA_OK &&
            (s = p->split_offsets.upload(host.split_offsets)) == RA_OK) {
            p->num_items = p->info.num_segments;
            auto is_long = [&](int32_t i) { return host.seg_bend[i] - host.seg_bbegin[i] > ra::kTileLongBlocks; };
            for (int32_t i = 0; i < p->num_items; ++i) p->part_long[0] += is_long(i);
            p->has_long = p->part_long[0] > 0;
            if (p->has_long) {
                try {
                    std::vector<int32_t> order;
                    order.reserve(p->num_items);
                    for (int pass = 0; pass < 2; ++pass)
                        for (int32_t i = 0; i < p->num_items; ++i)
                            if (is_long(i) == (pass == 0)) order.push_back(i);
                    s = p->item_order.upload(order);
                } catch (const std::bad_alloc&) {
                    s = ra::fail(RA_ERR_OUT_OF_MEMORY, "tile: host build out of memory");
                }
            }
        }
    }
    if (s != RA_OK) {
        delete p;
        return s;
    }
    p->info.build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    *out = p;
    return RA_OK;
}

ra_status ra_tile_plan_run(ra_tile_plan* p, const float* d_B, float* d_C, int32_t N, int32_t route,
                           ra_stream_t stream) {
    if (!p) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: plan is NULL");
    if (!p->info.active)
        return ra::fail(RA_ERR_INACTIVE_PLAN, "tile: plan is inactive (built with N < 16 or empty matrix)");
    if (N <= 0 || p->info.M == 0) return RA_OK;
    if (!d_B || !d_C) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: NULL B or C");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (route == RA_TILE_ROUTE_FP32) return ra::tile_f32_run(p, d_B, d_C, N, st);
    if (route != RA_TILE_ROUTE_F16 && route != RA_TILE_ROUTE_BF16)
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: unknown route");
    const bool bf16 = route == RA_TILE_ROUTE_BF16;
    if (bf16 != (p->info.value_dtype == RA_DTYPE_BF16))
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: route precision differs from the plan's value dtype");
    const int ldb = (N + 7) / 8 * 8;
    RA_TRY(p->bconv.ensure((size_t)p->info.K * ldb * sizeof(uint16_t), st));
    RA_TRY(launch_convert(d_B, p->bconv.get(), p->info.K, N, ldb, bf16, st));
    return run_common(p, p->bconv.get<uint16_t>(), ldb, bf16, d_C, N, st);
}

ra_status ra_tile_plan_run_lowp(ra_tile_plan* p, const void* d_Bh, int32_t ldb, int32_t b_dtype,
                                float* d_C, int32_t N, ra_stream_t stream) {
    if (!p) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: plan is NULL");
    if (!p->info.active)
        return ra::fail(RA_ERR_INACTIVE_PLAN, "tile: plan is inactive (built with N < 16 or empty matrix)");
    if (N <= 0 || p->info.M == 0) return RA_OK;
    if (!d_Bh || !d_C) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: NULL B or C");
    if (ldb < N || (ldb % 8) != 0 || !ra::aligned16(d_Bh))
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: low-precision B needs ldb >= N, ldb % 8 == 0, 16-byte alignment");
    const bool bf16 = b_dtype == RA_DTYPE_BF16;
    if (b_dtype != RA_DTYPE_F16 && !bf16) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: b_dtype must be F16 or BF16");
    if (bf16 != (p->info.value_dtype == RA_DTYPE_BF16))
        return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: B precision differs from the plan's value dtype");
    return run_common(p, static_cast<const uint16_t*>(d_Bh), ldb, bf16, d_C, N, reinterpret_cast<hipStream_t>(stream));
}

ra_status ra_tile_plan_get_info(const ra_tile_plan* p, ra_tile_info* info) {
    if (!p || !info) return ra::fail(RA_ERR_INVALID_ARGUMENT, "tile: NULL argument");
    *info = p->info;
    return RA_OK;
}

void ra_tile_plan_destroy(ra_tile_plan* p) { delete p; }

}  // extern "C"
