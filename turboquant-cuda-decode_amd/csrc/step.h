// The full decode step on the 16x16x32 matrix cores: query rotation, attention over the
// quantised cache and, where one workgroup holds a whole sequence, the output rows, in one
// launch; else part rows that merge_parts_kernel (stage2.h) turns into the output.
//
// The tile arithmetic is stage1_xdl.h's.  What differs from its kernel is how the work is cut:
// nobody but the merge reads the rows, so there are no splits.  A workgroup of vw * sw waves
// covers vw consecutive head parts (waves vi) with sw waves each (sub), which take consecutive
// runs of the workgroup's 16-token tiles and join their results in LDS.  The plan (step_plan.h)
// either gives every sequence one workgroup, or makes one list of the tiles of all sequences, of
// which workgroup x of the nx along it takes an equal stretch, across sequence ends if need be (a
// segment per sequence), so that ragged batches and batch sizes that do not divide the device keep
// the CUs about equally busy; where that ends no later, sequences get workgroups of their own.
// The cut is worked out in the kernel from seq_lens (step_cut.h); the grid depends on shapes alone.
// With one workgroup per sequence the longest sequence sets the time.
//
// Against num_splits rows of 129 floats per head this drops the mid_o traffic of all but one
// row per workgroup, the split ends inside the stream, and for lengths that are not a multiple
// of 16 num_splits the tiles that two splits share and the padding of each split; against a
// rotation launch it saves that launch (5 to 7 us at any size: staging 64 KB of rot_t).
//
// Measured, full step, before (rotation, Stage1 over the splits, Stage2; 256 sequences: one
// launch) and now: 64 x 4096 tokens with 32 / 8 heads 83.1 -> 67.0 us, AoS 97.6 -> 81.9, 64 of 512 to
// 8192 tokens 96.8 -> 76.0, 256 x 2048 116.8 -> 116.6, one of 32768 tokens 37.4 -> 19.4 (kernels 38.5 ->
// 17.1 and merge 4.8), 3-bit 48 x 4096 64.9 -> 53.8, FP8 keys with 64 heads, 24 of 1001 to 6001, 51.5 -> 41.1.
// What bounds it at these sizes is the tile loop's own issue and latency chain
// (stage1_xdl_kernel); first loads go out 4 us and the first four tiles are done 13 us after the
// launch starts, with every CU asking at once.
#pragma once
#include "stage1_xdl.h"
#include "step_cut.h"

namespace tq4 {
namespace xdl {

constexpr int kQRowFloats = kHeadDim + 4;  // LDS row of a rotated query (rows 16 bytes apart in bank)

struct StepArgs : CutArgs {
    const void *query;         // ROT: the bf16 / fp16 query; else fp32 rows, already rotated (FP8 keys: q_dtype rows)
    const float *rot_t;        // [D, D] (ROT)
    const float *centroids;    // [16], 3-bit keys [8], FP8 keys null
    const uint8_t *cache;
    const int32_t *block_table;
    const float *sinks;        // [Hq] or null
    float *parts;              // part rows (stage2.h); unused when whole
    void *out;
    float *lse;
    int64_t block_stride;
    float score_scale_log2;
    int q_dtype, out_dtype;
    int num_q_heads, num_kv_heads, block_size_log2, max_blocks, slot_pos, slot_head;
    int group, n_hp;           // q-heads per kv-head, head parts per kv-head
    int vw;                    // head parts per workgroup (a power of two)
    int whole;                 // workgroup x holds sequence x and writes its output rows
};

// LDS of a workgroup besides the K table: the waves' block-table entries; a part that holds, one after the other, the operands of
// the rotation and the waves' record stage buffers, then the rotated queries; at a segment's end
// the waves' results take the place of both.
constexpr int kPitPad = 2;   // floats: 8 rows of 16 nw + 2 floats are 16 banks apart (mod 64)
constexpr int kQRawPad = 16; // bytes
__host__ __device__ constexpr int pit_bytes(int nw) { return kHeadDim * (16 * nw + kPitPad) * 4; }
__host__ __device__ constexpr int qraw_bytes(int rows) { return rows * (2 * kHeadDim + kQRawPad); }
template <int LAYOUT, bool KF8, bool KB3, bool V3> __host__ __device__ constexpr int stage_bytes() {
    constexpr int rec = record_bytes<LAYOUT, KF8, KB3, V3>();
    // (3-bit: + 16 bytes, a 3-bit V dword of token 15, n = 15, reads 4 bytes past them)
    return LAYOUT != 0 ? 0 : KB3 ? 16 * rec + 16 : KF8 ? 16 * rec : 0;
}
// Bytes of the first part, and of all of it.
template <int LAYOUT, int G, bool ROT, bool KF8, bool KB3, bool V3>
__host__ __device__ constexpr int step_lds_low(int vw, int sw) {
    const int stage = vw * sw * stage_bytes<LAYOUT, KF8, KB3, V3>();
    const int rot = ROT ? pit_bytes(vw * sw) + qraw_bytes(vw * G) : 0;
    return stage > rot ? stage : rot;
}
template <int LAYOUT, int G, bool ROT, bool KF8, bool KB3, bool V3> constexpr int step_lds(int vw, int sw) {
    const int run = step_lds_low<LAYOUT, G, ROT, KF8, KB3, V3>(vw, sw) + (ROT ? vw * G * kQRowFloats * 4 : 0);
    const int join = sw > 1 ? vw * sw * G * (kHeadDim + 1) * 4 : 0;
    return vw * sw * kTableTiles * 4 + (run > join ? run : join);
}

// ---- K table, built by the waves of a workgroup together ------------------------------
// 4-bit keys: rows i = w (mod nw) (entries e = lane + 64 i, the pair (c[e & 15], c[e >> 4])); 3-bit
// keys: 64 entries (c[e & 7], c[e >> 3]), wave 0.
template <bool KB3> struct TableRows {
    float2 r[KB3 ? 1 : 256 / kWave];
};
template <bool KB3> __device__ __forceinline__ TableRows<KB3> load_table_rows(const float *centroids, int lane) {
    TableRows<KB3> v;
#pragma unroll
    for (int i = 0; i < (KB3 ? 1 : 256 / kWave); ++i) {
        const int e = lane + kWave * i;
        v.r[i] = KB3 ? float2{centroids[e & 7], centroids[e >> 3]} : float2{centroids[e & 15], centroids[e >> 4]};
    }
    return v;
}
template <bool KB3>
__device__ __forceinline__ void build_table_rows(uint32_t *tbl, const TableRows<KB3> &v, int lane, int w, int nw) {
#pragma unroll
    for (int i = 0; i < (KB3 ? 1 : 256 / kWave); ++i) {
        if ((i & (nw - 1)) != w)
            continue;
        const int e = lane + kWave * i;
        const uint32_t p_lo = split_f16(v.r[i].x), p_hi = split_f16(v.r[i].y);
        tbl[2 * e] = (p_lo & 0xFFFFu) | (p_hi << 16);
        tbl[2 * e + 1] = (p_lo >> 16) | (p_hi & 0xFFFF0000u);
    }
}

// ---- Query rotation --------------------------------------------------------------------
// The waves of a workgroup compute the rotated queries of its heads, q_rot = query @ rot_t,
// into LDS with the operands and the MFMA order of rotate_mfma_kernel, so the rows are
// bit-identical to that launch's: each query row scaled by the power of two that puts its
// largest |x| in [2^14, 2^15) (exact in f16 for fp16 / bf16 queries), rot_t as f16 hi + lo
// parts, D[rows 4g .. 4g+3][col n] of output column tile c per row tile.  The workgroup loads
// rot_t 16 nw columns at a time and its query rows once, whole lines and 16 bytes per lane, and
// hands them over through LDS; wave w takes column tile w of each chunk (8 waves: one chunk).
// Loads per wave straight into the operand layout (32 of rot_t, each half lines, and every wave
// all the query rows) kept a CU's 8 waves issuing for 3 us.
template <int G> struct RotLoads {
    uint4 pit[8];
    uint4 q[G / 4];
};
// Chunk `c` of rot_t: lane i of the workgroup's nw * 64 takes 16-byte piece i + 64 nw k of the
// chunk's 128 rows of 4 nw pieces.  (rot_t is an array of floats: its pieces are 4-byte aligned.)
template <int G>
__device__ __forceinline__ void rot_load_pit(RotLoads<G> &r, const float *__restrict__ rot_t, int c, int nw, int tid) {
    typedef uint32_t piece __attribute__((ext_vector_type(4), aligned(4)));
    const int per_row = 4 * nw, row = div_pos(tid, per_row), col = tid - row * per_row;  // 16 rows per load
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const piece v = *reinterpret_cast<const piece *>(rot_t + (16 * k + row) * kHeadDim + 16 * nw * c + 4 * col);
        r.pit[k] = uint4{v[0], v[1], v[2], v[3]};
    }
}
// The query rows row_base .. + n_rows - 1, 16 pieces each (n_rows <= G nw; spare lanes repeat the last piece).
template <int G>
__device__ __forceinline__ void rot_load_query(RotLoads<G> &r, const uint16_t *__restrict__ query, int64_t row_base,
                                               int n_rows, int nw, int tid) {
#pragma unroll
    for (int k = 0; k < G / 4; ++k)
        r.q[k] = reinterpret_cast<const uint4 *>(query + row_base * kHeadDim)[min(tid + 64 * nw * k, 16 * n_rows - 1)];
}
template <int G>
__device__ __forceinline__ void rot_store_pit(const RotLoads<G> &r, float *pit, int nw, int tid) {
    const int per_row = 4 * nw, row = div_pos(tid, per_row), col = tid - row * per_row;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        uint2 *p = reinterpret_cast<uint2 *>(pit + (16 * k + row) * (16 * nw + kPitPad) + 4 * col);
        p[0] = uint2{r.pit[k].x, r.pit[k].y};
        p[1] = uint2{r.pit[k].z, r.pit[k].w};
    }
}
// Max over the 16 lanes of a DPP row, in every lane.
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, dppf<0x121>(x));  // row_ror:1, 2, 4, 8
    x = fmaxf(x, dppf<0x122>(x));
    x = fmaxf(x, dppf<kRor4>(x));
    return fmaxf(x, dppf<kRor8>(x));
}
// The loaded rows scaled to f16 (a row's 16 pieces are in the 16 lanes of a DPP row), each with
// its exponent after its 128 elements.
template <typename InT, int G>
__device__ __forceinline__ void rot_store_query(const RotLoads<G> &r, unsigned char *qraw, int n_rows, int nw, int tid) {
    typedef InT in8 __attribute__((ext_vector_type(8)));
#pragma unroll
    for (int k = 0; k < G / 4; ++k) {
        const in8 p = __builtin_bit_cast(in8, r.q[k]);
        float amax = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            amax = fmaxf(amax, fabsf(to_float<InT>(p[j])));
        amax = row16_max(amax);
        const int e = (amax > 0.f && amax < __builtin_inff()) ? 15 - __builtin_amdgcn_frexp_expf(amax) : 0;
        half8 h;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            h[j] = (_Float16)__builtin_ldexpf(to_float<InT>(p[j]), e);
        const int i = tid + 64 * nw * k;
        if (i < 16 * n_rows) {
            unsigned char *row = qraw + (i >> 4) * (2 * kHeadDim + kQRawPad);
            *reinterpret_cast<half8 *>(row + 16 * (i & 15)) = h;
            if ((i & 15) == 0)
                *reinterpret_cast<int *>(row + 2 * kHeadDim) = e;
        }
    }
}
// Column tile w of chunk c for every row, into the LDS rows qbuf [n_rows][kQRowFloats].  B operand
// of step kb: rot_t rows 32kb + 8g + j, column 16w + n of the chunk, as f16 hi + lo; A operand of
// row tile t: elements 32kb + 8g .. +7 of row 16t + n (rows past the last one repeat it and are
// not stored).  At most 8 G rows, so G / 2 row tiles.
template <int G>
__device__ __forceinline__ void rot_column_tile(const float *pit, const unsigned char *qraw, float *qbuf, int w, int nw,
                                                int c, int n_rows, int n, int g) {
    constexpr int kRow = 2 * kHeadDim + kQRawPad;
    floatx4 acc[G / 2];
#pragma unroll
    for (int t = 0; t < G / 2; ++t)
        acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        half8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float v = pit[(32 * kb + 8 * g + j) * (16 * nw + kPitPad) + 16 * w + n];
            hi[j] = (_Float16)v;
            lo[j] = (_Float16)(v - (float)hi[j]);
        }
#pragma unroll
        for (int t = 0; t < G / 2; ++t) {
            if (16 * t >= n_rows)
                break;
            const half8 a = *reinterpret_cast<const half8 *>(qraw + min(16 * t + n, n_rows - 1) * kRow + 64 * kb + 16 * g);
            acc[t] = mfma(a, hi, acc[t]);
            acc[t] = mfma(a, lo, acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < G / 2; ++t) {
        if (16 * t >= n_rows)
            break;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * t + 4 * g + i;
            if (r < n_rows)
                qbuf[r * kQRowFloats + 16 * (c * nw + w) + n] =
                    __builtin_ldexpf(acc[t][i], -*reinterpret_cast<const int *>(qraw + r * kRow + 2 * kHeadDim));
        }
    }
}
// FP8 keys: dims 16g .. 16g+15 and 64 + 16g .. of an unrotated bf16 / fp16 query row (exact in
// fp32), read as the caller has it.
template <typename T>
__device__ __forceinline__ void load_query_rows_fp8(float4 (&qx)[8], const T *__restrict__ query, int64_t head_row,
                                                    int g) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    const T *qr = query + head_row * kHeadDim + 16 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const t8 v = *reinterpret_cast<const t8 *>(qr + 64 * (i >> 1) + 8 * (i & 1));
        qx[2 * i] = float4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
        qx[2 * i + 1] = float4{(float)v[4], (float)v[5], (float)v[6], (float)v[7]};
    }
}

// LDS accesses done, then the workgroup barrier.  KV loads stay in flight: no vmcnt wait,
// unlike __syncthreads.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- Outputs ------------------------------------------------------------------------------
// Output element conversion (the same roundings as Stage2's).
__device__ __forceinline__ void put_out(void *out, int dtype, int64_t i, float v) {
    if (dtype == kOutBf16)
        static_cast<__bf16 *>(out)[i] = (__bf16)v;
    else if (dtype == kOutF16)
        static_cast<_Float16 *>(out)[i] = (_Float16)v;
    else
        static_cast<float *>(out)[i] = v;
}

// What happens to a finished segment's rows: the output itself when the workgroup held the
// whole sequence (one row per head merges to itself: weight exp(0) = 1), else part row p, and
// from part 0 the count of parts.
struct RowSink {
    bool whole;
    int64_t row0;     // first head's row b * Hq + head
    int p, n_parts;
};
__device__ __forceinline__ void sink_lse(const StepArgs &a, const RowSink &s, int h, float v) {
    if (s.whole) {
        a.lse[s.row0 + h] = v;
        return;
    }
    float *l = part_lse(a.parts, (int64_t)a.batch * a.num_q_heads, s.row0 + h, a.num_splits);
    l[s.p] = part_lse_value(v);
    if (s.p == 0 && s.n_parts < a.num_splits)
        l[a.num_splits - 1] = part_count_mark(s.n_parts);
}
// The wave's rows from registers (heads nh .. G-1 are padding).
template <int G, bool V3>
__device__ __forceinline__ void emit_rows(const StepArgs &a, const RowSink &s, const State &st, const floatx4 (&acc)[8],
                                          const LaneConst &lc, int nh) {
    int h0;
    float o[G / 4][8], safe_l;
    finish_rows<G, V3>(st, acc, lc, h0, o, safe_l);
    typedef float float4a __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int k = 0; k < G / 4; ++k) {
        if (h0 + k >= nh)
            continue;
        if (s.whole) {
            const int64_t r = (s.row0 + h0 + k) * kHeadDim + 8 * lc.n;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                put_out(a.out, a.out_dtype, r + i, o[k][i]);
        } else {
            float *r = part_row(a.parts, s.row0 + h0 + k, a.num_splits, s.p) + 8 * lc.n;
            *reinterpret_cast<float4a *>(r) = float4a{o[k][0], o[k][1], o[k][2], o[k][3]};
            *reinterpret_cast<float4a *>(r + 4) = float4a{o[k][4], o[k][5], o[k][6], o[k][7]};
        }
    }
    if (lc.g == 0 && lc.n < nh)
        sink_lse(a, s, lc.n, lse_of(st.negm, safe_l));
}
// The rows of the sw waves of a head part joined in LDS: every wave leaves its rows and LSEs
// (-inf from a wave without tiles), then merges heads sub, sub + sw, ... of its part as
// merge_parts_kernel would.  buf: the workgroup's [waves][G][D] rows, then [waves][G] LSEs.
template <int G, bool V3>
__device__ __forceinline__ void join_rows(const StepArgs &a, const RowSink &s, const State &st, const floatx4 (&acc)[8],
                                          const LaneConst &lc, int nh, float *buf, int w, int vi, int sub, bool empty,
                                          int lane) {
    const int nw = a.vw * a.sw;
    float *lses = buf + nw * G * kHeadDim;
    int h0;
    float o[G / 4][8], safe_l;
    finish_rows<G, V3>(st, acc, lc, h0, o, safe_l);
    lds_barrier();  // the buffer's place held stage buffers and queries until here
#pragma unroll
    for (int k = 0; k < G / 4; ++k) {
        float4 *r = reinterpret_cast<float4 *>(buf + (w * G + h0 + k) * kHeadDim + 8 * lc.n);
        r[0] = float4{o[k][0], o[k][1], o[k][2], o[k][3]};
        r[1] = float4{o[k][4], o[k][5], o[k][6], o[k][7]};
    }
    if (lc.g == 0 && lc.n < G)
        lses[w * G + lc.n] = empty ? -INFINITY : lse_of(st.negm, safe_l);
    lds_barrier();
    for (int h = sub; h < nh; h += a.sw) {
        float mx = -INFINITY;
        for (int j = 0; j < a.sw; ++j)
            mx = fmaxf(mx, lses[(j * a.vw + vi) * G + h]);
        float a0 = 0.f, a1 = 0.f, wsum = 0.f;
        for (int j = 0; j < a.sw; ++j) {
            const int at = (j * a.vw + vi) * G + h;
            const float wt = expf(lses[at] - mx);
            // a wave without tiles weighs 0 and its row is 0
            a0 = fmaf(wt, buf[at * kHeadDim + 2 * lane], a0);
            a1 = fmaf(wt, buf[at * kHeadDim + 2 * lane + 1], a1);
            wsum += wt;
        }
        const float inv = 1.f / wsum;
        if (s.whole) {
            const int64_t r = (s.row0 + h) * kHeadDim + 2 * lane;
            put_out(a.out, a.out_dtype, r, a0 * inv);
            put_out(a.out, a.out_dtype, r + 1, a1 * inv);
        } else {
            float *r = part_row(a.parts, s.row0 + h, a.num_splits, s.p) + 2 * lane;
            r[0] = a0 * inv;
            r[1] = a1 * inv;
        }
        if (lane == 0)
            sink_lse(a, s, h, mx + logf(wsum));
    }
}

// The kernel.  ROT: it rotates the (bf16 / fp16) query itself.  KF8 / KB3 / V3: the presets, as
// in stage1_xdl_kernel.  Head parts are numbered
// kv-head by kv-head (part vh: kv-head vh / parts, heads G (vh % parts) .. of its group), so
// the heads of consecutive parts are consecutive.
template <int LAYOUT, int G, bool ROT, bool KF8 = false, bool KB3 = false, bool V3 = false>
__global__ __launch_bounds__(kWave *kStepWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void decode_step_kernel(const StepArgs a) {
    static_assert(!ROT || !KF8, "FP8 keys take the query unrotated");
    constexpr int TPL = G / 4;
    constexpr int RING = 4;
    constexpr int FIRST_SLOTS = 2;  // ring slots issued before the table and the q operands (see stage1_xdl_kernel)
    constexpr bool STG = KB3 && LAYOUT == 0, STG8 = KF8 && LAYOUT == 0;
    constexpr int kRec = record_bytes<LAYOUT, KF8, KB3, V3>();
    constexpr int kStage = stage_bytes<LAYOUT, KF8, KB3, V3>();
    using RK = std::conditional_t<STG8, RawRec3, std::conditional_t<KF8, RawK8, std::conditional_t<STG, RawRec, std::conditional_t<KB3, RawK3, RawK<LAYOUT>>>>>;
    // (the K table has a place of its own, known to the compiler: an address computed from the
    // dynamic base costs the loop 12 VALU per tile)
    __shared__ __align__(16) uint32_t ktab[KF8 ? 4 : KTable<LAYOUT>::words];
    extern __shared__ __align__(16) unsigned char dyn[];

    const int lane = threadIdx.x % kWave;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), nw = a.vw * a.sw;
    uint32_t *const blocks = reinterpret_cast<uint32_t *>(dyn) + w * kTableTiles;
    unsigned char *const work = dyn + nw * kTableTiles * 4;
    unsigned char *const recbuf = work + w * kStage;
    float *const pit = reinterpret_cast<float *>(work);
    unsigned char *const qraw = work + pit_bytes(nw);
    float *const qbuf = reinterpret_cast<float *>(work + step_lds_low<LAYOUT, G, ROT, KF8, KB3, V3>(a.vw, a.sw));
    int vg = blockIdx.x, x = blockIdx.y;
    const int nx = gridDim.y;
    if constexpr (LAYOUT == 1 || KF8 || KB3) {
        // head parts that share 128-byte lines on one XCD (see stage1_xdl_kernel)
        constexpr int kXcds = 8;
        if (gridDim.x > 1 && nx % kXcds == 0) {
            const int lin = blockIdx.x + gridDim.x * blockIdx.y, r = lin / kXcds;
            x = lin % kXcds + kXcds * (r / (int)gridDim.x);
            vg = r % (int)gridDim.x;
        }
    }
    // waves w and w + 4 share a SIMD: with eight head parts it gets parts 2s and 2s + 1, one even
    // and one odd kv-head (they read HBM at different speeds, see stage1_xdl_kernel)
    const int sub = a.vw == 8 ? 0 : div_pos(w, a.vw);
    const int vi = a.vw == 8 ? 2 * (w & 3) + (w >> 2) : w - sub * a.vw;
    const int group = a.group, n_hp = a.n_hp;
    const int vh = vg * a.vw + vi, kvh = div_pos(vh, n_hp);
    const int hb = kvh * group + (vh - kvh * n_hp) * G;      // the wave's first q-head
    const int nh = min(G, (kvh + 1) * group - hb);           // its real q-heads (the rest are padding)
    const int hl = min((lane & 15) & (G - 1), nh - 1);       // the lane's q-head (padding: a real one's)
    // the workgroup's heads, consecutive: h_first .. h_first + n_rows - 1
    const int v0 = vg * a.vw, v1 = v0 + a.vw - 1, kv0 = div_pos(v0, n_hp), kv1 = div_pos(v1, n_hp);
    const int h_first = kv0 * group + (v0 - kv0 * n_hp) * G;
    const int n_rows = min(kv1 * group + (v1 - kv1 * n_hp) * G + G, (kv1 + 1) * group) - h_first;
    const int block_size = 1 << a.block_size_log2, tl = a.block_size_log2 - 4;

    // What does not depend on the lengths goes out first, under the latency of reading them: the
    // first 64 lengths themselves, the K table's and the rotation's operands, and a guess (equal
    // lengths that fill the table) at the sequence and the wave's first tiles: its block-table
    // entries and query rows.  Where it turns out right, registers serve the first chunk and the
    // rotation, and nothing but the cut stands before the first KV loads.
    const int len_lane = a.seq_lens[min(lane, a.batch - 1)];
    TableRows<KB3> table_rows{};
    if constexpr (!KF8)
        table_rows = load_table_rows<KB3>(a.centroids, lane);
    const int per_seq = max(a.per_seq, 1);
    const int guess_b = a.whole ? x : min(div_pos(x, per_seq), a.batch - 1);
    int guess_tile;
    {
        const Run r = run_of(a.max_blocks << tl, a.whole ? 1 : per_seq, a.whole ? 0 : x - guess_b * per_seq);
        guess_tile = max(r.first, 0) + run_of(max(r.count, 0), a.sw, sub).first;
    }
    const int bt_guess = a.block_table[(int64_t)guess_b * a.max_blocks + min((guess_tile + lane) >> tl, a.max_blocks - 1)];
    RotLoads<G> rot;
    if constexpr (ROT) {
        rot_load_query(rot, static_cast<const uint16_t *>(a.query), (int64_t)guess_b * a.num_q_heads + h_first, n_rows,
                       nw, threadIdx.x);
        rot_load_pit(rot, a.rot_t, 0, nw, threadIdx.x);
    }
    // the head's sink logit (a dummy read when there are none, so the load is unconditional)
    const float sink = *(a.sinks ? a.sinks + hb + hl : reinterpret_cast<const float *>(a.seq_lens));

    Cut cut;
    bool single = true;  // the workgroup has no segment after this one
    if (a.whole) {
        cut.b = x;
        cut.len = a.seq_lens[x];
        cut.tiles = tiles_of(cut.len);
        cut.run = Run{0, cut.tiles};
        cut.p = 0;
        cut.n_parts = 1;
        if (cut.tiles == 0) {  // an empty sequence: what Stage2 writes for it (0 / 0 and ln 0)
            if (sub == 0) {
                const int64_t r0 = ((int64_t)x * a.num_q_heads + hb) * kHeadDim;
                for (int i = lane; i < nh * kHeadDim; i += kWave)
                    put_out(a.out, a.out_dtype, r0 + i, __builtin_nanf(""));
                if (lane < nh)
                    a.lse[(int64_t)x * a.num_q_heads + hb + lane] = -__builtin_inff();
            }
            return;
        }
    } else if (!first_segment(cut, a, nx, x, lane, len_lane, single)) {
        return;
    }

    LaneConst lc;
    lc.n = lane & 15;
    lc.g = lane >> 4;
    lc.tok_bit0 = (lc.n >> 2) & 1;
    lc.tok_bit1 = (lc.n >> 3) & 1;
    lc.upper = lc.n >= 8;
    lc.part_sel = lc.upper ? 0x07060302u : 0x05040100u;
    const LaneOffsets off =
        lane_offsets<LAYOUT, G, KF8, KB3, V3>(lc.n, lc.g, kvh, a.num_kv_heads, block_size, a.slot_pos, a.slot_head);
    const int tok0 = 4 * lc.g + TPL * (lc.n / G);  // the lane's first softmax token

    if constexpr (!KF8)
        build_table_rows<KB3>(ktab, table_rows, lane, w, nw);

    if constexpr (ROT)
        if (cut.b != guess_b)
            rot_load_query(rot, static_cast<const uint16_t *>(a.query), (int64_t)cut.b * a.num_q_heads + h_first,
                           n_rows, nw, threadIdx.x);

    for (bool first = true;; first = false) {
        // the wave's run of the segment; without tiles it takes a masked one along (its loads
        // are in bounds), so that every wave reaches the barriers
        const Run mine = run_of(cut.run.count, a.sw, sub);
        const int n_run = mine.count, t_lo = cut.run.first + min(mine.first, cut.run.count - 1);
        const int run_start = 16 * t_lo, run_end = n_run > 0 ? min(16 * (t_lo + n_run), cut.len) : run_start;
        const int total = max((n_run + RING - 1) & ~(RING - 1), RING);
        const int b = cut.b;
        // opaque, or the compiler hoists the operand conversions out of the segment loop and holds
        // them in registers (spilling) through the stream
        int rn = lane & 15, rg = lane >> 4, tid = threadIdx.x;
        asm volatile("" : "+v"(rn), "+v"(rg), "+v"(tid));
        if (!first && (ROT || a.sw > 1))
            lds_barrier();  // the last segment's LDS contents are no longer read

        State st{__FLT_MAX__, 0.f, 0.f, 1.f};
        if (a.sinks && t_lo == 0 && sub == 0) {
            // the first tokens start from the head's sink logit: max = sink, sum = 1 (one lane
            // per head, lane h, holds it; the sums are totalled over the lanes n = h (mod G))
            st.negm = -sink * kLog2e;
            st.l = lane < G ? 1.f : 0.f;
        }
        floatx4 acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
        half8 bq[8];
        float q_unscale = 1.f;

        const int32_t *bt = a.block_table + (int64_t)b * a.max_blocks;
        // base_lo / base_hi: the address of the 16-token piece at the lane's stream position (its KV
        // block plus the piece's offset), moff_lane: the SoA metadata offset relative to it.
        int mask_lane = 0, moff_lane = 0;
        uint32_t base_lo = 0, base_hi = 0;
        RK kr[RING];
        RawV<LAYOUT, TPL> vr[RING];
        __amdgpu_buffer_rsrc_t pos[RING];
        auto rsrc_at = [&](int j) {
            const uint64_t p = ((uint64_t)__builtin_amdgcn_readlane(base_hi, j & 63) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane(base_lo, j & 63);
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(p), 0, 0x7FFFFFFF, 0x00020000);
        };
        // (scheduling barriers: loads in program order, so each wait counts only later tiles')
        auto issue_kpos = [&](RK &r, const __amdgpu_buffer_rsrc_t &rsrc) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (KF8 || KB3)
                issue_k(r, rsrc, 0, off);
            else
                issue_k<LAYOUT>(r, rsrc, 0, off);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto issue_vpos = [&](RawV<LAYOUT, TPL> &r, const __amdgpu_buffer_rsrc_t &rsrc, int j) {
            const int moff = LAYOUT == 0 ? __builtin_amdgcn_readlane(moff_lane, j & 63) : 0;
            __builtin_amdgcn_sched_barrier(0);
            issue_v<LAYOUT, TPL, KF8, KB3, V3>(r, rsrc, 0, moff, off);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto issue_slots = [&](int j0, int last, int k0, int k1) {
#pragma unroll
            for (int k = 0; k < RING; ++k) {
                if (k < k0 || k >= k1)
                    continue;
                const auto rsrc = rsrc_at(min(j0 + k, last));
                issue_kpos(kr[k], rsrc);
                issue_vpos(vr[k], rsrc, min(j0 + k, last));
            }
        };
        // Stream position p lives in lane p mod 64: its tile, mask and address.  p: the lane's
        // position, blk: the block of its tile (past the run: of the last one).
        auto tile_at = [&](int p) { return t_lo + min(p, max(n_run, 1) - 1); };
        auto set_position = [&](int p, int blk, bool here) {
            const int tile = tile_at(p);
            const int toff = (16 * tile) & (block_size - 1);
            // the piece's first record: token toff of kv-head 0 (AoS: at toff * slot_pos)
            const int piece = LAYOUT == 0 ? toff * a.num_kv_heads * kRec : toff * a.slot_pos;
            const uint64_t at = reinterpret_cast<uint64_t>(a.cache) + (uint64_t)((int64_t)blk * a.block_stride) +
                                (uint64_t)piece;
            base_lo = here ? (uint32_t)at : base_lo;
            base_hi = here ? (uint32_t)(at >> 32) : base_hi;
            moff_lane = here ? (block_size - toff) * a.num_kv_heads * kRec + toff * 2 : moff_lane;
            mask_lane = here ? (p < n_run ? tile : -(1 << 24)) : mask_lane;  // padding: no valid token
        };
        // the block of tile t_lo + min(p, n_run - 1), from the table or, for the first 64, the guess
        auto block_at = [&](int p, bool may_guess) {
            if (may_guess && b == guess_b && t_lo == guess_tile)
                return __shfl(bt_guess, tile_at(p) - t_lo, kWave);
            return bt[tile_at(p) >> tl];
        };

        floatx4 sc;         // QK^T accumulator of the next tile
        std::conditional_t<KF8, K8, std::conditional_t<KB3, RawK3, uint4>> kn;  // K bytes of the next tile, in the MFMA layout
        float csq_tot = 0;  // AoS: ||c[idx]||^2 of token n of that tile
        uint32_t aw[4];
        // K bytes of a loaded tile in the MFMA layout; staged records also give its V codes
        auto take_k = [&](const RK &r, RawV<LAYOUT, TPL> &v) {
            if constexpr (STG)
                return stage_records<kRec, V3>(r, recbuf, off, v.v);
            else if constexpr (STG8)
                return stage_records(r, recbuf, off, v.v);
            else if constexpr (KF8 || KB3)
                return decode_k(r, off);
            else
                return decode_k<LAYOUT>(r, off);
        };
        auto look_up = [&](const auto &k) {
            if constexpr (KF8)
                return lookup_tile(k, ktab);
            else
                return lookup_tile<LAYOUT>(k, ktab);
        };
        // Stage j: softmax of position j, then QK^T of position j + 1; odd stages also run the
        // PV of positions (j - 1, j) (see stage1_xdl_kernel).
        auto stage = [&](int k, const RawV<LAYOUT, TPL> &vprev, const RawV<LAYOUT, TPL> &vcur, const RK &kafter,
                         RawV<LAYOUT, TPL> &vafter, int j) {
            const KOps e = look_up(kn);
            __builtin_amdgcn_sched_barrier(0);
            const TileV t = decode_v<LAYOUT, TPL>(vcur, off);
            const int t0 = 16 * __builtin_amdgcn_readlane(mask_lane, j & 63);
            const bool boundary = !(t0 >= run_start && t0 + 16 <= run_end);
            float dot[TPL], nf[TPL];
            bool valid[TPL];
            lane_dots<G>(sc, lc, dot);
#pragma unroll
            for (int q = 0; q < TPL; ++q) {
                valid[q] = (uint32_t)(t0 + tok0 + q - run_start) < (uint32_t)(run_end - run_start);
                if constexpr (LAYOUT == 0 || KF8)
                    nf[q] = half_at(t.norm, q) * q_unscale;
                else  // ||c[idx]||^2 of token tok0 + q: totals sit in lanes n = token (any row)
                    nf[q] = half_at(t.norm, q) * __builtin_amdgcn_rsqf(__shfl(csq_tot, tok0 + q, kWave) + 1e-16f) *
                            q_unscale;
            }
            if (k & 1)
                softmax_tile<G, true>(dot, nf, t, st, acc, lc, boundary, valid, aw[0], aw[1], aw[2], aw[3]);
            else
                softmax_tile<G, false>(dot, nf, t, st, acc, lc, boundary, valid, aw[0], aw[1], aw[0], aw[1]);
            if (k & 1) {
                const TileV ta = decode_v<LAYOUT, TPL>(vprev, off);
                sc = pv_qk<V3>(acc, aw, ta.v, t.v, e, bq);
            } else {
                sc = qk_tile(e, bq);
            }
            if constexpr (LAYOUT == 1 && !KF8)
                csq_tot = sum_xor16(sum_xor32(e.csq));
            kn = take_k(kafter, vafter);
        };

        // First loads, then (under them) the rotation, the K table and the q operands.
        const int blk0 = block_at(lane, first);
        float4 q_rows[8];
        if constexpr (!ROT) {
            const int64_t head_row = (int64_t)b * a.num_q_heads + hb + hl;
            if (KF8 && a.q_dtype == kOutBf16)
                load_query_rows_fp8(q_rows, static_cast<const __bf16 *>(a.query), head_row, rg);
            else if (KF8 && a.q_dtype == kOutF16)
                load_query_rows_fp8(q_rows, static_cast<const _Float16 *>(a.query), head_row, rg);
            else
                load_q_rows(q_rows, static_cast<const float *>(a.query), head_row, rg, KF8);
        }
        set_position(lane, blk0, true);
        issue_slots(0, total - 1, 0, FIRST_SLOTS);
        if constexpr (!KF8) {
            if constexpr (ROT) {
                if (a.q_dtype == kOutBf16)
                    rot_store_query<__bf16>(rot, qraw, n_rows, nw, tid);
                else
                    rot_store_query<_Float16>(rot, qraw, n_rows, nw, tid);
                for (int c = 0;; ++c) {
                    rot_store_pit(rot, pit, nw, tid);
                    lds_barrier();
                    rot_column_tile<G>(pit, qraw, qbuf, w, nw, c, n_rows, rn, rg);
                    if ((c + 1) * nw >= kHeadDim / 16)
                        break;
                    rot_load_pit(rot, a.rot_t, c + 1, nw, tid);
                    lds_barrier();  // the chunk is no longer read
                }
            }
            if (ROT || first)
                lds_barrier();
            if constexpr (ROT)
#pragma unroll
                for (int m = 0; m < 8; ++m)
                    q_rows[m] = *reinterpret_cast<const float4 *>(qbuf + (hb + hl - h_first) * kQRowFloats +
                                                                 32 * rg + 4 * m);
        }
        if (hl != ((lane & 15) & (G - 1)))  // padding head: a zero query
#pragma unroll
            for (int m = 0; m < 8; ++m)
                q_rows[m] = float4{0.f, 0.f, 0.f, 0.f};
        q_unscale = q_operands(bq, q_rows, lc.n, a.score_scale_log2);
        issue_slots(0, total - 1, FIRST_SLOTS, RING);

        for (int j0 = 0; j0 < total; j0 += kTableTiles) {
            const int last = min(j0 + kTableTiles, total) - 1;
            if (j0 > 0) {
                set_position(j0 + lane, block_at(j0 + lane, false), true);
                issue_slots(j0, last, 0, RING);
            }
            for (int i = 64; i <= last - j0; i += 64)
                blocks[i + lane] = (uint32_t)bt[tile_at(j0 + i + lane) >> tl];
            // one wave: its LDS accesses run in program order; only the compiler must not forward
            // a lane's own values
            asm volatile("" ::: "memory");
            {
                const KOps e = look_up(take_k(kr[0], vr[0]));
                sc = qk_tile(e, bq);
                if constexpr (LAYOUT == 1 && !KF8)
                    csq_tot = sum_xor16(sum_xor32(e.csq));
                kn = take_k(kr[1], vr[1]);
            }
            pos[0] = rsrc_at(min(j0 + RING, last));
            issue_kpos(kr[0], pos[0]);
            int j = j0;
            do {
                // every 32 positions the lanes whose positions are done take those 64 further on
                // (loads run at most 8 positions ahead)
                if ((j & 31) == 0 && j > j0 && j + 32 <= last) {
                    const int p = j + 32 + ((lane - j - 32) & 63);
                    set_position(p, (int)blocks[min(p, last) - j0], p < j + 64);
                }
#pragma unroll
                for (int k = 0; k < RING; ++k) {
                    stage(k, vr[(k + RING - 1) % RING], vr[k], kr[(k + 2) % RING], vr[(k + 2) % RING], j + k);
                    pos[(k + 1) % RING] = rsrc_at(min(j + k + 1 + RING, last));
                    issue_kpos(kr[(k + 1) % RING], pos[(k + 1) % RING]);
                    if (k & 1) {
                        issue_vpos(vr[k - 1], pos[(k + 3) % RING], min(j + k - 1 + RING, last));
                        issue_vpos(vr[k], pos[k % RING], min(j + k + RING, last));
                    }
                }
                j += RING;
            } while (j <= last);
        }
        const RowSink rows{a.whole != 0, (int64_t)b * a.num_q_heads + hb, cut.p, cut.n_parts};
        if (a.sw == 1)
            emit_rows<G, V3>(a, rows, st, acc, lc, nh);
        else
            join_rows<G, V3>(a, rows, st, acc, lc, nh, reinterpret_cast<float *>(work), w, vi, sub, n_run == 0, lane);
        if (a.whole || single || !next_segment(cut, a, x, true))
            return;
        if constexpr (ROT) {  // (here, not at the segment's start: there they would be live through the stream)
            rot_load_query(rot, static_cast<const uint16_t *>(a.query), (int64_t)cut.b * a.num_q_heads + h_first,
                           n_rows, nw, tid);
            rot_load_pit(rot, a.rot_t, 0, nw, tid);
        }
    }
}

}  // namespace xdl
}  // namespace tq4
