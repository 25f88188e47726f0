// Kernel parameter blocks and host-side launchers of the gfx950 kernels.
// Included by the kernel sources and by the C ABI (capi.hip); not installed.
#pragma once

#include <algorithm>

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mtlattn {

// CUs of the current device (cached per device; 256 if unknown)
int device_cus();

// Tensor geometry shared by every kernel (the scalar block of the reference's
// Params, src/ext.mm:44-57, with 64-bit row strides).
struct Geometry {
    const int* cu_q;
    const int* cu_kv;
    int64_t total_q, total_kv;
    int num_seqs, hq, hkv, g, d;
    float scale;
    int causal, window;
    const float* bias;            // nullptr = no bias
    int64_t bias_qs, bias_hs, bias_cols;
    int64_t bias_ss = -1;         // >= 0: bias rows per sequence (bias_row_offset)
    int64_t bias_rows = 0;        // rows per sequence block when bias_ss >= 0
};

// How the 16-bit flash forward cuts its work (make_fwd_plan): grid == 0: one
// workgroup per tile of query rows; else `grid` workgroups take pieces of the
// tiles' key tiles, merged afterwards.
struct FwdPlan {
    int grid = 0, nw = 0, hpw = 0, n_tiles = 0;   // waves and heads per workgroup, row tiles
    size_t bytes = 0;                             // workspace
};
FwdPlan make_fwd_plan(const Geometry& g, int max_q, int cus, size_t max_bytes);

struct FwdArgs {
    Geometry geo;
    const void* q; int64_t q_rs;
    const void* k; int64_t k_rs;
    const void* v; int64_t v_rs;
    void* o;                      // contiguous [total_q, hq, d]
    float* lse;                   // nullable [total_q, hq]
    // fp32 matrix-core forward only: f32_splits > 1 splits each workgroup's
    // key tiles over that many workgroups, with normalised fp32 partials and
    // their LSEs in f32_part (f32_fwd_part_floats floats), then merged
    float* f32_part = nullptr;
    int f32_splits = 1;
    // 16-bit flash forward only: split as plan says, with plan.bytes of scratch
    FwdPlan plan;
    void* split_ws = nullptr;
};

// Dense forward: [B, H, N, D] tensors by strides (elements; the head dim
// contiguous), o contiguous. geo: num_seqs = B, total_q = B * nq, hq, hkv, g, d,
// scale, causal and a bias by sequence and local row; no cu_seqlens. lens
// (nullable, nq == nkv): the first lens[b] tokens of batch b attend, the other
// query rows are written as 0.
struct DenseArgs {
    Geometry geo;
    const void* q; int64_t q_bs, q_hs, q_rs;
    const void* k; int64_t k_bs, k_hs, k_rs;
    const void* v; int64_t v_bs, v_hs, v_rs;
    void* o;
    const int* lens;
    int nq, nkv;
};
inline bool dense_head_dim(int d) { return d == 64 || d == 80 || d == 88 || d == 96 || d == 128; }

// Piece length of a split plan: the smallest c >= c0 for which mult times the
// pieces of c steps of all tiles (n[0 .. tiles) steps each, at least one piece a
// tile) are at most `limit`, or n_max if only whole tiles are; *wgs is that
// count of pieces. By bisection between the bounds that the sum of the steps
// gives: a plan is made on every call, and at 256 tiles of thousands of steps a
// search step by step took up to 85 ms.
inline int64_t plan_piece(const int64_t* n, int64_t tiles, int64_t mult, int64_t limit, int64_t c0, int64_t n_max,
                          int64_t* wgs) {
    int64_t sum = 0;
    for (int64_t i = 0; i < tiles; ++i) sum += n[i];
    auto count = [&](int64_t c) {
        int64_t x = 0;
        for (int64_t i = 0; i < tiles; ++i) x += n[i] > c ? (n[i] + c - 1) / c : 1;
        return x * mult;
    };
    int64_t hi = c0;
    if (c0 < n_max && (*wgs = count(c0)) > limit) {
        // lo does not fit; hi does, or is n_max
        int64_t lo = c0;
        hi = n_max;
        if (limit > 0) lo = std::max(lo, (sum * mult + limit - 1) / limit - 1);
        if (limit > tiles * mult) hi = std::min(hi, sum * mult / (limit - tiles * mult) + 1);
        while (hi - lo > 1) {
            const int64_t mid = (lo + hi) / 2;
            if (count(mid) > limit) lo = mid; else hi = mid;
        }
    }
    *wgs = count(hi);
    return hi;
}

// How the 16-bit dK/dV cuts its work (make_dkv_plan): pieces == 1: one
// workgroup per key block; else at most `pieces` pieces
// per key block on a grid of `grid` workgroups.
struct DkvPlan {
    int pieces = 1, grid = 0;
};
DkvPlan make_dkv_plan(const Geometry& g, int cus);
constexpr int kDkvPartTail = 64;   // floats past the partials (the piece length)
inline int64_t dkv_part_floats(int pieces, int64_t total_kv, int hkv, int d) {
    return pieces > 1 ? (int64_t)pieces * 2 * total_kv * hkv * d + kDkvPartTail : 0;
}

struct BwdArgs {
    Geometry geo;
    const void* q; int64_t q_rs;
    const void* k; int64_t k_rs;
    const void* v; int64_t v_rs;
    const void* dout; int64_t do_rs;
    const float* lse;             // [total_q, hq]
    const float* delta;           // [total_q, hq]
    void* dq;                     // [total_q, hq, d]
    void* dk;                     // [total_kv, hkv, d]
    void* dv;
    // 16-bit matrix-core kernels only: row strides of dq and of dk / dv
    // (0: contiguous)
    int64_t dq_rs = 0, dkv_rs = 0;
    int out_f32;                  // 1: dq/dk/dv are fp32, 0: input dtype
    // dQ only: with delta_out set, the dQ kernel computes delta = rowsum(dO * O)
    // itself from o (the forward's output) and writes it to delta_out for the
    // dK/dV kernel, in place of the separate preprocess (head dims 64 and 128)
    const void* o = nullptr; int64_t o_rs = 0;
    float* delta_out = nullptr;
    // fp32 matrix-core dQ and dK/dV only: f32_splits > 1 splits each
    // workgroup's work over that many workgroups, with fp32 partials in
    // f32_part (f32_dq_part_floats / f32_dkv_part_floats floats), which
    // launch_f32_bwd_finish adds in a fixed order; dQ also takes o / delta_out (delta in-kernel)
    float* f32_part = nullptr;
    int f32_splits = 1;
    // 16-bit dK/dV only: with dkv_plan.pieces > 1 a launch of dkv_plan.grid
    // workgroups takes pieces of the key blocks' work, with fp32 partials in
    // dkv_part (dkv_part_floats floats); the pass that adds them also clears
    // the rows of dq, dk and dv that no sequence owns and says so
    float* dkv_part = nullptr;
    DkvPlan dkv_plan;
    bool* cleared = nullptr;
};

struct DecodeArgs {
    Geometry geo;
    const void* q; int64_t q_rs;
    const void* k; int64_t k_rs;
    const void* v; int64_t v_rs;
    void* o;                      // contiguous [total_q, hq, d]
    float* lse;                   // nullable
    float* o_part;                // [hkv * head groups * slots * 16, d] (decode_workspace_rows)
    float* lse_part;              // [hkv * head groups * slots * 16]
    int num_splits;               // equal splits per sequence (used when chunk == 0)
    int chunk;                    // > 0: fixed KV chunk length (multiple of 32)
    int max_q;                    // bound on q lengths; heads_per_group * max_q <= 16
    int wg = 0;                   // 4 or 8: one workgroup of that many waves per item, not one wave;
                                  // with chunk == 0 and num_splits == 1 it writes o and lse, no partials
    // paged KV: k / v are caches [num_pages, page_size, hkv, d] (row strides
    // k_rs / v_rs per token), logical key j of sequence s in page
    // block_table[s * bt_stride + j / page_size]; block_table == nullptr:
    // contiguous K/V by cu_seqlens_kv
    const int* block_table = nullptr;
    int64_t bt_stride = 0;
    int page_size = 0, num_pages = 0;
};

// Launchers return hipSuccess or the launch error. `dtype` is MTLATTN_DTYPE_*.
hipError_t launch_fwd_mfma(int dtype, const FwdArgs& a, hipStream_t st);
hipError_t launch_fwd_dense(int dtype, const DenseArgs& a, hipStream_t st);
hipError_t launch_fwd_generic(int dtype, const FwdArgs& a, hipStream_t st);
hipError_t launch_bwd_preprocess(int dtype, const Geometry& geo, const void* o, int64_t o_rs,
                                 const void* dout, int64_t do_rs, float* delta, hipStream_t st);
hipError_t launch_bwd_dq_mfma(int dtype, const BwdArgs& a, hipStream_t st);
hipError_t launch_bwd_dkv_mfma(int dtype, const BwdArgs& a, hipStream_t st);
// dK/dV without a bias at head dims 80-128, one wave per SIMD (bwd_wide.hip);
// hipErrorNotSupported when the problem is not for it. type_code: BF16::code / F16::code.
hipError_t launch_bwd_dkv_wide(int type_code, const BwdArgs& a, hipStream_t st);
// Adds the partials of a split dK/dV launch (key blocks of kb keys, stages of
// qtl queries) into dk / dv and clears the rows of dq, dk and dv that no
// sequence owns.
hipError_t launch_dkv_finish(int type_code, const BwdArgs& a, int kb, int qtl, hipStream_t st);
hipError_t launch_bwd_dq_generic(int dtype, const BwdArgs& a, hipStream_t st);
hipError_t launch_bwd_dkv_generic(int dtype, const BwdArgs& a, hipStream_t st);
// fp32 inputs on the fp32 matrix cores (f32_mfma_head_dim, 16-byte aligned
// rows and outputs); dq / dk / dv are written as fp32
hipError_t launch_fwd_f32mfma(const FwdArgs& a, hipStream_t st);
hipError_t launch_bwd_dq_f32mfma(const BwdArgs& a, hipStream_t st);
hipError_t launch_bwd_dkv_f32mfma(const BwdArgs& a, hipStream_t st);
// The splits' partials of dq, or of dk and dv, added into them (splits 1:
// already written), and their rows that no sequence owns cleared. With both,
// dq is only cleared.
hipError_t launch_f32_bwd_finish(const BwdArgs& a, const float* part, int splits, bool dq, bool dkv, hipStream_t st);
// Rows of a [total_rows, row_bytes] tensor (row stride stride_bytes, 0:
// contiguous) outside [cu[0], cu[num_seqs]).
struct ZeroFill {
    void* ptr;
    int64_t row_bytes, total_rows;
    const int* cu;
    int64_t stride_bytes = 0;
};
// Zeroes those rows of up to three tensors in one launch.
hipError_t launch_zero_outside(const ZeroFill* fills, int n, int num_seqs, hipStream_t st);
hipError_t launch_decode(int dtype, const DecodeArgs& a, hipStream_t st);
hipError_t launch_pad_pack(int esize, int B, int N, int H, int D, const void* src, int64_t sb, int64_t sh,
                           int64_t sn, const int* lens, int* cu, void* dst, hipStream_t st);
hipError_t launch_pad_unpack(int esize, int B, int N, int H, int D, const void* src, const int* lens, const int* cu,
                             void* dst, int64_t sb, int64_t sh, int64_t sn, hipStream_t st);
hipError_t launch_content_differs(const void* a, const void* b, int64_t bytes, int* flag, hipStream_t st);

// Partial rows of the split-KV workspace (fp32 O rows of D values plus one
// LSE each): kv heads x head groups x work-item slots x 16.
inline int64_t decode_workspace_rows(int64_t total_kv, int num_seqs, int hkv, int n_hg, int chunk, int ns) {
    const int64_t slots = chunk > 0 ? total_kv / chunk + num_seqs + 1 : (int64_t)num_seqs * ns;
    return (int64_t)hkv * n_hg * slots * 16;
}

// Which head dims have MFMA kernels.
// head dims of the matrix-core flash kernels (fp16/bf16): 64 and 128 native,
// 80, 88, 96 on the 128-wide tile with the spare columns unused, 160 and 256
// on 256-wide tiles with the output columns produced in slices
inline bool mfma_head_dim(int d) {
    return d == 64 || d == 80 || d == 88 || d == 96 || d == 128 || d == 160 || d == 256;
}
// head dims of the fp32 matrix-core kernels (columns padded to a multiple
// of 32 with zeros)
inline bool f32_mfma_head_dim(int d) { return d > 0 && d <= 128 && d % 4 == 0; }
// grid x of the fp32 matrix-core kernels: 128-row tiles over every sequence
inline int64_t f32_row_tiles(int64_t total_rows, int num_seqs) { return total_rows / 128 + num_seqs + 1; }
inline int64_t f32_fwd_part_floats(int splits, int64_t total_q, int hq, int d) {
    return splits > 1 ? (int64_t)splits * total_q * hq * (d + 1) : 0;
}
inline int64_t f32_dq_part_floats(int splits, int64_t total_q, int hq, int d) {
    return splits > 1 ? (int64_t)splits * total_q * hq * d : 0;
}
inline int64_t f32_dkv_part_floats(int splits, int64_t total_kv, int hkv, int d) {
    return splits > 1 ? (int64_t)splits * 2 * total_kv * hkv * d : 0;
}
// head dims of the split-KV decode kernels
inline bool decode_head_dim(int d) { return d == 64 || d == 128; }

}  // namespace mtlattn
