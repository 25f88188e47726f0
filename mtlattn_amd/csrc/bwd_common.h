// Kernel parameters and small helpers shared by the 16-bit backward kernels
// (bwd.hip, bwd_wide.hip).
#pragma once

#include "common.h"
#include "kernels.h"

namespace mtlattn {
namespace {

struct BwdKParams {
    const uint16_t* q; const uint16_t* k; const uint16_t* v; const uint16_t* dout;
    const float* lse; const float* delta;
    void* dq; void* dk; void* dv;
    int64_t dq_rs, dkv_rs;             // their row strides
    const int* cu_q; const int* cu_kv;
    const float* bias;
    int64_t q_rs, k_rs, v_rs, do_rs;
    int64_t bias_qs, bias_hs, bias_cols, bias_ss, bias_rows;
    int64_t total_q, total_kv;
    int num_seqs, hq, hkv, g, hpw, n_tiles, n_hg;
    float scale, scale_log2;
    int causal, window;
    int seq_group;    // one-wave-per-SIMD dK/dV: sequences dispatched together
    int bias_v4;      // bias rows 16-byte aligned (pointer and strides)
    int bias_b32;     // 64 bias rows plus a row's columns span < 2^32 bytes (32-bit buffer offsets)
    const uint16_t* o; int64_t o_rs;   // forward output (dQ with delta_w)
    float* delta_w;   // non-null: the dQ kernel computes delta and writes it here
    // SPLIT dK/dV kernels: fp32 partials of up to max_pieces pieces of a key
    // block's stages, and the piece length the grid of `split_grid` workgroups
    // works with (written for the pass that adds the partials)
    float* part; int* piece_out; int max_pieces, split_grid;
};

// The query rows that a dK/dV workgroup visits: tiles of qtl rows from q_lo
// (on a grid aligned to qtl, so that workgroups of a sequence share tiles)
// that can see any of the keys k0 .. k0 + kb - 1.
struct QWalk {
    int q_lo, n_tiles;
};
__device__ inline QWalk query_walk(int k0, int kb, int coff, int q_len, int kv_len, int causal, int window, int qtl) {
    const int k_last = min(kv_len, k0 + kb) - 1;
    const int q_lo = causal ? max(0, k0 - coff) / qtl * qtl : 0;
    const int q_hi = window > 0 ? min(q_len, k_last - coff + window) : q_len;
    return QWalk{q_lo, q_hi > q_lo ? (q_hi - q_lo + qtl - 1) / qtl : 0};
}

// Offset of dK's (which = 0) or dV's (1) partial rows of piece z.
__device__ inline int64_t part_offset(int z, int which, int64_t total_kv, int64_t row) {
    return (2 * (int64_t)z + which) * total_kv * row;
}

// The piece of workgroup `id` of a split dK/dV launch (find_piece): pieces of
// the query stages of key tile t (KB keys) of kv head `group`. Pieces start at
// the same distances from the top of the walk in every block, so workgroups
// that run together read the same query tiles.
constexpr int kDkvMinPiece = 8;
template <int KB, int QTL>
__device__ inline bool dkv_piece(const BwdKParams& p, int id, SplitPiece& out) {
    auto stages = [&](int t) {
        const int s = find_seq_for_tile(p.cu_kv, p.num_seqs, KB, t, p.total_kv);
        const SeqRange qr = seq_range(p.cu_q, s, p.total_q), kr = seq_range(p.cu_kv, s, p.total_kv);
        const int q_len = qr.end - qr.start, kv_len = kr.end - kr.start;
        const int blk = t - tile_base(p.cu_kv, s, KB, p.total_kv);
        if (blk < 0 || blk * KB >= kv_len) return -1;
        return query_walk(blk * KB, KB, kv_len - q_len, q_len, kv_len, p.causal, p.window, QTL).n_tiles * p.g;
    };
    return find_piece(stages, p.n_tiles, p.hkv, p.split_grid, kDkvMinPiece, p.max_pieces, p.piece_out, id, out);
}

// Sum of the 8 products of one 16-byte chunk of O and dO. The preprocess and
// the dQ kernel's fused delta both use it and combine chunks in the same tree,
// so the two give bitwise equal deltas.
template <typename T>
__device__ inline float dot8(const u32x4_t a, const u32x4_t b) {
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc += lo16<T>(a[e]) * lo16<T>(b[e]) + hi16<T>(a[e]) * hi16<T>(b[e]);
    return acc;
}

template <typename T, bool OUT_F32>
__device__ inline void store4(void* base, int64_t off, float a, float b, float c, float d) {
    if (OUT_F32) {
        *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(base) + off) = f32x4_t{a, b, c, d};
    } else {
        st8(reinterpret_cast<uint16_t*>(base) + off, u32x2_t{T::pack2(a, b), T::pack2(c, d)});
    }
}

// Staged lse / delta columns as the dK/dV products use them: lse (which = 0)
// becomes -lse log2(e), with rows of no allowed key (lse = -inf) giving -inf
// so that every P of theirs is exp2(-inf) = 0; delta (which = 1) becomes -delta.
// First query tile (its first row) of a dK/dV workgroup's walk over the
// n tiles q_lo, q_lo + qtl, ... of its query range. The walk descends from
// there and, reaching q_lo, wraps to the top tile. Without a window it starts
// at the top tile: every workgroup of a sequence then reads the same (tile,
// head) at the same time from the top, and the L2 serves the repeats. Under
// a sliding window the ranges of neighbouring key blocks are shifted copies
// of equal length, so the walk starts at the tile whose index is a multiple
// of n: each tile X then comes at step (start - X) mod n in every workgroup
// whose range holds it, and co-resident workgroups again read it together.
__device__ inline int first_q_tile(int q_lo, int n, int qtl, bool cyclic) {
    if (!cyclic || n <= 0) return q_lo + (n - 1) * qtl;
    const int lo_t = q_lo / qtl;
    return q_lo + (n - lo_t % n) % n * qtl;
}

__device__ inline float neg_lse2(float v) { return v == kNegInf ? kNegInf : -v * kLog2e; }
__device__ inline void neg_col(float* x, int which) {
    const float v = *x;
    *x = which ? -v : neg_lse2(v);
}

// Whether a dK/dV launch with n_tiles key tiles takes the problem's split plan
// (made for the kernel that usually runs it: another one may have more tiles)
inline bool use_split(const BwdArgs& a, int64_t n_tiles) {
    return a.dkv_plan.pieces > 1 && a.dkv_part != nullptr && n_tiles <= 64 * kSplitChunks &&
           n_tiles * a.geo.hkv <= a.dkv_plan.grid;
}

BwdKParams make_params(const BwdArgs& a) {
    const Geometry& g = a.geo;
    BwdKParams p;
    p.q = (const uint16_t*)a.q; p.k = (const uint16_t*)a.k; p.v = (const uint16_t*)a.v;
    p.dout = (const uint16_t*)a.dout;
    p.lse = a.lse; p.delta = a.delta;
    p.dq = a.dq; p.dk = a.dk; p.dv = a.dv;
    p.dq_rs = a.dq_rs > 0 ? a.dq_rs : (int64_t)g.hq * g.d;
    p.dkv_rs = a.dkv_rs > 0 ? a.dkv_rs : (int64_t)g.hkv * g.d;
    p.cu_q = g.cu_q; p.cu_kv = g.cu_kv; p.bias = g.bias;
    p.q_rs = a.q_rs; p.k_rs = a.k_rs; p.v_rs = a.v_rs; p.do_rs = a.do_rs;
    p.bias_qs = g.bias_qs; p.bias_hs = g.bias_hs; p.bias_cols = g.bias_cols;
    p.bias_ss = g.bias_ss; p.bias_rows = g.bias_rows;
    p.total_q = g.total_q; p.total_kv = g.total_kv;
    p.num_seqs = g.num_seqs; p.hq = g.hq; p.hkv = g.hkv; p.g = g.g;
    p.hpw = 1;
    p.n_tiles = 0; p.n_hg = 0; p.seq_group = g.num_seqs;
    p.scale = g.scale; p.scale_log2 = g.scale * kLog2e;
    p.causal = g.causal; p.window = g.window > 0 ? g.window : 0;
    p.bias_b32 = g.bias != nullptr && (64 * g.bias_qs + g.bias_cols) * 4 < ((int64_t)1 << 32);
    p.bias_v4 = g.bias != nullptr && ((uintptr_t)g.bias % 16 == 0) && g.bias_qs % 4 == 0 && g.bias_hs % 4 == 0 &&
                (g.bias_ss < 0 || g.bias_ss % 4 == 0);
    p.o = (const uint16_t*)a.o; p.o_rs = a.o_rs;
    p.delta_w = a.delta_out;
    p.part = a.dkv_part; p.piece_out = nullptr; p.max_pieces = a.dkv_plan.pieces; p.split_grid = a.dkv_plan.grid;
    if (a.dkv_part != nullptr)
        p.piece_out = (int*)(a.dkv_part + dkv_part_floats(a.dkv_plan.pieces, g.total_kv, g.hkv, g.d) - kDkvPartTail);
    return p;
}

}  // namespace
}  // namespace mtlattn
