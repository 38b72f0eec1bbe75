// merkle.hip -- BLAKE3 column leaves and the binary Merkle tree over them,
// the commitment that closes the reference's Ligero commit
// (rust/volta-pcs/src/ligero.rs:595-621, rust/volta-pcs/src/merkle.rs:9-51).
//
// Leaf j is blake3 (the blake3 1.8.5 crate's unkeyed hash) of column j of the
// row-major matrix, read as little-endian u64 words row by row; an Fp2
// element contributes c0 then c1.  Inner nodes are blake3(left || right).
// The tree buffer holds 2 cols - 1 hashes level by level, root last.
//
// BLAKE3 cuts a column's byte stream into 1024-byte chunks (128 Fp rows or 64
// Fp2 rows) and joins chunk chaining values in a binary tree whose left
// subtrees are complete power-of-two blocks.  Any aligned power-of-two run of
// chunks is therefore an exact subtree, and a short run at the end is the
// left-complete subtree over what remains; the GPU builds the tree in such
// runs, bottom up:
//   column_groups: one thread per (column, run of up to 4 chunks).  A wave's
//     lanes are 64 consecutive columns, so every row read is one coalesced
//     512-byte (Fp) or 1 KiB (Fp2) segment.  The thread hashes its chunks in
//     order, loading the next block while it compresses the current one, and
//     joins them with two registers of pending values (no LDS, so occupancy
//     is set by registers alone).
//   merge_pass: one thread per (column, run of 16 values) folds them with an
//     eager join stack in LDS, repeated until one value per column is left;
//     the column's last join carries the ROOT flag.
//   merkle_subtrees: the pair hashes of the Merkle tree, up to ten levels of a
//     subtree per workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>

#include "context.hpp"
#include "gl64_shift.hpp"
#include "kernels.hpp"

namespace vmx {

namespace b3 {

constexpr uint32_t CHUNK_START = 1, CHUNK_END = 2, PARENT = 4, ROOT = 8;
constexpr std::array<uint32_t, 8> IV = {0x6A09E667u, 0xBB67AE85u, 0x3C6EF372u, 0xA54FF53Au,
                                        0x510E527Fu, 0x9B05688Cu, 0x1F83D9ABu, 0x5BE0CD19u};

// Message word order of each of the 7 rounds: round r + 1 reads word
// SCHED[r][PERM[i]] at position i (the specification's fixed permutation).
constexpr std::array<std::array<uint8_t, 16>, 7> make_schedule() {
    constexpr uint8_t perm[16] = {2, 6, 3, 10, 7, 0, 4, 13, 1, 11, 12, 5, 9, 14, 15, 8};
    std::array<std::array<uint8_t, 16>, 7> s{};
    for (int i = 0; i < 16; ++i) s[0][i] = static_cast<uint8_t>(i);
    for (int r = 1; r < 7; ++r)
        for (int i = 0; i < 16; ++i) s[r][i] = s[r - 1][perm[i]];
    return s;
}
constexpr auto SCHED = make_schedule();

__device__ __forceinline__ uint32_t rotr(uint32_t x, int n) { return (x >> n) | (x << (32 - n)); }

__device__ __forceinline__ void g(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d, uint32_t x, uint32_t y) {
    a = a + b + x;
    d = rotr(d ^ a, 16);
    c = c + d;
    b = rotr(b ^ c, 12);
    a = a + b + y;
    d = rotr(d ^ a, 8);
    c = c + d;
    b = rotr(b ^ c, 7);
}

// cv[s] <- the chaining value of compress(cv[s], m[s], counter, block_len,
// flags) for S independent states, their G functions interleaved so one
// lane keeps several dependency chains in flight.
template <int S>
__device__ __forceinline__ void compress_n(uint32_t (*cv)[8], const uint32_t (*m)[16], uint64_t counter,
                                           uint32_t block_len, uint32_t flags) {
    uint32_t v[S][16];
#pragma unroll
    for (int q = 0; q < S; ++q) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[q][i] = cv[q][i];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[q][8 + i] = IV[i];
        v[q][12] = static_cast<uint32_t>(counter);
        v[q][13] = static_cast<uint32_t>(counter >> 32);
        v[q][14] = block_len;
        v[q][15] = flags;
    }
    gl::static_for<0, 7>([&](auto rr) {
        constexpr auto s = SCHED[decltype(rr)::value];
#pragma unroll
        for (int q = 0; q < S; ++q) {
            g(v[q][0], v[q][4], v[q][8], v[q][12], m[q][s[0]], m[q][s[1]]);
            g(v[q][1], v[q][5], v[q][9], v[q][13], m[q][s[2]], m[q][s[3]]);
            g(v[q][2], v[q][6], v[q][10], v[q][14], m[q][s[4]], m[q][s[5]]);
            g(v[q][3], v[q][7], v[q][11], v[q][15], m[q][s[6]], m[q][s[7]]);
        }
#pragma unroll
        for (int q = 0; q < S; ++q) {
            g(v[q][0], v[q][5], v[q][10], v[q][15], m[q][s[8]], m[q][s[9]]);
            g(v[q][1], v[q][6], v[q][11], v[q][12], m[q][s[10]], m[q][s[11]]);
            g(v[q][2], v[q][7], v[q][8], v[q][13], m[q][s[12]], m[q][s[13]]);
            g(v[q][3], v[q][4], v[q][9], v[q][14], m[q][s[14]], m[q][s[15]]);
        }
    });
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < 8; ++i) cv[q][i] = v[q][i] ^ v[q][i + 8];
}

__device__ __forceinline__ void compress(uint32_t* cv, const uint32_t* m, uint64_t counter, uint32_t block_len,
                                         uint32_t flags) {
    compress_n<1>(reinterpret_cast<uint32_t(*)[8]>(cv), reinterpret_cast<const uint32_t(*)[16]>(m), counter,
                  block_len, flags);
}

// out[s] <- compress(IV, l[s] || r[s], 0, 64, flags) for S pairs: BLAKE3
// parent nodes (flags PARENT [| ROOT]) or, with CHUNK_START | CHUNK_END |
// ROOT, the hash of the 64 bytes l || r as a message (the Merkle pair hash).
template <int S>
__device__ __forceinline__ void join_n(uint32_t (*out)[8], const uint32_t (*l)[8], const uint32_t (*r)[8],
                                       uint32_t flags) {
    uint32_t m[S][16], cv[S][8];
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            m[q][i] = l[q][i];
            m[q][8 + i] = r[q][i];
            cv[q][i] = IV[i];
        }
    compress_n<S>(cv, m, 0, 64, flags);
#pragma unroll
    for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < 8; ++i) out[q][i] = cv[q][i];
}

__device__ __forceinline__ void join(uint32_t* out, const uint32_t* l, const uint32_t* r, uint32_t flags) {
    join_n<1>(reinterpret_cast<uint32_t(*)[8]>(out), reinterpret_cast<const uint32_t(*)[8]>(l),
              reinterpret_cast<const uint32_t(*)[8]>(r), flags);
}

__device__ __forceinline__ void store_hash(uint32_t* dst, const uint32_t* h) {
    using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
    reinterpret_cast<u32x4*>(dst)[0] = u32x4{h[0], h[1], h[2], h[3]};
    reinterpret_cast<u32x4*>(dst)[1] = u32x4{h[4], h[5], h[6], h[7]};
}

__device__ __forceinline__ void load_hash(uint32_t* h, const uint32_t* src) {
    using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
    const u32x4 a = reinterpret_cast<const u32x4*>(src)[0], b = reinterpret_cast<const u32x4*>(src)[1];
    h[0] = a.x, h[1] = a.y, h[2] = a.z, h[3] = a.w, h[4] = b.x, h[5] = b.y, h[6] = b.z, h[7] = b.w;
}

constexpr int LANES = 64;          // columns per column_groups workgroup (one wave)
constexpr size_t CHUNK_WORDS = 128; // u64 words per 1024-byte chunk

// W = u64 words per matrix element: 1 for Fp, 2 for Fp2.  Thread (column,
// g) hashes the chunks [g G, min(g G + G, chunks)) of its column, G <= 4, and
// joins them left-complete with two registers of pending values: chunks 0+1
// and 2+3 pair up, then the pairs; a short last group of 3 joins (0+1)+2.
// Writes the group's chaining value to out[(g cols + col) 8 ..], or with
// root set (one group per column) the column's leaf hash to out[col 8 ..].
// OFF32: the rows of a block span less than 4 GiB, so a lane's element is
// addressed as the block's uniform pointer plus a 32-bit byte offset.
template <int W, bool OFF32>
__global__ __launch_bounds__(LANES, 6) void column_groups(const uint64_t* __restrict__ m, size_t rows, size_t cols,
                                                       size_t chunks, size_t group, int root,
                                                       uint32_t* __restrict__ out) {
    const int lane = threadIdx.x;
    const size_t col = static_cast<size_t>(blockIdx.x) * LANES + lane;
    if (col >= cols) return;
    const size_t gi = blockIdx.y;
    const size_t c_begin = gi * group;
    const size_t c_end = min(chunks, c_begin + group);
    const size_t n_local = c_end - c_begin;  // 1..4
    const size_t words = rows * W;            // the column's u64 word stream
    const size_t row_stride = cols * W;
    const uint32_t lane_bytes = static_cast<uint32_t>(col * W * sizeof(uint64_t));  // used when OFF32
    // blocks of the group in stream order: only the column's last chunk can
    // be short, and it comes last, so block k starts at word (c_begin 16 + k) 8
    const size_t last_words = words - (c_end - 1) * CHUNK_WORDS;
    const size_t total = (n_local - 1) * 16 + (min(CHUNK_WORDS, last_words) + 7) / 8;

    // Blocks load in stream order, RB rows each.  OFF32: a buffer resource at
    // the block's first row, the lane's column as the 32-bit offset and the
    // row's distance as a scalar one, so a block costs no vector address
    // arithmetic and its addresses eight scalars (as 64-bit row pointers they
    // spilled scalars into vector lanes, 133 moves per pair of blocks; 1,531
    // rows x 4,096 columns 51 -> 49 us, the largest within 0.5%: the
    // compressions themselves bound those).
    constexpr int RB = 8 / W;
    const size_t row0 = c_begin * CHUNK_WORDS / W;
    const uint64_t* blk = m + row0 * row_stride;
    auto load_block = [&](size_t k, uint32_t* mw) {
        const size_t w0 = (c_begin * 16 + k) * 8;
        if (w0 + 8 <= words) {
            if constexpr (OFF32) {
                const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<uint64_t*>(blk), static_cast<short>(0), -1, 0x00020000);
                const uint32_t stride = static_cast<uint32_t>(row_stride * sizeof(uint64_t));
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    if constexpr (W == 1) {
                        const auto x = __builtin_amdgcn_raw_buffer_load_b64(r, lane_bytes, i * stride, 0);
                        mw[2 * i] = x[0], mw[2 * i + 1] = x[1];
                    } else {  // one 16-byte (c0, c1) load per row
                        const auto x = __builtin_amdgcn_raw_buffer_load_b128(r, lane_bytes, i * stride, 0);
                        mw[4 * i] = x[0], mw[4 * i + 1] = x[1], mw[4 * i + 2] = x[2], mw[4 * i + 3] = x[3];
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint64_t x = blk[(i / W) * row_stride + col * W + i % W];
                    mw[2 * i] = static_cast<uint32_t>(x);
                    mw[2 * i + 1] = static_cast<uint32_t>(x >> 32);
                }
            }
        } else {  // the column's last, partial block: zero past the end
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint64_t x = w0 + i < words ? blk[(i / W) * row_stride + col * W + i % W] : 0;
                mw[2 * i] = static_cast<uint32_t>(x);
                mw[2 * i + 1] = static_cast<uint32_t>(x >> 32);
            }
        }
        blk += RB * row_stride;
    };

    const uint32_t top = root ? PARENT | ROOT : PARENT;  // flags of the group's last join
    uint32_t cv[8], p0[8], p1[8];
    auto compress_block = [&](const uint32_t* mw, size_t k, int cb, int nb) {
        const size_t left = words - (c_begin * 16 + k) * 8;
        const uint32_t len = static_cast<uint32_t>(min<size_t>(8, left) * 8);
        uint32_t flags = (cb == 0 ? CHUNK_START : 0u) | (cb + 1 == nb ? CHUNK_END : 0u);
        if (chunks == 1 && cb + 1 == nb) flags |= ROOT;  // a one-chunk column: this block is the root
        compress(cv, mw, c_begin + k / 16, len, flags);
    };

    // Two block buffers alternate: the next block loads while the current one
    // compresses.  A full chunk has 16 blocks, so the next chunk's first block
    // always lands in `a`; only the column's last chunk can be shorter.
    uint32_t a[16], b[16];
    load_block(0, a);
    for (size_t lc = 0; lc < n_local; ++lc) {
        const size_t k0 = lc * 16;
        const int nb = static_cast<int>(min<size_t>(16, total - k0));
#pragma unroll
        for (int i = 0; i < 8; ++i) cv[i] = IV[i];
        for (int cb = 0; cb < nb; cb += 2) {
            if (k0 + cb + 1 < total) load_block(k0 + cb + 1, b);
            compress_block(a, k0 + cb, cb, nb);
            if (cb + 1 == nb) break;
            if (k0 + cb + 2 < total) load_block(k0 + cb + 2, a);
            compress_block(b, k0 + cb + 1, cb + 1, nb);
        }
        // chunk lc done: chunks 0 and 2 wait in p0 / p1, chunks 1 and 3 join them
        if ((lc & 1) == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) (lc == 0 ? p0 : p1)[i] = cv[i];
        } else {
            uint32_t l[8], j[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) l[i] = lc == 1 ? p0[i] : p1[i];
            join(j, l, cv, lc == 1 && n_local == 2 ? top : PARENT);
#pragma unroll
            for (int i = 0; i < 8; ++i) (lc == 1 ? p0 : p1)[i] = j[i];
        }
    }
    if (chunks == 1) {  // the single block chain already carried ROOT
        store_hash(out + col * 8, cv);
        return;
    }
    if (n_local >= 3) join(p0, p0, p1, top);  // (0+1) + 2  or  (0+1) + (2+3)
    store_hash(out + (root ? col : gi * cols + col) * 8, p0);
}

constexpr int FAN_IN = 16;      // values one merge_pass thread folds
constexpr int MERGE_DEPTH = 5;  // pending values of a left-complete fold of 16

// Thread (column, j) folds values [16 j, min(16 j + 16, k_in)) of its column
// (in[(i cols + col) 8 ..]) left-complete, joining complete power-of-two runs
// eagerly on a per-lane LDS stack; with final set this is the column's last
// fold and its top join carries ROOT.  k_in >= 2.
__global__ __launch_bounds__(LANES) void merge_pass(const uint32_t* __restrict__ in, size_t k_in, size_t cols,
                                                    int final, uint32_t* __restrict__ out) {
    __shared__ uint32_t stack[MERGE_DEPTH][8][LANES];
    const int lane = threadIdx.x;
    const size_t col = static_cast<size_t>(blockIdx.x) * LANES + lane;
    if (col >= cols) return;
    const size_t j = blockIdx.y;
    const size_t i0 = j * FAN_IN;
    const size_t n = min<size_t>(FAN_IN, k_in - i0);
    auto push = [&](int d, const uint32_t* h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) stack[d][i][lane] = h[i];
    };
    auto peek = [&](int d, uint32_t* h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = stack[d][i][lane];
    };
    int depth = 0;
    for (size_t t = 1; t <= n; ++t) {
        uint32_t h[8];
        load_hash(h, in + ((i0 + t - 1) * cols + col) * 8);
        push(depth++, h);
        if (t == n) break;  // the last value is joined in the fold below
        for (size_t u = t; (u & 1) == 0; u >>= 1) {
            uint32_t l[8], r[8], p[8];
            peek(depth - 1, r);
            peek(depth - 2, l);
            join(p, l, r, PARENT);
            depth -= 2;
            push(depth++, p);
        }
    }
    uint32_t acc[8];
    peek(--depth, acc);
    while (depth > 0) {
        uint32_t l[8];
        peek(--depth, l);
        join(acc, l, acc, PARENT | (depth == 0 && final ? ROOT : 0u));
    }
    store_hash(out + (final ? col : j * cols + col) * 8, acc);
}

constexpr int MERGE_THREADS = 256;
constexpr int MERGE_MAX = 2 * MERGE_THREADS;  // values per column merge_final handles

// The column's last fold when it has k_in <= 512 values (in[(i cols + col) 8
// ..]): the workgroup holds cpw = 256 / tpc columns (tpc = ceil(k_in / 2)
// rounded up to a power of two) and joins each column's values level by
// level in LDS, carrying an odd last value up unchanged (which builds the
// same left-complete tree); the last join carries ROOT.  Each level is one
// join deep.
__global__ __launch_bounds__(MERGE_THREADS) void merge_final(const uint32_t* __restrict__ in, int k_in, size_t cols,
                                                             int cpw, uint32_t* __restrict__ leaves) {
    __shared__ uint32_t node[MERGE_MAX][9];  // odd pitch: a join reads two neighbouring nodes
    const int t = threadIdx.x;
    const int per = MERGE_MAX / cpw;          // node slots per column
    const int tpc = MERGE_THREADS / cpw;      // threads per column
    // columns interleave across threads: a level's active threads (r < pairs)
    // are the first pairs * cpw, packed into as few waves as possible
    const int q = t % cpw, r = t / cpw;       // column within the workgroup, thread within the column
    const size_t col = static_cast<size_t>(blockIdx.x) * cpw + q;
    const bool live = q < cpw && col < cols;
    uint32_t(*mine)[9] = node + q * per;
    if (live)
        for (int i = r; i < k_in; i += tpc) {
            uint32_t h[8];
            load_hash(h, in + (static_cast<size_t>(i) * cols + col) * 8);
#pragma unroll
            for (int w = 0; w < 8; ++w) mine[i][w] = h[w];
        }
    __syncthreads();
    for (int count = k_in; count > 1;) {
        const int pairs = count / 2;
        uint32_t p[8];
        const bool act = live && r < pairs;
        if (act) {
            uint32_t l[8], rr[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) {
                l[w] = mine[2 * r][w];
                rr[w] = mine[2 * r + 1][w];
            }
            join(p, l, rr, PARENT | (count == 2 ? ROOT : 0u));
        }
        __syncthreads();
        if (act)
#pragma unroll
            for (int w = 0; w < 8; ++w) mine[r][w] = p[w];
        if (live && (count & 1) && r == pairs)  // carry the odd last value up unchanged
#pragma unroll
            for (int w = 0; w < 8; ++w) mine[pairs][w] = mine[count - 1][w];
        __syncthreads();
        count = pairs + (count & 1);
    }
    if (live && r == 0) {
        uint32_t h[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) h[w] = mine[0][w];
        store_hash(leaves + col * 8, h);
    }
}

constexpr uint32_t PAIR_FLAGS = CHUNK_START | CHUNK_END | ROOT;  // blake3 of a 64-byte message

// One compression split over a quad of lanes: lane i holds column i of the
// 4 x 4 state, the diagonal half-rounds rotate rows 1..3 across the quad (DPP),
// and the lane's 28 message words come from LDS at byte offsets that depend on
// i only.  A join is then about 270 instructions deep instead of 690, at 1.5
// times the total work: for the upper tree levels, whose few joins leave the
// machine idle and whose depth is the time.
struct Quad {
    uint32_t off[7][4];      // byte offsets of the lane's words: two per half-round
    uint32_t iva, ivb, len;  // IV[i], IV[4 + i] and the block length of state word 14
    bool flag_lane;          // lane 3 holds the flags (state word 15)
};

__device__ __forceinline__ Quad make_quad(uint32_t i) {
    Quad q;
    gl::static_for<0, 28>([&](auto z_) {
        constexpr int r = decltype(z_)::value / 4, j = decltype(z_)::value % 4, pos = j < 2 ? j : 6 + j;
        constexpr uint32_t c = (4u * SCHED[r][pos]) | (4u * SCHED[r][pos + 2]) << 8 | (4u * SCHED[r][pos + 4]) << 16 |
                               (4u * SCHED[r][pos + 6]) << 24;
        q.off[r][j] = (c >> (8 * i)) & 255u;
    });
    q.iva = i == 0 ? IV[0] : i == 1 ? IV[1] : i == 2 ? IV[2] : IV[3];
    q.ivb = i == 0 ? IV[4] : i == 1 ? IV[5] : i == 2 ? IV[6] : IV[7];
    q.len = i == 2 ? 64u : 0u;
    q.flag_lane = i == 3;
    return q;
}

template <int CTRL>
__device__ __forceinline__ uint32_t quad_perm(uint32_t x) {
    return static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(x), CTRL, 0xF, 0xF, true));
}

// Words i and 4 + i of compress(IV, the 16 words at msg, 0, 64, flags), for
// lane i of a quad whose four lanes are active and share msg (LDS).
__device__ __forceinline__ void quad_join(const Quad& q, const uint32_t* msg, uint32_t flags, uint32_t* lo,
                                          uint32_t* hi) {
    uint32_t w[7][4];
    gl::static_for<0, 28>([&](auto z_) {
        constexpr int r = decltype(z_)::value / 4, j = decltype(z_)::value % 4;
        w[r][j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(msg) + q.off[r][j]);
    });
    uint32_t a = q.iva, b = q.ivb, c = q.iva, d = q.flag_lane ? flags : q.len;
    constexpr int NEXT = 0x39, OPPOSITE = 0x4E, PREV = 0x93;  // lane i reads lane i + 1, i + 2, i + 3 (mod 4)
    gl::static_for<0, 7>([&](auto r_) {
        constexpr int r = decltype(r_)::value;
        g(a, b, c, d, w[r][0], w[r][1]);
        b = quad_perm<NEXT>(b);
        c = quad_perm<OPPOSITE>(c);
        d = quad_perm<PREV>(d);
        g(a, b, c, d, w[r][2], w[r][3]);
        b = quad_perm<PREV>(b);
        c = quad_perm<OPPOSITE>(c);
        d = quad_perm<NEXT>(d);
    });
    *lo = a ^ c;
    *hi = b ^ d;
}

constexpr int TREE_THREADS = 512;
constexpr int TREE_QUADS = TREE_THREADS / 4;
constexpr size_t TREE_MAX = 1024;  // nodes one workgroup takes at most
constexpr size_t TREE_SPAN = 256;  // nodes per workgroup while the level has more than TREE_MAX
constexpr int MSG_PITCH = 17;      // words per pair of children: 16 and a pad against bank conflicts

// Workgroup b builds the subtree over nodes [b span, (b + 1) span) of a level
// (len nodes at tree + off 8; span a power of two, 2 <= span <= TREE_MAX,
// dividing len) up to its root, staging levels through two LDS buffers and
// writing each to its place in the tree.  A level of more than TREE_QUADS
// joins takes one lane per join, the others a quad of lanes.  Column hash and
// tree of 24 rows x 256 columns 19.7 -> 14.5 us, 7 x 131,072 48 -> 28 us, against
// one launch per level down to 1,024 nodes and one lane per join throughout.
__global__ __launch_bounds__(TREE_THREADS) void merkle_subtrees(uint32_t* __restrict__ tree, size_t off, size_t len,
                                                               int span) {
    __shared__ uint32_t even[TREE_MAX / 2 * MSG_PITCH], odd[TREE_MAX / 4 * MSG_PITCH];
    const int t = threadIdx.x;
    const uint32_t i = t & 3;
    size_t base = static_cast<size_t>(blockIdx.x) * span;
    // node n sits in pair n / 2, half n & 1
    for (int n = t; n < span; n += TREE_THREADS) {
        uint32_t h[8];
        load_hash(h, tree + (off + base + n) * 8);
        uint32_t* dst = even + (n >> 1) * MSG_PITCH + 8 * (n & 1);
#pragma unroll
        for (int k = 0; k < 8; ++k) dst[k] = h[k];
    }
    const Quad quad = make_quad(i);
    uint32_t *cur = even, *up = odd;
    __syncthreads();
    for (int parents = span / 2; parents > 0; parents /= 2) {
        off += len;
        len /= 2;
        base /= 2;
        if (parents > TREE_QUADS) {
            if (t < parents) {
                uint32_t m[16], cv[8];
#pragma unroll
                for (int k = 0; k < 16; ++k) m[k] = cur[t * MSG_PITCH + k];
#pragma unroll
                for (int k = 0; k < 8; ++k) cv[k] = IV[k];
                compress(cv, m, 0, 64, PAIR_FLAGS);
                store_hash(tree + (off + base + t) * 8, cv);
                uint32_t* dst = up + (t >> 1) * MSG_PITCH + 8 * (t & 1);
#pragma unroll
                for (int k = 0; k < 8; ++k) dst[k] = cv[k];
            }
        } else {
            const int n = t >> 2;
            if (n < parents) {
                uint32_t lo, hi;
                quad_join(quad, cur + n * MSG_PITCH, PAIR_FLAGS, &lo, &hi);
                uint32_t* dst = up + (n >> 1) * MSG_PITCH + 8 * (n & 1) + i;
                dst[0] = lo;
                dst[4] = hi;
                uint32_t* node = tree + (off + base + n) * 8 + i;
                node[0] = lo;
                node[4] = hi;
            }
        }
        __syncthreads();
        uint32_t* const s = cur;
        cur = up;
        up = s;
    }
}

// paths[(q bits + l) 8 ..] = the level-l sibling of leaf idx[q]; zero for an
// index outside [0, leaves).
__global__ __launch_bounds__(256) void merkle_paths_kernel(const uint32_t* __restrict__ tree,
                                                           const uint32_t* __restrict__ idx,
                                                           uint32_t* __restrict__ paths, size_t leaves,
                                                           size_t queries, int bits) {
    const size_t z = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (z >= queries * bits) return;
    const size_t q = z / bits;
    const int level = static_cast<int>(z - q * bits);
    size_t i = idx[q];
    uint32_t h[8] = {};
    if (i < leaves) {
        size_t off = 0, len = leaves;
        for (int l = 0; l < level; ++l) {
            off += len;
            len >>= 1;
            i >>= 1;
        }
        load_hash(h, tree + (off + (i ^ 1)) * 8);
    }
    store_hash(paths + z * 8, h);
}

}  // namespace b3


// Chunks per column_groups thread: the most (4, 2 or 1) that still gives every
// SIMD its 6 waves, since longer runs leave fewer chaining values to store and
// join; below that the time is the run's own length and short runs win.  The
// whole tree with 4 / 2 / 1 chunks per thread, microseconds: 1,531 rows x 4,096
// columns 129 / 82 / 61; 3,000 x 8,192 136 / 125 / 109; 8,192 x 8,192 222 / 217 /
// 215; 8,192 x 16,384 385 / 380 / 380; above the line 2,080 x 131,072 705 / 716 /
// 751; 24,576 x 32,768 1,967 / 2,004 / 2,116; 65,536 x 8,192 1,331 / 1,351 / 1,410.
static size_t chunks_per_thread(const Context* c, size_t cols, size_t chunks) {
    const size_t cus = c->cu_count > 0 ? static_cast<size_t>(c->cu_count) : 256;
    const size_t full = cus * 4 * 6, waves = (cols + b3::LANES - 1) / b3::LANES;
    for (size_t g : {size_t{4}, size_t{2}}) {
        // half as long runs would exceed the launch grid's second dimension
        const bool limit = (chunks + g / 2 - 1) / (g / 2) > 65535;
        if (limit || waves * ((chunks + g - 1) / g) >= full) return std::min(g, chunks);
    }
    return 1;
}

int merkle_column_leaves(Context* c, const uint64_t* m, size_t rows, size_t cols, bool fp2, uint32_t* leaves) {
    const size_t w = fp2 ? 2 : 1;
    const size_t words = rows * w;
    const size_t chunks = (words + b3::CHUNK_WORDS - 1) / b3::CHUNK_WORDS;
    if (chunks > 4 * size_t{65535}) return fail_msg(c, "Merkle column too long (more than 2^18 BLAKE3 chunks)");
    // Workspace of runs of `g` chunks: column_groups' values, then each non-final merge
    // pass's (16x fewer).
    auto ws_bytes = [&](size_t g, size_t* bytes) {
        size_t slots = 0;
        for (size_t kk = (chunks + g - 1) / g; kk > 1; kk = (kk + b3::FAN_IN - 1) / b3::FAN_IN) slots += kk;
        return mul_ok(slots, cols * 32, bytes);
    };
    size_t group = chunks_per_thread(c, cols, chunks), bytes = 0;
    // Short runs leave more values: where the workspace for them is not to be had, as
    // inside a coarse timing scope, the longest runs do, which need the least (none up
    // to four chunks).
    if (!ws_bytes(group, &bytes) || !try_ws(c, WS_HASH, bytes)) {
        group = std::min<size_t>(4, chunks);
        if (!ws_bytes(group, &bytes)) return fail_msg(c, "Merkle workspace overflows size_t");
    }
    size_t k = (chunks + group - 1) / group;  // values per column after column_groups
    if (bytes && ensure_ws(c, WS_HASH, bytes)) return -1;
    uint32_t* buf = bytes ? ws<uint32_t>(c, WS_HASH) : nullptr;
    const dim3 grid(static_cast<unsigned>((cols + b3::LANES - 1) / b3::LANES), static_cast<unsigned>(k));
    const int is_root = k == 1 ? 1 : 0;
    uint32_t* gout = k == 1 ? leaves : buf;
    const bool off32 = cols <= 0xFFFFFFFFull / 64;  // a block is 64 bytes of every column
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(b3::LANES), 0, c->stream, m, rows, cols, chunks, group, is_root, gout);
    };
    if (fp2) off32 ? launch(b3::column_groups<2, true>) : launch(b3::column_groups<2, false>);
    else off32 ? launch(b3::column_groups<1, true>) : launch(b3::column_groups<1, false>);
    VMX_HIP(c, hipGetLastError());
    const uint32_t* in = buf;
    uint32_t* next = buf ? buf + k * cols * 8 : nullptr;
    while (k > static_cast<size_t>(b3::MERGE_MAX)) {  // 16-way passes down to a single workgroup's worth
        const size_t k_out = (k + b3::FAN_IN - 1) / b3::FAN_IN;
        hipLaunchKernelGGL(b3::merge_pass, dim3(static_cast<unsigned>((cols + b3::LANES - 1) / b3::LANES),
                                                static_cast<unsigned>(k_out)),
                           dim3(b3::LANES), 0, c->stream, in, k, cols, 0, next);
        VMX_HIP(c, hipGetLastError());
        in = next;
        next += k_out * cols * 8;
        k = k_out;
    }
    if (k > 1) {
        // threads per column: the first level's joins, rounded up to a power of two
        size_t tpc = 1;
        while (tpc < (k + 1) / 2) tpc *= 2;
        const int cpw = static_cast<int>(b3::MERGE_THREADS / tpc);
        hipLaunchKernelGGL(b3::merge_final, dim3(static_cast<unsigned>((cols + cpw - 1) / cpw)),
                           dim3(b3::MERGE_THREADS), 0, c->stream, in, static_cast<int>(k), cols, cpw, leaves);
        VMX_HIP(c, hipGetLastError());
    }
    return 0;
}

int merkle_tree_levels(Context* c, uint32_t* tree, size_t leaves) {
    size_t off = 0, len = leaves;
    while (len > 1) {
        const size_t span = len > b3::TREE_MAX ? b3::TREE_SPAN : len;
        hipLaunchKernelGGL(b3::merkle_subtrees, dim3(static_cast<unsigned>(len / span)), dim3(b3::TREE_THREADS), 0,
                           c->stream, tree, off, len, static_cast<int>(span));
        VMX_HIP(c, hipGetLastError());
        for (size_t n = span; n > 1; n /= 2) {
            off += len;
            len /= 2;
        }
    }
    return 0;
}

int merkle_paths(Context* c, const uint32_t* tree, size_t leaves, const uint32_t* idx, size_t queries,
                 uint32_t* paths) {
    int bits = 0;
    while ((size_t{1} << bits) < leaves) ++bits;
    const size_t total = queries * bits;
    hipLaunchKernelGGL(b3::merkle_paths_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0,
                       c->stream, tree, idx, paths, leaves, queries, bits);
    VMX_HIP(c, hipGetLastError());
    return 0;
}

}  // namespace vmx
