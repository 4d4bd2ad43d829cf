// Tip5 hashing kernels: row digests, pair hashing, Merkle trees, auth paths.
//
// The kernels run 16 sponges per wave, or four where that would leave SIMDs
// without a wave (tip5_dev.hpp).  State words 0..9 are the rate.
//
// Row hashing restates Tip5::hash_varlen (src/hash/tip5.cpp:246-282) over a
// column-major table (element (r, c) at c*rows + r, the reference GPU layout,
// include/gpu/kernels/row_hash_kernel.cuh:18-33): zero state, overwrite absorb
// of 10 elements per permutation, last block padded [rest, 1, 0...].  A wave
// reads 16 consecutive u64 (one 128-byte line) of four columns at a time.
//
// Merkle trees follow merkle_tree.cpp:41-61 (parent = hash_pair(left,right)).
// Node (level l, index i) of an n-leaf tree lives at base(l) + i with
//   level order (merkle_kernel.cu:60-102): base(l) = 2n - (2n >> l)
//   heap        (merkle_tree.cpp:12-33):   base(l) = n >> l      (1-indexed)
// Large levels take a launch each; below them a block hashes up to 64 parents (256
// in launches over many trees), keeps them in LDS and continues to their subtree
// root.
#include "tvh_internal.hpp"

namespace tvh {

using gl::u32;
using gl::u64;

// Sponge states are kept in Montgomery form (tip5_dev.hpp); digests leave
// canonical.  The kernels are templates over the wave's form Wv: 16 sponges
// (tip5::Wave) or four (tip5::QuadWave).
template <class Wv>
__device__ __forceinline__ void store_digest(u64* dst, const u64 (&s)[Wv::kWords], const Wv& W) {
#pragma unroll
    for (int v = 0; v < Wv::kWords; v++)
        if (W.word(v) < (u32)tip5::DIGEST) dst[W.word(v)] = tip5::from_m(s[v]);
}

// Segment lookup for multi-table launches (start[nseg] = total blocks).
__device__ __forceinline__ u32 find_seg(const u32* __restrict__ start, u32 nseg, u32 blk) {
    u32 lo = 0, hi = nseg;
    while (hi - lo > 1) {
        u32 mid = (lo + hi) >> 1;
        if (start[mid] <= blk) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Blocks of `threads` threads along the first axis of a hash_grid launch that has a
// second one, and the block's index (launches of the four-sponge form are short).
__host__ __device__ constexpr u64 grid_row(u32 threads) { return (1ull << 31) / threads; }
template <class Wv, u32 THREADS = kHashThreads>
__device__ __forceinline__ u64 grid_block() {
    if constexpr (Wv::kSponges == (u32)tip5::QUAD) return blockIdx.x;
    return blockIdx.y * grid_row(THREADS) + blockIdx.x;
}

// First sponge of the wave in block blk.
template <class Wv>
__device__ __forceinline__ u64 wave_first(u64 blk) {
    return (blk * (blockDim.x >> 6) + (threadIdx.x >> 6)) * Wv::kSponges;
}

// The lane's elements of a full rate block: elem(i) is element i (0..9), canonical.
template <class Wv>
constexpr int kRateWords = Wv::kWords < 3 ? Wv::kWords : 3;
template <class Wv, class F>
__device__ __forceinline__ void rate_elements(u64 (&x)[kRateWords<Wv>], const Wv& W, const F& elem) {
#pragma unroll
    for (int v = 0; v < kRateWords<Wv>; v++)
        x[v] = W.word(v) < (u32)tip5::RATE ? elem(W.word(v)) : 0;
}
// Absorbs them.
template <class Wv>
__device__ __forceinline__ void absorb(u64 (&s)[Wv::kWords], const Wv& W,
                                       const u64 (&x)[kRateWords<Wv>]) {
    constexpr int N = kRateWords<Wv>;
    u64 m[N];
    if constexpr (N >= 3) {
        gl::mask bad = 0;
        gl::to_mont_rare(m, x, bad);
        if (__builtin_expect(gl::in_mask(bad), 0)) {
#pragma unroll
            for (int i = 0; i < N; i++) m[i] = tip5::to_m(x[i]);
        }
    } else {
        m[0] = tip5::to_m(x[0]);
    }
#pragma unroll
    for (int v = 0; v < N; v++) s[v] = W.word(v) < (u32)tip5::RATE ? m[v] : s[v];
}

// Absorbs the padding block [rest elements, 1, 0...], rest < 10.
template <class Wv, class F>
__device__ __forceinline__ void absorb_last(u64 (&s)[Wv::kWords], const Wv& W, u32 rest, const F& elem) {
#pragma unroll
    for (int v = 0; v < kRateWords<Wv>; v++) {
        const u32 i = W.word(v);
        if (i < (u32)tip5::RATE)
            s[v] = i < rest ? tip5::to_m(elem(i)) : (i == rest ? tip5::kOneM : 0ull);
    }
}

// Absorbs `total` elements, elem(i), and permutes after each rate block; the
// elements past the last full block are left (their count is returned).
template <class Wv, class F>
__device__ __forceinline__ u32 absorb_blocks(u64 (&s)[Wv::kWords], const Wv& W, u32 total, const F& elem) {
    u32 used = 0;
    for (; used + tip5::RATE <= total; used += tip5::RATE) {
        u64 x[kRateWords<Wv>];
        rate_elements(x, W, [&](u32 i) { return elem(used + i); });
        absorb(s, W, x);
        tip5::permutation_m(s, W);
    }
    return total - used;
}

// rows x cols column-major table -> rows digests (5 u64 each, row-major).
template <class Wv>
__device__ __forceinline__ void hash_rows_body(const HashArgs& A, u64 blk, const Wv& W) {
    const u64 row = wave_first<Wv>(blk) + W.n;
    const u64 rows = A.rows;
    const u32 cols = A.cols;
    // lanes past the last row hash it again (they take part in the matrix products)
    const u64* p = A.tab + (row < rows ? row : rows - 1);
    auto elem = [&](u32 i) { return __builtin_nontemporal_load(p + (u64)i * rows); };
    u64 s[Wv::kWords] = {};
    const u32 rest = absorb_blocks(s, W, cols, elem);
    absorb_last(s, W, rest, [&](u32 i) { return elem(cols - rest + i); });
    tip5::permutation_m(s, W);
    if (row < rows) store_digest(A.dig + row * tip5::DIGEST, s, W);
}

template <class Wv>
__global__ void __launch_bounds__(kHashThreads, 4) k_hash_rows(HashArgs A) {
    __shared__ typename Wv::Tables T;
    tip5::load_tables(T);
    const Wv W = tip5::make_wave(T);
    __syncthreads();
    hash_rows_body(A, grid_block<Wv>(), W);
}

__global__ void __launch_bounds__(kHashThreads, 4) k_hash_rows_multi(
    const HashArgs* __restrict__ args, const u32* __restrict__ start, u32 nseg) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u32 blk = (u32)grid_block<tip5::Wave>();  // (surplus: the last table's, past its rows)
    u32 seg = find_seg(start, nseg, blk);
    HashArgs A = args[seg];
    hash_rows_body(A, blk - start[seg], W);
}

// Column-chunk absorption for the streaming ("frugal") commit: each row's
// hash_varlen sponge continues across chunks of columns.  The row's element
// stream is the npend elements left over from the previous chunks (pend,
// column-major by position) followed by this chunk's ccols columns; full rate
// blocks are absorbed by overwrite, the remainder is carried.  All rows have
// the same counts, so lanes never diverge.  State is column-major by word
// (state[i*rows + row]).  The FINAL chunk absorbs the padding block
// [rest, 1, 0...] and writes the canonical digest (tip5.cpp:246-282).  The
// carried state is in Montgomery form, the carried elements are canonical.
template <bool FINAL, class Wv>
__global__ void __launch_bounds__(kHashThreads, 4)
    k_absorb_chunk(const u64* __restrict__ chunk, u64 rows, u32 ccols, u64* __restrict__ state,
                   u64* __restrict__ pend, u32 npend, int first, u64* __restrict__ dig) {
    __shared__ typename Wv::Tables T;
    tip5::load_tables(T);
    const Wv W = tip5::make_wave(T);
    __syncthreads();
    const u64 row = wave_first<Wv>(grid_block<Wv>()) + W.n;
    const u64 r = row < rows ? row : rows - 1;  // lanes past the end repeat the last row
    u64 s[Wv::kWords];
#pragma unroll
    for (int v = 0; v < Wv::kWords; v++) s[v] = first ? 0ull : state[(u64)W.word(v) * rows + r];
    auto elem = [&](u32 j) -> u64 {
        return j < npend ? pend[(u64)j * rows + r] : chunk[(u64)(j - npend) * rows + r];
    };
    const u32 total = npend + ccols;
    const u32 rest = absorb_blocks(s, W, total, elem), used = total - rest;
    if (FINAL) {
        absorb_last(s, W, rest, [&](u32 i) { return elem(used + i); });
        tip5::permutation_m(s, W);
        if (row < rows) store_digest(dig + row * tip5::DIGEST, s, W);
    } else if (row < rows) {
        // carried elements: position i is read and written by the same lane
#pragma unroll
        for (int v = 0; v < kRateWords<Wv>; v++) {
            const u32 i = W.word(v);
            if (i < rest) pend[(u64)i * rows + row] = elem(used + i);
        }
#pragma unroll
        for (int v = 0; v < Wv::kWords; v++) state[(u64)W.word(v) * rows + row] = s[v];
    }
}

// Tip5 permutation of num states (16 u64 each, in place); outputs canonical.
template <class Wv>
__global__ void __launch_bounds__(kHashThreads, 4) k_permutation(u64* __restrict__ st, u64 num) {
    __shared__ typename Wv::Tables T;
    tip5::load_tables(T);
    const Wv W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first<Wv>(grid_block<Wv>()) + W.n;
    const u64* in = st + (i < num ? i : num - 1) * tip5::STATE;
    u64 s[Wv::kWords];
#pragma unroll
    for (int v = 0; v < Wv::kWords; v++) s[v] = tip5::to_m(in[W.word(v)]);
    tip5::permutation_m(s, W);
    if (i >= num) return;
#pragma unroll
    for (int v = 0; v < Wv::kWords; v++) st[i * tip5::STATE + W.word(v)] = tip5::from_m(s[v]);
}

// Rounds [first, first + count) of the permutation on num states (in place).
// trace (may be null) receives, per state, the input and the state after each
// of those rounds: trace[(i * (count + 1) + j) * 16 + k].  Outputs canonical.
// Without a trace (TRACED) a block takes its sets of 64 states in turn: its tables and
// operands (12 KB a wave) outweigh the states (2 KB) where there are few rounds.
template <bool TRACED>
__global__ void __launch_bounds__(kHashThreads) k_permutation_rounds(u64* __restrict__ st, u64 num,
                                                                     u32 first, u32 count,
                                                                     u64* __restrict__ trace) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    u64 blk = blockIdx.x;
    do {
        const u64 i = wave_first<tip5::Wave>(blk) + W.n;
        const bool live = i < num;
        const u64* in = st + (live ? i : num - 1) * tip5::STATE + W.g;
        u64* tr = TRACED && live ? trace + i * (count + 1) * tip5::STATE + W.g : nullptr;
        u64 s[tip5::WORDS];
#pragma unroll
        for (int v = 0; v < tip5::WORDS; v++) {
            const u64 x = in[4 * v];
            if (tr) tr[4 * v] = x;
            s[v] = tip5::to_m(x);
        }
        for (u32 r = 0; r < count; r++) {
            tip5::round_m(s, (int)(first + r), W);
            if (tr) {
#pragma unroll
                for (int v = 0; v < tip5::WORDS; v++)
                    tr[(r + 1) * tip5::STATE + 4 * v] = tip5::from_m(s[v]);
            }
        }
        if (live) {
#pragma unroll
            for (int v = 0; v < tip5::WORDS; v++) st[i * tip5::STATE + W.g + 4 * v] = tip5::from_m(s[v]);
        }
        blk += gridDim.x;
    } while (!TRACED && blk * kSpongesPerBlock < num);
}

// hash_pair: the two digests are words 0..9 (x: the lane's), the capacity is ones.
template <class Wv>
__device__ __forceinline__ void hash_pair(u64 (&s)[Wv::kWords], const Wv& W, const u64 (&x)[kRateWords<Wv>]) {
#pragma unroll
    for (int v = 0; v < Wv::kWords; v++) s[v] = tip5::kOneM;
    absorb(s, W, x);
    tip5::permutation_m(s, W);
}

// out[i] = hash_pair(left[i], right[i])  (Backend::hash_pairs, backend.hpp:110-115)
template <class Wv>
__global__ void __launch_bounds__(kHashThreads, 4) k_hash_pairs(const u64* __restrict__ left,
                                                                const u64* __restrict__ right,
                                                                u64* __restrict__ out, u64 count) {
    __shared__ typename Wv::Tables T;
    tip5::load_tables(T);
    const Wv W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first<Wv>(grid_block<Wv>()) + W.n;
    const u64 r = i < count ? i : count - 1;
    u64 s[Wv::kWords], x[kRateWords<Wv>];
    rate_elements(x, W, [&](u32 k) { return k < 5 ? left[5 * r + k] : right[5 * r + k - 5]; });
    hash_pair(s, W, x);
    if (i < count) store_digest(out + 5 * i, s, W);
}

// One launch of the Merkle build: children are the nodes of one level; each
// block hashes 2T children into T parents (T <= its waves' sponges) and
// continues for `levels` levels inside LDS.  Level j (1-based) parents go to
// dst[j-1] + index.
template <class Wv>
__device__ __forceinline__ void merkle_body(const MerkleArgs& A, u64 blk, const Wv& W, u64* buf) {
    const u32 first = (threadIdx.x >> 6) * Wv::kSponges;  // the wave's first parent
    const u32 t = first + W.n;
    u32 width = A.T;
    u64 s[Wv::kWords], x[kRateWords<Wv>];
    if (first < width) {  // (whole waves)
        const u64* c = A.src + 10 * (blk * width + (t < width ? t : 0));
        rate_elements(x, W, [&](u32 k) { return c[k]; });
        hash_pair(s, W, x);
    }
    for (u32 j = 0;; j++) {
        const bool last = j + 1 == A.levels;
        if (t < width) {
            u64* d = A.dst[j] + 5 * (blk * width + t);
#pragma unroll
            for (int v = 0; v < Wv::kWords; v++)
                if (W.word(v) < (u32)tip5::DIGEST) {
                    const u64 y = tip5::from_m(s[v]);
                    d[W.word(v)] = y;
                    if (!last) buf[5 * t + W.word(v)] = y;
                }
        }
        if (last) break;
        __syncthreads();  // this level's digests are in buf
        width >>= 1;
        if (first < width) rate_elements(x, W, [&](u32 k) { return buf[10 * (t < width ? t : 0) + k]; });
        __syncthreads();  // every read of buf precedes the next level's writes
        if (first < width) hash_pair(s, W, x);
    }
}

// One level, kSpongesPerBlock parents to a block.
__global__ void __launch_bounds__(kHashThreads) k_merkle_level(MerkleArgs A) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first<tip5::Wave>(grid_block<tip5::Wave>()) + W.n;
    const u64* c = A.src + 10 * i;
    u64 s[tip5::WORDS], x[3];
    rate_elements(x, W, [&](u32 k) { return c[k]; });
    hash_pair(s, W, x);
    store_digest(A.dst[0] + 5 * i, s, W);
}

// Levels of few parents, up to kQuadSponges to a block, four to a wave.
__global__ void __launch_bounds__(kMerkleThreads) k_merkle_subtrees(MerkleArgs A) {
    __shared__ tip5::QuadTables T;
    __shared__ u64 buf[kQuadSponges * 5];
    tip5::load_tables(T);
    const tip5::QuadWave W = tip5::make_wave(T);
    __syncthreads();
    merkle_body(A, blockIdx.x, W, buf);
}

__global__ void __launch_bounds__(kMerkleThreads) k_merkle_subtrees_multi(
    const MerkleArgs* __restrict__ args, const u32* __restrict__ start, u32 nseg) {
    __shared__ tip5::Tables T;
    __shared__ u64 buf[kMerkleThreads / 64 * tip5::GROUP * 5];
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u32 blk = (u32)grid_block<tip5::Wave, kMerkleThreads>();
    if (blockIdx.y && blk >= start[nseg]) return;  // surplus
    u32 seg = find_seg(start, nseg, blk);
    const MerkleArgs& A = args[seg];  // read in place: a private copy would spill dst[]
    merkle_body(A, blk - start[seg], W, buf);
}

// Gather: out[q] = node with heap index idx[q] (1 <= idx < 2n) of a tree in
// either layout.  Out-of-range indices produce zeros.
__global__ void k_gather_heap(const u64* __restrict__ tree, u64 n, u32 logn, int layout,
                              const u64* __restrict__ idx, u64 count, u64* __restrict__ out) {
    u64 q = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= count * 5) return;
    u64 h = idx[q / 5];
    if (h == 0 || h >= 2 * n) {
        out[q] = 0;
        return;
    }
    u64 pos = h;
    if (layout == TVH_TREE_LEVEL_ORDER) {
        u32 fl = 63 - __builtin_clzll(h);      // floor(log2 h)
        u32 level = logn - fl;                  // 0 = leaves
        u64 base_heap = n >> level;
        pos = (2 * n - ((2 * n) >> level)) + (h - base_heap);
    }
    out[q] = tree[pos * 5 + q % 5];
}

// ------------------------------------------------------------------ host side

// A sponge takes 4 threads or 16, and a launch can have 2^32 threads along one grid
// axis (more are cut off without an error): past 2^31 the blocks go on along the
// second one.  Kernels take grid_block() and leave out the last row's surplus.
static dim3 hash_grid(u64 blocks, u32 threads) {
    const u64 row = grid_row(threads);
    return blocks <= row ? dim3((u32)blocks) : dim3((u32)row, (u32)((blocks + row - 1) / row));
}

// The 16-sponge form, or the four-sponge one where that leaves few waves.
#define TVH_SPONGES(count, kernel, ...)                                                            \
    do {                                                                                           \
        if ((count) <= kQuadMaxSponges)                                                            \
            hipLaunchKernelGGL(kernel<tip5::QuadWave>, dim3(quad_blocks(count)), dim3(kHashThreads), \
                               0, st, __VA_ARGS__);                                                \
        else                                                                                       \
            hipLaunchKernelGGL(kernel<tip5::Wave>, hash_grid(sponge_blocks(count), kHashThreads), \
                               dim3(kHashThreads), 0, st, __VA_ARGS__);                            \
    } while (0)
template <class Wv>
constexpr auto k_absorb_chunk_final = k_absorb_chunk<true, Wv>;
template <class Wv>
constexpr auto k_absorb_chunk_more = k_absorb_chunk<false, Wv>;

int launch_hash_rows(const u64* tab, u64 rows, u64 cols, u64* dig, hipStream_t st) {
    if (rows == 0) return TVH_OK;
    if (cols > 0xFFFFFFFFull) return TVH_ERR_INVALID_ARG;
    const HashArgs A{tab, rows, (u32)cols, dig};
    TVH_SPONGES(rows, k_hash_rows, A);
    return check_launch();
}

int launch_absorb_chunk(const u64* chunk, u64 rows, u64 ccols, u64* state, u64* pend, u32 npend,
                        bool first, bool final_chunk, u64* dig, hipStream_t st) {
    if (rows == 0) return TVH_OK;
    if (final_chunk)
        TVH_SPONGES(rows, k_absorb_chunk_final, chunk, rows, (u32)ccols, state, pend, npend, (int)first, dig);
    else
        TVH_SPONGES(rows, k_absorb_chunk_more, chunk, rows, (u32)ccols, state, pend, npend, (int)first, dig);
    return check_launch();
}

// Fiat-Shamir sponge on a device-resident state (16 canonical u64), following
// the reference's device transcript (fiat_shamir_kernel.cu: fs_absorb_device_gpu
// pads [data..., 1, 0...] to a multiple of 10 and overwrites the rate before
// each permutation; squeeze reads the rate, then permutes).  One wave runs the
// whole absorption in one launch; its four sponges are the same one.
// mode 0 absorb, 1 squeeze, 2 init (zeros; a kernel rather than a memset so
// that the call can be captured in a graph).
__global__ void __launch_bounds__(64) k_sponge(u64* __restrict__ state,
                                               const u64* __restrict__ data, u64 len,
                                               u64* __restrict__ out, int mode) {
    if (mode == 2) {
        if (threadIdx.x < tip5::STATE) state[threadIdx.x] = 0;
        return;
    }
    __shared__ tip5::QuadTables T;
    tip5::load_tables(T);
    const tip5::QuadWave W = tip5::make_wave(T);
    u64 s[1] = {tip5::to_m(state[W.own])};
    __syncthreads();  // (also: every lane has read the state before lanes n = 0 write it)
    if (mode == 1) {
        if (W.n == 0 && W.own < (u32)tip5::RATE) out[W.own] = tip5::from_m(s[0]);
        tip5::permutation_m(s, W);
    } else {
        u64 base = 0;
        for (; base + tip5::RATE <= len; base += tip5::RATE) {
            u64 x[1];
            rate_elements(x, W, [&](u32 i) { return data[base + i]; });
            absorb(s, W, x);
            tip5::permutation_m(s, W);
        }
        absorb_last(s, W, (u32)(len - base), [&](u32 i) { return data[base + i]; });
        tip5::permutation_m(s, W);
    }
    if (W.n == 0) state[W.own] = tip5::from_m(s[0]);
}

int launch_sponge(u64* state, const u64* data, u64 len, u64* out, int mode, hipStream_t st) {
    hipLaunchKernelGGL(k_sponge, dim3(1), dim3(64), 0, st, state, data, len, out, mode);
    return check_launch();
}

// FRI codeword leaves (reference gpu_stark.cu:863-875): XFE i (3 limbs,
// interleaved) becomes the digest (c0, c1, c2, 0, 0) without hashing.
__global__ void k_xfe_leaves(const u64* __restrict__ xfe, u64 n, u64* __restrict__ leaves) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 a = xfe[3 * i], b = xfe[3 * i + 1], c = xfe[3 * i + 2];
    leaves[5 * i + 0] = a;
    leaves[5 * i + 1] = b;
    leaves[5 * i + 2] = c;
    leaves[5 * i + 3] = 0;
    leaves[5 * i + 4] = 0;
}

int launch_xfe_leaves(const u64* xfe, u64 n, u64* leaves, hipStream_t st) {
    if (n == 0) return TVH_OK;
    hipLaunchKernelGGL(k_xfe_leaves, dim3((u32)((n + 255) / 256)), dim3(256), 0, st, xfe, n,
                       leaves);
    return check_launch();
}

int launch_permutation(u64* states, u64 num, hipStream_t st) {
    if (num == 0) return TVH_OK;
    TVH_SPONGES(num, k_permutation, states, num);
    return check_launch();
}

int launch_permutation_rounds(u64* states, u64 num, u32 first, u32 count, u64* trace,
                              hipStream_t st) {
    if (num == 0) return TVH_OK;
    const u64 sets = (num + kSpongesPerBlock - 1) / kSpongesPerBlock;
    const dim3 tpb(kHashThreads);
    if (trace) {
        hipLaunchKernelGGL(k_permutation_rounds<true>, dim3((u32)sets), tpb, 0, st, states, num, first, count,
                           trace);
    } else {
        // eight blocks to a CU (one round of 2^20 states: 59 us, 86 with a block to every
        // 64; a trace's stores want those: 346 us for five rounds of 2^20, else 433)
        hipLaunchKernelGGL(k_permutation_rounds<false>, dim3((u32)(sets < 2048 ? sets : 2048)), tpb, 0, st,
                           states, num, first, count, trace);
    }
    return check_launch();
}

int launch_hash_pairs(const u64* l, const u64* r, u64* out, u64 count, hipStream_t st) {
    if (count == 0) return TVH_OK;
    TVH_SPONGES(count, k_hash_pairs, l, r, out, count);
    return check_launch();
}

u64 merkle_level_base(u64 n, u32 level, int layout) {
    return layout == TVH_TREE_HEAP ? (n >> level) : (2 * n - ((2 * n) >> level));
}

// Launch groups of the Merkle build of an n-leaf tree whose leaves are already
// at level 0: group g covers up to 9 levels; T parents per block at its first.
// A launch over many tables (multi) has one block size for all of them.  For a
// single tree, levels of at most kQuadMaxSponges parents go four to a wave.
int merkle_groups(u64* tree, u64 n, int layout, bool multi, std::vector<MerkleGroup>& groups) {
    groups.clear();
    u32 logn = log2u(n);
    u32 lvl = 0;
    while (lvl < logn) {
        u64 nchild = n >> lvl;
        u64 parents = nchild / 2;
        const bool wide = parents > (multi ? kMerkleSubtreeParents : kQuadMaxSponges);
        const u64 most = multi ? kMerkleSponges : wide ? kSpongesPerBlock : kQuadSponges;
        u32 T = (u32)(parents < most ? parents : most);  // parents is a power of two
        u32 maxlev = wide ? 1 : log2u(T) + 1;            // T = 256 -> 9 levels
        u32 levels = logn - lvl < maxlev ? logn - lvl : maxlev;
        MerkleGroup g;
        g.args.src = tree + 5 * merkle_level_base(n, lvl, layout);
        for (u32 j = 0; j < 9; j++)
            g.args.dst[j] = j < levels ? tree + 5 * merkle_level_base(n, lvl + j + 1, layout) : nullptr;
        g.args.levels = levels;
        g.args.T = T;
        g.quad = !multi && !wide;
        g.blocks = (u32)(parents / T);
        groups.push_back(g);
        lvl += levels;
    }
    return TVH_OK;
}

// Build levels 1..log2(n) of a tree whose leaves are already at level 0.
int launch_merkle_levels(u64* tree, u64 n, int layout, hipStream_t st) {
    std::vector<MerkleGroup> groups;
    merkle_groups(tree, n, layout, false, groups);
    for (const MerkleGroup& g : groups) {
        if (g.quad)  // (waves for the first level's parents)
            hipLaunchKernelGGL(k_merkle_subtrees, dim3(g.blocks),
                               dim3((g.args.T + tip5::QUAD - 1) / tip5::QUAD * 64), 0, st, g.args);
        else
            hipLaunchKernelGGL(k_merkle_level, hash_grid(g.blocks, kHashThreads), dim3(kHashThreads), 0,
                               st, g.args);
        int rc = check_launch();
        if (rc) return rc;
    }
    return TVH_OK;
}

int launch_hash_rows_multi(const HashArgs* d_args, const u32* d_start, u32 nseg, u32 blocks,
                           hipStream_t st) {
    if (!blocks) return TVH_OK;
    hipLaunchKernelGGL(k_hash_rows_multi, hash_grid(blocks, kHashThreads), dim3(kHashThreads), 0, st,
                       d_args, d_start, nseg);
    return check_launch();
}

int launch_merkle_multi(const MerkleArgs* d_args, const u32* d_start, u32 nseg, u32 blocks,
                        hipStream_t st) {
    if (!blocks) return TVH_OK;
    hipLaunchKernelGGL(k_merkle_subtrees_multi, hash_grid(blocks, kMerkleThreads),
                       dim3(kMerkleThreads), 0, st, d_args, d_start, nseg);
    return check_launch();
}

int launch_gather_heap(const u64* tree, u64 n, int layout, const u64* idx, u64 count, u64* out,
                       hipStream_t st) {
    if (count == 0) return TVH_OK;
    u64 total = count * 5;
    hipLaunchKernelGGL(k_gather_heap, dim3((u32)((total + 255) / 256)), dim3(256), 0, st, tree, n,
                       log2u(n), layout, idx, count, out);
    return check_launch();
}

}  // namespace tvh
