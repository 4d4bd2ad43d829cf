// Tip5 hashing kernels: row digests, pair hashing, Merkle trees, auth paths.
//
// Every kernel runs 16 sponges per wave (tip5_dev.hpp): lane 16g + n holds
// words 4v + g (v = 0..3) of sponge n.  State words 0..9 are the rate.
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
// Large levels take a launch each; below them a block hashes up to 256 parents,
// keeps them in LDS and continues to their subtree root.
#include "tvh_internal.hpp"

namespace tvh {

using gl::u32;
using gl::u64;

// Sponge states are kept in Montgomery form (tip5_dev.hpp); digests leave
// canonical.  Word 4v + g < 5 of the lane's sponge goes to dst[4v + g].
__device__ __forceinline__ void store_digest(u64* dst, const u64 s[tip5::WORDS],
                                             const tip5::Wave& W) {
    dst[W.g] = tip5::from_m(s[0]);
    if (W.g == 0) dst[4] = tip5::from_m(s[1]);
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

// First sponge of the wave: block blk of kSpongesPerBlock sponges.
__device__ __forceinline__ u64 wave_first(u64 blk) {
    return blk * kSpongesPerBlock + (threadIdx.x >> 6) * tip5::GROUP;
}

// Absorbs one full rate block: elem(i) is element i (0..9), canonical.
template <class F>
__device__ __forceinline__ void absorb(u64 s[tip5::WORDS], const tip5::Wave& W, const F& elem) {
    const u64 x[3] = {elem(W.g), elem(4 + W.g), W.g < 2 ? elem(8 + W.g) : 0};
    u64 m[3];
    gl::mask bad = 0;
    gl::to_mont_rare(m, x, bad);
    if (__builtin_expect(gl::in_mask(bad), 0)) {
#pragma unroll
        for (int i = 0; i < 3; i++) m[i] = tip5::to_m(x[i]);
    }
    s[0] = m[0];
    s[1] = m[1];
    s[2] = W.g < 2 ? m[2] : s[2];
}

// Absorbs the padding block [rest elements, 1, 0...], rest < 10.
template <class F>
__device__ __forceinline__ void absorb_last(u64 s[tip5::WORDS], const tip5::Wave& W, u32 rest,
                                            const F& elem) {
#pragma unroll
    for (int v = 0; v < 3; v++) {
        const u32 i = 4 * v + W.g;
        if (i < (u32)tip5::RATE)
            s[v] = i < rest ? tip5::to_m(elem(i)) : (i == rest ? tip5::kOneM : 0ull);
    }
}

// rows x cols column-major table -> rows digests (5 u64 each, row-major).
__device__ __forceinline__ void hash_rows_body(const HashArgs& A, u64 blk, const tip5::Wave& W) {
    const u64 row = wave_first(blk) + W.n;
    const u64 rows = A.rows;
    const u32 cols = A.cols;
    // lanes past the last row hash it again (they take part in the matrix products)
    const u64* p = A.tab + (row < rows ? row : rows - 1);
    u64 s[tip5::WORDS] = {0, 0, 0, 0};
    u32 used = 0;
    for (; used + tip5::RATE <= cols; used += tip5::RATE) {
        absorb(s, W, [&](u32 i) { return __builtin_nontemporal_load(p + (u64)(used + i) * rows); });
        tip5::permutation_m(s, W);
    }
    absorb_last(s, W, cols - used,
                [&](u32 i) { return __builtin_nontemporal_load(p + (u64)(used + i) * rows); });
    tip5::permutation_m(s, W);
    if (row < rows) store_digest(A.dig + row * tip5::DIGEST, s, W);
}

__global__ void __launch_bounds__(kHashThreads, 4) k_hash_rows(HashArgs A) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    hash_rows_body(A, blockIdx.x, W);
}

__global__ void __launch_bounds__(kHashThreads, 4) k_hash_rows_multi(
    const HashArgs* __restrict__ args, const u32* __restrict__ start, u32 nseg) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    u32 seg = find_seg(start, nseg, blockIdx.x);
    HashArgs A = args[seg];
    hash_rows_body(A, blockIdx.x - start[seg], W);
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
template <bool FINAL>
__global__ void __launch_bounds__(kHashThreads, 4)
    k_absorb_chunk(const u64* __restrict__ chunk, u64 rows, u32 ccols, u64* __restrict__ state,
                   u64* __restrict__ pend, u32 npend, int first, u64* __restrict__ dig) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u64 row = wave_first(blockIdx.x) + W.n;
    const u64 r = row < rows ? row : rows - 1;  // lanes past the end repeat the last row
    u64 s[tip5::WORDS];
#pragma unroll
    for (int v = 0; v < tip5::WORDS; v++) s[v] = first ? 0ull : state[(u64)(4 * v + W.g) * rows + r];
    auto elem = [&](u32 j) -> u64 {
        return j < npend ? pend[(u64)j * rows + r] : chunk[(u64)(j - npend) * rows + r];
    };
    const u32 total = npend + ccols;
    u32 used = 0;
    for (; used + tip5::RATE <= total; used += tip5::RATE) {
        absorb(s, W, [&](u32 i) { return elem(used + i); });
        tip5::permutation_m(s, W);
    }
    const u32 rest = total - used;
    if (FINAL) {
        absorb_last(s, W, rest, [&](u32 i) { return elem(used + i); });
        tip5::permutation_m(s, W);
        if (row < rows) store_digest(dig + row * tip5::DIGEST, s, W);
    } else if (row < rows) {
        // carried elements: position i is read and written by the same lane
#pragma unroll
        for (int v = 0; v < 3; v++) {
            const u32 i = 4 * v + W.g;
            if (i < rest) pend[(u64)i * rows + row] = elem(used + i);
        }
#pragma unroll
        for (int v = 0; v < tip5::WORDS; v++) state[(u64)(4 * v + W.g) * rows + row] = s[v];
    }
}

// Tip5 permutation of num states (16 u64 each, in place); outputs canonical.
__global__ void __launch_bounds__(kHashThreads, 4) k_permutation(u64* __restrict__ st, u64 num) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first(blockIdx.x) + W.n;
    const u64* in = st + (i < num ? i : num - 1) * tip5::STATE + W.g;
    u64 s[tip5::WORDS];
#pragma unroll
    for (int v = 0; v < tip5::WORDS; v++) s[v] = tip5::to_m(in[4 * v]);
    tip5::permutation_m(s, W);
    if (i >= num) return;
#pragma unroll
    for (int v = 0; v < tip5::WORDS; v++) st[i * tip5::STATE + W.g + 4 * v] = tip5::from_m(s[v]);
}

// Rounds [first, first + count) of the permutation on num states (in place).
// trace (may be null) receives, per state, the input and the state after each
// of those rounds: trace[(i * (count + 1) + j) * 16 + k].  Outputs canonical.
__global__ void __launch_bounds__(kHashThreads) k_permutation_rounds(u64* __restrict__ st, u64 num,
                                                                     u32 first, u32 count,
                                                                     u64* __restrict__ trace) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first(blockIdx.x) + W.n;
    const bool live = i < num;
    const u64* in = st + (live ? i : num - 1) * tip5::STATE + W.g;
    u64* tr = trace && live ? trace + i * (count + 1) * tip5::STATE + W.g : nullptr;
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
    if (!live) return;
#pragma unroll
    for (int v = 0; v < tip5::WORDS; v++) st[i * tip5::STATE + W.g + 4 * v] = tip5::from_m(s[v]);
}

// hash_pair: the two digests are words 0..9 (elem), the capacity is ones.
template <class F>
__device__ __forceinline__ void hash_pair(u64 s[tip5::WORDS], const tip5::Wave& W, const F& elem) {
    s[2] = s[3] = tip5::kOneM;
    absorb(s, W, elem);
    tip5::permutation_m(s, W);
}

// out[i] = hash_pair(left[i], right[i])  (Backend::hash_pairs, backend.hpp:110-115)
__global__ void __launch_bounds__(kHashThreads, 4) k_hash_pairs(const u64* __restrict__ left,
                                                                const u64* __restrict__ right,
                                                                u64* __restrict__ out, u64 count) {
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    __syncthreads();
    const u64 i = wave_first(blockIdx.x) + W.n;
    const u64 r = i < count ? i : count - 1;
    u64 s[tip5::WORDS];
    hash_pair(s, W, [&](u32 k) { return k < 5 ? left[5 * r + k] : right[5 * r + k - 5]; });
    if (i < count) store_digest(out + 5 * i, s, W);
}

// One launch of the Merkle build: children are the nodes of one level; each
// block hashes 2T children into T parents (16 per wave, T <= 16 waves) and
// continues for `levels` levels inside LDS.  Level j (1-based) parents go to
// dst[j-1] + index.
__device__ __forceinline__ void merkle_body(const MerkleArgs& A, u64 blk, const tip5::Wave& W,
                                            u64* buf) {
    const u32 first = (threadIdx.x >> 6) * tip5::GROUP;  // the wave's first parent
    const u32 t = first + W.n;
    u32 width = A.T;
    u64 s[tip5::WORDS];
    if (first < width) {  // (whole waves)
        const u64* c = A.src + 10 * (blk * width + (t < width ? t : 0));
        hash_pair(s, W, [&](u32 k) { return c[k]; });
    }
    for (u32 j = 0;; j++) {
        const bool last = j + 1 == A.levels;
        if (t < width) {
            u64* d = A.dst[j] + 5 * (blk * width + t);
            const u64 x = tip5::from_m(s[0]);
            d[W.g] = x;
            if (!last) buf[5 * t + W.g] = x;
            if (W.g == 0) {
                const u64 z = tip5::from_m(s[1]);
                d[4] = z;
                if (!last) buf[5 * t + 4] = z;
            }
        }
        if (last) break;
        __syncthreads();  // this level's digests are in buf
        width >>= 1;
        u64 in[3] = {0, 0, 0};
        if (first < width) {
            const u64* c = buf + 10 * (t < width ? t : 0);
            in[0] = c[W.g];
            in[1] = c[4 + W.g];
            if (W.g < 2) in[2] = c[8 + W.g];
        }
        __syncthreads();  // every read of buf precedes the next level's writes
        if (first < width) hash_pair(s, W, [&](u32 k) { return in[k >> 2]; });
    }
}

template <int THREADS>
__global__ void __launch_bounds__(THREADS) k_merkle_subtrees(MerkleArgs A) {
    __shared__ tip5::Tables T;
    __shared__ u64 buf[THREADS / 64 * tip5::GROUP * 5];
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
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
    u32 seg = find_seg(start, nseg, blockIdx.x);
    const MerkleArgs& A = args[seg];  // read in place: a private copy would spill dst[]
    merkle_body(A, blockIdx.x - start[seg], W, buf);
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

int launch_hash_rows(const u64* tab, u64 rows, u64 cols, u64* dig, hipStream_t st) {
    if (rows == 0) return TVH_OK;
    if (cols > 0xFFFFFFFFull) return TVH_ERR_INVALID_ARG;
    hipLaunchKernelGGL(k_hash_rows, dim3(sponge_blocks(rows)), dim3(kHashThreads), 0, st,
                       HashArgs{tab, rows, (u32)cols, dig});
    return check_launch();
}

int launch_absorb_chunk(const u64* chunk, u64 rows, u64 ccols, u64* state, u64* pend, u32 npend,
                        bool first, bool final_chunk, u64* dig, hipStream_t st) {
    if (rows == 0) return TVH_OK;
    const dim3 blocks(sponge_blocks(rows)), tpb(kHashThreads);
    if (final_chunk)
        hipLaunchKernelGGL(k_absorb_chunk<true>, blocks, tpb, 0, st, chunk, rows, (u32)ccols, state,
                           pend, npend, (int)first, dig);
    else
        hipLaunchKernelGGL(k_absorb_chunk<false>, blocks, tpb, 0, st, chunk, rows, (u32)ccols, state,
                           pend, npend, (int)first, dig);
    return check_launch();
}

// Fiat-Shamir sponge on a device-resident state (16 canonical u64), following
// the reference's device transcript (fiat_shamir_kernel.cu: fs_absorb_device_gpu
// pads [data..., 1, 0...] to a multiple of 10 and overwrites the rate before
// each permutation; squeeze reads the rate, then permutes).  One wave runs the
// whole absorption in one launch; its 16 sponges are the same one.
// mode 0 absorb, 1 squeeze, 2 init (zeros; a kernel rather than a memset so
// that the call can be captured in a graph).
__global__ void __launch_bounds__(64) k_sponge(u64* __restrict__ state,
                                               const u64* __restrict__ data, u64 len,
                                               u64* __restrict__ out, int mode) {
    if (mode == 2) {
        if (threadIdx.x < tip5::STATE) state[threadIdx.x] = 0;
        return;
    }
    __shared__ tip5::Tables T;
    tip5::load_tables(T);
    const tip5::Wave W = tip5::make_wave(T);
    u64 s[tip5::WORDS];
#pragma unroll
    for (int v = 0; v < tip5::WORDS; v++) s[v] = tip5::to_m(state[4 * v + W.g]);
    __syncthreads();  // (also: every lane has read the state before lanes n = 0 write it)
    if (mode == 1) {
#pragma unroll
        for (int v = 0; v < 3; v++)
            if (W.n == 0 && 4 * v + W.g < (u32)tip5::RATE) out[4 * v + W.g] = tip5::from_m(s[v]);
        tip5::permutation_m(s, W);
    } else {
        u64 base = 0;
        for (; base + tip5::RATE <= len; base += tip5::RATE) {
            absorb(s, W, [&](u32 i) { return data[base + i]; });
            tip5::permutation_m(s, W);
        }
        absorb_last(s, W, (u32)(len - base), [&](u32 i) { return data[base + i]; });
        tip5::permutation_m(s, W);
    }
    if (W.n == 0) {
#pragma unroll
        for (int v = 0; v < tip5::WORDS; v++) state[4 * v + W.g] = tip5::from_m(s[v]);
    }
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
    hipLaunchKernelGGL(k_permutation, dim3(sponge_blocks(num)), dim3(kHashThreads), 0, st, states,
                       num);
    return check_launch();
}

int launch_permutation_rounds(u64* states, u64 num, u32 first, u32 count, u64* trace,
                              hipStream_t st) {
    if (num == 0) return TVH_OK;
    hipLaunchKernelGGL(k_permutation_rounds, dim3(sponge_blocks(num)), dim3(kHashThreads), 0, st,
                       states, num, first, count, trace);
    return check_launch();
}

int launch_hash_pairs(const u64* l, const u64* r, u64* out, u64 count, hipStream_t st) {
    if (count == 0) return TVH_OK;
    hipLaunchKernelGGL(k_hash_pairs, dim3(sponge_blocks(count)), dim3(kHashThreads), 0, st, l, r, out,
                       count);
    return check_launch();
}

u64 merkle_level_base(u64 n, u32 level, int layout) {
    return layout == TVH_TREE_HEAP ? (n >> level) : (2 * n - ((2 * n) >> level));
}

// Launch groups of the Merkle build of an n-leaf tree whose leaves are already
// at level 0: group g covers up to 9 levels; T parents per block at its first.
// A launch over many tables (multi) has one block size for all of them.
int merkle_groups(u64* tree, u64 n, int layout, bool multi, std::vector<MerkleGroup>& groups) {
    groups.clear();
    u32 logn = log2u(n);
    u32 lvl = 0;
    while (lvl < logn) {
        u64 nchild = n >> lvl;
        u64 parents = nchild / 2;
        const bool wide = parents > kMerkleSubtreeParents;
        const u64 most = wide && !multi ? kSpongesPerBlock : kMerkleSponges;
        u32 T = (u32)(parents < most ? parents : most);  // parents is a power of two
        u32 maxlev = wide ? 1 : log2u(T) + 1;            // T = 256 -> 9 levels
        u32 levels = logn - lvl < maxlev ? logn - lvl : maxlev;
        MerkleGroup g;
        g.args.src = tree + 5 * merkle_level_base(n, lvl, layout);
        for (u32 j = 0; j < 9; j++)
            g.args.dst[j] = j < levels ? tree + 5 * merkle_level_base(n, lvl + j + 1, layout) : nullptr;
        g.args.levels = levels;
        g.args.T = T;
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
        if (g.args.T <= kSpongesPerBlock)
            hipLaunchKernelGGL(k_merkle_subtrees<kHashThreads>, dim3(g.blocks), dim3(kHashThreads), 0,
                               st, g.args);
        else
            hipLaunchKernelGGL(k_merkle_subtrees<kMerkleThreads>, dim3(g.blocks),
                               dim3(kMerkleThreads), 0, st, g.args);
        int rc = check_launch();
        if (rc) return rc;
    }
    return TVH_OK;
}

int launch_hash_rows_multi(const HashArgs* d_args, const u32* d_start, u32 nseg, u32 blocks,
                           hipStream_t st) {
    if (!blocks) return TVH_OK;
    hipLaunchKernelGGL(k_hash_rows_multi, dim3(blocks), dim3(kHashThreads), 0, st, d_args, d_start,
                       nseg);
    return check_launch();
}

int launch_merkle_multi(const MerkleArgs* d_args, const u32* d_start, u32 nseg, u32 blocks,
                        hipStream_t st) {
    if (!blocks) return TVH_OK;
    hipLaunchKernelGGL(k_merkle_subtrees_multi, dim3(blocks), dim3(kMerkleThreads), 0, st, d_args,
                       d_start, nseg);
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
