// Host side of the batched Goldilocks NTT and the coset low-degree extension:
// kernel variants and plans, the per-shape coset tables, launches, the
// synthetic fill and the XFE relayout.  The kernels themselves are in
// ntt_dev.hpp (device code) and ntt_step1.hip, ntt_step2.hip, lde_rows.hip,
// lde_step3.hip (instantiations and launchers).
#include <atomic>
#include <map>
#include <mutex>
#include <tuple>
#include <utility>

#include "ntt_dev.hpp"

namespace tvh {

// Constant tables pa/pb of one (logN, a, E, o, g).
__global__ void k_lde_consts(u64* pa, u64* pb, u32 a, u32 b, u32 E, const u64* beta, u64 ninv) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    u64 n1 = 1ull << a, n2 = 1ull << b;
    if (i < E * n1) {
        u64 s = i >> a, k1 = i & (n1 - 1);
        pa[i] = gl::mul(ninv, gl::pow(beta[s], k1));
    } else if (i < E * (n1 + n2)) {
        u64 j = i - E * n1;
        u64 s = j >> b, k2 = j & (n2 - 1);
        pb[j] = gl::pow(gl::pow(beta[s], n1), k2);
    }
}

// Synthetic uniform inputs: counter-based SplitMix64 finaliser of seed + (i+1)*gamma.
__global__ void k_fill_uniform(u64* d, u64 count, u64 seed) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    u64 z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    d[i] = z >= gl::P ? z - gl::P : z;
}

int launch_fill_uniform(u64* d, u64 count, u64 seed, hipStream_t st) {
    if (!count) return TVH_OK;
    hipLaunchKernelGGL(k_fill_uniform, dim3((u32)((count + 255) / 256)), dim3(256), 0, st, d,
                       count, seed);
    return check_launch();
}

// XFE interleaved <-> limb-major.  Interleaved: (c*len + r)*3 + k; limb-major: (3c + k)*len + r.
__global__ void k_xfe_relayout(const u64* __restrict__ src, u64* __restrict__ dst, u64 cols,
                               u64 len, int to_limb_major) {
    u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cols * len * 3) return;
    // i indexes the interleaved position
    u64 k = i % 3, cr = i / 3, r = cr % len, c = cr / len;
    u64 lm = (3 * c + k) * len + r;
    if (to_limb_major) dst[lm] = src[i];
    else dst[i] = src[lm];
}

// ---------------------------------------------------------------- host side

// Tuned variant per (log2 N, log2 E, width class); 0 = not set.
static std::atomic<int> g_variant[kMaxLogN + 1][5][kWidthClasses];

int lde_variant(u32 logN, u32 logE, u64 cols) {
    int v = (logN <= kMaxLogN && logE <= 4) ? g_variant[logN][logE][width_class(cols)].load() : 0;
    if (v) return v;
    // default (measured at 16, 88 and 379 columns, 2^8..2^21 rows, E = 1..16): up to
    // 2^14 codeword elements the whole transform in the shortest tile (2^12 x 379,
    // E = 4: 62 us, split 113; 2^10 x 379: 21 in 2^12 tiles, 31 in 2^14); above, the
    // shortest row tile with columns of 2^8, two passes (2^18 x 379: 4.32 ms, 4.66
    // and 4.72 in 2^13 and 2^14; 2^20 x 140: 6.3 in 2^14, 7.2 and 7.5 shorter).
    // Column tiles of 2^13, but 2^12 where those make fewer than four blocks a CU
    // (2^16 x 88: 197 against 204 us; 2^16 x 379: 983 against 916).
    const u32 all = logN + logE;
    // 2^26 codeword elements a column are refused by default (prepare_lde; the bound of
    // the 2^13 row tile does it): only a variant with the 2^14 row tile takes them.
    if (all >= 26) return LDE_SPLIT | 1 << 2 | LDE_ROW_HALF;
    const u32 b = logN < 20 ? logN - 8 : 12;
    const u32 row = all <= LOG_TILE ? all : b + logE;
    const int col = (cols << logN) < (1ull << 23) ? 2 : 1;
    return LDE_SPLIT | col << 2 | (row <= 12 ? LDE_ROW_QUARTER : row == 13 ? LDE_ROW_HALF : 0);
}

bool lde_variant_valid(int v) {
    int form = v & 3, tile = (v >> 2) & 3, half = (v >> 4) & 1, ihalf = (v >> 5) & 1,
        quarter = (v >> 6) & 1;
    return v == LDE_AUTO || (v < 128 && (form == LDE_WIDE || form == LDE_SPLIT) && tile <= 2 &&
                             half + ihalf + quarter <= (form == LDE_SPLIT));
}

int set_lde_variant(u32 logN, u32 logE, int v, int wc) {
    if (logN > kMaxLogN || logE > 4 || !lde_variant_valid(v) || wc >= kWidthClasses)
        return set_error(TVH_ERR_INVALID_ARG, "lde variant (%u, %u, %d)", logN, logE, v);
    for (int c = 0; c < kWidthClasses; c++)
        if (wc < 0 || c == wc) g_variant[logN][logE][c].store(v);
    return TVH_OK;
}

// Passes over LDS (or one product) of a transform of length 2^l.
static u32 passes(u32 l) { return l <= 4 ? 1 : l <= 8 ? 2 : 3; }

// N = N1 * N2, N1 = 2^a.  E * N2 <= 2^row_lt, N2 <= 4096: a row's E coset transforms
// share one tile (the row step overwrites its input row in place, so a row's cosets
// cannot be split over blocks; rows of 2^12 in four cosets go through a smaller tile
// one after the other, and keep to the same bound).  Within that the split with the
// fewest passes, then the longest rows (more contiguous bytes, fewer columns of
// the strided step).  A column step has at least 2^5 points (shorter ones leave
// part of the matrices idle) and, if it can, at most 2^9: longer ones leave less
// than a cache line of adjacent columns in a 2^13 tile (2^20 x 140, E = 4, in
// 2^13 row tiles: 7.2 ms with 2^9, 13.5 with 2^12).  Rows have at least 2^5
// elements too; where that cannot be (2^9 rows, E = 16, 2^12 tiles) the whole
// transform takes the next tile.  Above 2^12 columns the shape is refused (a > 12).
static u32 choose_split(u32 logN, u32 E, u32 row_lt) {
    u32 bmax = row_lt - log2u(E);
    if (bmax > 12) bmax = 12;
    if (logN <= bmax || logN < 10) return 0;
    if (logN - bmax > 12) return logN - bmax;
    u32 best = 0, cost = ~0u;
    for (u32 a = logN - bmax > 5 ? logN - bmax : 5; a <= 9 && a + 5 <= logN; a++) {
        const u32 c = passes(a) + passes(logN - a);
        if (c < cost) {
            cost = c;
            best = a;
        }
    }
    return best ? best : logN - bmax;
}

LaunchShape launch_shape(u32 lt, u32 logL, u32 log_per, u64 cols, bool flat, u32 log_e) {
    LaunchShape g;
    u32 log_nt;
    if (logL <= 4) {
        log_nt = kSmallTile - logL;
        g.threads = kSmallThreads;
    } else {
        log_nt = lt - logL - log_e;
        g.threads = 1u << (lt - 4);
        // (the pitch of Shape<LT, LOGL>, then two sets of accumulator starts)
        const u32 L = 1u << logL, lnt = lt - logL, unit = lnt >= 4 ? 1 : 16u >> lnt;
        const size_t pitch = unit * (((L + (L >> 4) + (L >> 8) + unit) / unit) | 1);
        g.lds = (pitch << lnt) * sizeof(u64) + 2 * 64 * sizeof(u32);
    }
    const u64 blocks = flat ? (cols + (1ull << log_nt) - 1) >> log_nt
                            : cols << (log_per > log_nt ? log_per - log_nt : 0);
    g.blocks = (u32)blocks;
    return g;
}

struct ConstKey {
    u32 logN, a, E;
    u64 toff, goff;
    int dev;
    bool operator<(const ConstKey& o) const {
        return std::tie(logN, a, E, toff, goff, dev) <
               std::tie(o.logN, o.a, o.E, o.toff, o.goff, o.dev);
    }
};
struct ConstVal {
    u64* pa;
    u64* pb;
};
static std::mutex g_const_mu;
static std::map<ConstKey, ConstVal> g_consts;
// At most this many tables (each <= E*(N1+N2)*8 <= 1 MB) are kept; the cache
// never evicts, since kernels in flight may read any entry.
constexpr size_t kMaxConstEntries = 256;

// The coset tables of one (shape, split, offsets) key: found in the cache, or
// computed now (one allocation and a wait on a private stream; tvh_lde_prepare
// does this ahead of time).
static int lde_consts(DeviceState* ds, u32 logN, u32 a, u32 E, u64 toff, u64 goff, ConstVal* out) {
    ConstKey key{logN, a, E, toff, goff, ds->device};
    std::lock_guard<std::mutex> lk(g_const_mu);
    auto it = g_consts.find(key);
    if (it != g_consts.end()) {
        *out = it->second;
        return TVH_OK;
    }
    if (g_consts.size() >= kMaxConstEntries)
        return set_error(TVH_ERR_RANGE,
                         "more than %zu distinct LDE shape/offset tables; release them with "
                         "tvh_lde_release_constants",
                         kMaxConstEntries);
    u32 b = logN - a;
    u64 n1 = 1ull << a, n2 = 1ull << b;
    u64 M = (u64)E << logN;
    u64 wM = gl::root_of_unity(log2u(M));
    u64 oinv = gl::inv(toff);
    u64 beta[16];
    u64 ws = 1;
    for (u32 s = 0; s < E; s++) {
        beta[s] = gl::mul(gl::mul(goff, ws), oinv);
        ws = gl::mul(ws, wM);
    }
    u64 ninv = gl::inv(1ull << logN);
    u64* mem = nullptr;
    size_t bytes = (E * (n1 + n2) + 16) * sizeof(u64);
    if (hipMalloc(&mem, bytes) != hipSuccess) return set_error(TVH_ERR_OOM, "lde constants");
    u64* dbeta = mem + E * (n1 + n2);
    hipStream_t st;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess)
        return set_error(TVH_ERR_DEVICE, "stream create");
    int rc = TVH_OK;
    if (hipMemcpyAsync(dbeta, beta, sizeof(beta), hipMemcpyHostToDevice, st) != hipSuccess)
        rc = set_error(TVH_ERR_DEVICE, "copy beta");
    if (!rc) {
        u64 total = E * (n1 + n2);
        hipLaunchKernelGGL(k_lde_consts, dim3((u32)((total + 255) / 256)), dim3(256), 0, st, mem,
                           mem + E * n1, a, b, E, dbeta, ninv);
        rc = check_launch();
    }
    if (!rc && hipStreamSynchronize(st) != hipSuccess) rc = set_error(TVH_ERR_DEVICE, "sync");
    (void)hipStreamDestroy(st);
    if (rc) {
        (void)hipFree(mem);
        return rc;
    }
    ConstVal v{mem, mem + E * n1};
    g_consts[key] = v;
    *out = v;
    return TVH_OK;
}

int lde_prepare_consts(u64 n, u64 m, u64 toff, u64 goff) {
    if (!is_pow2(n) || !is_pow2(m)) return set_error(TVH_ERR_NOT_POW2, "lde lengths");
    if (m < n) return set_error(TVH_ERR_INVALID_ARG, "target_len < trace_len");
    if (m / n > 16) return set_error(TVH_ERR_UNSUPPORTED, "expansion > 16");
    if (toff == 0 || toff >= gl::P || goff >= gl::P)
        return set_error(TVH_ERR_INVALID_ARG, "offsets must be canonical, trace offset nonzero");
    u32 logN = log2u(n);
    if (logN > 23) return set_error(TVH_ERR_UNSUPPORTED, "trace_len > 2^23");
    DeviceState* ds = current_device();
    if (!ds) return TVH_ERR_DEVICE;
    u32 E = (u32)(m / n);
    // every row tile a kernel variant can use (2^12..2^14 elements) gives its own split
    for (u32 lt = LOG_TILE - 2; lt <= LOG_TILE; lt++) {
        u32 a = choose_split(logN, E, lt);
        if (a > 12) continue;
        ConstVal cv;
        int rc = lde_consts(ds, logN, a, E, toff, goff, &cv);
        if (rc) return rc;
    }
    return TVH_OK;
}

int lde_release_consts() {
    std::lock_guard<std::mutex> lk(g_const_mu);
    if (hipDeviceSynchronize() != hipSuccess) return set_error(TVH_ERR_DEVICE, "device sync");
    for (auto& kv : g_consts) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        (void)hipSetDevice(kv.first.dev);
        (void)hipFree(kv.second.pa);
        (void)hipSetDevice(dev);
    }
    g_consts.clear();
    return TVH_OK;
}

int prepare_lde(const u64* trace, u64 cols, u64 n, const RandSpec& rs, u64 toff, u64 goff,
                u64 m, bool truncate, u64* out, LdePlan* P, bool batch) {
    P->k1 = P->k3 = false;
    P->k2_variant = lde_variant(log2u(n), log2u(m / (n ? n : 1)), cols);
    P->col_lt = batch ? kBatchColLt : LOG_TILE - ((P->k2_variant >> 2) & 3);
    P->row_lt = (P->k2_variant & LDE_ROW_QUARTER) ? LOG_TILE - 2
                : (P->k2_variant & LDE_ROW_HALF)  ? LOG_TILE - 1
                                                  : LOG_TILE;
    P->g1 = P->g2 = P->g3 = LaunchShape{};
    if (cols == 0) return TVH_OK;
    if (!is_pow2(n) || !is_pow2(m)) return set_error(TVH_ERR_NOT_POW2, "lde lengths");
    if (m < n) return set_error(TVH_ERR_INVALID_ARG, "target_len < trace_len");
    u64 E64 = m / n;
    if (E64 > 16) return set_error(TVH_ERR_UNSUPPORTED, "expansion > 16");
    if (rs.k > n) return set_error(TVH_ERR_UNSUPPORTED, "rand_len > trace_len");
    if (toff == 0 || toff >= gl::P || goff >= gl::P)
        return set_error(TVH_ERR_INVALID_ARG, "offsets must be canonical, trace offset nonzero");
    u32 logN = log2u(n), E = (u32)E64, logE = log2u(E64);
    if (logN > 23) return set_error(TVH_ERR_UNSUPPORTED, "trace_len > 2^23");
    DeviceState* ds = current_device();
    if (!ds) return TVH_ERR_DEVICE;
    u32 a = choose_split(logN, E, P->row_lt);
    if (batch) {  // the shapes that row tiles of 2^13 (wide form: 2^14) can take
        const u32 bound = (P->k2_variant & 3) == LDE_SPLIT ? LOG_TILE - 1 : LOG_TILE;
        if (a > 12 || choose_split(logN, E, bound) > 12) a = choose_split(logN, E, bound);
    }
    u32 b = logN - a;
    if (a > 12) return set_error(TVH_ERR_UNSUPPORTED, "split");
    ConstVal cv;
    int rc = lde_consts(ds, logN, a, E, toff, goff, &cv);
    if (rc) return rc;

    // K1: INTT step 1 (transforms (c, n2)); a size-1 step is the identity
    // map trace -> Y, so K2 then reads the trace itself.
    P->k1 = a > 0;
    if (P->k1) {
        P->s1 = Step1Args{trace, n, out, m, logN, a, E, 1, 0};
        P->g1 = launch_shape(P->col_lt, a, b, cols, false);
    }
    // K2: INTT step 2 + coset scaling + forward step 1
    {
        LdeArgs& A = P->s2;
        A.out = out;
        A.logN = logN;
        A.a = a;
        A.E = E;
        A.logE = logE;
        A.cols = cols;
        A.M = m;
        A.pa = cv.pa;
        A.pb = cv.pb;
        A.toff = toff;
        A.rs = rs;
        u64 gN = gl::pow(goff, n), oN = gl::pow(toff, n);
        u64 wE = gl::root_of_unity(logE), ws = 1;
        u64 nmod = n % gl::P;
        for (u32 s = 0; s < 16; s++) {
            u64 d = (truncate && E == 1) ? gl::neg(oN) : gl::sub(gl::mul(gN, ws), oN);
            A.delta_n[s] = gl::mul(d, nmod);
            ws = gl::mul(ws, wE);
        }
        A.src = P->k1 ? out : trace;
        A.src_col_stride = P->k1 ? m : n;
        A.src_row_stride = P->k1 ? ((u64)E << b) : 0;
        // Rows of 2^12 in four cosets: one after the other in a 2^12 tile (2^20 x 379:
        // 12.3 ms, 12.8 in one tile of 2^14).  More cosets leave rows of 2^11 and shorter
        // (choose_split), which share a tile: with two matrices to reload for each coset
        // they are slower one by one (2^18 x 379, E = 8: LDE 10.1 against 8.4 ms; 2^19 x
        // 264, E = 4: 7.6, 6.7).
        A.cosets = a > 0 && b == kCosetsLt && logE == 2 && !batch;
        A.log_c = 0;
        A.products = 0;
        if (b <= 4) {  // a = 0
            // waves for the whole GPU first, then up to 16 products each
            const u64 products = ((cols << (b + logE)) + kShortOut - 1) / kShortOut;
            const u64 waves = kShortThreads / 64;
            A.products = (u32)std::min<u64>(std::max<u64>(products >> 13, 1), 16);
            P->row_lt = kBatchShort;
            P->g2.blocks = (u32)((products + waves * A.products - 1) / (waves * A.products));
            P->g2.threads = kShortThreads;
            P->g2.lds = kShortLds;
        } else if (A.cosets) {  // whole runs to a block of step 3; 16 elements are a cache line
            const u32 log_nt = P->col_lt - a;
            A.log_c = log_nt > logE ? std::min(log_nt - logE, 4u) : 0;
            P->g2 = launch_shape(kCosetsLt, b, a, cols, false);
            P->g2.threads = kCosetsThreads;
            P->g2.lds += sizeof(u64) << kCosetsLt;
        } else {
            P->row_lt = std::max(b + logE, 12u);  // the shortest tile that holds a row's cosets
            P->g2 = launch_shape(P->row_lt, b, a, cols, a == 0, logE);
        }
    }
    // K3: forward step 2 for all cosets (identity when N1 = 1)
    P->k3 = a > 0;
    if (P->k3) {
        P->s3 = Step3Args{out, logN, a, logE, P->s2.log_c, m};
        P->g3 = launch_shape(P->col_lt, a, b + logE, cols, false);
    }
    return TVH_OK;
}

int launch_lde(const u64* trace, u64 cols, u64 n, const RandSpec& rs, u64 toff, u64 goff, u64 m,
               bool truncate, u64* out, hipStream_t st) {
    LdePlan P;
    int rc = prepare_lde(trace, cols, n, rs, toff, goff, m, truncate, out, &P, false);
    if (rc || cols == 0) return rc;
    DeviceState* ds = current_device();
    if (P.k1 && (rc = launch_k_step1(true, P.col_lt, P.g1, st, P.s1, ds->roots)))
        return rc;
    if ((rc = launch_k_lde_rows(P.row_lt, P.g2, st, P.s2, ds->roots))) return rc;
    if (P.k3 && (rc = launch_k_lde_step3(P.col_lt, P.g3, st, P.s3, ds->roots)))
        return rc;
    return TVH_OK;
}

int launch_lde_multi(int phase, const void* d_args, const u32* d_start, u32 nseg, u32 blocks,
                     size_t lds, hipStream_t st) {
    if (blocks == 0) return TVH_OK;
    DeviceState* ds = current_device();
    if (!ds) return TVH_ERR_DEVICE;
    switch (phase) {
        case LDE_PHASE_STEP1:
            return launch_k_step1_multi((const Step1Args*)d_args, d_start, nseg, blocks, lds, st,
                                        ds->roots);
        case LDE_PHASE_STEP3:
            return launch_k_lde_step3_multi((const Step3Args*)d_args, d_start, nseg, blocks, lds, st,
                                            ds->roots);
        default:
            return launch_k_lde_rows_multi(12 + phase - LDE_PHASE_ROWS, (const LdeArgs*)d_args, d_start,
                                           nseg, blocks, lds, st, ds->roots);
    }
}

// Scratch of the allocation-free NTT entry point (tvh_ntt_batched_noalloc_dev):
// one file-scope device array per GPU, held until the process ends.  Host
// code never passes `scratch` itself to a kernel (in host code the name is a
// host-side stand-in, not a device address): noalloc_scratch_setup resolves
// this device's address once, at set-up, and launches take that pointer.
static __device__ __align__(256) u64 scratch[kNoAllocScratchElems];

int noalloc_scratch_setup(DeviceState* ds) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return set_error(TVH_ERR_DEVICE, "no-allocation scratch address: %s", hipGetErrorString(e));
    ds->noalloc_scratch = (u64*)p;
    return TVH_OK;
}

u64 ntt_scratch_elems(u64 n, u64 cols) {
    // columns go through the scratch in groups of at most 2 GiB.  Every group
    // is one launch of each step, and each launch pays about one round of
    // blocks to fill and drain the GPU (~35 us at 2^20 rows, a tenth of a
    // 32-column launch), so the groups are made large; the cap bounds the
    // scratch (a 2^20 x 379 table takes two groups).
    u64 group = cols;
    u64 max_group = (2048ull << 20) / (n * sizeof(u64));
    if (max_group < 1) max_group = 1;
    if (group > max_group) group = max_group;
    return group * n;
}

int launch_ntt_batched(const u64* src, u64* dst, u64 n, u64 cols, bool inverse, u64* scratch,
                       u64 scratch_elems, hipStream_t st, const NttScale* scale) {
    if (cols == 0) return TVH_OK;
    if (scale && inverse) return set_error(TVH_ERR_INVALID_ARG, "input scaling of an inverse NTT");
    if (!is_pow2(n)) return set_error(TVH_ERR_NOT_POW2, "NTT size must be a power of 2");
    u32 logN = log2u(n);
    if (logN > kMaxLogN) return set_error(TVH_ERR_UNSUPPORTED, "NTT size > 2^24");
    DeviceState* ds = current_device();
    if (!ds) return TVH_ERR_DEVICE;
    // Split N = N1 * N2 and tiles, measured on MI355X over 2^13..2^24 rows and 4 to
    // 1000 columns.  N1 = 2^8, two passes, wherever N2 fits in 2^12 (2^16 x 379: 186
    // us, N1 = 2^7 220; 2^20 x 379: 3.89 ms, N1 = 2^9 4.34, 2^10 4.46).  Column tiles
    // of 2^13 elements (2^12 while those are fewer than four blocks a CU: 2^14 x 60 21
    // us, 25 in 2^13 tiles, 35 in 2^14; 2^14 beyond 2^22 rows, where 2^13 would hold 4
    // or 2 columns' transforms, 32 or 16 B segments).  The row step stores a block's
    // rows transposed, in runs as long as its row count: the shortest tile that holds
    // 8 rows.  Blocks of one column go to one XCD, whose L2 completes their cache
    // lines (column_on_xcd).  Shorter runs can be faster by themselves and slow down
    // the kernel that reads them next: evaluating a coset of 2^19 x 379 takes 2.17 ms
    // in column order, 2.07 as here, 1.97 in 2^13 tiles; with the row hashes after it
    // 4.54, 4.46 and 4.66.
    // Up to 2^12 rows the row step alone (2^10 x 100: 9.4 us in 2^12 tiles, 19.6 in
    // 2^14), the scaled form too.
    const u32 a = logN <= 12 ? 0 : logN <= 14 ? logN / 2 : logN <= 20 ? 8 : logN - 12;
    const u32 b = logN - a;
    const u32 col_lt = logN > 22 ? LOG_TILE : (cols << logN) < (1ull << 23) && a < 10 ? 12 : 13;
    const u32 row_lt = ntt_row_tile(b, a == 0);
    NttScaleDev S{};
    if (scale) {  // p1[n1] = base^(N2 n1), p2[n2] = base^n2
        if (!scale->tables) return set_error(TVH_ERR_INVALID_ARG, "no tables for the NTT scaling");
        S = NttScaleDev{scale->tables, scale->tables + (1ull << a), scale->rand, scale->k,
                        scale->delta};
        int rc;
        if ((a && (rc = launch_pow_table(scale->tables, gl::pow(scale->base, 1ull << b), 1ull << a, st))) ||
            (rc = launch_pow_table(scale->tables + (1ull << a), scale->base, 1ull << b, st)))
            return rc;
    }
    // step 1 writes each group of columns to the scratch, step 2 writes it back (the
    // row step alone needs no scratch, and asks for it all the same)
    u64 group = scratch_elems / n;
    if (!scratch || group == 0)
        return set_error(TVH_ERR_INVALID_ARG, "NTT scratch of %llu elements < n = %llu",
                         (unsigned long long)scratch_elems, (unsigned long long)n);
    if (group > cols) group = cols;
    u64 ninv = gl::inv(n % gl::P);
    int rc;
    for (u64 c0 = 0; c0 < cols; c0 += group) {
        u64 g = cols - c0 < group ? cols - c0 : group;
        const u64* sg = src + c0 * n;  // step 1 reads the group from src
        u64* d = dst + c0 * n;         // step 2 writes it to dst
        NttScaleDev Sg = S;
        if (Sg.rand) Sg.rand += c0 * Sg.k;  // the group's first column
        if (a) {
            const LaunchShape s1 = launch_shape(col_lt, a, b, g, false);
            Step1Args A{sg, n, scratch, n, logN, a, 1u, inverse ? ninv : 1, s1.blocks};
            rc = scale ? launch_k_step1_scaled(col_lt, s1, st, A, Sg, ds->roots)
                       : launch_k_step1(inverse, col_lt, s1, st, A, ds->roots);
            if (rc) return rc;
        }
        const LaunchShape s2 = launch_shape(row_lt, b, a, g, a == 0);
        rc = scale && !a ? launch_k_ntt_cols_scaled(s2, st, sg, d, logN, g, Sg, ds->roots)
                         : launch_k_ntt_step2(inverse, s2, st, a ? scratch : sg, d, logN, a, g, ninv, ds->roots);
        if (rc) return rc;
    }
    return TVH_OK;
}

// ---------------------------------------------------------------- DFT matrices
u32 dft_matrices_words() { return 4 * kDftWords; }

// Coefficient 2^x (0 <= x < 192, 2^96 = -1) of byte `b` of an element's low word
// in byte place pos < 12 (2^(8 pos), 2^96 = -1): +-2^(x mod 8) or 0.
static int unfolded(u32 x, u32 b, u32 pos) {
    u32 e = (x + 8 * b) % 192;
    const int sign = e >= 96 ? -1 : 1;
    if (e >= 96) e -= 96;
    return e / 8 == pos ? sign * (1 << (e % 8)) : 0;
}

void build_dft_matrices(bool inverse, u32* out) {
    typedef unsigned __int128 u128;
    for (u32 r = 1; r <= 4; r++, out += kDftWords) {
        const u32 sub = (1u << (4 - r)) - 1;
        for (u32 i = 0; i < kDftWords; i++) out[i] = 0;
        // output k from input j: w_(2^r)^(digit product) when their low bits agree
        auto power = [&](u32 k, u32 j) -> u32 {
            const u32 kj = ((k >> (4 - r)) * (j >> (4 - r))) % (1u << r);
            const u32 x = (39 * (64 >> r) * kj) % 192;  // w_64 = 2^39
            return inverse ? (192 - x) % 192 : x;
        };
        for (u32 k = 0; k < 16; k++) {
            // what the products leave out of output k: sum over j, b of
            // coefficient * 128 per byte, and of Q_s for -x = ~x + 1
            u64 total = 0, q_sum[4] = {0, 0, 0, 0};
            for (u32 j = 0; j < 16; j++) {
                if ((k & sub) != (j & sub)) continue;
                const u32 x = power(k, j);
                total = gl::add(total, gl::mul(gl::pow2_mod_p(x), kSignBits * 0x100000001ull));
                // lane 16 (j mod 4) + row of k (k = 4 (row mod 4) + row / 4), register j / 4
                const u32 at = (16 * (j & 3) + 4 * (k & 3) + (k >> 2)) * 4 + (j >> 2);
                for (u32 s = 0; s < 4; s++)
                    for (u32 b = 0; b < 4; b++) {
                        const int u0 = unfolded(x, b, s), u4 = unfolded(x, b, s + 4),
                                  u8 = unfolded(x, b, s + 8);
                        const int p = u0 - u8, q = u4 + u8, pq = u0 + u4;
                        out[s * 256 + at] |= (u32)(p & 255) << (8 * b);
                        out[(4 + s) * 256 + at] |= (u32)(q & 255) << (8 * b);
                        out[(8 + s) * 256 + at] |= (u32)(pq & 255) << (8 * b);
                        q_sum[s] = gl::add(q_sum[s], q < 0 ? gl::P - (u64)-q : (u64)q);
                    }
            }
            for (u32 s = 0; s < 4; s++) total = gl::add(total, gl::mul(q_sum[s], 1ull << (8 * s)));
            const u128 bias = (u128)kDftBias * (1 + (1ull << 16) + (1ull << 32) + (1ull << 48));
            const u64 c = gl::sub(total, (u64)(bias % gl::P));
            for (u32 q = 0; q < 4; q++)  // start[q][g = k mod 4][v = k / 4]
                out[kDftStarts + (q * 4 + (k & 3)) * 4 + (k >> 2)] =
                    kDftBias + (u32)((c >> (16 * q)) & 0xFFFF);
        }
    }
}

int set_lds_attribute(const std::vector<const void*>& kernels, int bytes) {
    for (const void* f : kernels)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
            return set_error(TVH_ERR_DEVICE, "LDS attribute");
    return TVH_OK;
}

int ntt_set_attributes() {
    const int bytes = 150 * 1024;
    int rc;
    if ((rc = set_attributes_step1(bytes)) || (rc = set_attributes_step2(bytes)) ||
        (rc = set_attributes_rows(bytes)) || (rc = set_attributes_step3(bytes)))
        return rc;
    return TVH_OK;
}

int launch_xfe_interleave(const u64* src, u64* dst, u64 cols, u64 len, bool to_limb_major,
                          hipStream_t st) {
    u64 total = cols * len * 3;
    if (!total) return TVH_OK;
    hipLaunchKernelGGL(k_xfe_relayout, dim3((u32)((total + 255) / 256)), dim3(256), 0, st, src,
                       dst, cols, len, (int)to_limb_major);
    return check_launch();
}

}  // namespace tvh
