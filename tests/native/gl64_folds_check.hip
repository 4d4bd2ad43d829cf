// Device check of the forms that set the unlikely borrow or carry aside
// (triton-vm-prover_amd/csrc/gl64.hpp: fold128_rare, mul_rare, mul_n, canon_n,
// to_mont_rare, join_half, join_rare), in the widths the kernels use, against
// unsigned __int128 arithmetic on the host.  Random operands take the borrow once
// in 2^32, so most of the operands here are made to: powers of two (the product's
// low half is zero), folds at the border of the carry, words of zeros and ones.
// Lanes and values that take it stand beside others that don't, in one wave; which
// of them are reported is checked as well as the results.
#include "gl64.hpp"

#include <cstdio>
#include <random>
#include <vector>

typedef unsigned __int128 u128;
using gl::u32;
using gl::u64;

constexpr int W = 4;  // operands a thread: a[4 i + v], b[4 i + v]

enum Op {
    OP_FOLD, OP_MUL1, OP_MUL2, OP_MUL3, OP_MUL4, OP_MUL1_JOINT, OP_MUL2_JOINT, OP_MUL3_JOINT, OP_MUL_N1,
    OP_MUL_N4, OP_MUL_N4_DIVERGENT, OP_CANON4, OP_TO_MONT3, OP_JOIN, OP_COUNT
};
static const char* kNames[OP_COUNT] = {"fold128_rare", "mul_rare<1>", "mul_rare<2>", "mul_rare<3>", "mul_rare<4>",
                                       "mul_rare<1> joint", "mul_rare<2> joint", "mul_rare<3> joint", "mul_n<1>",
                                       "mul_n<4>", "mul_n<4> in a branch", "canon_n<4>", "to_mont_rare<3>",
                                       "join"};

// r: result, mask of its own: with the reported values lowered by EPS
template <int N>
__device__ void mul_own(const u64* a, const u64* b, u64* r, u32* rep) {
    u64 x[N], y[N], z[N];
    gl::mask bad[N];
    for (int v = 0; v < N; v++) {
        x[v] = a[v];
        y[v] = b[v];
    }
    gl::mul_rare(z, x, y, bad);
    for (int v = 0; v < N; v++) {
        rep[v] = gl::in_mask(bad[v]);
        r[v] = rep[v] ? z[v] - gl::EPS : z[v];
    }
}
// one mask for all: a reported lane is done again
template <int N>
__device__ void mul_joint(const u64* a, const u64* b, u64* r, u32* rep) {
    u64 x[N], y[N], z[N];
    gl::mask bad = 0;
    for (int v = 0; v < N; v++) {
        x[v] = a[v];
        y[v] = b[v];
    }
    gl::mul_rare(z, x, y, bad);
    const bool again = gl::in_mask(bad);
    for (int v = 0; v < N; v++) {
        rep[v] = again;
        r[v] = again ? gl::mul_lazy(x[v], y[v]) : z[v];
    }
}
template <int N>
__device__ void mul_whole(const u64* a, const u64* b, u64* r) {
    u64 x[N], y[N], z[N];
    for (int v = 0; v < N; v++) {
        x[v] = a[v];
        y[v] = b[v];
    }
    gl::mul_n(z, x, y);
    for (int v = 0; v < N; v++) r[v] = z[v];
}

__global__ void k_ops(int op, const u64* __restrict__ a0, const u64* __restrict__ b0, u64* __restrict__ out,
                      u32* __restrict__ report, u32 n) {
    const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u64 a[W], b[W], r[W] = {0, 0, 0, 0};
    u32 rep[W] = {0, 0, 0, 0};
    for (int v = 0; v < W; v++) {
        a[v] = a0[W * i + v];
        b[v] = b0[W * i + v];
    }
    const gl::JoinConsts J = gl::join_consts();
    switch (op) {
        case OP_FOLD: {  // a + b * 2^64
            u32 h0[W], h1[W];
            gl::mask bad[W];
            for (int v = 0; v < W; v++) {
                h0[v] = (u32)b[v];
                h1[v] = (u32)(b[v] >> 32);
            }
            gl::fold128_rare(r, a, h0, h1, bad);
            for (int v = 0; v < W; v++) {
                rep[v] = gl::in_mask(bad[v]);
                if (rep[v]) r[v] -= gl::EPS;
            }
            break;
        }
        case OP_MUL1: mul_own<1>(a, b, r, rep); break;
        case OP_MUL2: mul_own<2>(a, b, r, rep); break;
        case OP_MUL3: mul_own<3>(a, b, r, rep); break;
        case OP_MUL4: mul_own<4>(a, b, r, rep); break;
        case OP_MUL1_JOINT: mul_joint<1>(a, b, r, rep); break;
        case OP_MUL2_JOINT: mul_joint<2>(a, b, r, rep); break;
        case OP_MUL3_JOINT: mul_joint<3>(a, b, r, rep); break;
        case OP_MUL_N1: mul_whole<1>(a, b, r); break;
        case OP_MUL_N4: mul_whole<4>(a, b, r); break;
        case OP_MUL_N4_DIVERGENT:
            if (a[0] & 1) mul_whole<4>(a, b, r);
            else mul_whole<4>(b, a, r);
            break;
        case OP_CANON4:
            for (int v = 0; v < W; v++) r[v] = a[v];
            gl::canon_n(r);
            break;
        case OP_TO_MONT3: {
            u64 x[3] = {a[0], a[1], a[2]}, y[3];
            gl::mask bad = 0;
            gl::to_mont_rare(y, x, bad);
            for (int v = 0; v < 3; v++) {
                rep[v] = gl::in_mask(bad);
                r[v] = rep[v] ? gl::to_mont(x[v]) : y[v];
            }
            break;
        }
        case OP_JOIN: {
            // byte places d[t] of 256^t: the pairs d[2s] + 256 d[2s + 1] are the 31-bit
            // numbers below, split with a negative first place in every other lane
            u32 d[8];
            const u32 pair[4] = {(u32)a[0] >> 1, (u32)a[1] >> 1, (u32)a[2] >> 1, (u32)a[3] >> 1};
            for (int s = 0; s < 4; s++) {
                const u32 low = i & 1 ? (pair[s] & 255) - 256 : pair[s] & 255;
                d[2 * s] = low;
                d[2 * s + 1] = (pair[s] - low) >> 8;
            }
            bool carry;
            const u64 x = gl::join_rare(J, gl::join_half(J, d[0], d[1], d[2], d[3]),
                                        gl::join_half(J, d[4], d[5], d[6], d[7]), carry);
            rep[0] = carry;
            r[0] = carry ? x + gl::EPS : x;
            break;
        }
        default: break;
    }
    for (int v = 0; v < W; v++) {
        out[W * i + v] = r[v];
        report[W * i + v] = rep[v];
    }
}

static u64 pmod(u128 v) { return (u64)(v % gl::P); }
// whether the fold of l + h * 2^64 takes the borrow that is set aside
static bool borrows(u64 l, u64 h) {
    const u128 u = (u128)l + (u128)(u32)h * gl::EPS;
    return u >> 64 == 0 && (u64)u < h >> 32;
}

int main() {
    const u32 n = 200001;  // a last wave in part
    const u64 P = gl::P;
    const u64 edge[] = {0, 1, 2, P - 1, P - 2, P, P + 1, 0xFFFFFFFFull, 0x100000000ull, 0x100000001ull,
                        P - 0x100000000ull, 0xFFFFFFFFFFFFFFFFull, 0xFFFFFFFF00000000ull,
                        0xFFFFFFFEFFFFFFFFull, 0x7FFFFFFFFFFFFFFFull};
    std::mt19937_64 rng(5);
    auto pick = [&](u32 power_share) -> u64 {
        if (rng() % 8 < power_share) return 1ull << (rng() & 63);
        const u32 k = (u32)(rng() % 4);
        return k == 0 ? edge[rng() % (sizeof(edge) / sizeof(edge[0]))] : rng();
    };
    std::vector<u64> a(W * n), b(W * n), out(W * n);
    std::vector<u32> rep(W * n);
    u64 *da = nullptr, *db = nullptr, *dout = nullptr;
    u32* drep = nullptr;
    if (hipMalloc(&da, W * n * 8ull) != hipSuccess || hipMalloc(&db, W * n * 8ull) != hipSuccess ||
        hipMalloc(&dout, W * n * 8ull) != hipSuccess || hipMalloc(&drep, W * n * 4ull) != hipSuccess) {
        printf("no device memory\n");
        return 2;
    }
    int total = 0;
    for (int op = 0; op < OP_COUNT; op++) {
        for (u32 j = 0; j < W * n; j++) {
            const u32 i = j / W;
            // waves without the borrow, with it in few lanes, and in most of them
            const u32 share = (i >> 6) % 3 == 0 ? 0 : (i >> 6) % 3 == 1 ? 2 : 6;
            a[j] = pick(share);
            b[j] = pick(share);
            if (op == OP_FOLD && rng() % 2) {  // round the carry out and the borrow
                const u32 h0 = (u32)(rng() % 3 ? rng() : rng() % 4), h1 = (u32)(rng() % 2 ? rng() : rng() % 4);
                b[j] = gl::mk64(h0, h1);
                a[j] = 0 - (u64)h0 * gl::EPS + rng() % 5 - 2 + (rng() % 2 ? h1 : 0);
            }
            if (op == OP_TO_MONT3 && rng() % 3 == 0) a[j] = gl::mk64((u32)(rng() % 3), (u32)rng());
            if (op == OP_JOIN) {  // places 4.. (the high half) at the border of the carry
                a[j] = rng() % 3 ? rng() : 0xFFFFFFFFull - rng() % 4;
                if (rng() % 4 == 0) a[j] = rng() % 4;
            }
        }
        if (op == OP_JOIN)
            for (u32 i = 0; i < n; i += 2) {  // H0 = C + D 2^16 mod 2^32 of ones: C = 0xFFFF.., D = 0xFFFF
                a[W * i + 2] = ((u64)(rng() % 0x8000) << 17) | 0x1FFFEull | (rng() & 1);
                a[W * i + 3] = (u64)((0xFFFF - (a[W * i + 2] >> 17)) & 0xFFFF) << 1 | (rng() & 0x7FFE0000ull);
            }
        if (hipMemcpy(da, a.data(), W * n * 8ull, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(db, b.data(), W * n * 8ull, hipMemcpyHostToDevice) != hipSuccess) {
            printf("copy failed\n");
            return 2;
        }
        hipLaunchKernelGGL(k_ops, dim3((n + 255) / 256), dim3(256), 0, 0, op, da, db, dout, drep, n);
        if (hipMemcpy(out.data(), dout, W * n * 8ull, hipMemcpyDeviceToHost) != hipSuccess ||
            hipMemcpy(rep.data(), drep, W * n * 4ull, hipMemcpyDeviceToHost) != hipSuccess) {
            printf("kernel or copy failed\n");
            return 2;
        }
        int bad = 0;
        u32 taken = 0;
        for (u32 i = 0; i < n; i++) {
            const u64 *x = &a[W * i], *y = &b[W * i], *r = &out[W * i];
            const u32* p = &rep[W * i];
            bool ok = true;
            auto product = [&](int v) { return (u128)x[v] * y[v]; };
            auto low = [&](int v) { return borrows((u64)product(v), (u64)(product(v) >> 64)); };
            auto products = [&](int width, bool own, bool joint) {
                bool any = false;
                for (int v = 0; v < width; v++) any |= low(v);
                for (int v = 0; v < width; v++) {
                    ok &= r[v] % P == pmod(product(v));
                    if (own) ok &= p[v] == (u32)low(v);
                    if (joint) ok &= p[v] == (u32)any;
                }
                taken += any;
            };
            switch (op) {
                case OP_FOLD:
                    for (int v = 0; v < W; v++) {
                        ok &= r[v] % P == pmod(((u128)y[v] << 64) | x[v]) && p[v] == (u32)borrows(x[v], y[v]);
                        taken += p[v];
                    }
                    break;
                case OP_MUL1: products(1, true, false); break;
                case OP_MUL2: products(2, true, false); break;
                case OP_MUL3: products(3, true, false); break;
                case OP_MUL4: products(4, true, false); break;
                case OP_MUL1_JOINT: products(1, false, true); break;
                case OP_MUL2_JOINT: products(2, false, true); break;
                case OP_MUL3_JOINT: products(3, false, true); break;
                case OP_MUL_N1: products(1, false, false); break;
                case OP_MUL_N4:
                case OP_MUL_N4_DIVERGENT: products(4, false, false); break;
                case OP_CANON4:
                    for (int v = 0; v < W; v++) {
                        ok &= r[v] == x[v] % P;
                        taken += x[v] >= P;
                    }
                    break;
                case OP_TO_MONT3: {
                    bool any = false;
                    for (int v = 0; v < 3; v++) any |= (u32)x[v] == 0 && x[v] >> 32;
                    for (int v = 0; v < 3; v++) ok &= r[v] % P == pmod((u128)x[v] * gl::EPS) && p[v] == (u32)any;
                    taken += any;
                    break;
                }
                default: {
                    u64 q[4];
                    for (int s = 0; s < 4; s++) q[s] = (u32)x[s] >> 1;
                    const u64 L = q[0] + (q[1] << 16), H = q[2] + (q[3] << 16);
                    ok = r[0] % P == pmod((u128)L + ((u128)H << 32));
                    taken += p[0];
                }
            }
            if (!ok && bad++ < 2)
                printf("%s, thread %u: (%016llx %016llx %016llx %016llx), (%016llx %016llx %016llx %016llx) -> "
                       "%016llx %016llx %016llx %016llx, reported %u%u%u%u\n",
                       kNames[op], i, (unsigned long long)x[0], (unsigned long long)x[1], (unsigned long long)x[2],
                       (unsigned long long)x[3], (unsigned long long)y[0], (unsigned long long)y[1],
                       (unsigned long long)y[2], (unsigned long long)y[3], (unsigned long long)r[0],
                       (unsigned long long)r[1], (unsigned long long)r[2], (unsigned long long)r[3], p[0], p[1],
                       p[2], p[3]);
        }
        printf("%s: %u rare, %d wrong\n", kNames[op], taken, bad);
        if (taken < 1000) {
            printf("%s: the rare case is not exercised\n", kNames[op]);
            bad++;
        }
        total += bad;
    }
    (void)hipFree(da);
    (void)hipFree(db);
    (void)hipFree(dout);
    (void)hipFree(drep);
    printf("folds bad=%d\n", total);
    return total != 0;
}
