// ntt_small.hip -- one-pass NTTs of rows of 2^8 .. 2^12 points in registers
// (NttPlan::forward, rust/volta-pcs/src/ntt.rs:34-61, and its inverse).
//
// n = 256 N1, N1 = 2^B (B = 0 .. 4), j = j1 + N1 j2 + 16 N1 j3 and
// k = k3 + 16 k2 + 256 k1 (j1, k1 < N1, the others < 16), m = j1 + N1 j2:
//   stage A (thread m of its row): the 16-point DFT over j3, then w_n^(k3 m);
//   stage B (thread (j1, k3)): the DFT over j2, then w_n^(16 j1 k2);
//   stage C (thread (k3, x), k2 = p + P x, P = 16 / N1): P DFTs of N1 points over j1.
// Every root inside the DFTs is a power of two (shifts only); two general
// multiplies per element.  A workgroup of 256 threads holds 4,096 elements (P
// rows), 16 per thread, which cross LDS twice (34 KiB, four workgroups per CU).
// The LDS kernel it takes over from (ntt_row_lds) runs B / 2 + 4 radix-2^2 rounds
// through LDS with three general multiplies per four elements each.
// Bound by VALU issue on large batches from 2^9 points on (0.88-0.89 of the cycles; 4.84
// TB/s of loads and stores dense at 2^12), by HBM at 2^8 (0.72; 5.56 TB/s).
// Before (ntt_row_lds) and now, us, at 2^26 points: n = 2^8 321 / 193, 2^9 347 / 196,
// 2^10 392 / 200, 2^11 449 / 209, 2^12 485 / 222; with the last three quarters of each
// row zero 301 / 150, 322 / 167, 363 / 172, 405 / 182, 446 / 191.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "context.hpp"
#include "gl64.hpp"
#include "gl64_shift.hpp"
#include "kernels.hpp"

namespace vmx {
namespace ns {

constexpr int THREADS = 256;
constexpr int E_W16 = 156;  // w_16 = 2^156

template <int B>
struct Shape {
    static constexpr int N1 = 1 << B;
    static constexpr int LOG_N = 8 + B;
    static constexpr int N = 256 * N1;
    static constexpr int M = 16 * N1;  // threads per row
    static constexpr int P = 16 / N1;  // rows per workgroup; stage-C DFTs per thread
    // First exchange: word (k3, m) of a row at k3 X1_PITCH + m; 17 N1 words apart, so
    // that 16 lanes (j1, k3) meet 16 banks.
    static constexpr int X1_PITCH = 17 * N1;
    static constexpr int X1_ROW = 16 * X1_PITCH;
    static constexpr int XBUF = P * X1_ROW;  // >= P N, the second exchange
    // Device table: T1[k3 M + m] = w_n^(k3 m), then T2[k2 N1 + j1] = w_n^(16 j1 k2).
    static constexpr int T1_WORDS = 16 * M;
    static constexpr int T2_WORDS = 16 * N1;
    static constexpr int TABLE_WORDS = T1_WORDS + T2_WORDS;
    // w_N1 as a power of two (w_2 = 2^96, w_4 = 2^48, w_8 = 2^120, w_16 = 2^156)
    static constexpr int E_WN1 = B == 1 ? 96 : B == 2 ? 48 : B == 3 ? 120 : 156;
};

constexpr uint64_t prefix_mask(int nz) {
    uint64_t m = 0;
    for (int j = 0; j < nz; ++j) m |= uint64_t{1} << gl::bitrev_c(j, 4);
    return m;
}

#if defined(__HIP_DEVICE_COMPILE__)
// A span of device memory at a uniform address: one 32-bit lane offset plus a
// scalar one per access; reads past its end give 0 and writes there are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t span(const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), static_cast<short>(0), static_cast<int>(bytes),
                                             0x00020000);
}
__device__ __forceinline__ uint64_t ld64(const __amdgpu_buffer_rsrc_t& r, uint32_t voff, uint32_t soff) {
    const auto t = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    return static_cast<uint64_t>(t[0]) | (static_cast<uint64_t>(t[1]) << 32);
}
#endif

// Sources: the elements m + M j3, j3 < NZ, of row g of the `live` rows from row0 on,
// into slot bitrev4(j3).  A group's rows are one span; what a lane reads past its own
// row is masked.
// SrcU64: x + row stride, len u64 then zeros; reversed (len = n), element (n - idx) mod n.
struct SrcU64 {
    const uint64_t* x;
    size_t stride;
    uint32_t len, rev_mask;  // n - 1 when reversed, else 0
    template <int M, int NZ>
    __device__ __forceinline__ void load(uint64_t* v, size_t row0, uint32_t live, uint32_t g, uint32_t m) const {
#if defined(__HIP_DEVICE_COMPILE__)
        const auto r = span(x + row0 * stride, ((live - 1) * stride + len) * 8);
        const uint32_t base = g * static_cast<uint32_t>(stride);
        uint64_t raw[NZ];
        gl::static_for<0, NZ>([&](auto j_) {
            constexpr uint32_t j = decltype(j_)::value * M;
            raw[decltype(j_)::value] = rev_mask ? ld64(r, (base + ((0u - m - j) & rev_mask)) * 8, 0) : ld64(r, (base + m) * 8, j * 8);
        });
        __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first use
        gl::static_for<0, NZ>([&](auto j_) {
            constexpr int j3 = decltype(j_)::value;
            v[gl::bitrev_c(j3, 4)] = m + M * j3 < len ? raw[j3] : 0;
        });
#endif
    }
};

// SrcMsg: lift(w) || pads || 0 (cols > 0; pads readable even when pad = 0).
struct SrcMsg {
    const int16_t* w;
    const uint64_t* pads;
    uint32_t cols, pad;
    template <int M, int NZ>
    __device__ __forceinline__ void load(uint64_t* v, size_t row0, uint32_t live, uint32_t g, uint32_t m) const {
#if defined(__HIP_DEVICE_COMPILE__)
        const auto rw = span(w + row0 * cols, size_t{live} * cols * 2), rp = span(pads + row0 * pad, size_t{live} * pad * 8);
        uint32_t h[NZ];
        uint64_t q[NZ];
        gl::static_for<0, NZ>([&](auto j_) {
            constexpr int j3 = decltype(j_)::value;
            const uint32_t idx = m + M * j3;
            h[j3] = __builtin_amdgcn_raw_buffer_load_b16(rw, (g * cols + m) * 2, M * j3 * 2, 0);
            q[j3] = ld64(rp, idx >= cols && idx - cols < pad ? (g * pad + idx - cols) * 8 : 0x7FFFFFF8u, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
        gl::static_for<0, NZ>([&](auto j_) {
            constexpr int j3 = decltype(j_)::value;
            // past the weights q is the pad, or 0 from past its span
            v[gl::bitrev_c(j3, 4)] =
                m + M * j3 < cols ? gl::from_i16(static_cast<int16_t>(static_cast<uint16_t>(h[j3]))) : q[j3];
        });
#endif
    }
};

// NZ: only j3 < NZ can be nonzero.  scale: 1, or the inverse's n^-1 (SCALED).
template <int B, int NZ, class Src, bool SCALED>
__global__ __launch_bounds__(THREADS, 4) void small_rows(Src src, size_t rows, const uint64_t* __restrict__ tab,
                                                         uint64_t* __restrict__ out, uint64_t scale) {
#if defined(__HIP_DEVICE_COMPILE__)
    using S = Shape<B>;
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    __shared__ uint64_t x[S::XBUF], t2[S::T2_WORDS];
    const uint32_t t = threadIdx.x;
    const uint32_t g = t / S::M, m = t % S::M;             // row of the workgroup, thread of the row
    const uint32_t j1 = m % S::N1, k3b = m / S::N1;        // stage B
    const uint32_t k3c = m & 15, xc = m >> 4;              // stage C
    if (t < S::T2_WORDS) t2[t] = tab[S::T1_WORDS + t];
    const auto tr = span(tab, size_t{S::T1_WORDS} * 8);
    const size_t groups = (rows + S::P - 1) / S::P;
    for (size_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const size_t row0 = grp * S::P;
        const uint32_t live = static_cast<uint32_t>(min(rows - row0, static_cast<size_t>(S::P)));
        uint64_t v[16], tw[16];
        gl::static_for<0, 16>([&](auto i_) { v[decltype(i_)::value] = 0; });
        src.template load<S::M, NZ>(v, row0, live, g, m);
        __builtin_amdgcn_sched_barrier(0);  // the twiddles load behind the DFT, not beside the inputs
        gl::static_for<1, 16>([&](auto k_) { tw[decltype(k_)::value] = ld64(tr, m * 8, decltype(k_)::value * S::M * 8); });
        gl::dit_pow2_sparse<4, E_W16, prefix_mask(NZ), 2, 32, 1>(v);  // only A[0] meets no twiddle
        uint64_t* x1 = x + g * S::X1_ROW;
        gl::static_for<0, 16>([&](auto k_) {
            constexpr int k3 = decltype(k_)::value;
            x1[k3 * S::X1_PITCH + m] = k3 ? gl::mul32x4(v[k3], tw[k3]) : v[0];
        });
        __syncthreads();
        gl::static_for<0, 16>([&](auto j_) {
            constexpr int j2 = decltype(j_)::value;
            v[gl::bitrev_c(j2, 4)] = x1[k3b * S::X1_PITCH + j1 + S::N1 * j2];
        });
        if constexpr (B == 0) {
            gl::dit_pow2<4, E_W16>(v);
        } else {
            gl::dit_pow2<4, E_W16, 2, 1>(v);  // only B[0] meets no twiddle
            __syncthreads();                  // the first exchange is read
            // word (k2, j1, k3) of a row, k3 rotated by P j1 within its 16 words: 16 lanes
            // (j1, k3) of a write and 16 lanes k3 of a read meet 16 banks
            uint64_t* x2 = x + g * S::N;
            gl::static_for<0, 16>([&](auto k_) {
                constexpr int k2 = decltype(k_)::value;
                x2[(k2 * S::N1 + j1) * 16 + ((k3b + S::P * j1) & 15)] =
                    k2 ? gl::mul32x4(v[k2], t2[k2 * S::N1 + j1]) : v[0];
            });
            __syncthreads();
            gl::static_for<0, S::P>([&](auto p_) {
                constexpr int p = decltype(p_)::value;
                uint64_t u[S::N1];
                gl::static_for<0, S::N1>([&](auto j_) {
                    constexpr int j = decltype(j_)::value;
                    u[gl::bitrev_c(j, B)] = x2[((p + S::P * xc) * S::N1 + j) * 16 + ((k3c + S::P * j) & 15)];
                });
                gl::dit_pow2<B, S::E_WN1>(u);
                gl::static_for<0, S::N1>([&](auto k_) { v[p + S::P * decltype(k_)::value] = u[decltype(k_)::value]; });
            });
        }
        // B > 0: X[k3 + 16 (p + P x) + 256 k1] in v[p + P k1]; B = 0: X[k3 + 16 k2] in v[k2];
        // rows past the last are past the span's end
        const auto o = span(out + row0 * S::N, size_t{live} * S::N * 8);
        const uint32_t off = (g * S::N + (B == 0 ? k3b : k3c + 16 * S::P * xc)) * 8;
        gl::static_for<0, 16>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            constexpr int k = B == 0 ? 16 * i : 16 * (i % S::P) + 256 * (i / S::P);
            const uint64_t y = SCALED ? gl::mul32x4(v[i], scale) : v[i];
            __builtin_amdgcn_raw_buffer_store_b64(v2u{static_cast<uint32_t>(y), static_cast<uint32_t>(y >> 32)}, o, off,
                                                  k * 8, 0);
        });
        __syncthreads();  // the next group rewrites the buffer
    }
#endif
}

template <int B>
__global__ void build_table(const uint64_t* __restrict__ fwd, uint64_t* __restrict__ tab) {
    using S = Shape<B>;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= S::TABLE_WORDS) return;
    const int e = idx < S::T1_WORDS ? (idx / S::M) * (idx % S::M)
                                    : 16 * ((idx - S::T1_WORDS) / S::N1) * ((idx - S::T1_WORDS) % S::N1);
    tab[idx] = e < S::N / 2 ? fwd[e] : gl::neg(fwd[e - S::N / 2]);
}

namespace {

template <int B>
int build(Context* c, TwiddleSet* t) {
    hipLaunchKernelGGL(build_table<B>, dim3((Shape<B>::TABLE_WORDS + 255) / 256), dim3(256), 0, c->stream,
                       static_cast<const uint64_t*>(t->fwd), t->grid);
    VMX_HIP(c, hipGetLastError());
    return 0;
}

template <int B, int NZ, class Src, bool SCALED>
int launch(Context* c, const Src& src, size_t rows, uint64_t* out, const uint64_t* tab, uint64_t scale) {
    const size_t groups = (rows + Shape<B>::P - 1) / Shape<B>::P;
    hipLaunchKernelGGL((small_rows<B, NZ, Src, SCALED>), dim3(static_cast<unsigned>(std::min<size_t>(groups, 1u << 20))),
                       dim3(THREADS), 0, c->stream, src, rows, tab, out, scale);
    VMX_HIP(c, hipGetLastError());
    return 0;
}

// The kernel whose stage A reads the fewest of its 16 inputs covering `extent`.
template <int B, class Src>
int run(Context* c, const Src& src, size_t extent, size_t rows, uint64_t* out, TwiddleSet* t, uint64_t scale) {
    if (ensure_grid_twiddles(c, t, size_t{Shape<B>::TABLE_WORDS} * sizeof(uint64_t), build<B>)) return -1;
    if (rows == 0) return 0;
    const size_t nz = (extent + Shape<B>::M - 1) / Shape<B>::M;
    if (scale != 1) {
        if constexpr (std::is_same<Src, SrcU64>::value) return launch<B, 16, Src, true>(c, src, rows, out, t->grid, scale);
        return fail_msg(c, "scaled message rows");
    }
    if (nz <= 4) return launch<B, 4, Src, false>(c, src, rows, out, t->grid, 1);
    if (nz <= 6) return launch<B, 6, Src, false>(c, src, rows, out, t->grid, 1);
    if (nz <= 8) return launch<B, 8, Src, false>(c, src, rows, out, t->grid, 1);
    return launch<B, 16, Src, false>(c, src, rows, out, t->grid, 1);
}

template <class Src>
int dispatch(Context* c, const Src& src, size_t extent, size_t rows, size_t n, uint64_t* out, TwiddleSet* t,
             uint64_t scale) {
    switch (n) {
        case 256: return run<0>(c, src, extent, rows, out, t, scale);
        case 512: return run<1>(c, src, extent, rows, out, t, scale);
        case 1024: return run<2>(c, src, extent, rows, out, t, scale);
        case 2048: return run<3>(c, src, extent, rows, out, t, scale);
        case 4096: return run<4>(c, src, extent, rows, out, t, scale);
        default: return 1;
    }
}

}  // namespace
// From here up a batch fills the chip.  Below 2^12 points ntt_row_lds has a shorter
// chain for smaller batches (more threads per element): before and now, us, dense and
// three quarters zero, at 2^19 points 2^8 6.2 / 6.8 and 6.2 / 5.8, 2^10 7.2 / 8.6 and
// 7.2 / 7.6, 2^11 8.2 / 8.9 and 8.4 / 8.0; at 2^20 2^8 9.3 / 7.4, 2^9 10.1 / 8.9,
// 2^10 10.8 / 9.2, 2^11 11.9 / 9.5.  At 2^12 one row alone is already faster
// (13.0 / 8.7; 13.2 / 7.9).
bool pays(size_t rows, size_t n) { return n == 4096 || rows >= (size_t{1} << 20) / n; }

}  // namespace ns

int ntt_small_u64_rows(Context* c, const uint64_t* in, size_t stride, size_t len, size_t rows, size_t n, uint64_t* out,
                       TwiddleSet* t, bool inverse) {
    if (n < 256 || n > 4096 || !ns::pays(rows, n) || len > n || (inverse && len != n) || !t->fwd) return 1;
    if (!t->grid && c->coarse_active) return 1;  // tables may not grow inside a coarse scope
    if (stride > (1u << 20)) return 1;  // a group's rows are one 32-bit span
    const ns::SrcU64 s{len ? in : t->fwd, len ? stride : 0, static_cast<uint32_t>(len),
                       inverse ? static_cast<uint32_t>(n - 1) : 0u};
    return ns::dispatch(c, s, len, rows, n, out, t, inverse ? gl::inv_host(gl::canon(n)) : 1) ? -1 : 0;
}

int ntt_small_msg_rows(Context* c, const int16_t* w, const uint64_t* pads, size_t cols, size_t pad, size_t rows, size_t n,
                       uint64_t* out, TwiddleSet* t) {
    if (n < 256 || n > 4096 || !ns::pays(rows, n) || cols == 0 || cols + pad > n || !t->fwd) return 1;
    if (!t->grid && c->coarse_active) return 1;
    const ns::SrcMsg s{w, pad ? pads : t->fwd, static_cast<uint32_t>(cols), static_cast<uint32_t>(pad)};
    return ns::dispatch(c, s, cols + pad, rows, n, out, t, 1) ? -1 : 0;
}

}  // namespace vmx
