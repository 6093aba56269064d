// KV page maintenance: token-major <-> page conversion, and the fused prepare
// step (RMSNorm + RoPE of q and k, fp16 append of k and v into the pages).
#include "kernels.hpp"
#include "prep.hpp"

#include <cmath>

namespace rs {
namespace {

// Token-major rows [count][kv_heads][D] (token first+t at row t) <-> pages.
// A block moves one (page, KV head) of K or of V, K's and V's blocks in one
// launch, KV heads fastest, so that neighbouring blocks share the 32 rows'
// lines.  The move is bound by HBM (read once, written once), so every thread
// moves 16-byte pieces of the pages:
//   K: a piece is 8 dims of one token on both sides.  Pages are accessed
//      contiguously, rows in 64-byte parts of 16 rows per wave instruction.
//   V: a piece is 8 tokens of one dim, so a thread takes VD dims of the 8
//      tokens of one key group (8 row accesses of 4 or 8 bytes, a wave
//      covering whole row parts) and transposes them in registers.
// Only tokens first .. first+count-1 are touched: other tokens' rows do not
// exist, and their page slots keep their values (of a V piece that holds such
// a token, four valid tokens are written at once, others value by value; a
// loop of loads and stores over that page took one block up to 31 rounds: 31
// tokens of 4 x 256 dims into pages 8.2 -> 3.9 us).  Buffers that are not
// 16-byte aligned move value by value throughout, four values in flight per
// thread, in eight blocks per page and head where the pages alone are few.
// Rows taken into pages are loaded non-temporally (each is read once: 39.5 ->
// 36.7 us); pages are loaded with the default policy (straight after their
// writes they are partly cached: 29.1 against 40.4 us non-temporally).
// 20,001 tokens of 4 x 256 dims (82 MB read and written each way), rocprof
// medians: 36.7 us into pages and 29.1 us back, 4.5 and 5.6 TB/s of read +
// write; four launches that moved value by value took 45-60 us each (207 us).
struct ConvertArgs {
    unsigned short *pages[2], *rows[2];   // K, V (both NULL on a side that is not moved)
    size_t head_stride;
    int kv_heads, first, count, page0, n_pages;
    bool whole;                           // 16-byte aligned buffers
    int parts;                            // blocks per (page, KV head, K or V): 1 or, unaligned, 8
};
constexpr int kConvertThreads = 256;
// Unaligned buffers: eight blocks per (page, KV head, K or V) where these are
// fewer than the CUs (1000 tokens of 8 x 128 dims, 512 pages and heads: 9.9 us in
// eight blocks each).
constexpr int kConvertBlocks = 256;

template <int D, bool TO_PAGES>
__global__ __launch_bounds__(kConvertThreads)
void convert_pages(ConvertArgs a) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int PAGE = 32 * D;
    const int sides = (a.pages[0] ? 1 : 0) + (a.pages[1] ? 1 : 0);
    const size_t blocks = (size_t)a.n_pages * a.kv_heads * sides * a.parts;
    const size_t row_stride = (size_t)a.kv_heads * D;
    for (size_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        const size_t ph = b / a.parts;
        const int h = (int)(ph % a.kv_heads);
        const size_t ps = ph / a.kv_heads;
        const int side = sides == 2 ? (int)(ps % 2) : a.pages[0] ? 0 : 1;
        const int page = a.page0 + (int)(sides == 2 ? ps / 2 : ps);
        unsigned short *pg = a.pages[side] + (size_t)h * a.head_stride + (size_t)page * PAGE;
        // Row of the page's token p: rows + p * row_stride (signed: the first
        // page may start before `first`).
        unsigned short *rows = a.rows[side] + ((long long)page * 32 - a.first) * (long long)row_stride + (size_t)h * D;
        const int lo = max(a.first - page * 32, 0);                          // valid tokens of the page: lo .. hi-1
        const int hi = (int)min((long long)a.first + a.count - (long long)page * 32, 32LL);
        if (!a.whole) {
            // Value by value, kBatch in flight per thread (pages and rows may
            // alias as far as the compiler knows, so it would wait for each).
            constexpr int kBatch = 4;
            const int p0 = (int)(b % a.parts) * (32 / a.parts), end = min(hi, p0 + 32 / a.parts) * D;
            for (int e0 = max(lo, p0) * D + threadIdx.x; e0 < end; e0 += kBatch * kConvertThreads) {
                unsigned short v[kBatch];
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int e = min(e0 + i * kConvertThreads, end - 1), p = e / D, d = e % D;
                    v[i] = TO_PAGES ? rows[p * row_stride + d]
                                    : pg[side ? v_page_offset(p, d, D) : k_page_offset(p, d, D)];
                }
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int e = e0 + i * kConvertThreads, p = e / D, d = e % D;
                    if (e >= end) break;
                    if (TO_PAGES) pg[side ? v_page_offset(p, d, D) : k_page_offset(p, d, D)] = v[i];
                    else rows[p * row_stride + d] = v[i];
                }
            }
        } else if (side == 0) {
            constexpr int PER = PAGE / 8 / kConvertThreads;
            u32x4 v[PER];
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int c = threadIdx.x + i * kConvertThreads;   // piece of the page
                const int p = c / (2 * D) * 16 + c % 16, d = c / 16 % (D / 8) * 8;
                if (p < lo || p >= hi) continue;
                v[i] = TO_PAGES ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(rows + p * row_stride + d))
                                : *reinterpret_cast<const u32x4 *>(pg + c * 8);
            }
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int c = threadIdx.x + i * kConvertThreads;
                const int p = c / (2 * D) * 16 + c % 16, d = c / 16 % (D / 8) * 8;
                if (p < lo || p >= hi) continue;
                if (TO_PAGES) *reinterpret_cast<u32x4 *>(pg + c * 8) = v[i];
                else *reinterpret_cast<u32x4 *>(rows + p * row_stride + d) = v[i];
            }
        } else {
            constexpr int VD = PAGE / 8 / kConvertThreads;   // dims per thread (4 or 2): D / VD threads per key group
            typedef unsigned short VP __attribute__((ext_vector_type(VD)));
            typedef unsigned short V8 __attribute__((ext_vector_type(8)));
            const int g = threadIdx.x / (D / VD), d = threadIdx.x % (D / VD) * VD;
            unsigned short *slots = pg + d / 16 * 512 + g * 128 + d % 16 * 8;
            VP x[8];
            V8 s[VD];
            if constexpr (!TO_PAGES) {
#pragma unroll
                for (int k = 0; k < VD; ++k) s[k] = *reinterpret_cast<const V8 *>(slots + k * 8);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int p = j / 4 * 16 + g * 4 + j % 4;   // slot j's token
                VP *row = reinterpret_cast<VP *>(rows + (TO_PAGES ? min(max(p, lo), hi - 1) : p) * row_stride + d);
                if constexpr (TO_PAGES) {
                    x[j] = __builtin_nontemporal_load(row);
                } else {
#pragma unroll
                    for (int k = 0; k < VD; ++k) x[j][k] = s[k][j];
                    if (p >= lo && p < hi) *row = x[j];
                }
            }
            if constexpr (TO_PAGES) {
                if (hi - lo == 32) {
#pragma unroll
                    for (int k = 0; k < VD; ++k) {
#pragma unroll
                        for (int j = 0; j < 8; ++j) s[k][j] = x[j][k];
                        *reinterpret_cast<V8 *>(slots + k * 8) = s[k];
                    }
                } else {
                    // Tokens outside lo .. hi-1 keep their slots, so what is
                    // not theirs is not written: four tokens at once where all
                    // of them are valid, else value by value.
                    typedef unsigned short V4 __attribute__((ext_vector_type(4)));
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int p0 = half * 16 + g * 4;
                        const bool all = p0 >= lo && p0 + 4 <= hi;
#pragma unroll
                        for (int k = 0; k < VD; ++k) {
                            unsigned short *dst = slots + k * 8 + half * 4;
                            if (all) {
                                *reinterpret_cast<V4 *>(dst) = V4{x[half * 4][k], x[half * 4 + 1][k],
                                                                  x[half * 4 + 2][k], x[half * 4 + 3][k]};
                            } else {
#pragma unroll
                                for (int j = 0; j < 4; ++j)
                                    if (p0 + j >= lo && p0 + j < hi) dst[j] = x[half * 4 + j][k];
                            }
                        }
                    }
                }
            }
        }
    }
}

template <bool TO_PAGES>
void convert(void *k_pages, void *v_pages, const void *k_rows, const void *v_rows,
             int kv_heads, int head_dim, int capacity, int first, int count,
             hipStream_t stream) {
    if (!count) return;
    ConvertArgs a = {};
    auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    a.whole = true;
    auto add = [&](int side, void *pages, const void *rows) {
        if (!pages || !rows) return;
        a.pages[side] = static_cast<unsigned short *>(pages);
        a.rows[side] = const_cast<unsigned short *>(static_cast<const unsigned short *>(rows));
        a.whole = a.whole && aligned(pages) && aligned(rows);
    };
    add(0, k_pages, k_rows);
    add(1, v_pages, v_rows);
    a.head_stride = (size_t)capacity * head_dim;
    a.kv_heads = kv_heads;
    a.first = first;
    a.count = count;
    a.page0 = first / kPageTokens;
    a.n_pages = (int)(((long long)first + count + kPageTokens - 1) / kPageTokens) - a.page0;
    const size_t blocks = (size_t)a.n_pages * kv_heads * ((a.pages[0] != nullptr) + (a.pages[1] != nullptr));
    a.parts = a.whole || blocks >= kConvertBlocks ? 1 : 8;
    const void *kernel = head_dim == 256 ? (const void *)&convert_pages<256, TO_PAGES>
                                         : (const void *)&convert_pages<128, TO_PAGES>;
    void *args[] = {&a};
    check(hipLaunchKernel(kernel, dim3((unsigned)std::min<size_t>(blocks * a.parts, 1u << 20)), dim3(kConvertThreads), args, 0,
                          stream));
}

// One wave per (head, token): heads 0..23 are query heads, 24..27 the KV
// heads (the reference's attn_prepare grid, src/kernels.cu:416-434), lane l
// owning dims l, 64+l, 128+l, 192+l.  Every global load is issued first and
// the RoPE angle computed while they are in flight.
__global__ __launch_bounds__(kWave)
void prepare_kernel(_Float16 *q_hilo, _Float16 *k_pages, _Float16 *v_pages, const float *q_gate,
                    const float *key, const float *value, const float *q_norm,
                    const float *k_norm, int position, size_t head_stride, float epsilon, int head0) {
    constexpr int D = kModelHeadDim, H = kModelQHeads, HKV = kModelKvHeads;
    static_assert(D == 4 * kWave, "four dims per lane");
    const int h = head0 + blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
    const bool is_q = h < H;
    const int kh = h - H;
    const float *src = is_q ? q_gate + ((size_t)t * H + h) * 2 * D : key + ((size_t)t * HKV + kh) * D;
    const float *gamma_src = is_q ? q_norm : k_norm;
    float x[1][4], gamma[4], v[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        x[0][w] = src[64 * w + lane];
        gamma[w] = gamma_src[64 * w + lane];
        v[w] = is_q ? 0.f : value[((size_t)t * HKV + kh) * D + 64 * w + lane];
    }
    float c[1] = {1.f}, s[1] = {0.f};
    if (lane < 32) rope_cos_sin(position + t, rope_freq(lane), c[0], s[0]);
    norm_rope_rows(x, gamma, c, s, epsilon, lane);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int d = 64 * w + lane;
        if (is_q) {
            const size_t idx = ((size_t)t * H + h) * D + d;
            const _Float16 hi = (_Float16)x[0][w];
            q_hilo[idx] = hi;
            q_hilo[(size_t)gridDim.y * H * D + idx] = (_Float16)(x[0][w] - (float)hi);
        } else {
            const int token = position + t;
            k_pages[(size_t)kh * head_stride + k_page_offset(token, d, D)] = cache_half(x[0][w]);
            v_pages[(size_t)kh * head_stride + v_page_offset(token, d, D)] = cache_half(v[w]);
        }
    }
}

// hi = fp16(q), lo = fp16(q - hi): q - hi is exact in fp32, so the two
// parts hold q to about 22 significant bits (|q| < 65504, error at most
// 2^-25 + 2^-22 |q| once lo falls into fp16's subnormal range).
__global__ __launch_bounds__(256)
void split_query(_Float16 *hi, _Float16 *lo, const float *q, size_t n) {
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const float x = q[e];
        const _Float16 h = (_Float16)x;
        hi[e] = h;
        lo[e] = (_Float16)(x - (float)h);
    }
}

// Copy of whole pages: for every KV head of K and of V, elements [0, n) of
// its run (the pages of tokens 0 .. n/D-1) from a cache of stride src_stride
// to one of stride dst_stride, both tensors in one launch (chunks of K's heads
// first, then V's).  Each thread moves kCopyUnroll 16-byte pieces of one
// head, all loads issued before the stores, non-temporal (every byte is
// touched once).  n is a whole number of pages, so per_head (16-byte pieces
// per head) is a multiple of 32 * D / 8 = 512 (D = 128) or 1024 (D = 256):
// the launch takes kCopyThreads threads when kCopyUnroll * kCopyThreads
// divides it, else half as many.  A sweep on the 139,264-token K and V
// prefix (4 KV heads, D = 256; per call, with a launch per tensor): 2 x 512
// 174.4 us, 4 x 256 177.7, 2 x 256 180.2, 4 x 128 184.8, 4 x 512 185.4,
// default-policy loads and stores 202.1.  One launch for both measured the
// same (176.47 against 176.81 us) and saves a launch per call.
constexpr int kCopyUnroll = 2, kCopyThreads = 512;
struct CopyArgs {
    uint4 *dst_k, *dst_v;
    const uint4 *src_k, *src_v;
    size_t dst_stride, src_stride, n;
    int kv_heads;
};
__global__ __launch_bounds__(kCopyThreads)
void copy_pages(CopyArgs a) {
    const size_t per_head = a.n / 8;   // uint4 per head
    const size_t chunk = (size_t)kCopyUnroll * blockDim.x;
    const size_t chunks = per_head / chunk * 2 * a.kv_heads;
    for (size_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        const size_t first = c * chunk;
        size_t h = first / per_head;
        const size_t i0 = first - h * per_head + threadIdx.x;
        const bool v_half = h >= (size_t)a.kv_heads;   // uniform per chunk
        if (v_half) h -= a.kv_heads;
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 *s = reinterpret_cast<const u32x4 *>((v_half ? a.src_v : a.src_k) + h * (a.src_stride / 8) + i0);
        u32x4 *d = reinterpret_cast<u32x4 *>((v_half ? a.dst_v : a.dst_k) + h * (a.dst_stride / 8) + i0);
        u32x4 v[kCopyUnroll];
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) v[u] = __builtin_nontemporal_load(s + u * blockDim.x);
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) __builtin_nontemporal_store(v[u], d + u * blockDim.x);
    }
}

}  // namespace

void launch_copy(void *dst_k, void *dst_v, const void *src_k, const void *src_v, int kv_heads,
                 int head_dim, int dst_capacity, int src_capacity, int pages, hipStream_t stream) {
    const size_t n = (size_t)pages * kPageTokens * head_dim;   // 16-bit elements per head
    if (!n) return;
    const int threads = (n / 8) % (kCopyUnroll * kCopyThreads) == 0 ? kCopyThreads : kCopyThreads / 2;
    require((n / 8) % (kCopyUnroll * threads) == 0, "page copy needs whole chunks of 16-byte pieces per head");
    const size_t chunks = n / 8 / (kCopyUnroll * threads) * 2 * kv_heads;
    const unsigned blocks = (unsigned)std::min<size_t>(chunks, 32768);
    CopyArgs a = {static_cast<uint4 *>(dst_k), static_cast<uint4 *>(dst_v), static_cast<const uint4 *>(src_k),
                  static_cast<const uint4 *>(src_v), (size_t)dst_capacity * head_dim,
                  (size_t)src_capacity * head_dim, n, kv_heads};
    hipLaunchKernelGGL(copy_pages, dim3(blocks), dim3(threads), 0, stream, a);
    check(hipGetLastError());
}

void launch_pack(void *k_pages, void *v_pages, const void *k_rows, const void *v_rows,
                 int kv_heads, int head_dim, int capacity, int first, int count,
                 hipStream_t stream) {
    convert<true>(k_pages, v_pages, k_rows, v_rows, kv_heads, head_dim, capacity, first, count, stream);
}

void launch_unpack(void *k_rows, void *v_rows, const void *k_pages, const void *v_pages,
                   int kv_heads, int head_dim, int capacity, int first, int count,
                   hipStream_t stream) {
    convert<false>(const_cast<void *>(k_pages), const_cast<void *>(v_pages), k_rows, v_rows,
                   kv_heads, head_dim, capacity, first, count, stream);
}

void launch_split_query(void *q_hilo, const float *q, size_t n, hipStream_t stream) {
    if (!n) return;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    _Float16 *hi = static_cast<_Float16 *>(q_hilo);
    hipLaunchKernelGGL(split_query, dim3(blocks), dim3(256), 0, stream, hi, hi + n, q, n);
    check(hipGetLastError());
}

void launch_prepare(void *q_hilo, void *k_pages, void *v_pages, const float *q_gate,
                    const float *key, const float *value, const float *q_norm,
                    const float *k_norm, int batch, int position, int capacity,
                    float epsilon, hipStream_t stream, bool keys_only) {
    const int head0 = keys_only ? kModelQHeads : 0;
    hipLaunchKernelGGL(prepare_kernel, dim3(kModelQHeads + kModelKvHeads - head0, batch),
                       dim3(kWave), 0, stream, static_cast<_Float16 *>(q_hilo),
                       static_cast<_Float16 *>(k_pages),
                       static_cast<_Float16 *>(v_pages), q_gate, key, value, q_norm, k_norm,
                       position, (size_t)capacity * kModelHeadDim, epsilon, head0);
    check(hipGetLastError());
}

}  // namespace rs
