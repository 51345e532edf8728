// Register sorting networks of the tiled top-K selection (geometry.hip), host- and device-callable so
// that a host program can check them (topk_check.cpp).
//
// A candidate is the 64-bit key (bits(d^2) << 32) | code: for d^2 >= 0 and codes >= 0 the unsigned key
// order is the (d^2, code) order of the reference's neighbour comparison (morton_types.cuh:68-72), and
// the empty entry (inf, INT_MAX) is the largest key.
#ifndef GDX_TOPK_H
#define GDX_TOPK_H

#include <hip/hip_runtime.h>

#include <cstdint>

#define GDX_TOPK_FN __host__ __device__ __forceinline__

namespace gdx {

constexpr uint64_t TOPK_EMPTY = (uint64_t(0x7f800000u) << 32) | uint64_t(0x7fffffffu);

// The smaller and the larger of two keys. Every key is at most (bits(inf) << 32) | 0xffffffff, so as the
// bits of a double it is non-negative and finite (the float's exponent ends below the double's last one),
// and such doubles order as their bits do, subnormal ones included: the device takes v_min_f64 and
// v_max_f64, one full-rate instruction each, where the integer form is a 64-bit compare and two selects
// each. The merges are a third of the top-K kernel's vector instructions: 22.1 ms with the integer form,
// 18.7 ms with these (1e7 records in 3D, K = 32, 16 keys a merge, before the box traversal). (Assembly because
// fmin of the language first quiets its operands, one more instruction per operand.)
GDX_TOPK_FN uint64_t key_min(uint64_t a, uint64_t b)
{
#ifdef __HIP_DEVICE_COMPILE__
    uint64_t r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return a < b ? a : b;
#endif
}

GDX_TOPK_FN uint64_t key_max(uint64_t a, uint64_t b)
{
#ifdef __HIP_DEVICE_COMPILE__
    uint64_t r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return a < b ? b : a;
#endif
}

GDX_TOPK_FN void cx_up(uint64_t &a, uint64_t &b)
{
    const uint64_t lo = key_min(a, b), hi = key_max(a, b);
    a = lo;
    b = hi;
}

// ascending sort of N keys (N a power of two) by Batcher's odd-even merges: 63 exchanges for 16 keys where a
// bitonic sort takes 80 (1e7 records in 3D, K = 32: 11.9 -> 11.2 ms)
template <int N>
GDX_TOPK_FN void odd_even_sort(uint64_t (&a)[N])
{
#pragma unroll
    for (int p = 1; p < N; p <<= 1)
    {
#pragma unroll
        for (int k = p; k > 0; k >>= 1)
        {
#pragma unroll
            for (int l = 0; l + k < N; ++l)
            {
                // l is the lower end of a pair of this step: the steps start at k mod p, in runs of k, and
                // stay within blocks of 2p
                const int j = l - k % p;
                if (j >= 0 && j % (2*k) < k && l / (2*p) == (l + k) / (2*p)) cx_up(a[l], a[l + k]);
            }
        }
    }
}

// ascending sort of a bitonic sequence of N keys
template <int N>
GDX_TOPK_FN void bitonic_merge(uint64_t (&a)[N])
{
#pragma unroll
    for (int j = N >> 1; j > 0; j >>= 1)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            const int l = i ^ j;
            if (l > i) cx_up(a[i], a[l]);
        }
    }
}

// L (K keys, ascending) becomes the K smallest keys of L and S (B keys, ascending): min(L[i], S[K-1-i])
// is bitonic and holds the K smallest of both (Batcher's merge), and one bitonic merge sorts it
template <int K, int B>
GDX_TOPK_FN void topk_merge_sorted(uint64_t (&L)[K], const uint64_t (&S)[B])
{
#pragma unroll
    for (int i = 0; i < K; ++i)
    {
        const int j = K - 1 - i;
        if (j < B) L[i] = key_min(L[i], S[j]);
    }
    bitonic_merge<K>(L);
}

}  // namespace gdx

#endif  // GDX_TOPK_H
