// Per-grain peak lists from per-peak labels: the peaks of each label in
// ascending order, as CSR (idx, off, owner), and the longest-first visiting
// order of the persistent refinement.  A counting sort: counts per label,
// their exclusive scan, a fill into each list in whatever order the atomics
// take, then each list sorted in LDS by a block of its own.  Five launches
// and one 16-byte read-back (the total and the longest list size the
// results), where nonzero, a 64-bit radix sort, bincount, gather and
// repeat_interleave took ~45 launches and four read-backs: one assignment
// round of 777 grains x 10^5 peaks with them 492 us, with these 172.  At that
// size it is bound by its launches (3 to 9 us each; the traffic is 1 MB).
#pragma once
#include "gs_kernels.h"

#define GS_LIST_LOCAL 8192      // labels counted in LDS at most (32 KB)
#define GS_LIST_SORT_MAX 16384  // entries of one list that are sorted in LDS (64 KB)

// counts[l] += 1 for every label in [0, K) (counts zeroed by the caller).
// LOCAL: counted in LDS (K ints) first, one global atomic per (block, label):
// atomics of many blocks on one counter go one after the other (100 003
// labels of 777 grains straight to memory: 24 us).
template <bool LOCAL>
__global__ __launch_bounds__(1024) void k_label_counts(const int* __restrict__ labels, int n, int K,
                                                       int* __restrict__ counts) {
    extern __shared__ int lcnt[];
    if (LOCAL) {
        for (int g = threadIdx.x; g < K; g += 1024) lcnt[g] = 0;
        __syncthreads();
    }
    for (long long k = (long long)blockIdx.x * 1024 + threadIdx.x; k < n;
         k += (long long)gridDim.x * 1024) {
        const int l = labels[k];
        if (l >= 0 && l < K) atomicAdd(LOCAL ? &lcnt[l] : &counts[l], 1);
    }
    if (LOCAL) {
        __syncthreads();
        for (int g = threadIdx.x; g < K; g += 1024)
            if (lcnt[g]) atomicAdd(&counts[g], lcnt[g]);
    }
}

// off[0..K] = exclusive scan of counts, cursor[g] = 0, info = {total, longest
// list}.  One block of GS_SCAN_THREADS, each thread a run of consecutive
// grains.
#define GS_SCAN_THREADS 1024
__global__ __launch_bounds__(GS_SCAN_THREADS) void k_list_offsets(const int* __restrict__ counts,
                                                                  int K, long long* __restrict__ off,
                                                                  int* __restrict__ cursor,
                                                                  long long* __restrict__ info) {
    __shared__ long long lsum[GS_SCAN_THREADS / GS_WAVE];
    __shared__ int lmax[GS_SCAN_THREADS / GS_WAVE];
    const int t = threadIdx.x, lane = t & (GS_WAVE - 1), wave = t / GS_WAVE;
    const int per = (K + GS_SCAN_THREADS - 1) / GS_SCAN_THREADS;
    const int a = min((long long)K, (long long)t * per), b = min(K, a + per);
    long long s = 0;
    int m = 0;
    for (int g = a; g < b; g++) {
        s += counts[g];
        m = max(m, counts[g]);
    }
    long long run = s;  // inclusive over the wave
    for (int o = 1; o < GS_WAVE; o <<= 1) {
        const long long v = __shfl_up(run, o, GS_WAVE);
        if (lane >= o) run += v;
        m = max(m, __shfl_xor(m, o, GS_WAVE));
    }
    if (lane == GS_WAVE - 1) lsum[wave] = run;
    if (lane == 0) lmax[wave] = m;
    __syncthreads();
    long long base = run - s;
    for (int w = 0; w < wave; w++) base += lsum[w];
    for (int g = a; g < b; g++) {
        off[g] = base;
        cursor[g] = 0;
        base += counts[g];
    }
    if (t == GS_SCAN_THREADS - 1) {  // its run is the last, or empty: base is the total
        off[K] = base;
        for (int w = 0; w < GS_SCAN_THREADS / GS_WAVE; w++) m = max(m, lmax[w]);
        info[0] = base;
        info[1] = m;
    }
}

// Peak numbers into their lists, in no particular order.  LOCAL: a block
// counts its labels in LDS (K ints), takes each list's room with one global
// atomic, and places its peaks from there.
template <bool LOCAL>
__global__ __launch_bounds__(1024) void k_list_fill(const int* __restrict__ labels, int n, int K,
                                                    const long long* __restrict__ off,
                                                    int* __restrict__ cursor,
                                                    int* __restrict__ idx) {
    extern __shared__ int lcnt[];
    const long long first = (long long)blockIdx.x * 1024 + threadIdx.x;
    const long long step = (long long)gridDim.x * 1024;
    if (LOCAL) {
        for (int g = threadIdx.x; g < K; g += 1024) lcnt[g] = 0;
        __syncthreads();
        for (long long k = first; k < n; k += step) {
            const int l = labels[k];
            if (l >= 0 && l < K) atomicAdd(&lcnt[l], 1);
        }
        __syncthreads();
        for (int g = threadIdx.x; g < K; g += 1024)
            if (lcnt[g]) lcnt[g] = atomicAdd(&cursor[g], lcnt[g]);
        __syncthreads();
    }
    for (long long k = first; k < n; k += step) {
        const int l = labels[k];
        if (l >= 0 && l < K)
            idx[off[l] + atomicAdd(LOCAL ? &lcnt[l] : &cursor[l], 1)] = (int)k;
    }
}

// Each list in ascending order (bitonic, padded to a power of two with
// INT_MAX in LDS, which holds the longest list's power of two), and the
// owner of every entry.  One block per list.
__global__ __launch_bounds__(GS_BLOCK) void k_list_sort(int* __restrict__ idx,
                                                        const long long* __restrict__ off,
                                                        int* __restrict__ owner) {
    extern __shared__ int lkey[];
    const int g = blockIdx.x;
    const long long o0 = off[g];
    const int n = (int)(off[g + 1] - o0);
    if (n == 0) return;
    int p = 1;
    while (p < n) p <<= 1;
    for (int i = threadIdx.x; i < p; i += GS_BLOCK) {
        lkey[i] = i < n ? idx[o0 + i] : 0x7fffffff;
        if (i < n) owner[o0 + i] = g;
    }
    for (int k = 2; k <= p; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int i = threadIdx.x; i < p / 2; i += GS_BLOCK) {
                const int lo = 2 * i - (i & (j - 1)), hi = lo + j;  // lo has bit j clear
                const int x = lkey[lo], y = lkey[hi];
                if ((x > y) == ((lo & k) == 0)) {
                    lkey[lo] = y;
                    lkey[hi] = x;
                }
            }
        }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += GS_BLOCK) idx[o0 + i] = lkey[i];
}

// order[r] = the grain whose list is r-th longest, equal lengths in grain
// order: a wave per grain counts the lists before it (64 lengths a step).
// 5 us at 5000 grains; the work is K^2, so the callers sort beyond
// GS_ORDER_MAX.
#define GS_ORDER_MAX 8192
__global__ __launch_bounds__(GS_BLOCK) void k_list_order(const long long* __restrict__ off, int K,
                                                         int* __restrict__ order) {
    const int g = (blockIdx.x * GS_BLOCK + threadIdx.x) / GS_WAVE;
    const int lane = threadIdx.x & (GS_WAVE - 1);
    if (g >= K) return;
    const long long len = off[g + 1] - off[g];
    int rank = 0;
    for (int j0 = 0; j0 < K; j0 += GS_WAVE) {
        const int j = j0 + lane;
        bool before = false;
        if (j < K) {
            const long long l = off[j + 1] - off[j];
            before = l > len || (l == len && j < g);
        }
        rank += __popcll(__ballot(before));
    }
    if (lane == 0) order[rank] = g;
}
