// Weights of the launches behind a short one, brought into the L2s beside it.
//
// A token is a chain of launches of which some (attention over a few hundred rows) are trips to memory one
// behind the other by a few workgroups, while memory has nothing to do.  Such a launch gets more workgroups, behind its own, that read
// the first weights of the launches behind it and drop them: they then lie in the L2 of the XCD whose workgroups will ask for them.
// Workgroups go to the XCDs in turn, launch by launch alike, so a unit's XCD is its number modulo eight; where that fails the weights
// lie in the memory-side cache, and nothing but time depends on it.
//
// 8 MB that a launch of 256 workgroups reads take 2.9 us from memory and 1.9 us from the L2s, 25 MB 5.6 and 2.9.  Beside attention behind 40 to
// 100 tokens, us of the launches that follow, without / with: Qwen3's gate and up (63 MB, 10 of them read ahead) 17.6 / 15.8, attention 6.7 / 7.2, 64
// tokens 14715 / 14130; Takosun's gate and up (50 MB, 8 ahead) 13.9 / 11.6, attention 5.5 / 5.8, 64 tokens 15630 / 15310.  How much: past 20 MB the
// launch waits for the reading (24 MB: Qwen3 14330, Takosun 15320; 32 MB 14470 and 15620), and fewer workgroups have too little under way (64
// workgroups, 16 MB: 14710, 15920).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace a81w41 {

struct WeightsAhead {
    static constexpr int kParts = 3;
    // Unit u, read by a workgroup of XCD u % 8: `bytes` bytes (a multiple of 16) at base + u / block * block_step + u % block * step, 16-byte
    // aligned, and as many `also` bytes further on, if that is not 0.
    struct Part {
        const uint8_t* base = nullptr;
        size_t block_step = 0, also = 0;
        unsigned step = 0, bytes = 0;
        int block = 1, count = 0;
        // 0: one place; else that many, the chosen experts' (of the token's row of `table`), slot_step bytes an expert
        int slots = 0;
        size_t slot_step = 0;
        // bytes from base to the end of what is read of one place
        size_t extent() const { return count ? (count - 1) / block * block_step + (size_t)((count - 1) % block) * step + also + bytes : 0; }
        size_t size() const { return (size_t)bytes * count * (also ? 2 : 1) * (slots ? slots : 1); }
    };
    Part part[kParts];
    static constexpr int kWorkgroups = 192;  // of 1024 threads; a multiple of 8
    static constexpr size_t kBytes = 20 << 20;
    int parts = 0;
    const int *ids = nullptr, *table = nullptr;
    int vocab = 0, top = 0, experts = 0;
    size_t room = kBytes;  // that parts may still be added for
    void add(const Part& p) {
        if (parts == kParts || !p.count || !p.bytes || p.size() > room) return;
        part[parts++] = p;
        room -= p.size();
    }
    int workgroups() const { return parts ? kWorkgroups : 0; }
};

#if defined(__HIPCC__)
// Workgroup `index` of `workgroups` additional ones, workgroup `linear` of the launch, of THREADS threads.  A wave takes 4 KB of a unit at a time.
template <int THREADS>
__device__ __forceinline__ void read_ahead(const WeightsAhead& w, int workgroups, int index, int linear) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int kLoads = 4, kWaves = THREADS / 64;
    const int turns = workgroups >> 3, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (index >> 3 >= turns) return;
    int n = (index >> 3) * kWaves + wave;
    for (int p = 0; p < w.parts; p++) {
        const WeightsAhead::Part& part = w.part[p];
        const int n16 = (int)(part.bytes >> 4), chunks = (n16 + 64 * kLoads - 1) / (64 * kLoads), pieces = part.also ? 2 : 1;
        const int of_slot = (part.count + 7) / 8 * pieces * chunks, total = of_slot * max(part.slots, 1);
        for (; n < total; n += turns * kWaves) {
            const int slot = n / of_slot, m = n - slot * of_slot, piece_of = m / chunks, chunk = m - piece_of * chunks;
            const int u = piece_of / pieces * 8 + (linear & 7);
            if (u >= part.count) continue;
            const uint8_t* from = part.base + u / part.block * part.block_step + u % part.block * (size_t)part.step + (piece_of % pieces) * part.also;
            if (part.slots) {
                const int id = min(max(w.ids[0], 0), w.vocab - 1);
                from += min(max(w.table[(size_t)id * w.top + slot], 0), w.experts - 1) * part.slot_step;
            }
            u32x4 v[kLoads];
#pragma unroll
            for (int j = 0; j < kLoads; j++) v[j] = reinterpret_cast<const u32x4*>(from)[min(chunk * 64 * kLoads + j * 64 + lane, n16 - 1)];
#pragma unroll
            for (int j = 0; j < kLoads; j++) asm volatile("" ::"v"(v[j]));
        }
        n -= total;
    }
}
#endif

}  // namespace a81w41
