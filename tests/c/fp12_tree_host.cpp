// Host build of vkzg_amd/csrc/fp12_tree.h for tests/test_fp12_tree.py: 32 threads
// stand for the lanes of a group, a lane exchange is a round of all of them.
// Reads 6 x 2 terms (real and imaginary part, 13 limbs each), prints the sums as
// the group's first quad's lanes 0 and 1 hold them.  Built with -ftrapv, so a limb
// that overflows its 32 bits aborts.
#define __host__
#define __device__
#define VKZG_DEV static inline
#include <pthread.h>

#include <cstdint>
#include <cstdio>
#include <thread>
#include <vector>

constexpr int kLanes = 32;
static pthread_barrier_t round_barrier;
static int32_t slot[kLanes];
static thread_local int lane;

// v of lane `from` (0 where that is none)
static int32_t exchange(int32_t v, int from) {
    slot[lane] = v;
    pthread_barrier_wait(&round_barrier);
    const int32_t r = from < 0 ? 0 : slot[from];
    pthread_barrier_wait(&round_barrier);
    return r;
}
static int32_t __shfl_xor(int32_t v, int mask) { return exchange(v, lane ^ mask); }
static int32_t row_dpp(int32_t v, int ctrl) {
    const int row = lane & ~15, l = lane & 15, n = ctrl & 15;
    if ((ctrl & ~15) == 0x120) return exchange(v, row + ((l - n) & 15));  // row_ror
    return exchange(v, l + n < 16 ? row + l + n : -1);                    // row_shl
}
#define __builtin_amdgcn_mov_dpp(v, ctrl, row_mask, bank_mask, bound) row_dpp(v, ctrl)

#include "../../vkzg_amd/csrc/fp12_tree.h"

using namespace vkzg_amd;

int main() {
    pthread_barrier_init(&round_barrier, nullptr, kLanes);
    for (;;) {
        Fp term[6][2], out[2];
        for (auto &t : term)
            for (Fp &c : t)
                for (int32_t &v : c.v)
                    if (std::scanf("%d", &v) != 1) return 0;
        std::vector<std::thread> lanes;
        for (int l = 0; l < kLanes; l++)
            lanes.emplace_back([&, l] {
                lane = l;
                const bool has = fp12_has_term((uint32_t)l) && (l & 3) < 2;
                const Fp v = fp12_tree(has ? term[fp12_term((uint32_t)l)][l & 3] : fp_zero());
                if (l < 2) out[l] = v;
            });
        for (auto &t : lanes) t.join();
        for (const Fp &o : out)
            for (int32_t v : o.v) std::printf("%d ", v);
        std::printf("\n");
    }
}
