// What every wave of the per-head norm and RoPE launch reads, for all small head counts: heads that exist, and the k weight only
// where there are k heads.
#include <cstdio>
#include <initializer_list>

#include "../turbo-fieldfare_amd/csrc/tf_epilogue_heads.hpp"

int main() {
    for (uint32_t q = 0; q <= 33; ++q)
        for (uint32_t kv = 0; kv <= 9; ++kv) {
            const tfk::EpilogueHeads heads = {q, kv};
            if (heads.count() == 0) continue;
            for (uint32_t per_wave : {1u, 2u, 4u, 8u}) {
                const uint32_t blocks = (heads.count() + 4 * per_wave - 1) / (4 * per_wave);
                for (uint32_t block = 0; block < blocks; ++block)
                    for (uint32_t wave = 0; wave < 4; ++wave)
                        for (uint32_t round = 0; round <= per_wave; ++round) {      // the last round: what a wave looks ahead to
                            const uint32_t h = block * 4 * per_wave + wave + 4 * round, r = heads.read(h);
                            const bool own = h >= heads.count() || r == h;
                            const bool weight = heads.takes_q_weight(h) ? q > 0 : kv > 0;
                            const bool right = h >= heads.count() || heads.takes_q_weight(h) == (h < q);
                            if (r >= heads.count() || !own || !weight || !right) {
                                std::printf("q %u kv %u head %u\n", q, kv, h);
                                return 1;
                            }
                        }
            }
        }
    std::printf("epilogue heads ok\n");
    return 0;
}
