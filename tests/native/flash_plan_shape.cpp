// The launch shape csrc/flash_plan.h gives a call: for every line "mode BH S_q S_kv
// causal keys keys_saves" (mode f32, bf16 or f32x3; keys: the keys shape may run)
// one line with whole, small, split, balanced or keys.  The call has the scratch
// the size queries ask for.
#define __host__
#define __device__
#include "flash_plan.h"

#include <iostream>
#include <string>

using namespace anima_hip;

int main()
{
    std::string mode;
    int64_t BH;
    int S_q, S_kv, causal, keys;
    float saves;
    while (std::cin >> mode >> BH >> S_q >> S_kv >> causal >> keys >> saves) {
        const FlashTimes &t = mode == "bf16" ? kTimesBF16 : mode == "f32x3" ? kTimesX3 : kTimesF32;
        FlashScratch s;
        s.part_bytes = flash_split_bytes(BH, S_q, S_kv, 128);
        s.balance_bytes = flash_balance_bytes(BH, S_q, S_kv, 128, t);
        s.keys = keys != 0;
        s.keys_saves = saves;
        if (s.balance_bytes > kMaxFlashBalanceBytes)
            return 1;
        const FlashPlan p = flash_plan(BH, S_q, S_kv, 128, t, causal != 0, s);
        std::cout << (p.keys         ? "keys"
                      : p.u > 0      ? "balanced"
                      : p.splits > 1 ? "split"
                      : p.waves == 4 ? "small"
                                     : "whole")
                  << "\n";
    }
    return 0;
}
