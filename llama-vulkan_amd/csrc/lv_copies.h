// lv_copies.h — which device copies of a LLaMA model's layer matrices a batched step works on, and in which order they are asked for.
//
// The prompt copy (lv_gemm.h, two bytes a weight) carries whole chunks of a long step: without it they go token by token, for the life of
// the model.  The short copy (lv_short.h, the file's size) makes what is left of a step, or a step of up to kMidTokens, faster, and is
// never worth the prompt copy's room.
#pragma once

namespace lv {

struct BatchCopies {
    bool batch;      // the step goes in batches
    bool mid;        // ... and its last one takes the products of lv_mid.h, on the short copy
};

// chunks: the step has whole chunks before its last batch; pays: that one is faster on the short copy.  prompt() and shorter() make a copy
// unless it is there already and say whether it is; room() says whether making the short copy leaves the prompt copy its room.
template <class Prompt, class Short, class Room>
inline BatchCopies batch_copies(bool chunks, bool pays, Prompt &&prompt, Short &&shorter, Room &&room)
{
    if (!chunks && pays && room() && shorter()) return {true, true};
    const bool whole = prompt(), mid = pays && (whole || !chunks) && shorter();
    return {whole || mid, mid};
}

}  // namespace lv
