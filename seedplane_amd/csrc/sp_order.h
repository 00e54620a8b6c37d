// Host bookkeeping of the persistent one-column step, apart from the runtime, so that it can be checked without a GPU.
#pragma once

namespace sp {

// The error word of the persistent step lies in pinned memory and is set by blocks that give up, possibly while other
// blocks of the same launch are still running and will set it again.  True once per failed launch: the word is cleared
// only after everything that may still set it has ended (wait).
template <class Wait>
bool take_error(volatile unsigned *word, Wait &&wait) {
    if (!word || *word == 0) return false;
    wait();
    *word = 0;
    return true;
}

}  // namespace sp
