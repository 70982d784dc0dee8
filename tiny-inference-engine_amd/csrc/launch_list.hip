// Runs launch lists (common.h): the launches of one layer, again for each of the layers of its shape.
#include "common.h"

// launches[i] takes its arguments at words[layer * words_a_layer + first[i]]. Returns the first status that is not
// TIE_OK and leaves in *failed which launch of a layer gave it; nothing is launched behind it.
extern "C" int tie_run_launch_list(const uintptr_t* launches, const int* first, int count, const uint64_t* words,
                                   int words_a_layer, int layers, int* failed) {
  if (launches == nullptr || first == nullptr || words == nullptr || failed == nullptr || count <= 0 || layers < 0)
    return TIE_BAD_ARGUMENT;
  for (int layer = 0; layer < layers; ++layer)
    for (int i = 0; i < count; ++i) {
      const auto launch = reinterpret_cast<int (*)(const uint64_t*)>(launches[i]);
      const int status = launch(words + static_cast<size_t>(layer) * words_a_layer + first[i]);
      if (status != TIE_OK) {
        *failed = i;
        return status;
      }
    }
  return TIE_OK;
}
