// The token-tile kernels of aq_qmv_tok.h for 8-bit codes.
#include "aq_qmv_tok.h"

namespace aq {

static const QmvTokEntry kEntries8[kTokPerWidth] = {AQ_QMVT_SET(8, 1)};
const QmvTokEntry* tok_entries_8() { return kEntries8; }

}  // namespace aq
