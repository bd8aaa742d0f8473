// The group launches (round_group.h) with tiles of sixteen rows.
#include "round_group.h"

namespace cavs {

template int group_fwd<GROUP_TREELSTM, true>(const GroupFwdArgs &a, void *stream);
template int group_bwd<GROUP_TREELSTM, true>(const GroupBwdArgs &a, void *stream);
template int group_fwd<GROUP_LSTM, true>(const GroupFwdArgs &a, void *stream);
template int group_bwd<GROUP_LSTM, true>(const GroupBwdArgs &a, void *stream);
template int group_fwd<GROUP_TREEFC, true>(const GroupFwdArgs &a, void *stream);
template int group_bwd<GROUP_TREEFC, true>(const GroupBwdArgs &a, void *stream);

}  // namespace cavs
