// Which of a field's two buffers holds each level's values is host state that
// changes while launches are issued: recording them into a graph changes it
// although nothing has run. RolesKeeper puts it back unless the recording ends
// well (without it, a level of odd flips would take the second buffer's old
// values for its own).
#pragma once

#include <cstddef>
#include <utility>
#include <vector>

namespace srmg {

// Fields: a vector of pointers (null ones allowed) to fields with a vector `cur`
template <class Fields>
class RolesKeeper {
    Fields &fields;
    std::vector<std::vector<unsigned char>> was;
    bool kept = false;

public:
    explicit RolesKeeper(Fields &f) : fields(f) {
        for (auto &p : f) {
            was.emplace_back();
            if (p) was.back().assign(p->cur.begin(), p->cur.end());
        }
    }
    RolesKeeper(const RolesKeeper &) = delete;
    RolesKeeper &operator=(const RolesKeeper &) = delete;
    // the recorded launches' roles stay
    void keep() { kept = true; }
    ~RolesKeeper() {
        if (kept) return;
        for (size_t i = 0; i < was.size() && i < fields.size(); i++)
            if (fields[i]) fields[i]->cur.swap(was[i]);
    }
};

}  // namespace srmg
