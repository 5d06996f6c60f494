// The default steps' choice of kernel by the batch's tiles, whatever a launch's group has
// of them: UNIT is the source with the rule, `size_rules TABLE INDEX TILES...` prints the
// first kernel of a launch of half the batch and of the whole of it, a line per TILES.
#include UNIT

#ifdef MOVE
namespace {
thread_local double s_move[1];   // of kernels that do not run here
}
namespace tmk { namespace {
thread_local double s_move[1];
} }
extern "C" int tm_perception_offsets(int, int32_t*, int) { return 0; }
#endif

int main(int argc, char** argv)
{
    int n = 0;
    const tmk::Variant* v = tmk::TABLE(&n);
    int at = -1;
    for (int i = 0; i < n; ++i)
        if (!strcmp(v[i].name, argv[1])) at = i;
    if (at < 0) return 2;
    std::string first;
    cpu_hip::on_launch = [&](const cpu_hip::Launch& l) {
        if (first.empty()) first = l.name;
    };
    for (int k = 2; k < argc; ++k)
        for (int part : {2, 1}) {
            tmk::ConsumerArgs a{};
            a.ptiles = atoi(argv[k]);
            a.ntiles = a.ptiles / part;
            first.clear();
            (v[at].fn_one ? v[at].fn_one : v[at].fn)(a, a.ntiles, nullptr);
            printf("%s\n", first.c_str());
        }
    return 0;
}
