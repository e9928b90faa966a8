# buildalt.sh <objects>: build _work/alt keeping its objects outside
cd /root/repo/_work/alt; [ -d /tmp/altbuild ] && mv /tmp/altbuild build
python3 - "$@" <<'P'
import sys, os, glob
for f in glob.glob('build/temp*/**/*.o', recursive=True):
    b = os.path.basename(f).replace('_hip.o','').replace('.o','')
    if b in sys.argv[1:]: os.remove(f)
P
python -c "import __graft_entry__ as g; g.build()" > /tmp/ba.log 2>&1; rc=$?; grep -n "error:" /tmp/ba.log | head; mv build /tmp/altbuild; echo rc $rc
